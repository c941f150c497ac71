"""Flat-tile conv kernel (conv_ring.hip) at the edges of its tiles: single
pixels, maps that leave tiles partly filled or span several images, one chunk
and odd chunk counts, one to nine time steps, the widest map of each staged
size, the pooled epilogue; against the CPU oracle, and against the 8x8-tile
kernel bit for bit (both accumulate in the same order)."""
import numpy as np
import pytest
import torch

import oracle
from catfuse_amd import runtime
from catfuse_amd.runtime import EPI_LIF, EPI_POOL, ConvLIFRunner
from choice import HALO, HALO_LEAN, RING, conv_choice
from parity import lif_parity

pytestmark = pytest.mark.gpu

# T, B, Cin, Cout, H, W, k: one round of workgroups but for the last two
SHAPES = [
    (4, 1, 64, 64, 7, 7, 3), (3, 2, 32, 32, 5, 9, 3), (6, 3, 96, 64, 13, 11, 3),
    (4, 1, 40, 64, 14, 14, 3), (8, 1, 33, 64, 16, 15, 3), (4, 1, 64, 64, 30, 30, 3),
    (1, 2, 64, 32, 1, 1, 3), (4, 17, 64, 64, 2, 2, 3), (9, 33, 33, 160, 3, 5, 3),
    (4, 1, 64, 64, 8, 8, 1), (4, 3, 96, 160, 14, 14, 1), (5, 1, 512, 64, 1, 1, 1),
    (2, 65, 300, 96, 1, 1, 1), (8, 4, 64, 64, 5, 7, 1), (1, 1, 32, 64, 3, 3, 1),
    (4, 1, 64, 64, 56, 56, 3), (5, 2, 33, 32, 9, 62, 3), (4, 3, 32, 96, 5, 31, 3),  # two slots
    (4, 30, 64, 704, 7, 7, 1),           # 64-channel tiles
    (4, 2, 64, 70, 7, 7, 3), (5, 1, 32, 5, 9, 9, 3), (4, 2, 64, 37, 8, 8, 1),
    (4, 30, 64, 690, 7, 7, 1),           # channels off 32 and off 64
    (4, 600, 64, 1024, 1, 1, 3), (5, 300, 33, 288, 2, 3, 3),   # two rounds of workgroups
]
POOLED = [(4, 1, 64, 64, 16, 16), (4, 3, 96, 64, 8, 8), (6, 5, 64, 64, 4, 4),
          (4, 33, 64, 96, 2, 2), (3, 2, 32, 32, 6, 4), (1, 4, 512, 512, 2, 2)]


# tau, v_th, v_reset, decay_input: the specialised hard reset off 0 and the generic
# neuron (tau not a power of two, soft reset, no input decay); NEURONS[-1] fires at rest
NEURONS = [(2.0, 0.3, 0.1, True), (3.0, 0.3, 0.0, True), (2.0, 0.3, None, True),
           (2.0, 0.3, 0.0, False), (2.0, 0.05, 0.1, True)]


def _layer(cuda, Ci, Co, k, seed=0, neuron=(2.0, 0.3, 0.0, True)):
    g = torch.Generator().manual_seed(seed)
    w = torch.randn(Co, Ci, k, k, generator=g) * (2.0 / (Co * k * k)) ** 0.5
    sc = torch.rand(Co, generator=g) * 0.4 + 0.8
    sh = torch.randn(Co, generator=g) * 0.1
    r = ConvLIFRunner(w.to(cuda), sc.to(cuda), sh.to(cuda), None, 1, k // 2, *neuron)
    return r, w, sc, sh


def _lazy(x, cuda):
    T, B, C, H, W = x.shape
    xp = runtime.pack_input(x.to(cuda).reshape(T * B, C, H, W))[0]
    return runtime.lazy_output((T, B, C, H, W), xp, torch.device(cuda))


def _tiled(r, x, v0, pool, ident):
    """The same launch through cf_conv_halo, which the dispatch of
    cf_conv_mfma passes over."""
    T, B, Ci, H, W = x.shape
    dev = x.device
    xp = x._cf_nhwc[0]
    Hs, Ws = (H // 2, W // 2) if pool else (H, W)
    cp = runtime.pad32(r.Cout)
    out = torch.empty((T * B, Hs, Ws, cp), dtype=torch.float16, device=dev)
    v = torch.empty((B, r.Cout, Hs, Ws), device=dev)
    p = runtime.ptr
    lib = runtime._hip.lib()
    rc = lib.cf_conv_halo(
        p(xp), p(r.w_packed), p(r.alpha), p(r.beta), p(v0), p(v), None, p(out), cp, None,
        p(ident), cp, 1, None, None, None, None, None, None, None, 0, None, x.numel(), 2.0, T, B,
        r.Cp, r.Cout, r.Coutp, H, W, H, W, r.KH, 1, r.KH // 2, 8, 8, 0,
        EPI_POOL if pool else EPI_LIF, *r.lif, runtime._hip.stream(dev))
    assert rc == 0
    return runtime.lazy_output((T, B, r.Cout, Hs, Ws), out, dev).clone(), v


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("ident,vin", [(False, False), (True, True)])
def test_flat_tiles(cuda, shape, ident, vin):
    T, B, Ci, Co, H, W, k = shape
    assert conv_choice(T, B, Ci, Co, H, W, k, ident=ident) == RING
    r, w, sc, sh = _layer(cuda, Ci, Co, k)
    g = torch.Generator().manual_seed(1)
    x = (torch.rand(T, B, Ci, H, W, generator=g) < 0.3).float()
    i0 = torch.randint(0, 3, (T, B, Co, H, W), generator=g).float() if ident else None
    v0 = torch.rand(B, Co, H, W, generator=g) * 0.25 if vin else None
    xl = _lazy(x, cuda)
    idl = _lazy(i0, cuda) if ident else None
    y, v = r.run_mfma(xl, None if v0 is None else v0.to(cuda), identity=idl)
    assert not bool(y._cf_nhwc[0][..., Co:].any())
    y, v = y.clone(), v.clone()
    ty, tv = _tiled(r, xl, None if v0 is None else v0.to(cuda), False,
                    idl._cf_nhwc[0] if ident else None)
    assert torch.equal(y, ty) and torch.equal(v, tv)
    z = oracle.conv2d(x.reshape(T * B, Ci, H, W), w, None, 1, k // 2)
    z = torch.as_tensor(np.asarray(z)).reshape(T, B, Co, H, W)
    z = (z * sc.view(-1, 1, 1) + sh.view(-1, 1, 1)).float()
    s_ref, v_ref, h_ref = oracle.lif_multistep(z, None if v0 is None else v0, tau=2.0,
                                               v_threshold=0.3)
    lif_parity((y - idl.clone() if ident else y).cpu().numpy(), v.cpu().numpy(), s_ref,
                        v_ref, h_ref, v_th=0.3)


@pytest.mark.parametrize("shape", POOLED)
@pytest.mark.parametrize("vin", [False, True])
def test_flat_tiles_pooled(cuda, shape, vin):
    T, B, Ci, Co, H, W = shape
    assert conv_choice(T, B, Ci, Co, H, W, 3, pool=True) == RING
    r = _layer(cuda, Ci, Co, 3)[0]
    g = torch.Generator().manual_seed(2)
    xl = _lazy((torch.rand(T, B, Ci, H, W, generator=g) < 0.3).float(), cuda)
    v0 = (torch.rand(B, Co, H // 2, W // 2, generator=g) * 0.25).to(cuda) if vin else None
    y, v = r.run_mfma(xl, v0, epilogue=EPI_POOL)
    ty, tv = _tiled(r, xl, v0, True, None)
    assert torch.equal(y.clone(), ty) and torch.equal(v.clone(), tv)
    assert 0 < float(y.mean()) < 1


@pytest.mark.parametrize("neuron", NEURONS)
@pytest.mark.parametrize("T,k,H,W,pool", [(6, 1, 5, 7, False), (5, 3, 9, 11, False), (4, 3, 8, 4, True)])
def test_flat_tiles_neurons(cuda, neuron, T, k, H, W, pool):
    """Every LIF specialisation of the flat-tile kernel, from a state, against the
    8x8-tile kernel bit for bit and the neuron as it is defined."""
    B, Ci, Co = 3, 64, 64
    r, w, sc, sh = _layer(cuda, Ci, Co, k, neuron=neuron)
    assert conv_choice(T, B, Ci, Co, H, W, k, pool=pool, lif=r.lif) == RING
    g = torch.Generator().manual_seed(4)
    x = (torch.rand(T, B, Ci, H, W, generator=g) < 0.3).float()
    xl = _lazy(x, cuda)
    Hs, Ws = (H // 2, W // 2) if pool else (H, W)
    v0 = torch.rand(B, Co, Hs, Ws, generator=g) * 0.25
    y, v = r.run_mfma(xl, v0.to(cuda), epilogue=EPI_POOL if pool else EPI_LIF)
    ty, tv = _tiled(r, xl, v0.to(cuda), pool, None)
    assert torch.equal(y.clone(), ty) and torch.equal(v.clone(), tv)
    z = torch.as_tensor(np.asarray(oracle.conv2d(x.reshape(T * B, Ci, H, W), w, None, 1, k // 2)))
    z = (z.reshape(T * B, Co, H, W) * sc.view(-1, 1, 1) + sh.view(-1, 1, 1)).float()
    if pool:
        z = torch.nn.functional.avg_pool2d(z, 2)
    tau, v_th, v_reset, decay = neuron
    s_ref, v_ref, h_ref = oracle.lif_multistep(z.reshape(T, B, Co, Hs, Ws), v0, tau=tau,
                                               v_threshold=v_th, v_reset=v_reset,
                                               decay_input=decay)
    lif_parity(ty.cpu().numpy(), tv.cpu().numpy(), s_ref, v_ref, h_ref, v_th=v_th)


@pytest.mark.parametrize("neuron", NEURONS)
@pytest.mark.parametrize("Co", [5, 70])
def test_channels_off_32_neurons(cuda, neuron, Co):
    """The 8x8-tile kernel off 32 channels with other neurons: those silent at rest
    take the lean epilogue and leave the copy's padding zero, whatever they reset
    to; all give the bits of the general epilogue with fp32 output."""
    T, B, Ci, H, W = 5, 2, 48, 19, 65
    r = _layer(cuda, Ci, Co, 3, neuron=neuron)[0]
    silent = neuron is not NEURONS[-1]
    assert conv_choice(T, B, Ci, Co, H, W, 3, lif=r.lif) == (HALO_LEAN if silent else HALO)
    g = torch.Generator().manual_seed(Co)
    xl = _lazy((torch.rand(T, B, Ci, H, W, generator=g) < 0.3).float(), cuda)
    v0 = (torch.rand(B, Co, H, W, generator=g) * 0.25).to(cuda)
    for v_in in (None, v0):
        y, v = r.run_mfma(xl, v_in)
        assert bool(y._cf_nhwc[0][..., Co:].any()) != silent
        gy, gv = r.run_mfma(xl, v_in, emit_nhwc=False)
        assert torch.equal(y.clone(), gy) and torch.equal(v.clone(), gv)


@pytest.mark.parametrize("k,pool", [(1, False), (3, False), (3, True)])
def test_flat_tiles_zero_input(cuda, k, pool):
    """StaticZero: an all-zero input gives the bias response on every route
    (elided with its count block known, computed without)."""
    r = _layer(cuda, 64, 64, k)[0]
    x = torch.zeros(4, 2, 64, 4, 4, device=cuda)
    r.run_mfma(x, epilogue=EPI_POOL if pool else EPI_LIF)     # bias response known
    y, v = r.run_mfma(x, epilogue=EPI_POOL if pool else EPI_LIF)
    ty, tv = _tiled(r, _lazy(x, cuda), None, pool, None)
    assert torch.equal(y.clone(), ty) and torch.equal(v.clone(), tv)


@pytest.mark.parametrize("Co", [1, 31, 40, 70, 170])
@pytest.mark.parametrize("k,stride,H,W,T,B", [(3, 1, 40, 33, 4, 3), (3, 2, 45, 61, 6, 2),
                                              (1, 2, 31, 30, 4, 2), (3, 1, 35, 64, 9, 1),
                                              (3, 1, 40, 65, 4, 3)])
@pytest.mark.parametrize("v_th", [0.3, -1.0])
def test_channels_off_32(cuda, Co, k, stride, H, W, T, B, v_th):
    """The 8x8-tile kernel at channel counts off 32: the spikes, the sums with
    an identity and the state equal the general epilogue's with fp32 output
    bit for bit, and with a neuron that is silent at rest (the lean epilogue;
    one that fires without drive takes the general one) channels past Cout are
    zero in the copy."""
    Ci = 48
    g = torch.Generator().manual_seed(Co)
    w = torch.randn(Co, Ci, k, k, generator=g) * (2.0 / (Co * k * k)) ** 0.5
    r = ConvLIFRunner(w.to(cuda), None, None, None, stride, k // 2, 2.0, v_th, 0.0, True)
    x = (torch.rand(T, B, Ci, H, W, generator=g) < 0.3).float()
    Ho, Wo = r.out_hw(H, W)
    i0 = torch.randint(0, 3, (T, B, Co, Ho, Wo), generator=g).float()
    for ident in (None, i0):
        if stride == 2 or W > 62:       # (else the flat-tile kernel may take it)
            assert conv_choice(T, B, Ci, Co, H, W, k, stride=stride, ident=ident is not None,
                               lif=(2.0, v_th, 0.0, 1, 1)) == (HALO_LEAN if v_th > 0 else HALO)
        for inp in (x, torch.zeros_like(x)):
            xl = _lazy(inp, cuda)
            y, v = r.run_mfma(xl, identity=None if ident is None else _lazy(ident, cuda))
            assert v_th < 0 or not bool(y._cf_nhwc[0][..., Co:].any())
            gy, gv = r.run_mfma(xl, identity=None if ident is None else ident.to(cuda),
                                emit_nhwc=False)
            assert torch.equal(y.clone(), gy) and torch.equal(v.clone(), gv)


@pytest.mark.parametrize("k,B,H", [(3, 1, 7), (1, 2, 8), (3, 3, 34)])
def test_wide_copy_keeps_its_padding(cuda, k, B, H):
    """An output copy whose pitch is wider than the channels need: channels
    past Cout are left as they were, the others equal the usual pitch's."""
    T, Ci, Co = 4, 64, 32
    r = _layer(cuda, Ci, Co, k)[0]
    dev = torch.device(cuda)
    g = torch.Generator().manual_seed(3)
    x = (torch.rand(T, B, Ci, H, H, generator=g) < 0.3).float().to(cuda)
    r.run_mfma(x)                                    # (packs the weights)
    xp = runtime.pack_input(x.reshape(T * B, Ci, H, H))[0]
    p = runtime.ptr
    outs = []
    for cp in (32, 64):
        out = torch.full((T * B, H, H, cp), 7.0, dtype=torch.float16, device=dev)
        v = torch.empty((B, Co, H, H), device=dev)
        rc = runtime._hip.lib().cf_conv_mfma(
            p(xp), p(r.w_packed), p(r.alpha), p(r.beta), None, p(v), None, p(out), cp, None, None,
            0, 1, None, None, None, None, None, None, None, 0, None, x.numel(), 2.0, T, B, r.Cp, Co,
            r.Coutp, H, H, H, H, k, k, 1, k // 2, B, 0, 0, 0, EPI_LIF, *r.lif,
            runtime._hip.stream(dev))
        assert rc == 0
        outs.append((out, v))
    assert torch.equal(outs[0][0], outs[1][0][..., :Co]) and torch.equal(outs[0][1], outs[1][1])
    assert bool((outs[1][0][..., Co:] == 7.0).all())
