"""Images whose state passes 2 GiB: the halo kernel's lean epilogue, whose byte
ranges end there, hands them to the general one, in single and paired launches
and from one-byte copies; against the same layer run over slices of its
channels, whose states are below it (a channel's sums do not depend on the
others), bit for bit."""
import pytest
import torch

from catfuse_amd import runtime
from catfuse_amd.runtime import ConvLIFRunner
from choice import HALO, HALO_LEAN, conv_choice

pytestmark = pytest.mark.gpu


def _runner(cuda, w, sc, sh, stride=1):
    return ConvLIFRunner(w.to(cuda), sc.to(cuda), sh.to(cuda), None, stride, w.shape[2] // 2, 2.0,
                         0.3, 0.0, True)


def _params(Co, Ci, k, seed):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(Co, Ci, k, k, generator=g) * 0.1, torch.rand(Co, generator=g) * 0.4 + 0.8,
            torch.randn(Co, generator=g) * 0.1)


def _input(cuda, n, dtype=torch.float16):
    g = torch.Generator(device=cuda).manual_seed(n)
    xp = (torch.rand(1, n, n, 32, device=cuda, generator=g) < 0.3).to(dtype)
    return runtime.lazy_output((1, 1, 32, n, n), xp, cuda)


def _check_slices(cuda, prm, x, n, stride, y, v, step):
    w, sc, sh = prm
    Co = w.shape[0]
    copy = y._cf_nhwc[0]
    assert copy.dtype == torch.float16 and not bool(copy[..., Co:].any())
    v = v.clone() if isinstance(v, runtime.ChannelState) else v
    for c in range(0, Co, step):
        s = slice(c, min(Co, c + step))
        k = w.shape[2]
        assert conv_choice(1, 1, 32, s.stop - c, n, n, k, stride=stride) == HALO_LEAN
        ys, vs = _runner(cuda, w[s], sc[s], sh[s], stride).run_mfma(x)
        assert torch.equal(copy[..., s], ys._cf_nhwc[0][..., :s.stop - c])
        assert torch.equal(v[:, s], vs)
    assert 0.01 < float(copy[0, ::7, ::7].float().mean()) < 0.9


@pytest.mark.parametrize("Co,step", [(100, 50), (128, 64)])
def test_state_past_2_gib(cuda, Co, step):
    n = 2400
    assert conv_choice(1, 1, 32, Co, n, n, 3) == HALO
    prm, x = _params(Co, 32, 3, Co), _input(cuda, n)
    y, v = _runner(cuda, *prm).run_mfma(x)
    _check_slices(cuda, prm, x, n, 1, y, v, step)


def test_pair_state_past_2_gib(cuda):
    n = 2888
    pa, pb = _params(288, 32, 3, 1), _params(64, 32, 1, 2)
    x = _input(cuda, n)
    ra, rb = _runner(cuda, *pa, stride=2), _runner(cuda, *pb, stride=2)
    ya, va, yb, vb = runtime.run_halo_pair(ra, rb, x)
    _check_slices(cuda, pa, x, n, 2, ya, va, 144)
    _check_slices(cuda, pb, x, n, 2, yb, vb, 64)


def test_byte_copy_widened_past_2_gib(cuda):
    n, Co = 2400, 128
    prm = _params(Co, 32, 3, 3)
    xb = _input(cuda, n, torch.uint8)
    runtime.set_spike_copy("u8")
    try:
        y, v = _runner(cuda, *prm).run_mfma(xb)
    finally:
        runtime.set_spike_copy("f16")
    _check_slices(cuda, prm, _input(cuda, n), n, 1, y, v, 64)
