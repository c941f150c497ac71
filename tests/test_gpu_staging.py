"""Staging passes between fp32 boundary tensors and the fp16 copies, at the
edges of their tiles: pixel counts off 64 and off 4, channels off 32 and 64,
single pixels and channels, values that fp16 cannot hold."""
import pytest
import torch

from catfuse_amd import runtime

pytestmark = pytest.mark.gpu


def _spikes(shape, cuda, seed=0):
    g = torch.Generator().manual_seed(seed)
    n = 1
    for d in shape:
        n *= d
    # (one float into its buffer: contiguous, not 16-byte aligned)
    x = torch.empty(n + 1, device=cuda)[1:].view(shape)
    return x.copy_(torch.randint(-3, 4, shape, generator=g))


def _status(cuda):
    return torch.zeros(1, dtype=torch.int32, device=cuda)


@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (3, 31, 1, 3), (2, 33, 5, 13), (2, 64, 8, 8),
                                   (3, 65, 7, 9), (2, 96, 9, 29), (1, 130, 3, 43),
                                   (5, 200, 45, 61)])
@pytest.mark.parametrize("act", [False, True])
def test_pack_input_edges(cuda, shape, act):
    x = _spikes(shape, cuda)
    x[x.abs() == 3] *= 0.25                       # quarters: exact in fp16
    NB, C, H, W = shape
    gs = max(8, -(-C // 32)) if act else 0
    nnz = runtime.count_block(x.device)
    st = _status(cuda)
    xp, a = runtime.pack_input(x, group_size=gs, nnz=nnz, status=st)
    want = torch.zeros((NB, H, W, runtime.pad32(C)), device=x.device, dtype=torch.float16)
    want[..., :C] = x.permute(0, 2, 3, 1).half()
    assert torch.equal(xp.view(want.shape), want)
    assert int(nnz[1]) == int((x != 0).sum())
    if act:
        bits = torch.zeros((NB, H, W), dtype=torch.int64, device=x.device)
        for g in range(-(-C // gs)):
            bits |= (x[:, g * gs:(g + 1) * gs] != 0).any(1).long() << g
        assert torch.equal(a.view(NB, H, W).long() & 0xffffffff, bits)
    assert int(st) == 0


# (16,385 rows of 31 on: both sides of where two chunks a thread begin, and
# 8-channel chunks of fp32 rows)
@pytest.mark.parametrize("rows,C", [(1, 1), (7, 31), (513, 64), (130, 100), (1030, 384),
                                    (16385, 31), (16384, 32), (16385, 100), (5500, 400),
                                    (32770, 257), (32769, 64)])
def test_pack_tokens_and_back(cuda, rows, C):
    x = _spikes((1, 1, rows, C), cuda, 1)
    cp = runtime.pad32(C)
    nnz = runtime.count_block(x.device)
    copy = runtime.pack_tokens(x, cp, nnz=nnz)
    want = torch.zeros((rows, cp), device=x.device, dtype=torch.float16)
    want[:, :C] = x.view(rows, C).half()
    assert torch.equal(copy.view(rows, cp), want)
    assert int(nnz[1]) == int((x != 0).sum())
    assert torch.equal(runtime.lazy_tokens((1, 1, rows, C), copy, x.device).clone(), x)


@pytest.mark.parametrize("where", [0, 63, 64, 2744 * 70 - 1])
@pytest.mark.parametrize("bad", [0.1, float("inf"), float("nan"), 1e30])
def test_pack_flags_what_fp16_cannot_hold(cuda, where, bad):
    for shape, pack in (((1, 70, 56, 49), runtime.pack_input),
                        ((1, 1, 2744, 70), lambda x, status: runtime.pack_tokens(x, 96, status=status))):
        x = torch.zeros(shape, device=cuda)
        x.view(-1)[where] = bad
        st = _status(cuda)
        pack(x, status=st)
        # an infinity is an fp16 value; what rounds or is no number is not
        assert int(st) == (0 if bad == float("inf") else runtime.STATUS_INEXACT_FP16)


@pytest.mark.parametrize("H,W,k,s,p", [(1, 1, 3, 2, 1), (7, 10, 3, 2, 1), (8, 9, 3, 2, 1),
                                       (7, 10, 3, 1, 1)])
def test_maxpool_order_with_nan(cuda, H, W, k, s, p):
    """Where a copy holds NaN (an identity's), the pool's result is that of a
    window walked by rows: its first value, and each later one that is greater
    (a NaN is only kept in the first place), at the borders too."""
    C = 40
    g = torch.Generator().manual_seed(H)
    v = torch.randint(0, 3, (2, 1, C, H, W), generator=g).float()
    u = torch.rand(v.shape, generator=g)
    v[u < 0.15], v[u > 0.9] = float("nan"), float("inf")
    nhwc = torch.zeros(2, H, W, runtime.pad32(C), dtype=torch.float16)
    nhwc[..., :C] = v.view(2, C, H, W).permute(0, 2, 3, 1).half()
    y = runtime.maxpool_nhwc(runtime.lazy_output(tuple(v.shape), nhwc.to(cuda), cuda), k, s, p)
    Ho, Wo = (H + 2 * p - k) // s + 1, (W + 2 * p - k) // s + 1
    want = torch.empty(2, 1, C, Ho, Wo)
    for oh in range(Ho):
        for ow in range(Wo):
            win = v[..., max(oh * s - p, 0):oh * s - p + k, max(ow * s - p, 0):ow * s - p + k]
            m, *rest = win.flatten(3).unbind(3)
            for q in rest:
                m = torch.where(q > m, q, m)
            want[..., oh, ow] = m
    assert torch.equal(y.cpu().nan_to_num(7.0), want.nan_to_num(7.0))


def _copies(NB, H, W, C, cp, dtype, cuda):
    g = torch.Generator(device=cuda).manual_seed(C)
    c = torch.randint(0, 4, (2, NB, H, W, cp), device=cuda, generator=g).to(dtype)
    c[..., C:] = 0
    return c[0].contiguous(), c[1].contiguous()


def _descs(alias, cuda):
    """Absent, written, all zero, an alias (the 16 bytes of a CfOutDesc)."""
    return [None] + [torch.tensor([k, alias.data_ptr() if k == 2 else 0], dtype=torch.int64,
                                  device=cuda) for k in (0, 1, 2)]


# both forms of the fp32 pass, tiles partly filled in pixels and channels (the last
# six: 64-channel tiles)
@pytest.mark.parametrize("NB,C,H,W", [
    (1, 1, 1, 1), (3, 33, 5, 13), (2, 64, 8, 8), (3, 65, 7, 9), (2, 96, 9, 29), (1, 130, 3, 43),
    (2, 70, 32, 32), (450, 100, 3, 3), (900, 33, 1, 1), (901, 64, 4, 4), (1500, 40, 1, 101),
    (47, 64, 17, 251), (4, 1000, 61, 64)])
def test_materialise_edges(cuda, NB, C, H, W):
    """The fp32 form of an fp16 copy read through every kind of descriptor, and
    of a byte copy."""
    lib, p, st = runtime._hip.lib(), runtime.ptr, runtime._hip.stream(cuda)
    cp = runtime.pad32(C) + (8 if C % 2 else 0)
    copy, other = _copies(NB, H, W, C, cp, torch.float16, cuda)
    out = torch.empty(NB, C, H, W, device=cuda)
    want = copy[..., :C].permute(0, 3, 1, 2).float()
    wants = (want, want, torch.zeros_like(want), other[..., :C].permute(0, 3, 1, 2).float())
    for d, w in zip(_descs(other, cuda), wants):
        out.fill_(-1.0)
        assert lib.cf_copy_to_f32(p(copy), p(d), p(out), NB, C, H, W, cp, 0, st) == 0
        assert torch.equal(out, w)
    out.fill_(-1.0)
    assert lib.cf_nhwc_to_nchw(p(copy), p(out), NB, C, H, W, cp, st) == 0
    assert torch.equal(out, want)
    out.fill_(-1.0)
    assert lib.cf_nhwc_to_nchw_u8(p(copy.to(torch.uint8)), p(out), NB, C, H, W, cp, st) == 0
    assert torch.equal(out, want)


@pytest.mark.parametrize("rows,C,pad", [(1, 1, 0), (33, 40, 0), (130, 100, 4), (5500, 400, 0),
                                        (32770, 257, 8), (32769, 64, 3)])
def test_materialise_tokens_edges(cuda, rows, C, pad):
    """The fp32 rows of a token-major copy read through every kind of descriptor."""
    lib, p, st = runtime._hip.lib(), runtime.ptr, runtime._hip.stream(cuda)
    cp = runtime.pad32(C) + pad
    copy, other = (t.view(rows, cp) for t in _copies(1, 1, rows, C, cp, torch.float16, cuda))
    out = torch.empty(rows, C, device=cuda)
    want = copy[:, :C].float()
    wants = (want, want, torch.zeros_like(want), other[:, :C].float())
    for d, w in zip(_descs(other, cuda), wants):
        out.fill_(-1.0)
        assert lib.cf_copy_to_f32(p(copy), p(d), p(out), rows, C, 1, 1, cp, 1, st) == 0
        assert torch.equal(out, w)
    out.fill_(-1.0)
    assert lib.cf_tokens_to_f32(p(copy), p(out), rows, C, cp, st) == 0
    assert torch.equal(out, want)
