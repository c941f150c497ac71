"""The one-launch spiking attention core at the edges of its tiles (token
counts around 16, 32, 64, 128 and 256, odd ones, step counts off the block of
four) against the CPU oracle: every sum is an integer, so results are equal bit
for bit; and the head Linear over a copy at the edges of its passes."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 15, 17, 33, 63, 64, 65, 127, 128, 129, 200, 255, 256])
@pytest.mark.parametrize("T,B,heads,cp_pad", [(1, 1, 1, 0), (5, 2, 3, 0), (4, 9, 1, 4)])
def test_attention_edges(cuda, N, T, B, heads, cp_pad):
    _check_attention(cuda, N, T, B, heads, cp_pad)


@pytest.mark.parametrize("N", [128, 129, 196, 255, 256])
@pytest.mark.parametrize("T,B,heads,cp_pad", [(1, 257, 1, 0), (2, 65, 4, 0), (5, 33, 8, 4)])
def test_attention_more_workgroups_than_cus(cuda, N, T, B, heads, cp_pad):
    """One step a block (more than 128 tokens, more workgroups than CUs)."""
    _check_attention(cuda, N, T, B, heads, cp_pad)


def _check_attention(cuda, N, T, B, heads, cp_pad):
    from catfuse_amd import runtime, snn
    C = 32 * heads
    g = torch.Generator().manual_seed(N + T)
    q, k, v = ((torch.rand(T, B, N, C, generator=g) < 0.4).float() for _ in range(3))
    th = max(0.5, 0.02 * N)
    lif = snn.LIFNode(step_mode="m", v_threshold=th)
    copy = runtime.pack_tokens(torch.cat([q, k, v], -1).to(cuda), 3 * C)
    s_ref, v_ref, _ = oracle.spike_attention_lif(q, k, v, heads, 0.125, lif)
    out, v_out = runtime.spike_attention_lif(copy, T, B, N, heads, (0, C, 2 * C), 0.125,
                                             v_threshold=th)
    np.testing.assert_array_equal(out.cpu().numpy(), s_ref)
    np.testing.assert_array_equal(v_out.cpu().numpy(), v_ref)
    if cp_pad:     # an output pitch off 8 channels: element stores
        cp = C + cp_pad
        o = torch.full((T * B * N, cp), 7.0, dtype=torch.float16, device=cuda)
        vo = torch.empty(B, N, C, device=cuda)
        p, lib = runtime.ptr, runtime._hip.lib()
        rc = lib.cf_spike_attention_lif(
            p(copy), p(copy), p(copy), 0, C, 2 * C, 3 * C, p(o), cp, None, p(vo), None, None, None,
            0, T, B, N, heads, 32, 0.125, 2.0, th, 0.0, 1, 1, runtime._hip.stream(o.device))
        assert rc == 0
        np.testing.assert_array_equal(o[:, :C].float().cpu().numpy().reshape(s_ref.shape), s_ref)
        assert bool((o[:, C:] == 7.0).all())      # channels past the heads are left alone
        assert torch.equal(vo, v_out)


@pytest.mark.parametrize("K,O", [(300, 21), (70000, 18)])
def test_linear_tokens_silent_rows(cuda, K, O):
    """Rows silent but for one spike (skipped groups of inputs at every output
    pass but the first), a wholly silent one, a copy recorded as all zero."""
    from catfuse_amd import runtime
    g = torch.Generator().manual_seed(K)
    at = [0, 63, 64, K // 2, K - 1]
    x = torch.zeros(1, len(at) + 1, K)
    x[0, range(len(at)), at] = 2.0
    w, b = torch.randn(O, K, generator=g), torch.randn(O, generator=g)
    copy = runtime.pack_tokens(x.to(cuda), runtime.pad32(K))
    y = runtime.linear_tokens(runtime.lazy_tokens(x.shape, copy, torch.device(cuda)), w.to(cuda),
                              b.to(cuda)).cpu()
    # one product of two, exact, and one addition
    assert torch.equal(y[0], torch.cat([b + 2.0 * w[:, at].t(), b[None]]))
    p, lib = runtime.ptr, runtime._hip.lib()
    zero = torch.tensor([1, 0], dtype=torch.int64, device=cuda)
    out, wg, bg = torch.empty(len(at) + 1, O, device=cuda), w.to(cuda), b.to(cuda)
    assert lib.cf_linear_tokens(p(copy), p(zero), p(wg), p(bg), p(out), len(at) + 1, K,
                                runtime.pad32(K), O, runtime._hip.stream(out.device)) == 0
    assert torch.equal(out.cpu(), b.expand(len(at) + 1, O))


@pytest.mark.parametrize("K,O", [(1, 1), (255, 10), (1024, 16), (1025, 17), (4096, 40), (5000, 3)])
def test_linear_tokens_edges(cuda, K, O):
    from catfuse_amd import runtime
    g = torch.Generator().manual_seed(K)
    x = torch.randint(0, 3, (2, 3, K), generator=g).float() * (torch.rand(2, 3, K, generator=g) < 0.3)
    x[..., 0] = 0.0
    w = torch.randn(O, K, generator=g)
    w[:, 0] = float("inf")              # behind a spike that never comes
    b = torch.randn(O, generator=g)
    xl = runtime.lazy_tokens((2, 3, K), runtime.pack_tokens(x.to(cuda), runtime.pad32(K)),
                             torch.device(cuda))
    y = runtime.linear_tokens(xl, w.to(cuda), b.to(cuda)).cpu()
    w[:, 0] = 0.0
    ref = x.double() @ w.double().t() + b.double()
    # K products of magnitude up to 2 max|w|, each rounded once or twice in fp32
    tol = 2.0 ** -23 * (K ** 0.5 + 8) * float(ref.abs().max().clamp(min=1)) * 4
    assert float((y.double() - ref).abs().max()) < tol
