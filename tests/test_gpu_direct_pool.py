"""The analog first stage's reset-free LIF (four steps of one image from the
initial state): equal, bit for bit, to the stepped LIF, which a state of zeros
passed in takes; neurons that fire at every first step and never, potentials on
the threshold, infinite and not-a-number pixels."""
import pytest
import torch

from catfuse_amd.runtime import ConvLIFRunner

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 3, 48, 32, 32), (2, 1, 16, 15, 17), (3, 4, 64, 7, 40)])
@pytest.mark.parametrize("tau", [1.0, 2.0, 4.0])
def test_reset_free_equals_stepped(cuda, shape, tau):
    B, Ci, Co, H, W = shape
    g = torch.Generator().manual_seed(H)
    w = torch.randn(Co, Ci, 3, 3, generator=g)
    w[0] = 0.0                             # channels on and around the threshold
    w[1] = 0.0
    sc, sh = torch.ones(Co), torch.randn(Co, generator=g) * 0.3
    sh[0], sh[1] = 1.0, 2.0
    r = ConvLIFRunner(w.to(cuda), sc.to(cuda), sh.to(cuda), None, 1, 1, tau, 1.0, 0.0, True)
    img = torch.randn(B, Ci, H, W, generator=g)
    img[0, 0, 1, 2], img[0, 0, 5, 9], img[0, 0, 6, 14] = float("inf"), float("nan"), 3e38
    x = img.to(cuda).unsqueeze(0).expand(4, B, Ci, H, W)
    y, v = r.run_direct_pool(x)
    ys, vs = r.run_direct_pool(x, torch.zeros(B, Co, H, W, device=cuda))
    assert torch.equal(y.clone(), ys.clone())
    assert torch.equal(v.view(torch.int32), vs.view(torch.int32)) or (
        torch.equal(torch.isnan(v), torch.isnan(vs)) and
        torch.equal(v.nan_to_num(7.0), vs.nan_to_num(7.0)))
    assert 0 < float(y.mean()) < 1
