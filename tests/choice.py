"""Which kernel a fused conv launch takes (cf_conv_mfma_choice), from its sizes
alone: pointers are placeholders, nothing is launched."""
import ctypes

from catfuse_amd import _hip
from catfuse_amd.runtime import EPI_LIF, EPI_POOL, pad32

GENERAL, HALO, HALO_LEAN, RING = range(4)


def conv_args(T, B, Ci, Co, H, W, k, stride=1, pool=False, ident=False, state=True, cp_out=None,
              cp_id=None, lif=(2.0, 0.3, 0.0, 1, 1)):
    p = 1 << 20
    a = _hip.ConvMfmaArgs()
    a.x = a.w_packed = a.alpha = a.beta = a.out_nhwc = p
    a.v_out = p if state else None
    a.identity_nhwc = p if ident else None
    a.identity_mode = 1
    a.cp_out = pad32(Co) if cp_out is None else cp_out
    a.cp_id = a.cp_out if cp_id is None else cp_id
    a.Coutp = max((Co + 63) // 64, (a.cp_out + 63) // 64) * 64
    a.sparse_threshold = 2.0
    a.T, a.B, a.Cp, a.Cout, a.H, a.W, a.KH, a.KW = T, B, pad32(Ci), Co, H, W, k, k
    a.stride, a.pad, a.x_img_tstride = stride, k // 2, B
    a.Ho, a.Wo = (H + 2 * a.pad - k) // stride + 1, (W + 2 * a.pad - k) // stride + 1
    a.numel = T * B * Ci * H * W
    a.epilogue = EPI_POOL if pool else EPI_LIF
    a.tau, a.v_th, a.v_reset, a.hard_reset, a.decay_input = lif
    return a


def conv_choice(*args, **kw):
    """The kernel's number, or None for a launch that is refused."""
    a, c = conv_args(*args, **kw), ctypes.c_int(-1)     # (held until the call returns)
    rc = _hip.lib().cf_conv_mfma_choice(ctypes.addressof(a), ctypes.addressof(c))
    assert rc in (0, 1)            # hipErrorInvalidValue
    return None if rc else c.value
