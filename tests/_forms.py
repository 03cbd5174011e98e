"""Which kernel the library takes for dk and dv of given sizes, asked without a GPU (fa_bwd_form)."""
import ctypes

import torch

from flash_mi355 import _cabi

NAMES = {_cabi.FA_FORM_KEYS: "keys", _cabi.FA_FORM_COLS: "cols", _cabi.FA_FORM_ROWS: "rows", _cabi.FA_FORM_PIPE: "pipe",
         _cabi.FA_FORM_SMALL: "small", _cabi.FA_FORM_FP32: "fp32"}
_DTYPES = {torch.bfloat16: _cabi.FA_DTYPE_BF16, torch.float16: _cabi.FA_DTYPE_FP16, torch.float32: _cabi.FA_DTYPE_FP32}


def dkdv_form(B, H, Hk, M, N, D, dtype, causal, kind="plain", window=0, prefix=0, nseq=0, whole=True, no_pair_wait=False):
    """(name, whether dq shares the launch), for fp32 (name, shape of dq, of dk/dv) where it does not.  kind: "plain", "doc", "heads" (ids per head), "qpos" (ids and positions), "block", "packed"."""
    buf = ctypes.create_string_buffer(4096)
    base = (ctypes.addressof(buf) + 255) & ~255   # never followed: the call looks at sizes, strides and alignment
    p = _cabi.FaParams()
    for f in ("q", "k", "v", "o", "lse", "dout", "dq", "dk", "dv", "delta", "workspace", "split_scratch"):
        setattr(p, f, base)
    p.workspace_bytes = p.split_scratch_bytes = 1 << 60
    p.B, p.H, p.Hk, p.M, p.N, p.D, p.causal, p.dtype, p.sm_scale = B, H, Hk, M, N, D, int(causal), _DTYPES[dtype], 0.1
    p.window, p.prefix = window, prefix
    for heads, rows, fields in ((H, M, ("q_stride", "o_stride", "do_stride", "dq_stride")), (Hk, N, ("k_stride", "v_stride", "dk_stride", "dv_stride"))):
        for f in fields:
            getattr(p, f)[:] = (heads * rows * D, rows * D, D, 1)
    if kind in ("doc", "heads", "qpos"):
        p.score_mode, p.eq, p.ek = _cabi.FA_SCORE_MODE1_DOC, base, base
        p.eq_stride[:] = (H * M, M if kind == "heads" else 0, 1)
        p.ek_stride[:] = (H * N, N if kind == "heads" else 0, 1)
        if kind == "qpos":
            p.qpos = base
    elif kind == "block":
        p.score_mode, p.eq = _cabi.FA_SCORE_MODE2_BLOCK, base
        p.eq_stride[:] = (0, 0, -(-N // 64))
    elif kind == "packed":
        p.score_mode, p.eq, p.ek, p.nseq = _cabi.FA_SCORE_MODE3_PACKED, base, base, nseq
    else:
        p.flags = _cabi.FA_FLAG_SPLIT_KEYS
    if no_pair_wait:
        p.flags |= _cabi.FA_FLAG_DEBUG_NO_PAIR_WAIT
    form = _cabi.lib().fa_bwd_form(ctypes.byref(p), int(whole))
    assert form > 0, _cabi.lib().fa_error_string(form)
    if dtype == torch.float32 and not form & _cabi.FA_FORM_WITH_DQ:   # ... and the shapes of dq's and dk/dv's workgroups
        return "fp32", (form >> 4) & 3, (form >> 6) & 3
    return NAMES[form & ~_cabi.FA_FORM_WITH_DQ], bool(form & _cabi.FA_FORM_WITH_DQ)
