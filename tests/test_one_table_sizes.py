"""Sizes of SBA_SAVE_ONE_TABLE: what the forward keeps and what the backward asks for beside it."""
import ctypes as C

import pytest

from flame_amd import _lib

ONE_TABLE = 0x4f4e4531


@pytest.mark.parametrize("dtype,head_dim,seq_len,takes", [
    (_lib.SBA_DTYPE_BF16, 64, 4096, True), (_lib.SBA_DTYPE_F16, 128, 129, True), (_lib.SBA_DTYPE_BF16, 128, 128, False),
    (_lib.SBA_DTYPE_BF16, 256, 4096, False), (_lib.SBA_DTYPE_F32, 64, 4096, False)])
def test_sizes_and_refusals(dtype, head_dim, seq_len, takes):
    lib = _lib.load()
    p = _lib.SbaParams()
    p.struct_size = C.sizeof(p)
    p.dtype, p.n_seq, p.n_heads, p.seq_len, p.total_tokens, p.head_dim, p.scale = dtype, 1, 16, seq_len, seq_len, head_dim, 0.125
    whole, recomputing = lib.sba_workspace_bytes(C.byref(p)), lib.sba_bwd_scratch_bytes(C.byref(p))
    p.workspace = 256
    beside_whole = lib.sba_bwd_scratch_bytes(C.byref(p))
    p.workspace = None
    for other in (1, 2, -1):                                     # (any other value means what 1 does)
        p.save_for_backward = other
        assert lib.sba_workspace_bytes(C.byref(p)) == whole
    p.save_for_backward = ONE_TABLE
    kept = lib.sba_workspace_bytes(C.byref(p))
    assert kept == (whole // 2 if takes else whole)
    assert lib.sba_bwd_scratch_bytes(C.byref(p)) == recomputing  # (nothing kept: the same as ever)
    p.workspace = 256
    assert lib.sba_bwd_scratch_bytes(C.byref(p)) == beside_whole + (whole - kept)
    # the forward and the backward refuse less
    for name in ("q", "k", "v", "o", "d_o", "dq", "dk", "dv"):
        setattr(p, name, _lib.SbaTensor(1 << 20, 0, 0, 16 * head_dim))
    p.rem = _lib.SbaVector(1 << 20, 0, 0)
    p.workspace_bytes = kept - 1
    assert lib.sba_fwd(C.byref(p)) == -4 and lib.sba_bwd(C.byref(p)) == -4
