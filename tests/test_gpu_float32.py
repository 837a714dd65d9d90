"""The fp32 matrix-core kernels at the edges of their row groups (32), key blocks (64), row blocks (128: one wave or four per
sweep) and key-owner steps (256), against the oracle."""
import pytest
import torch

from oracle import sb_oracle as O
from helpers import cu_from_lengths, max_abs, randn, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("current", [False, True])
@pytest.mark.parametrize("lens", [[1], [2], [31], [32], [33], [64], [65], [127], [128], [129], [160], [161], [255], [256], [257],
                                  [385], [1, 128, 64, 3], [1, 300, 64, 129, 33]])
def test_float32_against_the_oracle(lens, current, D):
    from flame_amd import sb_attn_varlen
    H, N = 3, sum(lens)
    q, k, v, do = (randn((H, N, D), 700 + i, 0.5 if i < 3 else 1.0) for i in range(4))
    dr = randn((H, N), 705, 1.0)
    cu = cu_from_lengths(lens)
    qg, kg, vg = (x.cuda().requires_grad_(True) for x in (q, k, v))
    o, rem = sb_attn_varlen(qg, kg, vg, cu.cuda(), max(lens), attend_current=current)
    got = torch.autograd.grad((o, rem), (qg, kg, vg), (do.cuda(), dr.cuda()))
    ref = O.sb_attn_grads_oracle(q, k, v, do, dr, cu_seqlens=cu.tolist(), attend_current=current)
    assert max_abs(o.cpu(), ref[0]) <= 1e-5 and max_abs(rem.cpu(), ref[1]) <= 1e-5
    for g, r in zip(got, ref[2:]):
        assert rel_l2(g.cpu(), r) <= (2e-5 if r.norm() > 0 else 0.0)


# Key blocks whose steps two workgroups share: lengths around the cut (256 and 512 queries) and a pack of cut and whole sweeps,
# the two passes as one call and as two, the second of them twice.
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("lens", [[256], [257], [511], [512], [513], [640], [769], [700, 1, 256, 300, 130]])
def test_key_blocks_of_two_workgroups(lens, D):
    import ctypes as C
    from flame_amd import _lib, sb_attn_varlen
    H, N = 2, sum(lens)
    q, k, v, do = (randn((H, N, D), 720 + i, 0.5 if i < 3 else 1.0) for i in range(4))
    cu = cu_from_lengths(lens)
    qg, kg, vg = (x.cuda().requires_grad_(True) for x in (q, k, v))
    o, rem = sb_attn_varlen(qg, kg, vg, cu.cuda(), max(lens))
    got = torch.autograd.grad(o, (qg, kg, vg), do.cuda())
    ref = O.sb_attn_grads_oracle(q, k, v, do, None, cu_seqlens=cu.tolist())
    for g, r in zip(got, ref[2:]):
        assert rel_l2(g.cpu(), r) <= 2e-5
    if len(lens) > 1:
        return
    T = lens[0]
    lib = _lib.load()
    x = [t.cuda().view(1, H, T, D) for t in (q, k, v, do)]
    out = [torch.full_like(x[0], float("nan")) for _ in range(4)]
    rem = torch.empty(1, H, T, device="cuda")
    p = _lib.SbaParams()
    p.struct_size = C.sizeof(p)
    p.n_seq, p.n_heads, p.seq_len, p.total_tokens, p.head_dim, p.dtype = 1, H, T, T, D, 0
    p.scale = D ** -0.5
    p.stream = torch.cuda.current_stream().cuda_stream
    for name, t in zip(("q", "k", "v", "d_o", "o", "dq", "dk", "dv"), x + out):
        setattr(p, name, _lib.tensor4(t))
    p.rem = _lib.SbaVector(rem.data_ptr(), *rem.stride()[:2])
    scratch = torch.empty(lib.sba_bwd_scratch_bytes(C.byref(p)), dtype=torch.uint8, device="cuda")
    p.bwd_scratch, p.bwd_scratch_bytes = scratch.data_ptr(), scratch.numel()
    for phase in (1, 2, 2):
        p.bwd_phases = phase
        _lib.check(lib.sba_bwd(C.byref(p)), "sba_bwd")
    for g, whole in zip(out[1:], got):
        assert torch.equal(g.view_as(whole), whole)
