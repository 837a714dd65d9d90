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


# Gradients that go where the two workgroups of a key block still read (dK and dV in the places of K and V), into host memory that the GPU
# has mapped, and from a scratch without room for two workgroups' sums: nothing but their finished rows is ever written there.
@pytest.mark.parametrize("T,D", [(700, 64), (513, 128)])
def test_where_the_gradients_of_shared_key_blocks_go(T, D):
    import ctypes as C
    from flame_amd import _lib
    lib, H = _lib.load(), 2
    x = [randn((1, H, T, D), 740 + i, 0.5 if i < 3 else 1.0).cuda() for i in range(4)]
    rem = torch.empty(1, H, T, device="cuda")

    def backward(k, v, dk, dv, without_room=False):
        p = _lib.SbaParams()
        p.struct_size = C.sizeof(p)
        p.n_seq, p.n_heads, p.seq_len, p.total_tokens, p.head_dim, p.dtype = 1, H, T, T, D, 0
        p.scale = D ** -0.5
        p.stream = torch.cuda.current_stream().cuda_stream
        dq = torch.empty_like(x[0])
        for name, t in (("q", x[0]), ("k", k), ("v", v), ("d_o", x[3]), ("dq", dq), ("dk", dk), ("dv", dv)):
            setattr(p, name, _lib.tensor4(t))
        whole = lib.sba_bwd_scratch_bytes(C.byref(p))
        sums = 4 * H * T * D * 4
        assert whole >= sums                    # (the problem is one whose key blocks are shared)
        n = whole - (sums + 255) // 256 * 256 if without_room else whole
        scratch = torch.full((n + 4096,), 0x5a, dtype=torch.uint8, device="cuda")
        p.bwd_scratch, p.bwd_scratch_bytes = scratch.data_ptr(), n
        _lib.check(lib.sba_bwd(C.byref(p)), "sba_bwd")
        torch.cuda.synchronize()
        assert bool((scratch[n:] == 0x5a).all())
        p.bwd_scratch_bytes = whole - (sums + 255) // 256 * 256 - 1
        assert lib.sba_bwd(C.byref(p)) == -4
        return dk, dv

    new = lambda: torch.full_like(x[1], float("nan"))
    want = backward(x[1], x[2], new(), new())
    ref = O.sb_attn_grads_oracle(*(t.cpu() for t in x), None)[3:]
    for g, r in zip(want, ref):
        assert rel_l2(g.cpu(), r) <= 2e-5
    k, v = x[1].clone(), x[2].clone()
    for g, w in zip(backward(k, v, k, v), want):
        assert torch.equal(g, w)
    host = [torch.full(x[1].shape, float("nan")).pin_memory() for _ in range(2)]
    for g, w in zip(backward(x[1], x[2], *host), want):
        assert torch.equal(g, w.cpu())
    for g, r in zip(backward(x[1], x[2], new(), new(), without_room=True), ref):
        assert rel_l2(g.cpu(), r) <= 2e-5
