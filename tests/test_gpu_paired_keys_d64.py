"""The paired key-owner kernel at head_dim 64 (its own number of waves per SIMD and workgroups per CU) at the edges of its 64-key blocks and
64-query steps: against the oracle, and against the kernel with one workgroup per key block."""
import pytest
import torch

from oracle import sb_oracle as O
from helpers import cu_from_lengths, max_abs, randn, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (40, torch.bfloat16), (64, torch.float16)])
@pytest.mark.parametrize("current", [False, True])
@pytest.mark.parametrize("lens", [[129], [191], [192], [193], [255], [256], [257], [577], [1, 321, 64, 65, 0, 200, 130]])
def test_paired_kernel_at_head_dim_64(lens, current, D, dtype, monkeypatch):
    from flame_amd import sb_attn_varlen
    H, N = 2, sum(lens)
    q, k, v, do = (randn((H, N, D), 970 + i, 0.5 if i < 3 else 1.0, dtype) for i in range(4))
    dr = randn((H, N), 975, 1.0, dtype)
    cu = cu_from_lengths(lens)
    qg, kg, vg = (x.cuda().requires_grad_(True) for x in (q, k, v))

    def run(kernel):
        monkeypatch.setenv("SBA_DKV_KERNEL", kernel)
        o, rem = sb_attn_varlen(qg, kg, vg, cu.cuda(), max(lens), attend_current=current)
        return torch.autograd.grad((o, rem), (qg, kg, vg), (do.cuda(), dr.cuda()))

    ref = O.sb_attn_grads_oracle(q, k, v, do, dr, cu_seqlens=cu.tolist(), attend_current=current)[2:]
    plain = run("plain")
    for kernel in ("pair", "pairq"):                            # (scores of scaled K and of the dQ pass's scaled q)
        for g, other, r in zip(run(kernel), plain, ref):        # (the bounds of the other packed tests of these kernels)
            assert max_abs(g.float().cpu(), r) <= 5e-2 and rel_l2(g.float().cpu(), r) <= 2e-2
            assert rel_l2(g.float(), other.float()) <= 2e-2
