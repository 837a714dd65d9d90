"""The paired key-owner kernel with workgroups of two and of four pairs of waves, at the edges of their key blocks: against the
oracle, and bit for bit against each other (they add the same products in the same order)."""
import pytest
import torch

from oracle import sb_oracle as O
from helpers import cu_from_lengths, max_abs, randn, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,dtype", [(72, torch.bfloat16), (96, torch.float16), (128, torch.bfloat16)])
@pytest.mark.parametrize("current", [False, True])
@pytest.mark.parametrize("lens", [[129], [191], [192], [193], [255], [256], [257], [577], [1, 321, 64, 65, 200, 130]])
def test_two_and_four_pairs_of_waves(lens, current, D, dtype, monkeypatch):
    from flame_amd import sb_attn_varlen
    H, N = 2, sum(lens)
    q, k, v, do = (randn((H, N, D), 940 + i, 0.5 if i < 3 else 1.0, dtype) for i in range(4))
    cu = cu_from_lengths(lens)
    qg, kg, vg = (x.cuda().requires_grad_(True) for x in (q, k, v))

    def run(kernel):
        monkeypatch.setenv("SBA_DKV_KERNEL", kernel)
        o, _ = sb_attn_varlen(qg, kg, vg, cu.cuda(), max(lens), attend_current=current)
        return torch.autograd.grad(o, (qg, kg, vg), do.cuda())

    two = run("pair")
    assert all(torch.equal(a, b) for a, b in zip(two, run("pair4")))
    ref = O.sb_attn_grads_oracle(q, k, v, do, None, cu_seqlens=cu.tolist(), attend_current=current)[2:]
    for g, r in zip(two, ref):          # (the bounds of the other packed tests of these kernels)
        assert max_abs(g.float().cpu(), r) <= 5e-2 and rel_l2(g.float().cpu(), r) <= 2e-2
