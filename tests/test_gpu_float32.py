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
