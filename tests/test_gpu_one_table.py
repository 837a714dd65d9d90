"""A budget that holds one of the forward's two carry tables: the forward keeps that one and the dQ pass makes the other
(16-bit types at head dims up to 128, sequences of more than 128 tokens; shorter ones repeat the forward's sweep)."""
import pytest
import torch

from flame_amd import _lib, sb_attn, sb_attn_varlen
from oracle import sb_oracle as O
from helpers import cu_from_lengths, randn, rel_l2

pytestmark = pytest.mark.gpu

# of the gradients, against the oracle: that of the whole tables (tests/test_gpu_parity.py)
TOL = {torch.bfloat16: 5e-2, torch.float16: 6.25e-3}


@pytest.fixture
def budget():
    yield _lib.set_workspace_budget
    _lib.set_workspace_budget(None)


def _table_bytes(lens, H):
    return 4 * 128 * H * sum(n * (n + 1) for n in ((length + 127) // 128 for length in lens))


# one row block and several, ragged ones, a large grid (one sweep per workgroup) and small ones (two segments), documents
@pytest.mark.parametrize("lens,H,D,dtype,current", [
    ([129], 2, 128, torch.bfloat16, False),
    ([193], 2, 96, torch.float16, True),
    ([1000], 4, 128, torch.bfloat16, False),
    ([1000], 4, 80, torch.bfloat16, False),
    ([100, 128, 3], 2, 128, torch.bfloat16, False),
    ([1000], 4, 64, torch.bfloat16, True),
    ([500] * 16, 16, 64, torch.float16, False),
    ([130, 1, 64, 700, 257], 3, 40, torch.bfloat16, False),
    ([500] * 16, 16, 128, torch.bfloat16, False),
    ([500] * 16, 16, 72, torch.float16, True),
    ([130, 1, 64, 700, 257], 3, 128, torch.float16, False),
    ([130, 1, 64, 700, 257], 3, 88, torch.bfloat16, True)])
def test_one_kept_table_against_the_oracle_and_both(lens, H, D, dtype, current, budget):
    N, dense = sum(lens), len(set(lens)) == 1
    scale = 1.0 if D in (64, 128) else 0.5                             # (sweeps that end, and that do not)
    q, k, v, do = (randn((H, N, D), 740 + i, scale if i < 3 else 1.0, dtype) for i in range(4))
    dr = randn((H, N), 745, 1.0, dtype)
    cu = cu_from_lengths(lens)
    results = []
    for nbytes in (float("inf"), 1.5 * _table_bytes(lens, H)):
        budget(nbytes)
        qg, kg, vg = (x.cuda().requires_grad_(True) for x in (q, k, v))
        if dense:
            b = lambda t: t.view(H, len(lens), lens[0], *t.shape[2:]).transpose(0, 1)
            o, rem = sb_attn(b(qg), b(kg), b(vg), attend_current=current)
            got = torch.autograd.grad((o, rem), (qg, kg, vg), (b(do.cuda()), b(dr.cuda())))
            o, rem = (x.transpose(0, 1).reshape(H, N, *x.shape[3:]) for x in (o, rem))
        else:
            o, rem = sb_attn_varlen(qg, kg, vg, cu.cuda(), max(lens), attend_current=current)
            got = torch.autograd.grad((o, rem), (qg, kg, vg), (do.cuda(), dr.cuda()))
        results.append((o, rem, *got))
    both, one = results
    assert torch.equal(both[0], one[0]) and torch.equal(both[1], one[1])
    # the carries differ by the rounding of a product in fp32, the gradients by single roundings to 16 bits that this tips
    for x, y in zip(both[2:], one[2:]):
        assert rel_l2(y.float(), x.float()) <= TOL[dtype] / 50
    ref = O.sb_attn_grads_oracle(q, k, v, do, dr, cu_seqlens=cu.tolist(), attend_current=current, compute_dtype=torch.float32)
    for g, r in zip(one[2:], ref[2:]):
        assert rel_l2(g.float().cpu(), r) <= TOL[dtype]
