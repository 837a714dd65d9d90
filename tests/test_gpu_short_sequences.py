"""The one-kernel backward of sequences that fit one workgroup, at the edges of its tiles, against the oracle and against the
two-pass kernels."""
import pytest
import torch

from oracle import sb_oracle as O
from helpers import cu_from_lengths, max_abs, randn, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("current", [False, True])
@pytest.mark.parametrize("lens", [[1], [2], [16], [17], [32], [33], [63], [64], [65], [66], [96], [97], [127], [128],
                                  [1, 128, 64, 65, 3, 127, 33, 96], [70, 40] * 70])
def test_short_sequences_against_the_oracle(lens, current, D):
    from flame_amd import sb_attn_varlen
    H, N = (3 if len(lens) < 100 else 16), sum(lens)
    q, k, v, do = (randn((H, N, D), 900 + i, 0.5 if i < 3 else 1.0, torch.bfloat16) for i in range(4))
    dr = randn((H, N), 905, 1.0, torch.bfloat16)
    cu = cu_from_lengths(lens)
    qg, kg, vg = (x.cuda().requires_grad_(True) for x in (q, k, v))
    o, rem = sb_attn_varlen(qg, kg, vg, cu.cuda(), max(lens), attend_current=current)
    got = torch.autograd.grad((o, rem), (qg, kg, vg), (do.cuda(), dr.cuda()))
    ref = O.sb_attn_grads_oracle(q, k, v, do, dr, cu_seqlens=cu.tolist(), attend_current=current)[2:]
    for g, r in zip(got, ref):
        assert max_abs(g.float().cpu(), r) <= 5e-2 and rel_l2(g.float().cpu(), r) <= (2e-2 if r.norm() > 0 else 0.0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,D", [(128, 64), (65, 64), (100, 128)])
def test_short_dense_batches_agree_with_the_two_passes(T, D, dtype, monkeypatch):
    # many sequences (several per compute unit), strided inputs (column slices of one tensor)
    from flame_amd import sb_attn
    B, H = 40, 16
    qkv = (torch.randn(B, T, 3 * H * D, device="cuda", generator=torch.Generator("cuda").manual_seed(7)) * 0.5).to(dtype)
    do = torch.randn(B, H, T, D, device="cuda", generator=torch.Generator("cuda").manual_seed(8)).to(dtype)

    def run():
        x = qkv.clone().requires_grad_(True)
        q, k, v = (t.unflatten(-1, (H, D)).transpose(1, 2) for t in x.split(H * D, dim=-1))
        o, _ = sb_attn(q, k, v)
        return torch.autograd.grad(o, x, do)[0]

    one = run()
    assert torch.equal(one, run())
    monkeypatch.setenv("SBA_DKV_KERNEL", "own" if D == 128 else "pair")
    assert rel_l2(one.float(), run().float()) <= (4e-3 if dtype == torch.bfloat16 else 5e-4)
