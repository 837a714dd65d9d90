"""16-bit rows of 72 .. 96 columns on the matrix-core kernels without padding: against the oracle, inside tensors whose other
columns are NaN (nothing outside the rows may be read or written), on the small-grid, large-grid and short-sequence kernels."""
import pytest
import torch

from oracle import sb_oracle as O
from helpers import cu_from_lengths, max_abs, randn, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,dtype", [(72, torch.bfloat16), (80, torch.bfloat16), (88, torch.float16), (96, torch.bfloat16),
                                     (96, torch.float16)])
@pytest.mark.parametrize("B,H,T", [(1, 2, 1), (2, 2, 65), (1, 2, 128), (1, 2, 129), (2, 3, 333), (1, 2, 1100)])
def test_rows_between_64_and_96_columns_against_the_oracle(B, H, T, D, dtype):
    from flame_amd import sb_attn
    q, k, v, do = (randn((B, H, T, D), 700 + i, 0.5 if i < 3 else 1.0, dtype) for i in range(4))
    dr = randn((B, H, T), 705, 1.0, dtype)

    def inside_nans(t):                            # rows of 104 elements, the last 104 - D of them NaN
        wide = torch.full(t.shape[:-1] + (104,), float("nan"), dtype=dtype, device="cuda")
        wide[..., :D] = t.cuda()
        return wide[..., :D]

    qg, kg, vg = (inside_nans(x).requires_grad_(True) for x in (q, k, v))
    for current in (False, True):
        o, rem = sb_attn(qg, kg, vg, attend_current=current)
        got = (o, rem) + torch.autograd.grad((o, rem), (qg, kg, vg), (inside_nans(do), dr.cuda()))
        ref = O.sb_attn_grads_oracle(q, k, v, do, dr, attend_current=current)
        scale = 1.0 if dtype == torch.bfloat16 else 0.125
        for g, r in zip(got, ref):
            assert g.shape == r.shape and max_abs(g.float().cpu(), r) <= 5e-2 * scale * max(1.0, float(r.abs().max()))
            assert rel_l2(g.float().cpu(), r) <= 2e-2 * scale or r.norm() == 0


@pytest.mark.parametrize("D", [80, 96])
def test_packs_of_rows_below_96_columns_match_zero_padded_rows(D, monkeypatch):
    # a pack of several workgroups per compute unit; recomputed carries give the same bits
    from flame_amd import sb_attn_varlen
    lens = [700, 1, 64, 129, 2000, 333, 5, 128] * 4
    H, N = 12, sum(lens)
    cu = cu_from_lengths(lens).cuda()
    q, k, v, do = (randn((H, N, D), 710 + i, 0.5 if i < 3 else 1.0, torch.bfloat16).cuda() for i in range(4))

    def run(pad):
        ins = [torch.nn.functional.pad(x, (0, pad)).requires_grad_(True) for x in (q, k, v)]
        o, rem = sb_attn_varlen(*ins, cu, max(lens), inv_temp=D ** -0.5)
        return [t[..., :D] if t.dim() == 3 else t for t in (o, rem, *torch.autograd.grad(o, ins, torch.nn.functional.pad(do, (0, pad))))]

    rows, padded = run(0), run(128 - D)
    for a, b in zip(rows, padded):
        assert rel_l2(a.float(), b.float()) <= 1e-3
    monkeypatch.setenv("SBA_RECOMPUTE_CARRIES", "1")
    assert all(torch.equal(a, b) for a, b in zip(rows, run(0)))
