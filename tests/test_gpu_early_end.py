"""Sweeps that end where nothing is left of any row's stick: bit for bit the results of the full sweeps, in every kernel."""
import pytest
import torch

from oracle import sb_oracle as O
from helpers import cu_from_lengths, rel_l2

pytestmark = pytest.mark.gpu


def _inputs(H, lead, T, D, dtype, seed):
    """Heads whose mean logit lies between 0 and -6, and between stretches of 96 rows another sharpness, so that neighbouring
    row blocks end their sweeps far from each other; the longest sweeps of the last heads never end."""
    g = torch.Generator("cuda").manual_seed(seed)
    c = (torch.linspace(0, 6, H, device="cuda") * D ** 0.5 / D).sqrt()[:, None, None]
    rows = (torch.arange(T, device="cuda") // 96 % 3)[:, None] * 0.5 + 0.4
    q = torch.randn(lead + (H, T, D), device="cuda", generator=g) * 0.5 + c * rows
    k = torch.randn(lead + (H, T, D), device="cuda", generator=g) * 0.5 - c
    v = torch.randn(lead + (H, T, D), device="cuda", generator=g) * 0.5
    do = torch.randn(lead + (H, T, D), device="cuda", generator=g)
    dr = torch.randn(lead + (H, T), device="cuda", generator=g)
    return tuple(x.to(dtype) for x in (q, k, v, do, dr))


def _run(x, lens, current):
    from flame_amd import sb_attn, sb_attn_varlen
    q, k, v = (t.detach().requires_grad_(True) for t in x[:3])
    if lens is None:
        o, rem = sb_attn(q, k, v, attend_current=current)
    else:
        o, rem = sb_attn_varlen(q, k, v, cu_from_lengths(lens).cuda(), max(lens), attend_current=current)
    return (o.detach(), rem.detach()) + torch.autograd.grad((o, rem), (q, k, v), x[3:])


CASES = [  # B, H, T or lengths, D, dtype, options
    (1, 4, 2048, 64, torch.bfloat16, {}),
    (1, 4, 2048, 64, torch.bfloat16, {"SBA_RECOMPUTE_CARRIES": "1"}),
    (1, 4, 2048, 64, torch.bfloat16, {"SBA_FWD_GROUPS": "2"}),
    (1, 4, 2047, 64, torch.bfloat16, {"SBA_DKV_KERNEL": "pair"}),
    (1, 4, 2047, 64, torch.bfloat16, {"SBA_DKV_KERNEL": "pairq"}),
    (1, 4, 2047, 64, torch.float16, {"SBA_DKV_KERNEL": "plain"}),
    (1, 4, 2047, 64, torch.bfloat16, {"SBA_DKV_KERNEL": "stream8"}),
    (3, 16, 1537, 64, torch.bfloat16, {}),
    (1, 4, 9001, 64, torch.bfloat16, {}),
    (4, 16, 1100, 128, torch.float16, {}),
    (1, 4, 2100, 128, torch.bfloat16, {"SBA_RECOMPUTE_CARRIES": "1"}),
    (1, 4, 1601, 256, torch.bfloat16, {}),
    (1, 4, 1601, 64, torch.float32, {}),
    (1, 4, 1001, 128, torch.float32, {"SBA_RECOMPUTE_CARRIES": "1"}),
    (0, 4, [1, 700, 129, 2500, 64, 1000], 64, torch.bfloat16, {}),
    (0, 16, [900, 700, 129, 2500, 64, 1000, 333] * 6, 64, torch.bfloat16, {}),
    (0, 4, [1, 700, 129, 1500, 64], 80, torch.bfloat16, {}),
    (0, 4, [1, 700, 129, 1500, 64], 64, torch.float32, {}),
]


@pytest.mark.parametrize("current", [False, True])
@pytest.mark.parametrize("B,H,T,D,dtype,options", CASES)
def test_same_bits_as_full_sweeps(B, H, T, D, dtype, options, current, monkeypatch):
    for name, value in options.items():
        monkeypatch.setenv(name, value)
    lens = T if isinstance(T, list) else None
    x = _inputs(H, (B,) if B else (), sum(T) if lens else T, D, dtype, 40 + D)
    short = _run(x, lens, current)
    monkeypatch.setenv("SBA_FULL_SWEEPS", "1")
    for a, b in zip(short, _run(x, lens, current)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("D", [64, 128])
def test_against_the_oracle(D):
    T = 900
    x = _inputs(3, (1,), T, D, torch.bfloat16, 7)
    got = _run(x, None, False)
    ref = O.sb_attn_grads_oracle(*(t.cpu() for t in x))
    for a, b in zip(got, ref):
        assert rel_l2(a.float().cpu(), b) <= 2e-2


@pytest.mark.parametrize("B,T,D,dtype", [
    (1, 1100, 64, torch.bfloat16),         # two steps an iteration
    (5, 1100, 64, torch.bfloat16),         # one step
    (1, 1100, 128, torch.float16),
    (1, 1100, 64, torch.float32),
])
def test_a_gradient_of_rem_that_is_no_number_shows_where_the_stick_is_used_up(B, T, D, dtype, monkeypatch):
    # the first head (logits near 0) uses its stick up within some 150 keys; inf * 0 and NaN * 0 of a row whose sweep ended are NaN
    x = list(_inputs(4, (B,), T, D, dtype, 11))
    dr = x[4]
    dr[0, 0, 700], dr[0, 0, 901], dr[0, 0, 1099] = float("inf"), float("nan"), -float("inf")
    dq, dk = _run(x, None, False)[2:4]
    monkeypatch.setenv("SBA_FULL_SWEEPS", "1")
    full = _run(x, None, False)[2]
    assert torch.equal(dq.isnan(), full.isnan()) and torch.equal(dq.nan_to_num(7), full.nan_to_num(7))
    assert bool(dq[0, 0, [700, 901, 1099]].isnan().all())
    assert bool(dk[0, 0, [690, 890, 1090]].isnan().all())        # the keys that these rows still reach


# with room for one of the forward's two tables, the other made by the dQ pass on its way
@pytest.mark.parametrize("B,H,T,D,dtype", [
    (1, 4, 2047, 64, torch.bfloat16),
    (3, 16, 1100, 64, torch.float16),
    (1, 4, 2100, 128, torch.float16),
    (1, 4, 1500, 80, torch.bfloat16),
    (0, 4, [1, 700, 129, 2500, 64, 1000], 64, torch.bfloat16),
    (0, 4, [1, 700, 129, 1500, 64], 128, torch.bfloat16),
    (0, 4, [1, 700, 129, 1500, 64], 96, torch.float16),
])
def test_same_bits_as_full_sweeps_with_one_kept_table(B, H, T, D, dtype, monkeypatch):
    from flame_amd import _lib
    lens = T if isinstance(T, list) else None
    x = _inputs(H, (B,) if B else (), sum(T) if lens else T, D, dtype, 60 + D)
    one = 4 * 128 * H * sum(n * (n + 1) for n in ((t + 127) // 128 for t in (lens or [T] * B)))
    kept = []

    def note(t):
        if t.dtype == torch.uint8:
            kept.append(t.numel())
        return t

    try:
        _lib.set_workspace_budget(1.5 * one)
        with torch.autograd.graph.saved_tensors_hooks(note, lambda t: t):
            _run(x, lens, False)
        assert kept == [one]
        short = _run(x, lens, False)
        monkeypatch.setenv("SBA_FULL_SWEEPS", "1")
        full = _run(x, lens, False)
    finally:
        _lib.set_workspace_budget(None)
    for a, b in zip(short, full):
        assert torch.equal(a, b)
