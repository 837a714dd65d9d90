"""Launches whose workgroups draw their jobs from queues against the same with a workgroup per job: the same kernels' arithmetic, bit for
bit, with barely more jobs than workgroups and with several rounds, queues in heads and in sequences, and every way of keeping the carries."""
import pytest
import torch

from helpers import cu_from_lengths, randn

pytestmark = pytest.mark.gpu

CASES = [
    # (sequences, heads, tokens or document lengths, D, dtype)
    (1, 16, 4100, 128, torch.bfloat16),              # 528 workgroups of 512
    (9, 3, 2500, 128, torch.float16),                # fewer heads than queues: the sequences hold them
    (2, 3, 6100, 96, torch.bfloat16),                # neither heads nor sequences enough: nothing is drawn
    (2, 24, 2500, 64, torch.bfloat16),               # 960 workgroups, three a CU in the dQ pass
    (1, 8, [0, 3000, 1, 129, 128, 64, 127, 5000, 700], 80, torch.bfloat16),
    (1, 40, [1, 3000, 0, 129, 128, 64, 65], 64, torch.float16),
]


def _run(case, current=False):
    from flame_amd import sb_attn, sb_attn_varlen
    B, H, tokens, D, dtype = case
    packed = isinstance(tokens, list)
    lead = (H, sum(tokens)) if packed else (B, H, tokens)
    q, k, v = (randn(lead + (D,), 960 + i, 0.5, dtype).cuda().requires_grad_(True) for i in range(3))
    do, drem = randn(lead + (D,), 963, 1.0, dtype).cuda(), randn(lead, 964, 1.0, dtype).cuda()
    cu = cu_from_lengths(tokens).cuda() if packed else None

    def step():
        o, rem = sb_attn_varlen(q, k, v, cu, max(tokens), attend_current=current) if packed else sb_attn(q, k, v, attend_current=current)
        return (o, rem) + torch.autograd.grad((o, rem), (q, k, v), (do, drem))
    return step


@pytest.mark.parametrize("keeps", ["both tables", "one table", "nothing"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: f"B{c[0]}-H{c[1]}-D{c[3]}")
def test_drawn_jobs_give_the_same_bits(case, keeps, monkeypatch):
    from flame_amd import _lib
    monkeypatch.setenv("SBA_DQ_KERNEL", "lean")
    monkeypatch.setenv("SBA_DKV_KERNEL", "pair" if case[3] > 64 else "own")
    if keeps == "nothing":
        monkeypatch.setenv("SBA_RECOMPUTE_CARRIES", "1")
    step = _run(case, current=keeps == "one table")
    try:
        if keeps == "one table":
            B, H, tokens = case[:3]
            lens = tokens if isinstance(tokens, list) else [tokens] * B
            columns = sum(n * (n + 1) for n in ((t + 127) // 128 for t in lens))
            _lib.set_workspace_budget(1.5 * columns * H * 128 * 4)
        monkeypatch.setenv("SBA_DRAW", "0")
        want = step()
        monkeypatch.setenv("SBA_DRAW", "1")
        for _ in range(2):
            for a, b in zip(want, step()):
                assert torch.equal(a, b)
    finally:
        _lib.set_workspace_budget(None)


def test_drawn_jobs_captured_in_a_graph(monkeypatch):
    monkeypatch.setenv("SBA_DRAW", "1")
    step = _run(CASES[0])
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = step()
    for _ in range(3):
        want = step()
        for t in captured:
            t.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(captured, want))
