"""Launches whose workgroups draw their jobs from queues against the same with a workgroup per job: the same kernels' arithmetic, bit for
bit, with barely more jobs than workgroups and with several rounds, queues in heads and in sequences, and every way of keeping the carries."""
import pytest
import torch

from helpers import cu_from_lengths, randn

pytestmark = pytest.mark.gpu

CASES = [
    # (sequences, heads, tokens or document lengths, D, dtype)
    (1, 16, 5500, 128, torch.bfloat16),              # 688 workgroups of 512, in all three passes
    (1, 16, 4100, 128, torch.bfloat16),              # 528 of 512 (the forward takes its two segments)
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
    monkeypatch.setenv("SBA_DKV_KERNEL", "pair")
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


# (heads, tokens, D, row-owner workgroups a CU, key-owner workgroups a CU, whether the forward draws)
@pytest.mark.parametrize("H,T,D,row_slots,key_slots,forward", [(16, 5500, 128, 2, 2, True), (12, 8000, 96, 2, 2, True), (16, 4100, 128, 2, 2, False), (24, 4500, 64, 3, 3, False)])
def test_queues_are_drawn_from(H, T, D, row_slots, key_slots, forward, monkeypatch):
    # Called through the C ABI, where the tables are at hand: the queues' counters (entries 32 and 48 of the first row block's last column, heads
    # 0 to 7) say that the jobs behind the first round were drawn, also by a key-owner pass that is called by itself, and more than once.
    import ctypes as C
    import math
    from flame_amd import _lib
    lib = _lib.load()
    monkeypatch.setenv("SBA_DQ_KERNEL", "lean")
    monkeypatch.setenv("SBA_DKV_KERNEL", "pair")
    q, k, v, do = (randn((1, H, T, D), 980 + i, 0.5 if i < 3 else 1.0, torch.bfloat16).cuda() for i in range(4))
    p = _lib.SbaParams()
    p.struct_size = C.sizeof(_lib.SbaParams)
    p.dtype = _lib.SBA_DTYPE_BF16
    p.n_seq, p.n_heads, p.seq_len, p.total_tokens, p.head_dim = 1, H, T, T, 128 if D == 96 else D
    p.columns = D if D == 96 else 0
    p.scale = 1.0 / math.sqrt(D)
    p.q, p.k, p.v = _lib.tensor4(q), _lib.tensor4(k), _lib.tensor4(v)
    p.stream = torch.cuda.current_stream().cuda_stream
    p.save_for_backward = 1
    ws = torch.empty(int(lib.sba_workspace_bytes(C.byref(p))) // 4, dtype=torch.int32, device="cuda")
    scratch = torch.empty(int(lib.sba_bwd_scratch_bytes(C.byref(p))) // 4, dtype=torch.int32, device="cuda")
    p.workspace, p.workspace_bytes = ws.data_ptr(), 4 * ws.numel()
    p.bwd_scratch, p.bwd_scratch_bytes = scratch.data_ptr(), 4 * scratch.numel()
    row_blocks = (T + 127) // 128
    stride = row_blocks * (row_blocks + 1) * 128
    rtab, gtab = ws[ws.numel() // 2:], scratch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    untouched = -7

    def counters(table, entry):
        return [int(table[128 + entry + i * stride]) for i in range(8)]

    def behind_first_round(jobs, slots):
        return [len(range(i, jobs, 8)) - (slots * cus & ~7) // 8 for i in range(8)]

    def run(draw, phases):
        monkeypatch.setenv("SBA_DRAW", draw)
        ws.fill_(untouched)
        scratch.fill_(untouched)
        out = [torch.full_like(q, math.nan) for _ in range(4)]
        rem = torch.full((1, H, T), math.nan, dtype=q.dtype, device="cuda")
        p.o, p.dq, p.dk, p.dv = (_lib.tensor4(t) for t in out)
        p.rem = _lib.SbaVector(rem.data_ptr(), rem.stride(0), rem.stride(1))
        p.d_o = _lib.tensor4(do)
        _lib.check(lib.sba_fwd(C.byref(p)), "sba_fwd")
        taken = [counters(rtab, 32)]
        for phase in phases:
            p.bwd_phases = phase
            if phase == 2:
                out[2].fill_(math.nan)
                out[3].fill_(math.nan)
            _lib.check(lib.sba_bwd(C.byref(p)), "sba_bwd")
            taken += [counters(gtab, 32), counters(gtab, 48)]
        return out + [rem], taken

    want, taken = run("0", [0])
    assert taken == [[untouched] * 8, [untouched] * 8, [0] * 8]
    for phases in ([0], [1, 2, 2]):
        got, taken = run("1", phases)
        for a, b in zip(got, want):
            assert torch.equal(a, b)
        for at, (jobs, slots) in ((0, (row_blocks * H, row_slots)), (1, (row_blocks * H, row_slots)), (-1, (2 * row_blocks * H, key_slots))):
            if at or forward:
                # every workgroup has taken a ticket behind its last job, too, from a queue that was empty by then
                assert all(n >= least > 0 for n, least in zip(taken[at], behind_first_round(jobs, slots))), (at, taken)
            else:
                assert taken[at] == [untouched] * 8


def test_drawn_jobs_on_two_streams(monkeypatch):
    monkeypatch.setenv("SBA_DRAW", "1")
    steps = [_run(CASES[0]), _run(CASES[0], current=True)]
    wants = [step() for step in steps]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in steps]
    got = []
    for _ in range(2):
        for stream, step in zip(streams, steps):
            with torch.cuda.stream(stream):
                got.append(step())
    torch.cuda.synchronize()
    for i, out in enumerate(got):
        assert all(torch.equal(a, b) for a, b in zip(out, wants[i % 2]))
