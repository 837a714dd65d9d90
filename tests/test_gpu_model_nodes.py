"""The native nodes of the language model (csrc/sba_torch_model.cpp) against the module-by-module path with the same weights in
fp32, and clipping with AdamW against torch's own."""
import pytest
import torch
import torch.nn.functional as F

from helpers import cu_from_lengths, rel_l2

pytestmark = pytest.mark.gpu


# hidden sizes at and off the 256 columns a wave keeps per register group, one to many rows, both head dims
@pytest.mark.parametrize("hidden,heads,B,T,lens,dtype", [
    (64, 1, 1, 1, None, torch.bfloat16),
    (256, 4, 2, 33, None, torch.bfloat16),
    (320, 5, 1, 700, [130, 7, 500, 63], torch.bfloat16),
    (512, 4, 3, 257, None, torch.float16),
    (1024, 16, 1, 1500, [1, 1499], torch.float16),
    (2048, 32, 1, 129, None, torch.bfloat16),
])
def test_block_and_head_and_loss_match_the_modules(hidden, heads, B, T, lens, dtype, monkeypatch):
    from flame_amd import fused
    from flame_amd.modeling_sba import SBAConfig, SBAForCausalLM
    torch.manual_seed(hidden + T)
    m = SBAForCausalLM(SBAConfig(hidden_size=hidden, num_heads=heads, num_hidden_layers=2, vocab_size=1000,
                                 initializer_range=hidden ** -0.5)).cuda()
    with torch.no_grad():
        for p in m.parameters():
            if p.dim() == 1:
                p.add_(0.1 * torch.randn_like(p))
    ids = torch.randint(0, 1000, (B, T), device="cuda")
    labels = ids.clone()
    labels[:, T // 2] = -100
    kwargs = {} if lens is None else {"cu_seqlens": cu_from_lengths(lens).cuda(), "max_seqlen": max(lens)}

    def run(grads=True):
        m.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=dtype):
            loss, logits = m(ids, labels=labels, **kwargs)
        if T == 1 or not grads:
            return loss, logits, {}
        loss.backward()
        return loss, logits, {n: p.grad for n, p in m.named_parameters()}

    taken = []
    block = fused.block
    with monkeypatch.context() as mp:
        mp.setattr(fused, "block", lambda *a: taken.append(block(*a)) or taken[-1])
        loss, logits, grads = run()
    assert len(taken) == 2 and all(y is not None for y in taken)
    with torch.no_grad():
        assert torch.equal(run(False)[1], logits)
    with monkeypatch.context() as mp:
        for name in ("block", "head", "next_token_loss"):
            mp.setattr(fused, name, lambda *a, **k: None)
        loss_ref, logits_ref, grads_ref = run()
    tol = 2e-2 if dtype == torch.bfloat16 else 4e-3
    assert rel_l2(logits.float(), logits_ref.float()) <= tol
    assert T == 1 or abs(float(loss) - float(loss_ref)) <= tol
    for n in grads:
        assert grads[n].dtype == torch.float32 and grads[n].shape == grads_ref[n].shape
        assert rel_l2(grads[n], grads_ref[n]) <= 2 * tol, n


# vocabularies off the 8 columns of a 16-byte chunk, also one to seven columns past a tile of 256
@pytest.mark.parametrize("vocab", [1004, 1009, 1025])
def test_ragged_vocabularies_match_the_modules(vocab, monkeypatch):
    from flame_amd import fused
    from flame_amd.modeling_sba import SBAConfig, SBAForCausalLM
    torch.manual_seed(vocab)
    m = SBAForCausalLM(SBAConfig(hidden_size=128, num_heads=2, num_hidden_layers=1, vocab_size=vocab, initializer_range=0.1)).cuda()
    ids = torch.randint(0, vocab, (2, 65), device="cuda")

    def run():
        m.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            loss, logits = m(ids, labels=ids)
        loss.backward()
        return loss, logits, {n: p.grad for n, p in m.named_parameters()}

    loss, logits, grads = run()
    with monkeypatch.context() as mp:
        for name in ("block", "head", "next_token_loss"):
            mp.setattr(fused, name, lambda *a, **k: None)
        loss_ref, logits_ref, grads_ref = run()
    assert rel_l2(logits.float(), logits_ref.float()) <= 2e-2 and abs(float(loss) - float(loss_ref)) <= 2e-2
    for n in grads:
        assert rel_l2(grads[n], grads_ref[n]) <= 4e-2, n
    # every row of the weight's gradient on its own: none may hold another one's
    assert (grads["lm_head.weight"] - grads_ref["lm_head.weight"]).norm(dim=1).max() <= 4e-2 * grads_ref["lm_head.weight"].norm(dim=1).max()


def test_weight_gradient_of_an_unaligned_buffer():
    # a gradient of the logits that a caller cut out of a larger buffer of its own
    from flame_amd import fused
    torch.manual_seed(0)
    norm, lm_head = torch.nn.RMSNorm(64).cuda(), torch.nn.Linear(64, 264, bias=False).cuda()
    x = torch.randn(1, 37, 64, device="cuda")
    buf = torch.randn(37 * 264 + 3, device="cuda").to(torch.bfloat16)
    d = buf[3:].view(1, 37, 264)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        logits = fused.head(x, norm, lm_head)
    logits.backward(d)
    ref = d[0].float().t() @ F.rms_norm(x[0], (64,), norm.weight, torch.finfo(torch.float32).eps).detach().to(torch.bfloat16).float()
    assert rel_l2(lm_head.weight.grad, ref) <= 1e-2


def test_hooks_and_other_modules_keep_the_module_path():
    from flame_amd import fused
    from flame_amd.modeling_sba import SBAConfig, SBAForCausalLM
    m = SBAForCausalLM(SBAConfig(hidden_size=128, num_heads=2, num_hidden_layers=1, vocab_size=64)).cuda()
    x = torch.randn(1, 5, 128, device="cuda")
    blk = m.model.layers[0]
    assert fused.block(blk, x, {}) is None                       # no autocast
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert fused.block(blk, x, {}) is not None
        seen = []
        hook = blk.mlp.down_proj.register_forward_hook(lambda *a: seen.append(1))
        assert fused.block(blk, x, {}) is None
        blk(x)
        assert seen == [1]
        hook.remove()
        assert fused.block(blk, x.to(torch.bfloat16), {}) is None
        blk.attn.attn_fn = lambda q, k, v, t: (q, None)
        assert fused.block(blk, x, {}) is None


@pytest.mark.parametrize("rows,len_,classes", [(1, 1, 8), (6, 3, 2048), (7, 7, 2056), (40, 10, 32000)])
def test_loss_edges_against_torch(rows, len_, classes):
    from flame_amd import fused
    torch.manual_seed(classes)
    logits = (4 * torch.randn(rows // len_, len_, classes, device="cuda")).to(torch.bfloat16)
    logits[0, 0, : classes // 2] = -float("inf")
    labels = torch.randint(classes // 2, classes, (rows // len_, len_), device="cuda")
    a, b = (logits.clone().requires_grad_(True) for _ in range(2))
    got = fused.next_token_loss(a, labels)
    shifted = torch.cat((labels[:, 1:], torch.full_like(labels[:, :1], -100)), 1)
    ref = F.cross_entropy(b.float().view(rows, -1), shifted.view(-1), ignore_index=-100)
    if len_ == 1:
        assert torch.isnan(got) and torch.isnan(ref)             # no row counts
        return
    (3 * got).backward()
    (3 * ref).backward()
    assert abs(float(got) - float(ref)) <= 1e-5 * float(ref)
    assert rel_l2(a.grad.float(), b.grad.float()) <= 5e-3


def test_loss_of_logits_off_a_16_byte_boundary():
    from flame_amd import fused
    torch.manual_seed(0)
    buf = torch.randn(2 * 9 * 264 + 3, device="cuda").to(torch.bfloat16)
    labels = torch.randint(0, 264, (2, 9), device="cuda")
    a = buf[3:].view(2, 9, 264).requires_grad_()
    b = a.detach().clone().requires_grad_()
    assert a.data_ptr() % 16 and b.data_ptr() % 16 == 0
    with torch.no_grad():
        assert torch.equal(fused.next_token_loss(a, labels), fused.next_token_loss(b, labels))
    for x in (a, b):
        fused.next_token_loss(x, labels).backward()
    assert torch.equal(a.grad, b.grad)


@pytest.mark.parametrize("max_norm", [1e-2, 1e6])
def test_clip_and_adamw_in_one_pass_matches_torch(max_norm):
    # lengths around the four values of a load and the chunk a workgroup takes; two parameter groups, one weight without gradient
    from flame_amd import fused
    sizes = [1, 3, 4, 1023, 16383, 16384, 16385, 50000]
    runs = []
    for native in (True, False):
        torch.manual_seed(0)
        ps = [torch.nn.Parameter(torch.randn(n, device="cuda")) for n in sizes] + [torch.nn.Parameter(torch.ones(5, device="cuda"))]
        opt = torch.optim.AdamW([{"params": ps[:4], "lr": 1e-2, "weight_decay": 0.3}, {"params": ps[4:]}], lr=1e-3,
                                betas=(0.9, 0.95), eps=1e-8, fused=True)
        sched = torch.optim.lr_scheduler.LambdaLR(opt, lambda s: 1.0 / (s + 1))
        norms = []
        for step in range(4):
            for p in ps[:-1]:
                p.grad = torch.randn_like(p)
            norm = fused.clip_and_step(ps, opt, max_norm) if native else None
            assert (norm is not None) == (native and step > 0)   # the first step sets the state up
            if norm is None:
                norm = torch.nn.utils.clip_grad_norm_(ps, max_norm)
                opt.step()
            sched.step()
            norms.append(float(norm))
        runs.append((norms, [p.detach() for p in ps], [p.grad for p in ps[:-1]],
                     [opt.state[p][k] for p in ps[:-1] for k in ("exp_avg", "exp_avg_sq", "step")]))
    (na, pa, ga, sa), (nb, pb, gb, sb) = runs
    assert all(abs(x - y) <= 1e-5 * y for x, y in zip(na, nb))
    for a, b in zip(pa + ga + sa, pb + gb + sb):
        assert torch.allclose(a, b, rtol=2e-5, atol=1e-7)


def test_clip_and_step_leaves_a_captured_step_to_the_optimizer():
    # which refuses it without `capturable`: nothing of the step may be in the graph
    from flame_amd import fused
    ps = [torch.nn.Parameter(torch.ones(1000, device="cuda"))]
    opt = torch.optim.AdamW(ps, lr=1e-2, fused=True)
    ps[0].grad = torch.ones_like(ps[0])
    opt.step()
    before = [t.clone() for t in (ps[0], *(opt.state[ps[0]][k] for k in ("exp_avg", "exp_avg_sq", "step")))]
    x = torch.ones(8, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = x + 1
        assert fused.clip_and_step(ps, opt, 1.0) is None
        with pytest.raises(RuntimeError, match="capturable"):
            opt.step()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, x + 1)
    after = [ps[0], *(opt.state[ps[0]][k] for k in ("exp_avg", "exp_avg_sq", "step"))]
    assert all(torch.equal(a, b) for a, b in zip(before, after))
    assert fused.clip_and_step(ps, opt, 1.0) is not None         # and outside of a capture it is taken again


def test_forward_mode_tangents_are_kept_or_refused():
    # a dual input that needs no gradient: the operator says that it has no such derivative, the model's other parts have one
    from torch.autograd import forward_ad
    from flame_amd import fused, sb_attn, sb_attn_varlen
    from flame_amd.modeling_sba import SBAConfig, SBAForCausalLM, next_token_loss
    torch.manual_seed(0)
    m = SBAForCausalLM(SBAConfig(hidden_size=128, num_heads=2, num_hidden_layers=1, vocab_size=256)).cuda()
    m.requires_grad_(False)
    rand = lambda *s: torch.randn(*s, device="cuda")
    x, tx, logits, tl = rand(1, 9, 128), rand(1, 9, 128), rand(1, 9, 256), rand(1, 9, 256)
    ids = torch.randint(0, 256, (1, 9), device="cuda")
    with forward_ad.dual_level():
        q = rand(1, 2, 9, 64).to(torch.bfloat16)
        for i in range(3):
            args = [q, q, q]
            args[i] = forward_ad.make_dual(q, torch.ones_like(q))
            with pytest.raises(NotImplementedError):
                sb_attn(*args)
            with pytest.raises(NotImplementedError):
                sb_attn_varlen(*(a[0] for a in args), torch.tensor([0, 4, 9], dtype=torch.int32), 5)
        sb_attn(q, q, q)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            dual = forward_ad.make_dual(x, tx)
            assert fused.block(m.model.layers[0], dual, {}) is None
            with pytest.raises(NotImplementedError):
                m.model.layers[0](dual)
            assert fused.head(dual, m.model.norm, m.lm_head) is None
            assert fused.head(x, m.model.norm, m.lm_head) is not None
        half = logits.to(torch.bfloat16)
        loss, got = forward_ad.unpack_dual(next_token_loss(forward_ad.make_dual(half, tl.to(torch.bfloat16)), ids))
    leaf = half.float().requires_grad_()
    want, = torch.autograd.grad(F.cross_entropy(leaf[0, :-1], ids[0, 1:]), leaf)
    assert got is not None and abs(float(got) - float((want * tl.to(torch.bfloat16).float()).sum())) <= 1e-5 * float(want.norm() * tl.norm())


def test_gradients_of_gradients_are_right_or_refused():
    from flame_amd.modeling_sba import SBAConfig, SBAForCausalLM, next_token_loss
    torch.manual_seed(0)
    labels = torch.randint(0, 264, (2, 9), device="cuda")
    labels[0, 3] = -100
    a = torch.randn(2, 9, 264, device="cuda").to(torch.bfloat16).transpose(0, 1).contiguous().transpose(0, 1).requires_grad_()
    b = a.detach().float().requires_grad_()
    w = torch.randn(2, 9, 264, device="cuda")
    shifted = torch.cat((labels[:, 1:], torch.full_like(labels[:, :1], -100)), 1)
    first, second = [], []
    for x, loss in ((a, 3 * next_token_loss(a, labels)),
                    (b, 3 * F.cross_entropy(b.reshape(18, -1), shifted.view(-1), ignore_index=-100))):
        g, = torch.autograd.grad(loss, x, create_graph=True)
        first.append(g.detach().float())
        second.append(torch.autograd.grad((g.float() * w).sum(), x)[0].float())
    # bf16 values of both: 2^-9 each, and of the second one's incoming gradient, which is rounded the same way
    assert rel_l2(first[0], first[1]) <= 5e-3 and rel_l2(second[0], second[1]) <= 1e-2

    m = SBAForCausalLM(SBAConfig(hidden_size=128, num_heads=2, num_hidden_layers=1, vocab_size=264, initializer_range=0.1)).cuda()
    ids = torch.randint(0, 264, (1, 40), device="cuda")
    params = list(m.parameters())

    def loss():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            return m(ids, labels=ids)[0]

    plain = torch.autograd.grad(loss(), params)
    kept = torch.autograd.grad(loss(), params, create_graph=True)
    for p, x, y in zip(params, plain, kept):
        assert rel_l2(y, x) <= 1e-2                              # (the logits' gradient rounds elsewhere)
        if p is not m.model.embeddings.weight:
            with pytest.raises(RuntimeError, match="differentiate once"):
                torch.autograd.grad(y.square().sum(), params, retain_graph=True, allow_unused=True)
            with pytest.raises(RuntimeError, match="differentiate once"):
                y.sum().backward(retain_graph=True)

    # one weight alone, behind gradients that depend on nothing
    blk = m.model.layers[0].requires_grad_(False)
    wq = blk.attn.q_proj.weight.requires_grad_()
    x = torch.randn(1, 40, 128, device="cuda")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = blk(x)
    g, = torch.autograd.grad(y, wq, torch.ones_like(y), create_graph=True)
    with pytest.raises(RuntimeError, match="differentiate once"):
        torch.autograd.grad(g.sum(), wq)


def test_frozen_weights_cost_no_gradients():
    # every single weight of a block and its head, the norms, a few together, the input alone: the same gradients as when all are
    # asked for, and no memory for the others'
    from flame_amd import fused
    from flame_amd.modeling_sba import SBAConfig, SBAForCausalLM
    torch.manual_seed(0)
    m = SBAForCausalLM(SBAConfig(hidden_size=256, num_heads=4, num_hidden_layers=1, vocab_size=512, initializer_range=0.06)).cuda()
    blk = m.model.layers[0]
    x = torch.randn(1, 100, 256, device="cuda")
    dy, dl = torch.randn(1, 100, 256, device="cuda"), torch.randn(1, 100, 512, device="cuda").to(torch.bfloat16)

    def grads(weights, with_x):
        leaves = dict(weights, x=x.clone()) if with_x else dict(weights)
        for p in m.parameters():
            p.requires_grad_(False)
        for t in leaves.values():
            t.requires_grad_(True)
        xin = leaves.get("x", x)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            head = any(n == "norm" or n == "lm_head" for n in weights)
            out, d = (fused.head(xin, m.model.norm, m.lm_head), dl) if head else (fused.block(blk, xin, {}), dy)
        before = torch.cuda.memory_stats()["allocated_bytes.all.allocated"]
        got = torch.autograd.grad(out, list(leaves.values()), d)
        return dict(zip(leaves, got)), torch.cuda.memory_stats()["allocated_bytes.all.allocated"] - before

    own = dict(blk.named_parameters())
    names = list(own)
    for weights, picks in (
            (own, [[n] for n in names] + [[], ["attn.q_proj.weight", "attn.v_proj.weight"], ["attn.k_proj.weight", "mlp.up_proj.weight"]]),
            ({"norm": m.model.norm.weight, "lm_head": m.lm_head.weight}, [["norm"], ["lm_head"]])):
        full, bytes_full = grads(weights, True)
        for pick in picks:
            for with_x in (True, False) if pick else (True,):
                got, used = grads({n: weights[n] for n in pick}, with_x)
                assert set(got) == set(pick) | ({"x"} if with_x else set())
                for n, g in got.items():
                    assert rel_l2(g, full[n]) <= 1e-5, (pick, n)      # fp32 sums, perhaps in another number of splits
                # (a norm's gradient comes with its input's, k's lies between q's and v's)
                spared = [n for n in weights if n not in pick and weights[n].dim() == 2]
                if pick == ["attn.q_proj.weight", "attn.v_proj.weight"]:
                    spared.remove("attn.k_proj.weight")
                assert used <= bytes_full - sum(weights[n].numel() * 4 for n in spared), pick


def test_observed_and_transformed_operators_keep_the_module_path():
    from torch.utils.flop_counter import FlopCounterMode
    from flame_amd import fused
    from flame_amd.modeling_sba import SBAConfig, SBAForCausalLM, next_token_loss

    class Other(torch.Tensor):
        pass

    torch.manual_seed(0)
    m = SBAForCausalLM(SBAConfig(hidden_size=128, num_heads=2, num_hidden_layers=1, vocab_size=64)).cuda()
    ids = torch.randint(0, 64, (1, 20), device="cuda")
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16), FlopCounterMode(display=False) as counter:
        m(ids)
    block = 4 * 128 ** 2 + 3 * 128 * m.model.layers[0].mlp.gate_proj.weight.shape[0]
    assert counter.get_total_flops() == 2 * 20 * (block + 128 * 64)
    logits = torch.randn(3, 1, 20, 64, device="cuda").to(torch.bfloat16)
    each = torch.func.vmap(lambda x: next_token_loss(x, ids))(logits)
    grads = torch.func.grad(lambda x: next_token_loss(x, ids))(logits[0])
    leaf = logits.clone().requires_grad_()
    want = [next_token_loss(x, ids) for x in leaf]
    want[0].backward()
    for a, b in zip(each, want):
        assert abs(float(a) - float(b.detach())) <= 1e-5 * float(b.detach())
    assert rel_l2(grads.float(), leaf.grad[0].float()) <= 5e-3
    assert fused.next_token_loss(logits[0].as_subclass(Other), ids) is None
    x = torch.randn(1, 20, 128, device="cuda")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert fused.head(x, m.model.norm, m.lm_head) is not None
        assert fused.head(x.as_subclass(Other), m.model.norm, m.lm_head) is None
