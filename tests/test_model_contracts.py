"""Which calls the language model's native nodes take, decided on the host: no GPU needed."""
import pytest
import torch

from flame_amd import _lib, fused


class _Native:
    """Stands in for the native module and notes what it is asked for."""
    max_norm_width = 2048

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        return lambda *a: self.calls.append(name) or name


@pytest.fixture
def native(monkeypatch):
    n = _Native()
    monkeypatch.setattr(_lib, "native", lambda: n)
    return n


@pytest.mark.parametrize("vocab,taken", [(1000, True), (1004, False), (1009, False), (32001, False)])
def test_head_takes_vocabularies_of_whole_chunks(vocab, taken, native, monkeypatch):
    monkeypatch.setattr(fused, "_compute_dtype", lambda x: torch.bfloat16)
    x, norm, lm_head = torch.randn(1, 3, 64), torch.nn.RMSNorm(64), torch.nn.Linear(64, vocab, bias=False)
    assert (fused.head(x, norm, lm_head) is not None) == taken
    assert native.calls == (["head"] if taken else [])


def test_weight_gradients_outside_their_contract_are_refused():
    grad = _lib.native().weight_grad                  # every one of these is refused before anything is launched
    rows = lambda cols, off=0: torch.zeros(64 * 2048, dtype=torch.bfloat16)[off:off + 16 * cols].view(16, cols)
    for d, x in [(rows(1009), rows(64)), (rows(1004), rows(64)), (rows(257), rows(64)), (rows(64), rows(60)),
                 (rows(64, off=1), rows(64)), (rows(64), rows(64, off=4)), (rows(72)[:, :64][:0], rows(64)[:0]),
                 (torch.zeros(16, 68, dtype=torch.bfloat16)[:, :64], rows(64))]:
        with pytest.raises(RuntimeError, match="bad shape"):
            grad(d, x)


def test_weights_of_other_shapes_are_left_to_the_modules_to_refuse(native, monkeypatch):
    from flame_amd.modeling_sba import SBABlock, SBAConfig
    from oracle import sb_oracle as O
    monkeypatch.setattr(fused, "_compute_dtype", lambda x: torch.bfloat16)
    cfg = SBAConfig(hidden_size=128, num_heads=2, intermediate_size=192)
    x = torch.randn(1, 5, 128)
    assert fused.block(SBABlock(cfg, 0), x, {}) is not None
    for name, shape in (("attn_norm", (136,)), ("mlp_norm", (64,)), ("attn.q_proj", (136, 128)), ("attn.k_proj", (128, 120)),
                        ("attn.v_proj", (64, 128)), ("attn.o_proj", (128, 64)), ("mlp.gate_proj", (192, 64)), ("mlp.up_proj", (200, 128)),
                        ("mlp.down_proj", (128, 184))):
        blk = SBABlock(cfg, 0)
        monkeypatch.setattr(blk.attn, "attn_fn", lambda q, k, v, t: O.sb_attn_oracle(q, k, v))
        with pytest.raises((RuntimeError, ValueError)):
            m = blk.get_submodule(name)
            m.weight = torch.nn.Parameter(torch.randn(shape))
            if "norm" in name:
                m.normalized_shape = shape
            blk.attn.attn_fn = fused.sb_attn                      # as far as fused.block() can tell, a usual block
            assert fused.block(blk, x, {}) is None
            blk.attn.attn_fn = lambda q, k, v, t: O.sb_attn_oracle(q, k, v)
            blk(x)
    norm, wide, head = torch.nn.RMSNorm(128), torch.nn.RMSNorm(136), torch.nn.Linear(128, 64, bias=False)
    assert fused.head(x, norm, head) is not None
    assert fused.head(x, wide, head) is None and fused.head(x, norm, torch.nn.Linear(136, 64, bias=False)) is None


def _adamw_after_one_step():
    p = torch.nn.Parameter(torch.ones(4))
    opt = torch.optim.AdamW([p], lr=1e-3, fused=True)
    p.grad = torch.ones(4)
    opt.step()
    return p, opt


def test_clip_and_step_leaves_hooked_optimizers_alone(native):
    from torch.optim.optimizer import register_optimizer_step_post_hook, register_optimizer_step_pre_hook
    p, opt = _adamw_after_one_step()
    for register in (register_optimizer_step_pre_hook, register_optimizer_step_post_hook,
                     opt.register_step_pre_hook, opt.register_step_post_hook):
        hook = register(lambda *a: None)
        assert fused.clip_and_step([p], opt, 1.0) is None and not native.calls
        hook.remove()
    assert fused.clip_and_step([p], opt, 1.0) is not None and native.calls == ["clip_and_step"]


def test_the_backbone_is_called_where_a_hook_or_a_compiled_call_would_see_it(monkeypatch):
    from torch.nn.modules.module import register_module_forward_hook, register_module_full_backward_hook
    from flame_amd.modeling_sba import SBAConfig, SBAForCausalLM, SBAModel
    from oracle import sb_oracle as O
    m = SBAForCausalLM(SBAConfig(hidden_size=64, num_hidden_layers=1, num_heads=1, vocab_size=40))
    m.model.layers[0].attn.attn_fn = lambda q, k, v, t: O.sb_attn_oracle(q, k, v)
    ids, seen = torch.randint(0, 40, (1, 6)), []
    note = lambda mod, *a: seen.append(type(mod)) and None
    assert fused.plain(m.model, SBAModel)
    for register in (register_module_forward_hook, register_module_full_backward_hook):
        hook = register(note)
        assert not fused.plain(m.model, SBAModel)
        m(ids, labels=ids)[0].backward()
        hook.remove()
        assert seen.count(SBAModel) == 1
        seen.clear()
    monkeypatch.setattr(m.model, "_compiled_call_impl", lambda *a, **k: seen.append(SBAModel) or m.model.forward(*a, **k))
    m(ids)
    assert seen == [SBAModel]


def test_clip_and_step_leaves_other_tensor_classes_and_observed_steps_alone(native):
    from torch.utils._python_dispatch import TorchDispatchMode

    class Other(torch.Tensor):
        pass

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    p, opt = _adamw_after_one_step()
    with Mode():
        assert fused.clip_and_step([p], opt, 1.0) is None
    plain = p.grad
    p.grad = plain.as_subclass(Other)
    assert fused.clip_and_step([p], opt, 1.0) is None
    p.grad = plain
    opt.state[p]["exp_avg"] = opt.state[p]["exp_avg"].as_subclass(Other)
    assert fused.clip_and_step([p], opt, 1.0) is None and not native.calls


# The projection kernels' entries by themselves: what the kernels take for granted is refused before anything is launched.
@pytest.mark.parametrize("change,error,says", [
    ({"x": torch.zeros(4, 64)}, TypeError, "float16"),
    ({"w": torch.zeros(32, 64, dtype=torch.float16)}, TypeError, "float16"),
    ({"w": torch.zeros(32, 96, dtype=torch.bfloat16)}, ValueError, "share k"),
    ({"x": torch.zeros(64, 4, dtype=torch.bfloat16).t()}, ValueError, "dense"),
    ({"residual": None}, ValueError, "residual"),
    ({"residual": torch.zeros(4, 16)}, ValueError, "residual"),
    ({"residual": torch.zeros(4, 32, dtype=torch.bfloat16)}, TypeError, "residual"),
    ({"out": torch.zeros(4, 16)}, ValueError, "out"),
    ({"out": torch.zeros(32, 4).t()}, ValueError, "out"),
    ({"out": torch.zeros(4, 32, dtype=torch.bfloat16)}, TypeError, "out"),
    ({"epilogue": 3, "out": torch.zeros(4, 64, dtype=torch.bfloat16), "w": torch.zeros(64, 32, dtype=torch.bfloat16), "rows_w": True}, ValueError, "pre"),
    ({"epilogue": 4}, RuntimeError, "epilogue"),
    ({"tile": 6}, RuntimeError, "tile"),
    ({}, ValueError, "GPU only"),
])
def test_what_the_projection_kernels_take_for_granted_is_checked(change, error, says):
    from flame_amd import _lib
    a = dict(tile=2, x=torch.zeros(4, 64, dtype=torch.bfloat16), w=torch.zeros(32, 64, dtype=torch.bfloat16), rows_w=False, epilogue=1,
             residual=torch.zeros(4, 32), pre=None, out=torch.zeros(4, 32))
    a.update(change)
    with pytest.raises(error, match=says):
        _lib.native().project_with(**a)
    if not set(change) - {"x", "w", "residual"} and a["residual"] is not None:
        with pytest.raises(error, match=says):
            _lib.native().project_add(a["x"], a["w"], a["residual"])
