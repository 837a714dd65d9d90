"""When a call of the language model runs on the native nodes of csrc/sba_torch_model.cpp, and the calls themselves.

The nodes compute what the modules' own forward() does under autocast (fp32 weights and residual stream, 16-bit products, fp32
normalisation) with the modules' parameters, in one autograd node per block.  They are taken when nothing outside could tell:
plain modules without hooks, fp32 parameters on the GPU of the shapes that belong together, autocast to a 16-bit type, no tracing, and
nobody who observes or transforms the operators.  Everything else runs module by module.
"""
from __future__ import annotations

import torch
import torch.nn as nn
from torch.nn.modules import module as _module
from torch.optim import optimizer as _optimizer

from . import _lib
from .stickbreaking_attention import profiling, sb_attn, sb_attn_varlen

_HALF = (torch.bfloat16, torch.float16)


def _observed() -> bool:
    """Someone looks at the operators of this thread one by one (a dispatch mode: tracing, counting, selective checkpointing) or
    transforms them (torch.func); a kernel launched beside them would be missed."""
    return torch._C._len_torch_dispatch_stack() > 0 or torch._C._functorch.peek_interpreter_stack() is not None


def _tensor(t) -> bool:
    """A tensor itself, and not of a class that may mean something else by its operators."""
    return type(t) is torch.Tensor or type(t) is nn.Parameter


def _compute_dtype(x: torch.Tensor):
    """The 16-bit type that products run in, or None where the native nodes do not apply."""
    if not x.is_cuda or x.dtype != torch.float32 or x.dim() != 3 or x.numel() == 0 or not profiling.native():
        return None
    if not _tensor(x) or _observed():
        return None
    if not torch.is_autocast_enabled("cuda"):
        return None
    t = torch.get_autocast_dtype("cuda")
    return t if t in _HALF else None


def plain(m: nn.Module, kind: type) -> bool:
    """A module of exactly this class whose call is its class's forward() and nothing else."""
    return (type(m) is kind and not m._forward_hooks and not m._forward_pre_hooks and not m._backward_hooks
            and not m._backward_pre_hooks and "forward" not in m.__dict__ and m._compiled_call_impl is None
            and not (_module._global_forward_hooks or _module._global_forward_pre_hooks
                     or _module._global_backward_hooks or _module._global_backward_pre_hooks))


def _weight(m: nn.Module, like: torch.Tensor, *shape: int):
    """The fp32 weight of this shape of a plain module without bias, contiguous on x's device; None otherwise (the module says what
    is wrong with another shape)."""
    w = m.weight
    if type(w) is not nn.Parameter or w.dtype != torch.float32 or w.device != like.device or not w.is_contiguous() or w.shape != shape:
        return None
    return w if getattr(m, "bias", None) is None else None


def _eps(norm: nn.RMSNorm) -> float:
    return torch.finfo(torch.float32).eps if norm.eps is None else norm.eps


def _norm_fits(norm: nn.Module, width: int) -> bool:
    return (plain(norm, nn.RMSNorm) and tuple(norm.normalized_shape) == (width,) and width % 8 == 0
            and width <= _lib.native().max_norm_width)


def block(blk: nn.Module, x: torch.Tensor, kwargs: dict):
    """SBABlock.forward() as one node, or None."""
    t = _compute_dtype(x)
    if t is None:
        return None
    attn, mlp, width = blk.attn, blk.mlp, x.shape[2]
    if not (plain(attn, blk.attention_class) and plain(mlp, blk.mlp_class) and _norm_fits(blk.attn_norm, width)
            and _norm_fits(blk.mlp_norm, width)):
        return None
    if attn.attn_fn is not sb_attn or attn.attn_varlen_fn is not sb_attn_varlen or not attn.fuse_qkv or attn.head_dim not in (64, 128) \
            or attn.head_dim * attn.num_heads != width or kwargs.get("attention_mask") is not None:
        return None
    cu_seqlens = kwargs.get("cu_seqlens")
    if cu_seqlens is not None and x.shape[0] != 1:
        return None                              # the layer says what is wrong with that
    inner = mlp.gate_proj.weight.shape[0]
    if inner % 8:
        return None
    square, ws = (width, width), []
    for m, shape in ((blk.attn_norm, (width,)), (attn.q_proj, square), (attn.k_proj, square), (attn.v_proj, square), (attn.o_proj, square),
                     (blk.mlp_norm, (width,)), (mlp.gate_proj, (inner, width)), (mlp.up_proj, (inner, width)), (mlp.down_proj, (width, inner))):
        w = _weight(m, x, *shape) if (type(m) is nn.RMSNorm or plain(m, nn.Linear)) else None
        if w is None:
            return None
        ws.append(w)
    max_len = kwargs.get("max_seqlen")
    return _lib.native().block(x, ws, attn.num_heads, _eps(blk.attn_norm), _eps(blk.mlp_norm), t, cu_seqlens,
                               x.shape[1] if max_len is None else int(max_len))


def head(x: torch.Tensor, norm: nn.Module, lm_head: nn.Module):
    """lm_head(norm(x)) as one node, or None."""
    t = _compute_dtype(x)
    if t is None or not (_norm_fits(norm, x.shape[2]) and plain(lm_head, nn.Linear)):
        return None
    n, w = _weight(norm, x, x.shape[2]), _weight(lm_head, x, lm_head.weight.shape[0], x.shape[2])
    # a vocabulary that is no multiple of 8 is not for the kernel of the weight's gradient (weight_grads_fit() in sba_model.h)
    if n is None or w is None or w.shape[0] % 8:
        return None
    return _lib.native().head(x, n, w, _eps(norm), t)


def next_token_loss(logits: torch.Tensor, labels: torch.Tensor, ignore: int = -100):
    """Mean cross-entropy of 16-bit logits [B, T, V] against the labels shifted left by one (the last position of a row
    ignored), or None."""
    if not (logits.is_cuda and logits.dtype in _HALF and logits.dim() == 3 and logits.shape[-1] % 8 == 0 and labels.numel() > 0
            and labels.dtype == torch.int64 and labels.device == logits.device and labels.shape == logits.shape[:2]
            and _tensor(logits) and _tensor(labels) and profiling.native() and not _observed()):
        return None
    return _lib.native().next_token_loss(logits, labels, ignore)


def clip_and_step(params, opt, max_norm: float):
    """Gradient clipping to `max_norm` over `params` and opt.step(), in one pass over the weights; returns the gradients' norm,
    or None, with nothing done, where that is not what the two calls would do one after the other."""
    if type(opt) is not torch.optim.AdamW or opt._optimizer_step_pre_hooks or opt._optimizer_step_post_hooks \
            or _optimizer._global_optimizer_pre_hooks or _optimizer._global_optimizer_post_hooks:
        return None
    step_fn = opt.__dict__.get("step")           # a learning-rate scheduler's wrapper notes that a step was taken
    if step_fn is not None and not getattr(step_fn, "_wrapped_by_lr_sched", False):
        return None
    if getattr(opt, "grad_scale", None) is not None or getattr(opt, "found_inf", None) is not None or _observed():
        return None
    params = list(params)
    ids = {id(p) for p in params}
    ps, gs, ms, vs, steps, group_of, groups = [], [], [], [], [], [], []
    for i, group in enumerate(opt.param_groups):
        lr, betas = group["lr"], group["betas"]
        if group["amsgrad"] or group["maximize"] or group["capturable"] or group["differentiable"] or not group["fused"] \
                or not all(isinstance(h, float) for h in (lr, *betas, group["eps"])):
            return None
        groups.append([lr, float(group["weight_decay"]), betas[0], betas[1], group["eps"]])
        for p in group["params"]:
            if p.grad is None:
                continue
            state = opt.state.get(p)
            if id(p) not in ids or not state:    # a first step sets up its state
                return None
            if not (_tensor(p) and _tensor(p.grad) and _tensor(state["exp_avg"])):       # (sharded weights, say)
                return None
            ps.append(p)
            gs.append(p.grad)
            ms.append(state["exp_avg"])
            vs.append(state["exp_avg_sq"])
            steps.append(state["step"])
            group_of.append(i)
    if not ps or len(ps) != sum(p.grad is not None for p in params):
        return None
    norm = _lib.native().clip_and_step(ps, gs, ms, vs, steps, group_of, groups, float(max_norm))
    if norm is not None:
        opt._opt_called = True
    return norm
