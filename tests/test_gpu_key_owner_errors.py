"""Errors of dK and dV against 64 bits where the paired key-owner kernel stands in the stream's place at head_dim 64 (launches that hang on
their longest sweeps): no larger than the stream's, whose scores have the operand that the forward's carries were made from."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _inputs(H, T, logits, dtype):
    g = torch.Generator("cuda").manual_seed(31)
    q, k, v, do = (torch.randn(1, H, T, 64, device="cuda", generator=g) for _ in range(4))
    if logits == "far":                 # mean -6, standard deviation 2: long sticks
        shift = math.sqrt(6 / 8)
        q, k = 0.5 * q + shift, 0.5 * k - shift
    else:                               # mean 0, standard deviation 3
        q, k = math.sqrt(3) * q, math.sqrt(3) * k
    return [t.to(dtype) for t in (q, k, v, do)]


def _gradients_64(q, k, v, do):
    """dK, dV of one head's [T, 64] tensors."""
    q, k, v, do = (t.double() for t in (q, k, v, do))
    T, scale = q.shape[0], 1 / math.sqrt(q.shape[1])
    i = torch.arange(T, device=q.device)
    sees = i[None, :] < i[:, None]
    z = scale * (q @ k.t().contiguous())
    stays = torch.where(sees, torch.nn.functional.logsigmoid(-z), 0.0)
    a = torch.where(sees, torch.exp(torch.nn.functional.logsigmoid(z) + stays.flip(-1).cumsum(-1).flip(-1) - stays), 0.0)
    g = a * (do @ v.t().contiguous())
    dz = torch.where(sees, scale * (g - torch.sigmoid(z) * g.cumsum(-1)), 0.0)
    return dz.t().contiguous() @ q, a.t().contiguous() @ do


# (kernel, heads, tokens): the paired kernel by name, and where the library takes it by itself (384 row blocks)
@pytest.mark.parametrize("kernel,H,T", [("pairq", 4, 2048), ("", 16, 3072)])
@pytest.mark.parametrize("logits", ["far", "wide"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_no_further_off_than_the_stream(kernel, H, T, logits, dtype, monkeypatch):
    from flame_amd import sb_attn
    q, k, v, do = _inputs(H, T, logits, dtype)
    reference = [_gradients_64(*(t[0, h] for t in (q, k, v, do))) for h in range(4)]

    def errors(name):
        monkeypatch.delenv("SBA_DKV_KERNEL", raising=False)
        if name:
            monkeypatch.setenv("SBA_DKV_KERNEL", name)
        qkv = [t.clone().requires_grad_(True) for t in (q, k, v)]
        grads = torch.autograd.grad(sb_attn(*qkv)[0], qkv, do)[1:]
        return [math.sqrt(sum(float((got[0, h].double() - ref[i]).square().sum()) for h, ref in enumerate(reference)) /
                          sum(float(ref[i].square().sum()) for ref in reference)) for i, got in enumerate(grads)]

    mine, stream = errors(kernel), errors("other")
    print("dK %.3e (stream %.3e)  dV %.3e (stream %.3e)" % (mine[0], stream[0], mine[1], stream[1]), flush=True)
    # The same operands are rounded in both; what is left is the order of the 32-bit sums, 1e-6 of values whose 16-bit
    # roundings are 1e-3 (bf16) and 1e-4 (f16) off.
    for a, b in zip(mine, stream):
        assert a <= 1.01 * b
