"""Which key-owner kernel a launch at head_dim 64 gets on both sides of the line between the resident stream and the paired kernel (which sum in
different orders, so that their bits tell them apart): few heads with long sweeps stay with the stream."""
import pytest
import torch

from helpers import cu_from_lengths

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel,H,lens", [
    ("other", 4, [12288]), ("other", 4, [16384]), ("other", 8, [6144]), ("other", 2, [16384, 8192]), ("other", 8, [4096, 2048]),
    ("other", 4, [4096] + [100] * 100), ("other", 8, [2500] + [128] * 40), ("pairq", 8, [2048] + [256] * 50), ("pairq", 16, [4096]), ("pairq", 4, [8192, 8192]), ("pairq", 16, [2048, 1024, 500, 400]),
    ("pair", 16, [1024] * 4), ("pair", 16, [600] * 20)], ids=lambda x: str(x)[:24])
def test_key_owner_kernel(kernel, H, lens, monkeypatch):
    from flame_amd import sb_attn_varlen
    g = torch.Generator("cuda").manual_seed(5)
    q, k, v, do = (torch.randn(H, sum(lens), 64, device="cuda", generator=g).bfloat16() for _ in range(4))
    q, k, v = ((0.5 * t).requires_grad_(True) for t in (q, k, v))
    cu = cu_from_lengths(lens).cuda()

    def run(name):
        monkeypatch.delenv("SBA_DKV_KERNEL", raising=False)
        if name:
            monkeypatch.setenv("SBA_DKV_KERNEL", name)
        return torch.autograd.grad(sb_attn_varlen(q, k, v, cu, max(lens))[0], (k, v), do)

    def same(a, b):
        return all(torch.equal(x, y) for x, y in zip(a, b))

    got, each = run(""), {name: run(name) for name in ("other", "pair", "pairq")}
    assert [name for name, grads in each.items() if same(got, grads)] == [kernel]
