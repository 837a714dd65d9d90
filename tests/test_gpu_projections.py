"""The projection kernels of the language model (csrc/sba_gemm.hip) against fp32 products."""
import pytest
import torch
import torch.nn.functional as F

from helpers import rel_l2

pytestmark = pytest.mark.gpu


# one row to several rounds of tiles per workgroup, sizes off the tiles' 128 and 256, k from one stage up and off 64
@pytest.mark.parametrize("m,n,k,dtype", [
    (1, 16, 32, torch.bfloat16),
    (129, 144, 96, torch.bfloat16),
    (255, 272, 160, torch.float16),
    (1000, 1040, 1024, torch.bfloat16),
    (8190, 1008, 192, torch.bfloat16),      # 128 x 256 tiles, one round
    (8190, 3056, 64, torch.bfloat16),       # 128 x 256 tiles, three rounds of one stage
    (8200, 1040, 448, torch.float16),
    (4090, 4080, 64, torch.bfloat16),       # 256 x 256 tiles, one stage
    (8200, 4112, 320, torch.bfloat16),
    (4100, 8080, 128, torch.float16),
])
def test_projections_and_what_follows_them(m, n, k, dtype):
    from flame_amd import _lib
    native = _lib.native()
    g = torch.Generator("cuda").manual_seed(m + n + k)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = rand(m, k + 8).to(dtype)[:, :k]
    w = (rand(n, k) / k ** 0.5).to(dtype)
    w_cols = w.t().contiguous()
    tol = 4e-3 if dtype == torch.bfloat16 else 6e-4

    def same(got, want, kind):
        assert got.dtype == kind and got.shape == want.shape
        assert rel_l2(got.float(), want) <= tol
        assert float((got.float() - want).abs().max()) <= 4 * tol * float(want.abs().max())

    y = x.float() @ w.float().t()
    same(native.project(x, w, False), y, dtype)
    same(native.project(x, w_cols, True), y, dtype)
    residual = rand(m, n)
    same(native.project_add(x, w, residual), residual + y, torch.float32)

    a, pre = native.project_swiglu(x, w)
    same(pre, y, dtype)
    gate, up = pre.float().chunk(2, dim=1)
    same(a, F.silu(gate) * up, dtype)

    pre = rand(m, 2 * n).to(dtype)
    leaf = pre.float().requires_grad_()
    gate, up = leaf.chunk(2, dim=1)
    (F.silu(gate) * up).backward(y)
    same(native.project_swiglu_grad(x, w_cols, pre), leaf.grad, dtype)
