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


# every tile's kernel where it can go wrong: one token, edges of 64, 128 and 256, fewer stages of 64 k than groups that share them out,
# a last stage of 32 k, more tiles than workgroups
@pytest.mark.parametrize("tile", range(6))
@pytest.mark.parametrize("m,n,k,dtype", [
    (1, 16, 32, torch.bfloat16),
    (65, 80, 64, torch.float16),
    (127, 144, 160, torch.bfloat16),
    (257, 272, 224, torch.bfloat16),
    (300, 528, 1088, torch.bfloat16),
    (4100, 4112, 128, torch.bfloat16),
])
def test_every_tile_of_the_projections(m, n, k, dtype, tile):
    from flame_amd import _lib
    native = _lib.native()
    assert native.projection_tiles == 6
    g = torch.Generator("cuda").manual_seed(m + n + k)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    x = rand(m, k + 8).to(dtype)[:, :k]
    w = (rand(n, k) / k ** 0.5).to(dtype)
    w_cols = w.t().contiguous()
    residual, pre = rand(m, n), rand(m, 2 * n).to(dtype)
    # the sums are fp32: what is left is the rounding to 16 bits, half a unit in the last place, and of a few intermediate 16-bit values
    tol = 4e-3 if dtype == torch.bfloat16 else 6e-4
    y = x.float() @ w.float().t()
    leaf = pre.float().requires_grad_()
    gate, up = leaf.chunk(2, dim=1)
    (F.silu(gate) * up).backward(y)
    y_gate, y_up = y.to(dtype).float().chunk(2, dim=1)
    store, add, glu, glu_back = range(4)
    taken = 0
    for rows_w, epilogue, out, want in (
            (False, store, torch.empty(m, n, device="cuda", dtype=dtype), y),
            (True, store, torch.empty(m, n, device="cuda", dtype=dtype), y),
            (False, add, torch.empty(m, n, device="cuda"), residual + y),
            (False, glu, torch.empty(m, n // 2, device="cuda", dtype=dtype), F.silu(y_gate) * y_up),
            (True, glu_back, torch.empty(m, 2 * n, device="cuda", dtype=dtype), leaf.grad)):
        out.fill_(float("nan"))
        both = {add: (residual, None), glu_back: (None, pre)}.get(epilogue, (None, None))
        if not native.project_with(tile, x, w_cols if rows_w else w, rows_w, epilogue, *both, out):
            continue
        taken += 1
        assert rel_l2(out.float(), want) <= tol, (rows_w, epilogue)
    assert taken or (tile < 2 and k % 64)


# tiles of 224 and 256 rows (4096 x 1024 and 512 x 512 fill more of the chip with the taller ones), their edges, contractions off 32 and shared out
@pytest.mark.parametrize("m,n,k,dtype", [
    (8, 8, 1, torch.bfloat16),
    (232, 264, 33, torch.float16),
    (448, 520, 700, torch.bfloat16),
    (512, 512, 1100, torch.bfloat16),
    (4096, 1016, 290, torch.bfloat16),
    (1032, 2824, 1000, torch.bfloat16),
])
def test_weight_gradients(m, n, k, dtype):
    from flame_amd import _lib
    g = torch.Generator("cuda").manual_seed(m + n + k)
    a = torch.randn(k, m, generator=g, device="cuda").to(dtype)
    b = torch.randn(k, n, generator=g, device="cuda").to(dtype)
    got = _lib.native().weight_grad(a, b)
    assert got.dtype == torch.float32
    # products of 16-bit values are exact in fp32, their sums carry at most k roundings of 2^-24
    assert rel_l2(got.double(), a.double().t() @ b.double()) <= 1e-5


# workgroups that share a tile's contraction: one token, edges of 128 and 256, shares of one stage, a last share that is shorter
@pytest.mark.parametrize("tile", [0, 1])
@pytest.mark.parametrize("m,n,k,splits,dtype", [
    (1, 16, 128, 2, torch.bfloat16),
    (257, 272, 448, 7, torch.float16),
    (300, 528, 640, 3, torch.bfloat16),
    (1030, 1008, 4096, 5, torch.bfloat16),
])
def test_shared_contractions(m, n, k, splits, dtype, tile):
    from flame_amd import _lib
    g = torch.Generator("cuda").manual_seed(m + n + k)
    x = torch.randn(m, k + 8, generator=g, device="cuda").to(dtype)[:, :k]
    w = (torch.randn(k, n, generator=g, device="cuda") / k ** 0.5).to(dtype)
    out = torch.full((m, n), float("nan"), device="cuda", dtype=dtype)
    assert _lib.native().project_with(tile, x, w, True, 0, None, None, out, splits)
    # fp32 sums: what is left is the rounding of the result, half a unit in the last place
    assert rel_l2(out.float(), x.float() @ w.float()) <= (4e-3 if dtype == torch.bfloat16 else 6e-4)


def test_the_input_gradient_of_a_head_is_shared_out():
    from flame_amd import _lib
    g = torch.Generator("cuda").manual_seed(5)
    x = torch.randn(700, 16000, generator=g, device="cuda").bfloat16()
    w = (torch.randn(16000, 512, generator=g, device="cuda") / 126).bfloat16()
    assert rel_l2(_lib.native().project(x, w, True).float(), x.float() @ w.float()) <= 4e-3


# the product is added to the residual as its fp32 sum, for contractions that the kernels take as they are and for others: rounded to 16
# bits first it would be off by a thousandth (bf16) or a ten-thousandth
@pytest.mark.parametrize("m,n,k,dtype", [(65, 80, 64, torch.bfloat16), (300, 512, 1000, torch.bfloat16), (257, 64, 8, torch.float16), (1, 128, 328, torch.float16)])
def test_the_residual_meets_an_unrounded_product(m, n, k, dtype):
    from flame_amd import _lib
    g = torch.Generator("cuda").manual_seed(m + n + k)
    x = torch.randn(m, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(n, k, generator=g, device="cuda") / k ** 0.5).to(dtype)
    residual = torch.randn(m, n, generator=g, device="cuda")
    got = _lib.native().project_add(x, w, residual)
    # products of 16-bit values are exact in fp32, their sums carry at most k + 1 roundings of 2^-24
    assert rel_l2(got.double(), residual.double() + x.double() @ w.double().t()) <= 1e-5
