"""The projection + row kernels that a forward with gradients runs (K and V written out and kept)
against the fused kernels: the same K and V bits, the same sums in the same order, so every output
but the scale gradients (sums over tokens in another order) is equal bit for bit.

Scale gradients: both are fp32 sums of the same n terms t_i = a_i x_i K_i, each within
n * 2^-24 * sum |t_i| of the exact one (a few ulps more for the products), so their difference is
held to twice that; sum |t_i| is bounded by sqrt(n) times the columns' 2-norm, and the terms here
are random in sign: |difference| <= 1e-5 * 2-norm over columns covers n = 2049 with a wide margin
against observed 2e-7."""
import pytest
import torch

from micro_engram_fork_amd import MicroEngram, ops
from micro_engram_fork_amd._lib import ME_GATE_SCALAR, ME_GATE_SCALAR_SQRT

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(n, d, m, mode, dtype, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    r = lambda *s, std=1.0: (torch.randn(*s, generator=g, device=DEV) * std).to(dtype)
    scales = (r(d, std=0.1), r(d, std=0.1)) if mode == ME_GATE_SCALAR_SQRT else (None, None)
    return (r(n, d), r(n, m, std=0.05), r(d, m, std=0.05), r(d, m, std=0.05), *scales,
            torch.rand(n, generator=g, device=DEV) > 0.1, r(n, d, std=1e-3))


# model dims: one group of 8 columns, one column past a 224-column tile, an odd number of 112-column
# halves, every step count of the row kernels (up to 24, 48 and 72 groups of 112), past them (8072);
# more than 64 tokens, where the projection sums over k in the fused kernel's order
@pytest.mark.parametrize("n,d,m,mode", [
    (65, 8, 192, ME_GATE_SCALAR_SQRT), (66, 112, 192, ME_GATE_SCALAR), (257, 232, 192, ME_GATE_SCALAR_SQRT),
    (513, 1032, 512, ME_GATE_SCALAR_SQRT), (2049, 336, 256, ME_GATE_SCALAR_SQRT),
    (255, 2688, 256, ME_GATE_SCALAR_SQRT), (256, 2696, 256, ME_GATE_SCALAR), (300, 5376, 1536, ME_GATE_SCALAR_SQRT),
    (69, 5384, 192, ME_GATE_SCALAR_SQRT), (70, 8064, 192, ME_GATE_SCALAR_SQRT), (70, 8072, 192, ME_GATE_SCALAR_SQRT)])
def test_rows_equal_fused_bf16(n, d, m, mode):
    x, mem, wk, wv, dq, dk, keep, g = _case(n, d, m, mode, torch.bfloat16)
    fused = ops.gate_residual(x, mem, wk, wv, dq, dk, mode, keep, True, True)
    kv = ops.kv_proj(mem, wk, wv)
    rows = ops.gate_rows(x, kv[:, :d], kv[:, d:], dq, dk, mode, keep, True, True)
    if d <= 8064:
        for a, b in zip(fused, rows):
            assert torch.equal(a, b)
    stats = fused[2]
    want = ops.gate_backward(g, x, mem, wk, wv, dq, dk, mode, keep, stats)
    got = ops.gate_rows_backward(g, x, kv[:, :d], kv[:, d:], dq, dk, mode, keep, stats)
    if d <= 8064:
        for a, b in zip(want[:3], got[:3]):
            assert torch.equal(a, b)
    for a, b in zip(want[3:], got[3:]):
        assert (a - b).norm() <= 1e-5 * a.norm() + 1e-12


def _check_proj(n, d, m, dtype):
    _, mem, wk, wv, *_ = _case(n, d, m, ME_GATE_SCALAR, dtype, seed=n)
    kv = ops.kv_proj(mem, wk, wv)
    ref = torch.cat([mem.double() @ wk.double().t(), mem.double() @ wv.double().t()], dim=1)
    mag = torch.cat([mem.double().abs() @ wk.double().abs().t(), mem.double().abs() @ wv.double().abs().t()], dim=1)
    # an fp32 sum of m products (each rounded once more in fp32), then one rounding to bf16
    rounding = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    assert bool(((kv.double() - ref).abs() <= rounding * ref.abs() + (m + 1) * 2.0 ** -24 * mag).all())


# token counts around the switches between the projection's tiles (by the tiles they make: 32 x 32,
# 64 x 64, 64 x 96, 256 x 96, 256 x 128, then 64 x 128 or 256 x 224) and memory widths of whole and partial slabs
@pytest.mark.parametrize("n", [64, 65, 192, 193, 256, 257, 512, 513, 768, 1025])
@pytest.mark.parametrize("d,m", [(5376, 192), (264, 1536), (2048, 200), (5320, 136)])
def test_kv_proj_tiles(n, d, m):
    _check_proj(n, d, m, torch.bfloat16)


# many tokens of memory rows that are no whole slabs (64 x 128 tiles past every one-round tile), with a row end
# inside a slab and columns that end inside a tile
def test_kv_proj_many_tokens_of_partial_slabs():
    _check_proj(1153, 5320, 136, torch.bfloat16)


# the few-token kernel (bf16 up to 32 tokens, fp32 up to 64): every count of 16-token blocks and its edges, columns
# that end inside a 16-column block, memory rows of one part of a slab, of fewer slabs than waves, of partial slabs,
# of each slab count per wave (2, 4, 6, 8, 12) and past its widest (3200)
@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("d,m", [(8, 16), (24, 192), (1032, 200), (40, 896), (264, 1536), (16, 2048), (8, 3072), (8, 3200)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_kv_proj_few_tokens(n, d, m, dtype):
    _check_proj(n, d, m, dtype)


# fp32 past the few-token kernel: fp32 MFMAs on tiles of 32 x 64 and 32 x 128 (the last two), split products on
# 64 x 64 (1000 tokens) and 64 x 128, by the tiles they make; memory rows of whole and partial slabs, columns and
# tokens that end inside a tile
@pytest.mark.parametrize("n,d,m", [(65, 264, 1536), (300, 1024, 200), (700, 1032, 96), (1000, 1024, 36), (1025, 1024, 64),
                                   (2049, 520, 4), (1025, 2056, 200), (257, 3576, 36), (800, 2560, 100)])
def test_kv_proj_fp32_tiles(n, d, m):
    _check_proj(n, d, m, torch.float32)


@pytest.mark.parametrize("n,d", [(70, 64), (700, 1032), (1000, 1024), (1025, 2056)])
def test_kv_proj_fp32_values_of_any_size(n, d):
    # rows and columns scaled by 2^-40 .. 2^40: the split is exact at every exponent, so the bound of
    # _check_proj holds relative to each element's own magnitudes
    m = 64
    g = torch.Generator(device=DEV).manual_seed(3)
    scale = lambda k: 2.0 ** torch.randint(-40, 41, (k, 1), generator=g, device=DEV).float()
    mem = torch.randn(n, m, generator=g, device=DEV) * scale(n)
    wk, wv = (torch.randn(d, m, generator=g, device=DEV) * scale(d) for _ in range(2))
    kv = ops.kv_proj(mem, wk, wv).double()
    w = torch.cat([wk, wv]).double().t().contiguous()
    ref, mag = mem.double() @ w, mem.double().abs() @ w.abs()
    assert bool(((kv - ref).abs() <= 2.0 ** -24 * ref.abs() + (m + 1) * 2.0 ** -24 * mag).all())


# values under about 2^-110 have no three bf16 parts: fp32 MFMAs, split products on both their tiles; memory
# rows of whole and partial k-steps, a tiny row, a tiny column and single tiny values among others
@pytest.mark.parametrize("n,d,m", [(70, 64, 64), (1000, 1024, 64), (1000, 1024, 36), (1025, 2056, 64), (1025, 2056, 200)])
@pytest.mark.parametrize("exponent", [-104, -112, -124, -140, -146])
def test_kv_proj_fp32_tiny_values(n, d, m, exponent):
    g = torch.Generator(device=DEV).manual_seed(5)
    r = lambda *s: torch.randn(*s, generator=g, device=DEV)
    mem, wk, wv = r(n, m), r(d, m), r(d, m)
    tiny = 2.0 ** exponent
    mem[n - 1] = (r(m).double() * tiny).float()
    mem[3, 5] = tiny * 1.2345678
    wk[d - 1] = (r(m).double() * tiny).float()
    wv[7] *= 2.0 ** 20
    wv[9, m - 1] = tiny
    kv = ops.kv_proj(mem, wk, wv).double()
    w = torch.cat([wk, wv]).double().t().contiguous()
    ref, mag = mem.double() @ w, mem.double().abs() @ w.abs()
    # each of the m products and sums is rounded once in fp32, at 2^-149 where it is subnormal
    bound = 2.0 ** -24 * ref.abs() + (m + 1) * 2.0 ** -24 * mag + (m + 1) * 2.0 ** -149
    assert bool(((kv - ref).abs() <= bound).all())


@pytest.mark.parametrize("n,d", [(70, 64), (700, 1032), (1000, 1024), (1025, 2056)])
def test_kv_proj_fp32_infinities_and_nan(n, d):
    # where a value is infinite or NaN, so is what the products give, and nothing else changes
    m = 64
    g = torch.Generator(device=DEV).manual_seed(4)
    mem = torch.randn(n, m, generator=g, device=DEV)
    wk, wv = (torch.randn(d, m, generator=g, device=DEV) for _ in range(2))
    clean = ops.kv_proj(mem, wk, wv)
    mem[5, 7], mem[n - 1, m - 1], mem[40, 3] = float("inf"), float("nan"), float("-inf")
    wk[11, 2], wv[d - 1, 0], wv[3] = float("-inf"), float("nan"), 0.0
    mem[41] = torch.finfo(torch.float32).max
    kv = ops.kv_proj(mem, wk, wv)
    w = torch.cat([wk, wv]).double().t().contiguous()
    ref = mem.double() @ w
    ref = torch.where(ref.abs() > torch.finfo(torch.float32).max, ref.sign() * float("inf"), ref)
    near = torch.zeros_like(ref, dtype=torch.bool)
    near[41] = True  # sums of the largest values may overflow on the way
    assert bool(((torch.isnan(ref) == torch.isnan(kv)) | near).all())
    assert bool(((torch.isinf(ref) == torch.isinf(kv)) | near).all())
    same = torch.isfinite(ref) & ~near
    err = (kv.double() - ref).abs() <= 1e-4 + 1e-4 * ref.abs()
    assert bool((err | ~same).all())
    rows = [i for i in range(n) if i not in (5, 40, 41, n - 1)]
    cols = [j for j in range(2 * d) if j not in (11, 2 * d - 1, d + 3)]
    assert (kv[rows][:, cols] - clean[rows][:, cols]).abs().max() <= 1e-4


def _make(dtype, d, tables=6, dim=32):
    torch.manual_seed(d)
    eng = MicroEngram(model_dim=d, table_size=257, engram_dim=dim, num_heads=tables // 2, orders=(2, 3),
                      vocab_size=1000, gate="scalar_sqrt")
    torch.nn.init.normal_(eng.value.weight, std=0.1)
    return eng.to(device=DEV, dtype=dtype).train()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hidden_dtype", [torch.bfloat16, torch.float32])
def test_kept_and_recomputed_gradients_agree(dtype, hidden_dtype):
    # above keep_kv_bytes the backward recomputes K and V; both give the same gradients
    n, d = 300, 264
    eng = _make(dtype, d)
    ids = torch.randint(0, 1000, (1, n), device=DEV)
    g = torch.randn(1, n, d, device=DEV).to(hidden_dtype) * 1e-2
    hidden = torch.randn(1, n, d, device=DEV).to(hidden_dtype)
    grads = []
    for limit in (1 << 30, 0):
        eng.keep_kv_bytes = limit
        eng.zero_grad(set_to_none=True)
        h = hidden.clone().requires_grad_(True)
        out = eng(h, ids)
        assert (out.grad_fn is not None)
        out.backward(g)
        grads.append([out.detach(), h.grad] + [p.grad for p in eng.parameters()])
    # bf16: K, V, dK and dV round the same values, differing by their sums' order; near s = 0 the
    # square root's slope carries that into a token's gradients, hence 5e-2 of the 2-norm there
    tol = 5e-2 if torch.bfloat16 in (dtype, hidden_dtype) else 5e-3
    for a, b in zip(*grads):
        assert a.dtype == b.dtype and (a.double() - b.double()).norm() <= tol * b.double().norm() + 1e-12


# hidden states and projections of two dtypes whose values fit bf16: the sums are those of one dtype, and results
# differ by their own rounding only. Model dims of each step count of the row kernels and their edges; 1100 tokens
# are more than one per workgroup of the backward
@pytest.mark.parametrize("n,d,mode", [
    (37, 8, ME_GATE_SCALAR_SQRT), (37, 112, ME_GATE_SCALAR), (1100, 232, ME_GATE_SCALAR_SQRT), (37, 2688, ME_GATE_SCALAR_SQRT),
    (37, 2696, ME_GATE_SCALAR), (37, 5376, ME_GATE_SCALAR_SQRT), (37, 5384, ME_GATE_SCALAR_SQRT), (37, 8064, ME_GATE_SCALAR_SQRT)])
@pytest.mark.parametrize("hidden_dtype,dtype", [(torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32)])
def test_rows_of_two_dtypes(n, d, mode, hidden_dtype, dtype):
    x, mem, wk, wv, dq, dk, keep, g = _case(n, d, 64, mode, torch.bfloat16)
    k, v = mem @ wk.t(), mem @ wv.t()
    want = ops.gate_rows(x, k, v, dq, dk, mode, keep, True, True)
    grads = ops.gate_rows_backward(g, x, k, v, dq, dk, mode, keep, want[2])
    xm, gm, km, vm = x.to(hidden_dtype), g.to(hidden_dtype), k.to(dtype), v.to(dtype)
    got = ops.gate_rows(xm, km, vm, dq, dk, mode, keep, True, True)
    back = ops.gate_rows_backward(gm, xm, km, vm, dq, dk, mode, keep, want[2])
    assert torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])  # gates and sums
    assert all(torch.equal(a.bfloat16(), b) for a, b in zip(back[1:3], grads[1:3]))  # of K and V: one rounding
    assert all((a - b).norm() <= 1e-5 * b.norm() + 1e-12 for a, b in zip(back[3:], grads[3:]))
    if hidden_dtype == torch.bfloat16:
        assert torch.equal(got[0], want[0]) and torch.equal(back[0], grads[0])
    else:  # bf16 rounds the term and the sum: at most 2^-8 of each
        for a, b, base in ((got[0], want[0], xm), (back[0], grads[0], gm)):
            assert bool(((a - b.float()).abs() <= 2.0 ** -8 * ((a - base).abs() + a.abs()) * 1.01 + 1e-30).all())
