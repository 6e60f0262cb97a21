"""me_dense_table_grads against zeros + a scatter of the unique rows' sums, bit for bit: widths of
16-byte chunks and not, one workgroup's rows and several (32 KB each, at most 1024 rows), tables
without a gradient, without any touched row, with every row touched, of one row, and more unique rows
than one step of the search covers (64, and 64 * 64)."""
import pytest
import torch

from micro_engram_fork_amd import MicroEngram, ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("dim", [1, 3, 8, 20, 64, 128, 4096, 9000])
def test_dense_table_grads(dtype, dim):
    g = torch.Generator(device=DEV).manual_seed(dim)
    big = 9001 if dim <= 128 else 50
    table_rows = [big, 1, 1023, 1025, 70, 130, 1]
    touched = [5000 if dim <= 128 else 17, 1, 0, 65, 70, 64, 0]
    local, bounds = [], [0]
    for r, t in zip(table_rows, touched):
        t = min(t, r)
        local.append(torch.randperm(r, generator=g, device=DEV)[:t].sort().values)
        bounds.append(bounds[-1] + t)
    local = torch.cat(local + [torch.full((11,), 1 << 40, device=DEV)])  # past the count: unset
    sums = torch.randn(bounds[-1] + 11, dim, generator=g, device=DEV)
    info = torch.tensor([bounds[-1]] + bounds, device=DEV)
    need = [True, True, True, True, False, True, True]
    got = ops.dense_table_grads(local, sums, info, [(r, dim) for r in table_rows], dtype, need)
    for k, (r, a, b) in enumerate(zip(table_rows, bounds, bounds[1:])):
        if not need[k]:
            assert got[k] is None
            continue
        want = torch.zeros(r, dim, device=DEV)
        want[local[a:b]] = sums[a:b]
        assert torch.equal(got[k], want.to(dtype))


@pytest.mark.parametrize("n", [0, 1, 33])
def test_frozen_tables_and_empty_batch(n):
    # tables that take no gradient get none; an empty batch leaves zeros
    torch.manual_seed(n)
    eng = MicroEngram(model_dim=32, table_size=97, engram_dim=8, num_heads=2, vocab_size=500).to(DEV)
    torch.nn.init.normal_(eng.value.weight, std=0.1)
    eng.tables[1].weight.requires_grad_(False)
    idx = eng.hash_ids(torch.randint(0, 500, (1, n), device=DEV))
    rows = eng.lookup(idx)
    grads = [torch.randn_like(r) for r in rows]
    torch.autograd.backward(rows, grads)
    for k, table in enumerate(eng.tables):
        if k == 1:
            assert table.weight.grad is None
            continue
        want = torch.zeros(97, 8, device=DEV).index_add_(0, idx[k].reshape(-1), grads[k].reshape(-1, 8))
        assert torch.allclose(table.weight.grad, want, rtol=1e-6, atol=1e-6)
