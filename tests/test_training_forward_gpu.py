"""MicroEngram.forward with gradients hashes and reads the rows in one launch; inject on hash_ids's list does
so in two. Both give the same output and gradients, bit for bit, and calls the fused read does not
take (replaced hash_ids or lookup, tables of another size than the hash's) go where they went."""
import pytest
import torch

from micro_engram_fork_amd import MicroEngram

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _make(dtype=torch.bfloat16, shard=False, **kw):
    torch.manual_seed(0)
    eng = MicroEngram(model_dim=64, table_size=301, engram_dim=16, num_heads=2, orders=(2, 3), vocab_size=500,
                      gate="scalar_sqrt", **kw)
    torch.nn.init.normal_(eng.value.weight, std=0.1)
    eng = eng.to(device=DEV, dtype=dtype).train()
    if shard:
        eng.shard_rows(0, 1)
        for p in eng.row_shards:
            p._sparse_rows = True
    return eng


def _both(eng, ids, pos, dtype, call):
    g = torch.Generator(device=DEV).manual_seed(1)
    hidden = torch.randn(*ids.shape, 64, generator=g, device=DEV).to(dtype)
    gout = torch.randn(*ids.shape, 64, generator=g, device=DEV).to(dtype)
    for p in eng.all_parameters():
        p.grad = None
        p.sparse_grad = None
    h = hidden.clone().requires_grad_(True)
    out = call(h)
    out.backward(gout)
    res = [out.detach(), h.grad] + [p.grad for p in eng.parameters()]
    return res + [t for p in (eng.row_shards or []) for t in (p.sparse_grad or ())]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shard", [False, True])
@pytest.mark.parametrize("batch,seq,positions", [(1, 1, None), (3, 37, None), (2, 65, "row"), (2, 65, "each")])
def test_forward_equals_inject_of_hash_ids(dtype, shard, batch, seq, positions):
    eng = _make(dtype, shard)
    ids = torch.randint(0, 500, (batch, 2 * seq), device=DEV)[:, ::2]  # strided ids
    pos = {None: None, "row": torch.arange(seq, device=DEV),
           "each": torch.randint(0, 4, (batch, seq), device=DEV)}[positions]
    a = _both(eng, ids, pos, dtype, lambda h: eng(h, ids, pos))
    b = _both(eng, ids, pos, dtype, lambda h: eng.inject(h, eng.hash_ids(ids, pos)))
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert (x is None) == (y is None) and (x is None or torch.equal(x, y))


def test_replaced_methods_and_table_sizes_keep_their_route():
    ids = torch.randint(0, 500, (1, 9), device=DEV)
    hidden = torch.randn(1, 9, 64, device=DEV).bfloat16()
    eng = _make()
    seen = []
    eng.hash_ids = lambda i, p=None: seen.append("hash") or MicroEngram.hash_ids(eng, i, p)
    eng(hidden, ids)
    eng.lookup = lambda idx: seen.append("lookup") or MicroEngram.lookup(eng, idx)
    eng(hidden, ids)
    assert seen == ["hash", "hash", "lookup"]
    # a smaller table than the hash's: its missing rows read as zeros
    eng = _make()
    full = eng.tables[1].weight.detach().clone()
    eng.tables[1] = torch.nn.Embedding(200, 16, _weight=full[:200].clone()).to(DEV)
    idx = eng.hash_ids(ids)
    assert torch.equal(eng(hidden, ids), eng.inject(hidden, idx))
    assert torch.equal(eng(hidden[:, :0], ids[:, :0]), hidden[:, :0])


def test_missing_rows_of_a_smaller_table_are_zeros_without_gradients():
    # the prefill and the decode step, whose fused reads do not look for a table's end
    eng = _make().eval()
    rows = eng.tables[1].weight.detach()[:200].clone()
    eng.tables[1] = torch.nn.Embedding(200, 16, _weight=rows).to(DEV)
    ids = torch.randint(0, 500, (1, 64), device=DEV)
    hidden = torch.randn(1, 64, 64, device=DEV).bfloat16()
    idx = eng.hash_ids(ids)[1].reshape(-1)
    want = torch.where((idx < 200)[:, None], rows[idx.clamp(max=199)], torch.zeros((), dtype=rows.dtype, device=DEV))
    assert bool((idx >= 200).any())
    with torch.no_grad():
        assert torch.equal(eng.hashed_memory(ids)[:, 16:32], want)
        prev = torch.stack([ids[0].roll(k) for k in range(3)], dim=1)
        read = eng.hash_prev(prev)
        assert torch.equal(eng.inject(hidden, read), eng.inject(hidden, [i.clone() for i in read]))
