"""Calls that do not fit are refused before any kernel is launched: the ops' checks run here on CPU tensors
with the launches recorded instead of made."""
import pytest
import torch

from micro_engram_fork_amd import MicroEngram, ops
from micro_engram_fork_amd._lib import ME_GATE_SCALAR, ME_GATE_SCALAR_SQRT


@pytest.fixture
def launches(monkeypatch):
    """The names of the library calls made, none of which reaches the library."""
    seen = []
    monkeypatch.setattr(ops, "require_gpu", lambda *tensors: torch.device("cpu"))
    monkeypatch.setattr(ops, "stream_of", lambda device: 0)
    monkeypatch.setattr(ops, "call", lambda name, *args: seen.append(name))
    cached = [f for f in vars(ops).values() if hasattr(f, "cache_clear")]  # workspace sizes: none was computed here
    for f in cached:
        f.cache_clear()
    yield seen
    for f in cached:
        f.cache_clear()


def _engram(d, dtype=torch.float32, gate="scalar_sqrt", **kw):
    kw = dict(dict(table_size=97, engram_dim=8, num_heads=2, orders=(2, 3), vocab_size=500), **kw)
    return MicroEngram(d, gate=gate, **kw).to(dtype).train()


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("gate", ["scalar", "scalar_sqrt"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [64, 96, 120, 192])
def test_hidden_of_another_width_is_refused(launches, width, dtype, gate, grad):
    eng = _engram(128, dtype, gate)
    hidden = torch.zeros(48, width, dtype=dtype)
    mem = torch.zeros(48, 32, dtype=dtype, requires_grad=grad)
    with torch.set_grad_enabled(grad), pytest.raises(ValueError, match="does not match"):
        eng.gate_residual(hidden, mem)
    assert launches == []
    with torch.set_grad_enabled(grad), pytest.raises(ValueError, match="does not match"):
        eng.gate_residual(torch.zeros(47, 128, dtype=dtype), mem)  # another number of tokens
    assert launches == []
    with torch.set_grad_enabled(grad):
        eng.gate_residual(torch.zeros(48, 128, dtype=dtype), mem)
    assert launches == ["me_kv_proj", "me_gate_rows"]


def test_row_kernels_refuse_rows_that_do_not_fit(launches):
    n, d = 48, 64
    x, stats = torch.zeros(n, d), torch.zeros(n, 4)
    k, q = torch.zeros(n, d), torch.zeros(d)
    both = [lambda k, v, q, s: ops.gate_rows(x, k, v, q, s, ME_GATE_SCALAR_SQRT, None, True),
            lambda k, v, q, s: ops.gate_rows_backward(x, x, k, v, q, s, ME_GATE_SCALAR_SQRT, None, stats)]
    wide = torch.zeros(n, 4 * d)
    for call in both:
        for kk, vv in ((k, wide[:, d:]), (wide[:, :d], wide[:, 2 * d:]), (k, k[:16]), (k[:16], k), (k[:, :32], k)):
            with pytest.raises(ValueError, match="do not match"):
                call(kk, vv, q, q)
        for qq, ss in ((q[:32], q), (q, q[:32]), (torch.zeros(2 * d), q)):
            with pytest.raises(ValueError, match="do not match"):
                call(k, k, qq, ss)
    with pytest.raises(ValueError, match="does not match"):
        ops.gate_rows_backward(x[:16], x, k, k, None, None, ME_GATE_SCALAR, None, stats)
    assert launches == []
    for call in both:  # halves of one buffer, and rows of any shape that holds n rows of d
        call(wide[:, :d], wide[:, d:2 * d], q, q)
        call(k.view(4, 12, d), k, q, q)
    assert launches == ["me_gate_rows"] * 2 + ["me_gate_rows_backward_workspace_size"] + ["me_gate_rows_backward"] * 2


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("tables", [3, 5])
def test_a_table_count_other_than_the_hashes_is_refused(launches, tables, grad):
    # the fused reads take the tables' addresses from a host array as long as the hash's table list
    eng = _engram(64)
    rows = [eng.tables[k % 4] for k in range(tables)]
    eng.tables = torch.nn.ModuleList(rows)
    hidden, ids = torch.zeros(1, 6, 64), torch.zeros(1, 6, dtype=torch.long)
    with torch.set_grad_enabled(grad), pytest.raises(ValueError, match="tables for the row ids"):
        eng(hidden, ids)
    with torch.no_grad(), pytest.raises(ValueError, match="tables for the row ids"):
        eng.hash_prev(torch.zeros(6, 3, dtype=torch.long))
    with pytest.raises(ValueError, match="table orders"):
        ops.hash_ids(ids, None, eng.canon, eng.mults, eng._table_orders, eng.table_rows[:3], 0)
    assert launches == []


def test_a_table_that_ends_before_its_row_ids_is_read_by_the_gather(launches):
    # the fused reads take every row id below the hash's row count to be in the table; the gather looks
    eng = _engram(64).eval()
    eng.tables[2] = torch.nn.Embedding(50, 8)
    ids = torch.zeros(1, 6, dtype=torch.long)
    with torch.no_grad():
        eng.hashed_memory(ids)
        eng.hash_prev(torch.zeros(6, 3, dtype=torch.long))
    assert launches == ["me_hash_ngrams", "me_gather", "me_hash_prev", "me_gather"]
    launches.clear()
    eng.tables[2] = torch.nn.Embedding(150, 8)
    with torch.no_grad():
        eng.hashed_memory(ids)
        eng.hash_prev(torch.zeros(6, 3, dtype=torch.long))
    assert launches == ["me_hash_gather", "me_hash_prev_gather"]


def test_unaligned_operands_with_gradients_are_copied_once(monkeypatch):
    # hidden, the output's gradient and the scales on odd addresses: both row kernels get copies they can read
    # 16 bytes at a time (else they take one column per lane)
    calls = {}
    monkeypatch.setattr(ops, "require_gpu", lambda *tensors: torch.device("cpu"))
    monkeypatch.setattr(ops, "stream_of", lambda device: 0)
    monkeypatch.setattr(ops, "call", lambda name, *args: calls.setdefault(name, args))
    odd = lambda *shape: torch.zeros(1 + torch.Size(shape).numel())[1:].view(shape)
    n, d = 24, 64
    w, scale, keep = torch.zeros(d, 32), odd(d), None
    x, g, stats = odd(n, d), odd(n, d), torch.zeros(n, 4)
    assert all(t.data_ptr() % 16 for t in (x, g, scale))
    kv = ops.gate_residual_rows(x, odd(n, 32), w, w, scale, scale, ME_GATE_SCALAR_SQRT, keep, True, True, True)[3]
    ops.gate_rows_backward(g, x, kv[:, :d], kv[:, d:], scale, scale, ME_GATE_SCALAR_SQRT, keep, stats)
    ops.gate_rows_backward_workspace_bytes.cache_clear()
    forward, backward = calls["me_gate_rows"], calls["me_gate_rows_backward"]
    assert all(p % 16 == 0 for p in (*(forward[i] for i in (0, 4, 5, 8, 9)), *(backward[i] for i in (0, 4, 5, 8, 9, 13))))
    # rows that are no multiple of 16 bytes gain nothing from a copy
    x, k = odd(n, 36), torch.zeros(n, 36)
    calls.clear()
    ops.gate_rows_backward(x, x, k, k, None, None, ME_GATE_SCALAR, keep, stats)
    ops.gate_rows_backward_workspace_bytes.cache_clear()
    assert calls["me_gate_rows_backward"][0] == x.data_ptr()


@pytest.mark.parametrize("d", [64, 36])
def test_an_output_whose_consumer_gives_no_gradient_leaves_gradients(launches, d):
    # what the engram's parameters get then is a gradient (of zeros), as from a gradient of zeros
    class NoGradient(torch.autograd.Function):
        @staticmethod
        def forward(ctx, x):
            return x.sum()

        @staticmethod
        def backward(ctx, grad):
            return None

    eng = _engram(d)
    out = eng.gate_residual(torch.zeros(12, d), torch.zeros(12, 32))
    NoGradient.apply(out).backward()
    assert "me_gate_rows_backward" in launches
    for p in (eng.key.weight, eng.value.weight, eng.q_scale, eng.k_scale):
        assert p.grad is not None and p.grad.shape == p.shape


@pytest.mark.parametrize("d,n,dtype,kept", [
    (8064, 1030, torch.bfloat16, True), (8072, 512, torch.bfloat16, True), (8072, 513, torch.bfloat16, False),
    (8072, 513, torch.float32, True)])
def test_rows_past_one_pass_of_the_row_kernels_keep_k_and_v_for_few_tokens(launches, d, n, dtype, kept):
    eng = _engram(d, dtype)
    eng.gate_residual(torch.empty(n, d, dtype=dtype), torch.empty(n, 32, dtype=dtype)).sum().backward()
    assert (launches[:2] == ["me_kv_proj", "me_gate_rows"]) == kept
    assert ("me_gate_residual" in launches) == (not kept) and ("me_gate_backward" in launches) == (not kept)


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("name", ["hash_ids", "inject", "lookup"])
def test_forward_goes_through_replaced_methods(launches, name, grad):
    # set on the instance or overridden by a subclass, with and without gradients
    seen = []

    def replacement(self, *args, **kwargs):
        seen.append(name)
        return getattr(MicroEngram, name)(self, *args, **kwargs)

    kw = dict(table_size=97, engram_dim=8, num_heads=2, orders=(2, 3), vocab_size=500, gate="scalar_sqrt")
    subclass = type("Sub", (MicroEngram,), {name: replacement})(64, **kw)
    instance = _engram(64)
    setattr(instance, name, lambda *a, **k: replacement(instance, *a, **k))
    hidden, ids = torch.zeros(1, 6, 64), torch.zeros(1, 6, dtype=torch.long)
    for eng in (subclass, instance):
        with torch.set_grad_enabled(grad):
            eng(hidden, ids)
    assert seen == [name, name]
