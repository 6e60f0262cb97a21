"""Adam on parameters of one column (the scale deltas: a thread per row) against the oracle, with the
bounds of the other kernel shapes (tests/test_rows_gpu.py), and the clip's norm read from the sum of
squares as torch's fp32 square root of it."""
import numpy as np
import pytest
import torch
from test_rows_gpu import _adam_case, _assert_bf16_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 255, 256, 257, 400])
@pytest.mark.parametrize("rowwise", [True, False])
@pytest.mark.parametrize("lazy", [True, False])
def test_one_column_adam_matches_oracle(n, rowwise, lazy):
    (p, m, v), (pr, mr, vr) = _adam_case(torch.bfloat16, rowwise, D=1, R=600, n=n, lazy=lazy, zero_rows=lazy)
    _assert_bf16_close(p, pr, frac=1e-2)
    _assert_bf16_close(m, mr, frac=1e-2)
    if rowwise:
        assert torch.allclose(v, vr, rtol=1e-6, atol=0)
    else:
        _assert_bf16_close(v, vr, frac=1e-2)


def test_host_square_root_is_torch_s():
    g = torch.Generator(device="cuda").manual_seed(0)
    s = torch.cat([torch.rand(4096, generator=g, device="cuda") * 10.0 ** k for k in range(-30, 30, 3)])
    s = torch.cat([s, torch.tensor([0.0, float("inf"), float("nan")], device="cuda")])
    want = s.sqrt().cpu().numpy()
    assert np.array_equal(np.sqrt(s.cpu().numpy()), want, equal_nan=True)
