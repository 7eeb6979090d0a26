"""Norms and softmax of wide, unaligned and few rows (csrc/rows_wide.hip) against the oracle.

Widths at the edges of the vectors per thread (4 x 64, 256 and 1,024 threads) and of the dispatch:
one vector, a last vector moved back by 1-3 columns, the widest row and one past it (which stays on
the element-wise kernels); row counts on both sides of the wave / workgroup line. Bounds as in
test_gpu_norms.py and test_gpu_softmax.py: the arithmetic per element is the same, and a row's sum
over W waves has no more rounding steps than the one-wave sum."""
import numpy as np
import pytest
import torch

import cdna4
import oracle
from gpu_util import DEV

pytestmark = pytest.mark.gpu

SHAPES = [(5, 4), (70, 5), (9, 67), (1300, 255), (1300, 257), (6, 513), (512, 768), (513, 769), (1100, 1023),
          (1024, 1025), (1025, 1030), (1030, 2047), (3, 2049), (2, 4093), (3, 4097), (2, 8192), (2, 8195),
          (3, 16383), (2, 16385), (1, 32767), (2, 32770), (1, 65533), (1, 65536), (1, 65537)]


def _x(M, H, offset):
    x = oracle.normal(M * 13 + H, M * H, 0.0, 2.0).reshape(M, H)
    buf = torch.full((M * H + offset,), float("nan"), device=DEV)
    buf[offset:] = torch.from_numpy(x).to(DEV).reshape(-1)
    return x, buf[offset:].reshape(M, H)


@pytest.mark.parametrize("M,H", SHAPES)
def test_norms_and_softmax(M, H):
    offset = H % 4   # rows of 4-byte alignment also where H % 4 == 0 would hide it
    x, X = _x(M, H, offset)
    guard = torch.full((M * H + 8,), 7.0, device=DEV)
    out = guard[4:4 + M * H].reshape(M, H)
    g, b = oracle.uniform(1, H, 0.5, 1.5), oracle.uniform(2, H)
    got = cdna4.layernorm_f32(X, torch.from_numpy(g).to(DEV), torch.from_numpy(b).to(DEV), 1e-5, out).cpu().numpy()
    np.testing.assert_allclose(got, oracle.layernorm(x, g, b, 1e-5), rtol=1e-4, atol=2e-5)
    _, wb = oracle.round16(oracle.normal(H, H, 1.0, 0.1), oracle.F16)
    W = torch.from_numpy(wb.view(np.int16)).view(torch.float16).to(DEV)
    got = cdna4.rmsnorm_f32(X, W, 1e-6, out).cpu().numpy()
    np.testing.assert_allclose(got, oracle.rmsnorm(x, wb, 1e-6), rtol=1e-5, atol=1e-5)
    ref = oracle.softmax_rows(x).astype(np.float64)
    bound = ref * (1e-6 + 1.2e-7 * (x.max(axis=1, keepdims=True).astype(np.float64) - x)) + 1e-37
    got = cdna4.softmax_rows_f32(X, out).cpu().numpy()
    assert np.all(np.abs(got.astype(np.float64) - ref) <= bound)
    assert torch.all(guard[:4] == 7.0) and torch.all(guard[4 + M * H:] == 7.0)   # nothing past the rows
    got = cdna4.softmax_rows_f32(X, X).cpu().numpy()                             # in place
    assert np.all(np.abs(got.astype(np.float64) - ref) <= bound)


@pytest.mark.parametrize("H", [1001, 6001])
def test_softmax_masked_rows(H):
    # -inf entries, a row with one finite value, the type's lowest value, and a row with a NaN
    x = oracle.normal(H, 4 * H, 0.0, 2.0).reshape(4, H)
    x[0, 1::2] = -np.inf
    x[1] = -np.inf
    x[1, H - 1] = 3.0
    x[2, :-2] = np.finfo(np.float32).min
    x[3, H - 2] = np.nan
    got = cdna4.softmax_rows_f32(torch.from_numpy(x).to(DEV)).cpu().numpy()
    want = np.exp(x[:3].astype(np.float64) - x[:3].max(axis=1, keepdims=True))
    want /= want.sum(axis=1, keepdims=True)
    np.testing.assert_allclose(got[:3], want, rtol=1e-5, atol=1e-37)
    assert np.isnan(got[3]).all()


@pytest.mark.parametrize("M,H", [(1100, 260), (1100, 1024), (1030, 2048)])
def test_rows_at_any_element_equal_aligned_rows(M, H):
    # One wave per row in both cases, the same columns per lane and the same order of the sums: the
    # start of the rows may not change a bit (M above the line of few rows).
    x = torch.from_numpy(oracle.normal(M + H, M * H, 0.0, 2.0)).to(DEV)
    g, b = torch.from_numpy(oracle.uniform(1, H, 0.5, 1.5)).to(DEV), torch.from_numpy(oracle.uniform(2, H)).to(DEV)
    buf = torch.empty(M * H + 1, device=DEV)
    buf[1:] = x
    X, U = x.reshape(M, H), buf[1:].reshape(M, H)
    assert torch.equal(cdna4.softmax_rows_f32(U), cdna4.softmax_rows_f32(X))
    assert torch.equal(cdna4.layernorm_f32(U, g, b, 1e-5), cdna4.layernorm_f32(X, g, b, 1e-5))
