"""Batches with per-row settings where some rows have no top-k (finished by one
workgroup, or split over several), with and without the kept-set output."""
import numpy as np
import pytest

from llima_amd import workloads as wl
from .test_gpu_parity import _sample_both, _say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("V", [37, 4096, 4097, 20001, 128256])
@pytest.mark.parametrize("keep", [False, True])
def test_mixed_rows(gpu, oracle, dtype, V, keep):
    """Every kind of row without top-k (top-p, min-p, both, neither, penalties
    of either sign, +inf values, all -inf, a single finite value, an infinite
    temperature) beside top-k and greedy rows; a chunk with one value and rows
    that are not 16-byte aligned."""
    _say("sample mixed", dtype, V, keep)
    rng = np.random.default_rng(V + keep)
    B, H = 14, 96
    x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(3.0)).astype(np.float32)
    x[5] = -np.inf
    x[6, rng.integers(0, V, 3)] = np.inf
    x[7] = -np.inf
    x[7, V - 1] = 1.5
    x[8, ::3] = np.nan
    hist = rng.integers(0, V, size=(B, H)).astype(np.int32)
    rows = dict(temperature=[1.0, 0.8, 1.3, 1.0, 0.7, 1.0, 1.0, 1.0, 0.9, 1.0, 0.0, 1.0, np.inf, 1.0],
                top_k=[0, 0, 0, 0, 0, 0, 0, 0, 0, 20, 0, 5, 0, 0],
                top_p=[0.9, 1.0, 0.95, 0.5, 1.0, 0.9, 0.9, 0.9, 0.97, 0.95, 1.0, 1.0, 1.0, 0.999],
                min_p=[0.0, 0.1, 0.02, 0.3, 0.0, 0.0, 0.0, 0.0, 0.0, 0.05, 0.0, 0.0, 0.0, 0.0],
                repetition_penalty=[1.0, 1.0, 1.2, 1.0, 1.0, 0.8, 1.0, 1.0, 1.1, 1.15, 1.0, 1.0, 1.0, 0.9])
    for _ in range(2):
        _sample_both(gpu, oracle, x if dtype == "f32" else wl.f32_to_bf16_bits(x),
                     rng.random(B).astype(np.float32), None, history=hist, cfg_rows=rows,
                     want_keep=keep)
