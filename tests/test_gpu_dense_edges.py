"""The dense path (no top-k, no mask) on rows whose values or temperature are
infinite, beside ordinary rows: ids, probabilities and kept sets are the
oracle's."""
import numpy as np
import pytest

from llima_amd import workloads as wl
from .test_gpu_parity import _sample_both, _say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("V", [37, 4096, 20001])
@pytest.mark.parametrize("keep", [False, True])
def test_dense_infinite_temperature(gpu, oracle, dtype, V, keep):
    """A row may have temperature +inf: a finite logit then gives 0 and an
    infinite one no value.  Rows of infinite logits alone have no token (no bin
    of theirs holds a value: the boundary bin must still be one); others draw
    uniformly from their finite logits, also where a chunk has none."""
    _say("sample dense infinite temperature", dtype, V, keep)
    rng = np.random.default_rng(V)
    B = 7
    x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(3.0)).astype(np.float32)
    x[0] = -np.inf
    x[0, V // 2] = np.inf                                  # +inf and -inf alone
    x[1] = np.inf
    x[2, ::3] = np.inf                                     # finite values beside both
    x[2, 1::3] = -np.inf
    x[3, :min(V - 1, 8192)] = np.inf                       # chunks without a finite value
    x[4, :V - 1] = -np.inf                                 # one finite value
    x[5, ::2] = np.nan
    rows = dict(temperature=[np.inf] * (B - 1) + [1.0], top_p=[0.9, 0.9, 0.9, 0.5, 0.9, 1.0, 0.95],
                min_p=[0.0, 0.0, 0.0, 0.0, 0.0, 0.1, 0.0])
    for _ in range(2):
        _sample_both(gpu, oracle, x if dtype == "f32" else wl.f32_to_bf16_bits(x),
                     rng.random(B).astype(np.float32), None, cfg_rows=rows, want_keep=keep)


@pytest.mark.parametrize("keep", [False, True])
@pytest.mark.parametrize("V", [40, 4096, 12300])
def test_dense_infinite_maximum(gpu, oracle, V, keep):
    """Rows whose maximum is +inf: 1, 64 and 65 infinities in one chunk (a
    window stages at most 64 values), spread over the chunks, all of a chunk's
    other values few enough to fit beside them, and every value infinite."""
    _say("sample dense infinite maximum", V, keep)
    rng = np.random.default_rng(V)
    B = 7
    x = (rng.standard_normal((B, V), dtype=np.float32) * np.float32(3.0)).astype(np.float32)
    for b, n in ((0, 1), (1, 64), (2, 65)):
        x[b, rng.permutation(min(V, 4096))[:n]] = np.inf
    x[3, ::17] = np.inf
    x[4] = -np.inf
    x[4, :20] = 1.0
    x[4, 5] = np.inf
    x[5] = np.inf
    for p in (0.3, 0.9):
        _sample_both(gpu, oracle, x, rng.random(B).astype(np.float32),
                     dict(temperature=0.8, top_p=p), want_keep=keep)
