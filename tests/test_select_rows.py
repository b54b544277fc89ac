"""Top-k row selection at the edges of its variants: row lengths around the registers' 2048 and 16384
scores and past them, k of 1, n - 1 and n, ties that cross waves and the threshold, infinities and NaN (GPU)."""
import numpy as np
import pytest
import torch

from oracle import compaction_oracle as co
from unifiedkv_amd import compaction

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 65, 511, 513, 2047, 2048, 2049, 4097, 16384, 16385, 40000])
@pytest.mark.parametrize("kind", ["uniform", "ties", "constant", "special"])
def test_rows_match_the_oracle(cuda, n, kind):
    rng = np.random.default_rng(n)
    s = rng.random((3, n), dtype=np.float32)
    if kind == "ties":
        s = np.floor(s * 5).astype(np.float32) - 2.0
    elif kind == "constant":
        s[:] = -3.5
    elif kind == "special":
        pick = np.array([np.nan, np.inf, -np.inf, 0.0, -0.0, 1e-45, -1e-45, 3.4e38], np.float32)
        s = np.where(rng.random((3, n)) < 0.3, rng.choice(pick, (3, n)), s - 0.5).astype(np.float32)
    for k in sorted({1, max(1, n // 5), max(1, n - 1), n}):
        got = compaction.select_blocks(torch.from_numpy(s).to(cuda), k).cpu().numpy()
        np.testing.assert_array_equal(got, co.select_topk(s, k), err_msg=f"{kind} n={n} k={k}")
