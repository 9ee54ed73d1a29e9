"""The LBVH at the sizes where its launches change: the sort by ranks with its
64-box tiles and a wave per node, the radix sort and the level by level merge; with tied codes,
signed zeros and NaN coordinates. Byte-identical to the oracle's host build."""
import numpy as np
import pytest

from test_gpu_lbvh import _boxes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 63, 65, 128, 4095, 4096, 8191, 8192, 8193, 30001])
@pytest.mark.parametrize("kind", ["random", "tied", "odd"])
def test_lbvh_sizes(pkg, oracle, dev, n, kind):
    rng = np.random.default_rng(n)
    b = _boxes(rng, n)
    if kind == "tied":
        g = rng.integers(0, 3, (n, 3)).astype(np.float32)
        b = np.concatenate([g, g + 1], axis=1)
    elif kind == "odd":
        b = _boxes(rng, n, 1.0)
        b[rng.random((n, 6)) < 0.3] = np.float32(0.0)
        b[rng.random((n, 6)) < 0.3] = np.float32(-0.0)
        b[rng.random((n, 6)) < 0.01] = np.float32(np.nan)
    nodes, order = pkg.build_tlas_fast(b)
    onodes, oorder = oracle.lbvh_tlas(b)
    assert np.array_equal(order, oorder)
    assert np.array_equal(nodes, onodes)
