"""The order of the top-k over fp16 logits at the edges of its integer keys and of its passes."""
import numpy as np
import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import ops

pytestmark = pytest.mark.gpu


# less than a chunk, a chunk and one, more candidates than one merge round (512), more chunks than the shared statistics
@pytest.mark.parametrize("V", [9, 4097, 300001, 1100000])
@pytest.mark.parametrize("k", [1, 8])
def test_order(dev, V, k):
    rng = np.random.default_rng(V)
    x = rng.integers(-40, 40, (3, V)).astype(np.float16) / 8        # ties everywhere
    x[0, rng.integers(0, V, 1)] = np.nan                            # never picked
    x[1, :] = -np.inf
    x[1, [V - 1, 2, V // 2]] = [0.0, -0.0, -1.0]                    # equal zeros, then -inf by index
    x[2, rng.integers(0, V, 4)] = np.float16(65504)
    idx, score = ops.logsoftmax_topk(torch.from_numpy(x).to(dev), k, mode=0)
    key = np.where(np.isnan(x), -np.inf, x.astype(np.float32))
    for r in range(3):
        order = np.lexsort((np.arange(V), np.isnan(x[r]), -key[r]))[:k]
        assert np.array_equal(idx[r].cpu().numpy(), order), r
