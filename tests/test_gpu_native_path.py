"""The native host path (csrc/host.cpp) and the kernels that came with it, against the forms they stand beside."""
import numpy as np
import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import eagle, ops
from oracle import tree_oracle as to
from util import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("root_dtype", [np.int32, np.int64])
@pytest.mark.parametrize("depth,total", [(0, 1), (0, 8), (1, 31), (1, 32), (4, 62), (5, 39), (7, 63), (15, 63)])
def test_tree_layout_from_lists(dev, depth, total, root_dtype):
    """Per-level lists read where they are, the packed retrieve rows: equal to the oracle, with frequent score ties."""
    k, rng = 8, np.random.default_rng(100 * depth + total)
    cu = np.sort(-rng.integers(0, 6, k).astype(np.float16))[::-1]
    scores, parents, chosen = [cu[None, None]], [np.zeros(1, np.int32)], np.arange(k)
    cur = cu
    for i in range(depth):
        parents.append((chosen + 1 + k * k * max(0, i - 1) + (k if i else 0)).astype(np.int32))
        c = (cur[:, None] - np.sort(rng.integers(0, 4, (k, k)), axis=1)).astype(np.float16)
        chosen = np.argsort(-c.reshape(-1).astype(np.float32), kind="stable")[:k]
        cur = c.reshape(-1)[chosen]
        scores.append(c[None])
    tokens = [rng.integers(0, 1000, s.shape).astype(np.int32) for s in scores]
    root = np.array([[7]], root_dtype)
    print(f"depth {depth} total {total}", flush=True)
    got = eagle.process_draft_tree([to_dev(s, dev) for s in scores], [to_dev(t, dev) for t in tokens],
                                   [to_dev(p, dev) for p in parents], to_dev(root, dev), k, total)
    pos, midx, toks, mask = (v.float().cpu().numpy() if v.dtype == torch.bfloat16 else v.cpu().numpy() for v in got)
    flat = [np.concatenate([v.reshape(-1) for v in part]) for part in (scores, tokens, parents)]
    dpos, dmidx, dtoks, bits = eagle.process_draft_tree_device(
        *(to_dev(v, dev) for v in flat), to_dev(root.astype(np.int32).reshape(-1), dev), k, total)
    assert np.array_equal(pos, dpos.cpu().numpy()) and np.array_equal(midx, dmidx.cpu().numpy())
    assert np.array_equal(toks, dtoks.cpu().numpy()[None]) and toks[0, 0] == 7
    assert np.array_equal(mask, eagle.bits_to_mask(bits).float().cpu().numpy())
    want = to.post_process_draft_tree(pos, total, midx)
    got = eagle.post_process_draft_tree(to_dev(pos, dev), total, to_dev(midx, dev))
    assert got.is_contiguous() and np.array_equal(got.cpu().numpy(), want)
