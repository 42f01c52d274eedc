"""Picking the candidates of a tree over every split of the ranking, and the wait for the shape of the paths."""
import numpy as np
import pytest
import torch

from mlx_eagle_spec_decoding_tree_amd import eagle
from oracle import tree_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C", [1, 7, 31, 32, 33, 127, 128, 129, 256, 257, 384, 385, 512, 513, 1000, 1024])
def test_picks_are_the_first_in_stable_descending_order(dev, C):
    rng = np.random.default_rng(C)
    for levels in (3, 60, 5000):               # few distinct scores: ties decide
        s = rng.integers(0, levels, C).astype(np.float16) - np.float16(levels // 2)
        if C > 7:
            s[rng.integers(0, C, 3)] = np.array([np.inf, -np.inf, np.nan], np.float16)
        total = min(63, C)
        key = np.where(np.isnan(s), np.float16(-np.inf), s).astype(np.float32)
        want = np.sort(np.argsort(-key, kind="stable")[:total])
        out = eagle.process_draft_tree_device(torch.from_numpy(s).to(dev), torch.arange(C, dtype=torch.int32, device=dev) + 5,
                                              torch.zeros(C, dtype=torch.int32, device=dev),
                                              torch.tensor([1], dtype=torch.int32, device=dev), 1, total)
        assert np.array_equal(out[2].cpu().numpy()[1:] - 5, want), levels


def test_paths_behind_other_work_and_on_other_streams(dev):
    """The call returns finished rows whether the kernel runs at once or long after the host has stopped watching."""
    rng = np.random.default_rng(9)
    side = torch.cuda.Stream()
    for case in range(12):
        total = int(rng.integers(2, 64))
        midx = np.array([int(rng.integers(0, i + 1)) for i in range(total)], np.int32)
        depth = np.zeros(total + 1, np.int32)
        for i, p in enumerate(midx):
            depth[i + 1] = depth[p] + 1
        want = tree_oracle.post_process_draft_tree(depth, total, midx)
        pos, idx = torch.from_numpy(depth).to(dev), torch.from_numpy(midx).to(dev)
        torch.cuda.synchronize()
        with torch.cuda.stream(side if case % 2 else torch.cuda.current_stream()):
            if case % 3 == 0:
                torch.cuda._sleep(2_000_000)   # about a millisecond
            got = eagle.post_process_draft_tree(pos, total, idx)
        # (read on this thread's own stream, which nothing made wait for the other)
        assert np.array_equal(got.cpu().numpy(), want), case
