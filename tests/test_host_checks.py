"""Arguments that are checked before anything runs on a device (no GPU needed)."""
import ctypes
import random

import pytest
import torch

from brainstorm_amd import _lib
from brainstorm_amd._C import router as c_router
from brainstorm_amd.router.fabric._impl import FusedCombineFabric


def test_weighted_compact_combine_refuses_scores_with_fewer_columns_than_paths():
    """The weight of an entry is the score of its cell on its path: a score matrix without a column for every
    path has none for some of them."""
    cells, k, paths = 6, 2, 4
    ids = torch.tensor([[0, 3]] * cells, dtype=torch.int32)
    vector = torch.ones(cells * k, dtype=torch.int32)
    route = c_router.CompactRoute(ids, None, vector[:paths], vector[:paths], vector.view(cells, k), vector, paths, None)
    fabric = FusedCombineFabric(1, transform=True)
    with pytest.raises(RuntimeError, match="3 columns for 4 paths"):
        fabric._combine_compact(torch.ones(cells * k, 8), route, None, torch.ones(cells, paths - 1), None)


def _walk_of(E, P, K, N):
    workgroups = ctypes.c_int()
    walk = _lib.lib().brt_hip_grouped_gemm_walk(E, P, K, N, ctypes.byref(workgroups))
    return walk, workgroups.value


@pytest.mark.parametrize("E,P,K,N,walk", [
    (8, 30732, 128, 4096, 2), (6, 19356, 192, 2040, 2), (12, 24576, 320, 2000, 2), (5, 86400, 320, 768, 3),
    (2, 80040, 192, 520, 3), (3, 80200, 128, 1272, 5),
    (16, 32768, 1024, 1792, 1), (16, 32768, 1024, 1024, 2), (16, 32768, 1088, 1024, 1), (16, 32768, 4096, 2048, 2), (16, 32768, 4160, 2048, 1),
])
def test_which_lists_of_tiles_are_walked(E, P, K, N, walk):
    """Two column tiles, or three or five where two do not divide their number, up to K = 4096 (1024 with few of them) in whole K-steps."""
    assert _walk_of(E, P, K, N)[0] == walk
    assert _walk_of(E, P, K + 8, N)[0] == 1


def test_lists_of_tiles_that_are_walked_have_their_workgroups():
    """For any loads: a workgroup for the column tiles that it walks, one for every other tile, four for one that is cut, and one for the tags of
    rows that no path owns."""
    rng = random.Random(7)
    walked = 0
    for _ in range(6000):
        E, K, N = int(2 ** rng.uniform(0, 8)), 64 * rng.randint(2, 64), 8 * int(2 ** rng.uniform(0, 10))
        mean, skew = 2 ** rng.uniform(6, 14), rng.choice([0, 0.3, 1, 2.5])
        loads = [int(mean * 2 ** rng.gauss(0, skew)) * (rng.random() < 0.9) for _ in range(E)]
        if rng.random() < 0.3:
            loads = [v // 256 * 256 + rng.choice([0, 0, 1, 128]) for v in loads]
        P = sum(loads) + rng.choice([0, 0, 1, 1000])
        tiles_n = -(-N // 256)
        tiles = sum(-(-v // 256) for v in loads) * tiles_n
        if P == 0 or tiles > 1 << 22:
            continue
        walk, workgroups = _walk_of(E, P, K, N)
        for tags in (0, 1):
            cut = _lib.lib().brt_hip_grouped_gemm_tiles_cut((ctypes.c_int32 * E)(*loads), E, P, N, tags)
            whole = tiles - cut
            walkers = whole // 256 // walk * 256 if walk > 1 else 0
            used = walkers + whole - walkers * walk + 4 * cut
            assert used + (tags and P > sum(loads)) <= workgroups, (loads, P, K, N, tags)
            walked += walkers > 0
    assert walked > 1000


def test_walks_of_bad_sizes():
    for sizes in ((0, 1, 64, 8), (1, 0, 64, 8), (1, 1, 0, 8), (1, 1, 64, 0)):
        assert _walk_of(*sizes)[0] == -1  # BRT_E_INVALID
    assert _lib.lib().brt_hip_grouped_gemm_walk(1, 1, 64, 8, None) == -1
