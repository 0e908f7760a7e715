"""Arguments that are checked before anything runs on a device (no GPU needed)."""
import pytest
import torch

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
