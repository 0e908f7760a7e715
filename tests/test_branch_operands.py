"""The table of branch pointers that a grouped linear kernel keeps between calls (host side, no GPU needed)."""
import pytest
import torch

import brainstorm_amd.jit as jit


def _pointers(table):
    return table.tolist()


def test_a_failed_conversion_leaves_no_table_of_freed_copies(monkeypatch):
    """fp32 branches are read through bf16 copies.  If converting other branches fails (out of memory), the
    kept table still has to be the one of copies that are alive, or be made again."""
    alive = {}

    def convert(t):
        if fail:
            raise MemoryError("no room for the copy")
        copy = t.to(torch.bfloat16)
        alive[copy.data_ptr()] = copy
        return copy

    monkeypatch.setattr(jit, "_to_bf16", convert)
    first = [torch.randn(4, 8) for _ in range(3)]
    other = [torch.randn(4, 8) for _ in range(3)]
    operands = jit._BranchOperands("weights")
    fail = False
    operands.get(first, 0, 1, 3)
    fail = True
    with pytest.raises(MemoryError):
        operands.get(other, 0, 1, 3)
    fail = False
    table = operands.get(first, 0, 1, 3)
    assert [c.data_ptr() for c in operands.copies] == _pointers(table)
    for p, t in zip(_pointers(table), first):
        assert torch.equal(alive[p], t.to(torch.bfloat16))
    table = operands.get(other, 0, 1, 3)
    assert [c.data_ptr() for c in operands.copies] == _pointers(table)
    for p, t in zip(_pointers(table), other):
        assert torch.equal(alive[p], t.to(torch.bfloat16))
