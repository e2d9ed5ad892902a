"""Host side of the layer calls: the bit widths passed with the expert tables."""
import torch

from helios_glm53flash_amd import moe


def _experts(bits):
    """A 128 x 128 ExpertSet on the CPU (the tables only hold addresses)."""
    tr = [[torch.zeros((8, 8, 16 * b), dtype=torch.int16) for b in bits] for _ in range(3)]
    v = [[torch.ones(128, dtype=torch.float16) for _ in bits] for _ in range(3)]
    return moe.ExpertSet(128, 128, tr, v, v, [list(bits) for _ in range(3)])


def test_call_bits_follow_the_tables():
    ex = _experts((2, 2, 2))
    assert ex.tables().bits_mask == 0 and ex.call_bits() == (2, 2, 2)
    ex.bits = [[3, 3, 3]] * 3
    ex._tables = None  # a rebuild of the tables takes the new widths with it
    assert ex.tables().bits_mask == 0 and ex.call_bits() == (3, 3, 3)
    mixed = _experts((2, 3, 2))
    assert mixed.tables().bits_mask == 0b1100 and mixed.call_bits() == (0, 0, 0)


def test_call_bits_with_tables_set_by_a_loader():
    ex = _experts((4, 4))
    ex._tables = object()  # the checkpoint loader builds the tables itself
    assert ex.call_bits() == (4, 4, 4)
