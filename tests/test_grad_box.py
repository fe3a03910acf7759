"""The sums of one ring chunk's dK / dV (GradBox in csrc/host.cpp), on CPU tensors: who writes, who adds, whose block leaves as
the total, and that nothing of one backward pass is left for the next.  The native nodes and the Python ones share it."""
import os

import pytest
import torch


@pytest.fixture()
def box():
    from picotron_amd import _lib
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built here")
    return _lib.host().GradBox()


def chunk(layout):
    k, v = (torch.zeros(2, 3, 8, 4, dtype=torch.bfloat16) for _ in range(2))
    if layout == "heads_inside":                   # [B,S,H,D] memory, as a projection leaves it
        k, v = (torch.zeros(2, 8, 3, 4, dtype=torch.bfloat16).transpose(1, 2) for _ in range(2))
    elif layout == "gaps":
        k, v = (torch.zeros(2, 3, 8, 12, dtype=torch.bfloat16)[..., :4] for _ in range(2))
    elif layout == "different":
        v = torch.zeros(2, 8, 3, 4, dtype=torch.bfloat16).transpose(1, 2)
    return k, v


@pytest.mark.parametrize("layout", ["plain", "heads_inside", "gaps", "different"])
def test_the_last_of_the_readers_gets_the_totals(box, layout):
    k, v = chunk(layout)
    box.readers = 3
    for backward_pass in range(2):
        first = box.claim(k, v, True, True)
        assert not first.add and first.final_dk is None
        assert first.dk.dtype == first.dv.dtype == torch.float32 and first.dk.shape == k.shape
        second = box.claim(k, v, True, True)
        assert second.add and second.final_dk is None and second.dk.data_ptr() == first.dk.data_ptr() and second.dv.data_ptr() == first.dv.data_ptr()
        last = box.claim(k, v, True, True)
        assert last.add and last.dk.data_ptr() == first.dk.data_ptr()
        for total, like in ((last.final_dk, k), (last.final_dv, v)):
            assert total.dtype == torch.bfloat16 and total.shape == like.shape
            assert total.stride() == (like.stride() if layout in ("plain", "heads_inside") else torch.empty(like.shape).stride())
        left = box.take()
        assert left.dk is None and left.dv is None and left.final_dk.data_ptr() == last.final_dk.data_ptr()
        again = box.take()                          # nothing is delivered twice
        assert again.dk is again.dv is again.final_dk is again.final_dv is None and box.arrived == 0 and box.dk is None


def test_one_reader_writes_the_totals_without_sums(box):
    k, v = chunk("plain")
    box.readers = 1
    only = box.claim(k, v, True, True)
    assert only.dk is None and only.dv is None and not only.add and only.final_dk is not None


@pytest.mark.parametrize("whole,rounds,readers", [(True, True, 3), (True, False, 2), (False, True, 2)])
def test_sums_are_handed_back_where_no_block_completes_them(box, whole, rounds, readers):
    """A part of the readers in this pass, a dtype the kernel cannot round to, or one ring step at a time."""
    k, v = chunk("plain")
    box.readers = readers
    first, second = (box.claim(k, v, whole, rounds) for _ in range(2))
    assert not first.add and second.add and second.final_dk is None
    first.dk.fill_(1)
    left = box.take()
    assert left.final_dk is None and bool((left.dk == 1).all()) and left.dv.data_ptr() == first.dv.data_ptr()
    assert box.claim(k, v, whole, rounds).add is False
