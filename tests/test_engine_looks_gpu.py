"""Entries that become one ticket each where they are looked at, beside entries that do not: sizes around the 16 descriptors
that are one ticket always and the 32 that are while eight submissions are in flight, empty ones and ones of several tickets
among them, one at a time and several to a call, with tickets sized by backlog and of a fixed size."""
import pytest

import test_engine_carried_gpu as carried

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_ticket", [0, 4, 64])
@pytest.mark.parametrize("per_call", [1, 2, 5, 17])
@pytest.mark.parametrize("other", [0, 17, 32, 33, 100])
def test_small_entries_among_others(pkg, hip, oracle, monkeypatch, other, per_call, per_ticket):
    monkeypatch.setattr(carried, "COUNTS", [16, other, 1, 16, 16, 2, other, other, 5, 16, 16, 16, 16, 16, 16, other])
    carried.small_lists(pkg, hip, oracle, "mapped", per_call, descs_per_ticket=per_ticket)
