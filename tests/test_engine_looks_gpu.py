"""Entries that become one ticket each where they are looked at, beside entries that do not: sizes around the 16 descriptors
that are one ticket always and the 32 that are while eight submissions are in flight, empty ones and ones of several tickets
among them, one at a time and several to a call, with tickets sized by backlog and of a fixed size.  And long runs of entries
of several tickets, which are taken 64 at a time, broken at the ends of sixteen and elsewhere by one that is not like them."""
import pytest

import test_engine_carried_gpu as carried

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_ticket", [0, 4, 64])
@pytest.mark.parametrize("per_call", [1, 2, 5, 17])
@pytest.mark.parametrize("other", [0, 17, 32, 33, 100])
def test_small_entries_among_others(pkg, hip, oracle, monkeypatch, other, per_call, per_ticket):
    monkeypatch.setattr(carried, "COUNTS", [16, other, 1, 16, 16, 2, other, other, 5, 16, 16, 16, 16, 16, 16, other])
    carried.small_lists(pkg, hip, oracle, "mapped", per_call, descs_per_ticket=per_ticket)


@pytest.mark.parametrize("per_ticket", [0, 3])
@pytest.mark.parametrize("usual", [33, 70, 130])
@pytest.mark.parametrize("other", [0, 1, 64, 600])
def test_long_runs_of_entries_of_several_tickets(pkg, hip, oracle, monkeypatch, other, usual, per_ticket):
    counts = [usual] * 160
    for at in (5, 31, 32, 63, 90, 111, 159):
        counts[at] = other
    monkeypatch.setattr(carried, "COUNTS", counts)
    for per_call in (160, 48):
        carried.small_lists(pkg, hip, oracle, "mapped", per_call, descs_per_ticket=per_ticket)
