"""CPU-only: a stack of WaveNet blocks in two halves never returns while work on the stream beside the caller's is not waited for."""
import pytest

from __graft_entry__ import load_package

FORK, EARLIER, LATER, JOIN = range(4)


@pytest.mark.parametrize("blocks", [1, 2, 5])
def test_order_without_errors(blocks):
    assert load_package().capi.probe_halves_order(blocks) == (True, [FORK, EARLIER, LATER] * blocks + [JOIN])


@pytest.mark.parametrize("fails", range(10))
def test_an_error_leaves_nothing_unjoined(fails):
    """Whichever step of three blocks fails: nothing is launched behind it, and the caller's stream waits for the one beside, if that has been
    handed anything."""
    ok, steps = load_package().capi.probe_halves_order(3, fails)
    assert not ok
    whole = [FORK, EARLIER, LATER] * 3 + [JOIN]
    # (the stream beside has nothing to wait for where the very first hand-over failed, and the wait itself is not tried twice)
    assert steps == whole[:fails + 1] + ([JOIN] if 0 < fails < 9 else [])
