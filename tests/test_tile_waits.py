"""Kernels whose workgroups wait for lower-numbered ones without a start-order
ticket (the single-pass block scan, the radix passes of small tiles).  The
hardware deals workgroups out to the eight XCDs in turn and starts each XCD's in
order, so a wait ends once the lowest unfinished workgroup of every waiting
kernel finds a place on its XCD.  A process has four hardware queues: the
waiting workgroups of three kernels must not fill an XCD's 32 CUs, in any
mixture, and a wait must outlast the work that other streams hold the device
with."""
import itertools

from tests.kernel_resources import constant, kernel_resources, workgroups_per_cu

XCDS, CUS_PER_XCD, QUEUES = 8, 32, 4


def test_other_streams_cannot_fill_an_xcd_with_waiting_workgroups():
    res = kernel_resources()
    waiting = {"k_bscan<2>": constant("kScanTilesOnePass"),
               "k_bscan<3>": constant("kScanTilesOnePass"),
               f"k_onesweep<{constant('kRadixSmallItems')}>": constant("kRadixSmallTiles")}
    share = {k: tiles / XCDS / (CUS_PER_XCD * workgroups_per_cu(res[k]))
             for k, tiles in waiting.items()}  # of an XCD, by one launch
    for mix in itertools.combinations_with_replacement(share, QUEUES - 1):
        assert sum(share[k] for k in mix) < 1.0, mix


def test_larger_sorts_take_a_ticket():
    import os

    from tests.kernel_resources import CSRC
    with open(os.path.join(CSRC, "mpm_kernels.hip")) as f:
        source = f.read()
    body = source[source.index("LBTicket lb_acquire("):]
    body = body[:body.index("\n}")]
    assert "if (ntiles <= kRadixSmallTiles)" in body
    assert "atomicAdd(&st->tile_ctr" in body


def test_waits_are_bounded_by_seconds():
    # a poll is a device-scope load and a sleep: half a microsecond at the least
    assert constant("kWaitLimit") * 0.5e-6 > 2.0
