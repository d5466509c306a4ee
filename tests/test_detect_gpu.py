"""Detectors across forwards: where the candidates of a result are suppressed -- inside the forward, behind it on the device, on the host --
and what runs between two forwards must not show in the boxes.  Every result is compared with the one a network gives that has run nothing
else (the same kernels: a load takes the tile choices of an earlier load of the same plan), bit for bit."""
import numpy as np
import pytest

import netutil as nu
from msnhnet_amd import netapi, zoo

pytestmark = pytest.mark.gpu


def same(got, want):
    return len(got) == len(want) and all(np.array_equal(a, b, equal_nan=True) for a, b in zip(got, want))


BETWEEN = {
    "headroom": lambda m, x: m.fp16_headroom(x),
    "profile_each_op": lambda m, x: m.profile_each_op(2),
    "profile_ops": lambda m, x: m.profile_ops(-1, 3),
}


@pytest.mark.parametrize("what", sorted(BETWEEN))
def test_launches_between_forwards_leave_no_candidates(what):
    """a network whose forwards suppress their own candidates (at most 1008 cells here) takes a slot's counts for zero when it starts: the
    launches of the headroom check and of the profiles append to counts too, and must not append to those"""
    size, batch = 128, 2
    net, binp, g = nu.model("yolov5s", batch, size, seed=3)
    xs = [zoo.seeded_input(batch, 3, size, size, seed=s) for s in (4, 5)]
    want = [netapi.Net(net, binp, fp16=True).run_yolo(x) for x in xs]
    assert all(len(b) > 0 for w in want for b in w)
    m = netapi.Net(net, binp, fp16=True)
    print("between forwards:", what, flush=True)
    for rounds in range(2):
        for first in (0, 1):                       # (either slot is the one that was used last)
            assert same(m.run_yolo(xs[first]), want[first])
            assert same(m.run_yolo(xs[1]), want[1])
            BETWEEN[what](m, xs[1])
            for i in (0, 1, 0):
                assert same(m.run_yolo(xs[i]), want[i]), (rounds, first, i)
