"""Detectors across forwards: where the candidates of a result are suppressed -- inside the forward, behind it on the device, on the host --
and what runs between two forwards must not show in the boxes.  Every result is compared with the one a network gives that has run nothing
else (the same kernels: a load takes the tile choices of an earlier load of the same plan), bit for bit."""
import numpy as np
import pytest
import torch

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


@pytest.mark.parametrize("what", ["profile_each_op", "profile_ops"])
@pytest.mark.parametrize("nms", [0, 1, 2])
def test_profiles_leave_outstanding_results_alone(what, nms, monkeypatch):
    """two results on their way, a profile, then the fetches: the profile's launches append to a set of their own, wherever the results are
    suppressed (nms 1: inside their forwards) and also where rows are still fetched from the device afterwards (a short prefix on the host path)"""
    size, batch = 128, 2
    net, binp, g = nu.model("yolov5s", batch, size, seed=3)
    xs = [zoo.seeded_input(batch, 3, size, size, seed=s) for s in (4, 5)]
    want = [netapi.Net(net, binp, fp16=True).run_yolo(x) for x in xs]
    xd = [torch.from_numpy(x).cuda() for x in xs]
    torch.cuda.synchronize()
    monkeypatch.setenv("MSNH_YOLO_ROWS_PREFIX", "8")
    netapi.set_device_nms(nms)
    try:
        m = netapi.Net(net, binp, fp16=True)
        print("outstanding results:", what, nms, flush=True)
        for rounds in range(3):
            for t in xd:
                m.enqueue(t.data_ptr())
            BETWEEN[what](m, xs[1])
            with pytest.raises(netapi.MsnhnetError, match="outstanding"):
                m.fp16_headroom(xs[0])
            for w in want:
                assert same(m.fetch_yolo(), w), rounds
    finally:
        netapi.set_device_nms(1)


def test_layer_dumps_wait_for_outstanding_results():
    """the layer-by-layer run uses the first slot: refused, before it writes anything, while a result in that slot is outstanding"""
    size, batch = 128, 2
    net, binp, g = nu.model("yolov5s", batch, size, seed=3)
    xs = [zoo.seeded_input(batch, 3, size, size, seed=s) for s in (4, 5)]
    m = netapi.Net(net, binp, fp16=True, dump_layers=True)
    want = [m.run_yolo(x) for x in xs]
    xd = torch.from_numpy(xs[0]).cuda()
    torch.cuda.synchronize()
    m.enqueue(xd.data_ptr())
    with pytest.raises(netapi.MsnhnetError, match="outstanding"):
        m.run_yolo(xs[1])
    assert same(m.fetch_yolo(), want[0])
    assert same(m.run_yolo(xs[1]), want[1])
