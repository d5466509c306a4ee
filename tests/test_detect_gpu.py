"""Detectors across forwards: where the candidates of a result are suppressed -- inside the forward, behind it on the device, on the host --
and what runs between two forwards must not show in the boxes.  Every result is compared with the one a network gives that has run nothing
else (the same kernels: a load takes the tile choices of an earlier load of the same plan), bit for bit."""
import os
import re

import numpy as np
import pytest
import torch

import netutil as nu
from msnhnet_amd import netapi, zoo

pytestmark = pytest.mark.gpu


def same(got, want):
    return len(got) == len(want) and all(np.array_equal(a, b, equal_nan=True) for a, b in zip(got, want))


GRID, CLASSES, LOGIT = 32, 3, 20.0          # a scene network's head: GRID x GRID cells, three anchors; pixel value v stands for the logit LOGIT * (v - 0.5)


def scene_net(batch, tag=""):
    """a detector whose only convolution (8 x 8, stride 8) hands the pixels on as logits: value m of anchor a in a cell is pixel m of the first
    row of the cell's patch in channel a -- any scene can be painted"""
    per = 5 + CLASSES
    g = zoo.GraphWriter(batch, 3, 8 * GRID, 8 * GRID)
    g.conv(3 * per, k=8, stride=8, bn=0, act="none")
    g.yolo([14, 17, 22, 31, 40, 26], class_num=CLASSES)
    g.yoloout([1], conf=0.5, nms=0.45)
    w = np.zeros((3 * per, 3, 8, 8), np.float32)
    for a in range(3):
        for m in range(per):
            w[a * per + m, a, 0, m] = LOGIT
    path = os.path.join(nu.workdir(), f"scenes_b{batch}{tag}")
    with open(path + ".msnhnet", "w") as f:
        f.write(g.text())
    np.concatenate([w.ravel(), np.full(3 * per, -LOGIT / 2, np.float32)]).tofile(path + ".msnhbin")
    return path + ".msnhnet", path + ".msnhbin"


def scene(counts, seed):
    """a batch with counts[b] candidates in image b, of all classes, many of them overlapping"""
    per, cells = 5 + CLASSES, 3 * GRID * GRID
    rng = np.random.default_rng(seed)
    x = np.zeros((len(counts), 3, GRID, 8, GRID, 8), np.float32)
    for b, n in enumerate(counts):
        t = rng.uniform(-2.0, 2.0, (cells, per))
        t[:, 4] = -6.0
        t[rng.permutation(cells)[:n], 4] = rng.uniform(0.5, 6.0, n)
        t[:, 2:4] *= 0.5
        v = (t / LOGIT + 0.5).reshape(3, GRID, GRID, per)
        x[b, :, :, 0, :, :per] = v
    return x.reshape(len(counts), 3, 8 * GRID, 8 * GRID)


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


def recorded(m):
    return int(re.search(r"(\d+) forwards recorded", m.load_detail()).group(1))


def test_forwards_are_recorded_before_they_are_needed():
    """a load records every forward that its network replays (a detector: two copy-back slots, the suppression inside and behind), so that neither
    the first batches nor the first crowded scene wait for it; a group's instances the same, over the weights they share"""
    net, binp = scene_net(2)
    quiet, crowded = scene((300, 900), 1), scene((1500, 2500), 2)
    m = netapi.Net(net, binp)
    assert recorded(m) == 4
    for x in (quiet, quiet, crowded, crowded, crowded, quiet, quiet, quiet):
        assert all(len(b) > 0 for b in m.run_yolo(x))
    assert recorded(m) == 4
    xd = [torch.from_numpy(x).cuda() for x in (quiet, crowded, quiet)]
    torch.cuda.synchronize()
    want = [m.run_yolo(x) for x in (quiet, crowded, quiet)]
    grp = netapi.NetGroup(net, binp, instances=2, depth=2)
    try:
        assert [recorded(n) for n in grp.nets] == [4, 4]
        grp.prime(xd[0].data_ptr())
        for i in (0, 1, 2, 1, 1, 1, 0, 0, 0, 2, 1):
            grp.submit(xd[i].data_ptr())
            assert same(grp.fetch(), want[i])
        assert [recorded(n) for n in grp.nets] == [4, 4]
    finally:
        grp.close()
    netapi.set_device_nms(0)
    try:
        m = netapi.Net(net, binp)
        assert recorded(m) == 2
        m.run_yolo(quiet)
    finally:
        netapi.set_device_nms(1)
    assert same(m.run_yolo(quiet), want[0]) and same(m.run_yolo(quiet), want[0])      # (a form that the settings did not allow before: recorded now)
    assert recorded(m) == 4
    assert recorded(netapi.Net(*nu.model("resnet18", 1, 224, seed=3)[:2])) == 1
    small = netapi.Net(*nu.model("resnet18", 1, 64, seed=3)[:2])                       # (its 7 x 7 pool does not fit a 2 x 2 tensor: loads, does not run)
    assert recorded(small) == 0
    with pytest.raises(netapi.MsnhnetError, match="window larger"):
        small.run_classify(zoo.seeded_input(1, 3, 64, 64, 1))


QUIET, CROWDED = [(0, 700, 1024), (1024, 3, 900), (500, 0, 1)], [(1025, 20, 3000), (1100, 1500, 2048), (10, 3072, 1024), (2049, 1024, 1025)]


@pytest.mark.parametrize("depth", [1, 2])
@pytest.mark.parametrize("own_stream", [True, False])
def test_scenes_that_cross_the_line_both_ways(depth, own_stream):
    """candidate counts on both sides of 1024 in one batch and from batch to batch, long enough for the suppression to go inside, behind and inside
    again several times: the boxes are the host's, wherever they were suppressed"""
    net, binp = scene_net(3)
    counts = QUIET + CROWDED
    xs = [scene(c, 10 + i) for i, c in enumerate(counts)]
    netapi.set_device_nms(0)
    try:
        host = netapi.Net(net, binp)
        want = [host.run_yolo(x) for x in xs]
        for i, c in enumerate(counts):
            host.run_yolo(xs[i])
            assert [len(host.yolo_candidates(b)) for b in range(3)] == list(c)
    finally:
        netapi.set_device_nms(1)
    assert all(len(np.unique(b[:, 6])) == CLASSES for b in want[3][2:])
    xd = [torch.from_numpy(x).cuda() for x in xs]
    torch.cuda.synchronize()
    m = netapi.Net(net, binp)
    m.set_copy_on_forward_stream(not own_stream)
    rng = np.random.default_rng(7)
    order = [0, 1, 3, 0, 4, 2, 5, 6, 6]
    for rounds in range(3):
        order += list(rng.integers(0, 3, 12)) + [3 + rounds, 6, 3, 1, 4]           # a quiet stretch, then back and forth
    order += list(rng.integers(0, len(xs), 40)) + [0] * 70 + [5, 0, 0]
    print("crossing", depth, own_stream, flush=True)
    sent = 0
    for k, i in enumerate(order):
        while sent < len(order) and sent < k + depth:
            m.enqueue(xd[order[sent]].data_ptr())
            sent += 1
        assert same(m.fetch_yolo(), want[i]), (k, i)
    assert recorded(m) == 4
