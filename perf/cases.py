"""Performance cases of the inference path: whole networks through the NetBuilder binding (`msnhnet_amd.netapi`).

A case is one network in one data type, at one batch and input size, fed in one of the ways a program feeds it, and a pass is what such a
program does per batch (or, for a group of instances, per burst of batches): hand the input over, run the forward, have the logits or
the boxes in host memory.  `feed` says where the input is before the call:

  device   float32 NCHW in device memory (a producer on the GPU writes there): enqueue(pointer), fetch
  host     float32 NCHW in host memory, the calling convention of runClassifyGPU / runYoloGPU: run_classify / run_yolo
  image    8-bit HWC pictures in host memory, resized or letterboxed on the device: set_input_image[_u8] per picture, enqueue, fetch

Architectures, sizes and data types are those of the benchmark configurations and of the other graphs `msnhnet_amd.zoo` writes.
"""
import math
import os
import tempfile
from collections import OrderedDict

import numpy as np
import torch

from msnhnet_amd import netapi, zoo

WEIGHT_SEED = 1
CLASSIFIERS = ("resnet18", "resnet50", "mobilenetv2")
DETECTORS = ("yolov3_tiny", "yolov5s", "yolov3", "yolov4")
PRE_TRANSFORMED = 3                                     # MSNH_PRE_TRANSFORMED of include/msnh_hip.h: (u / 255 - mean) / std
MEAN, STD = (0.485, 0.456, 0.406), (0.229, 0.224, 0.225)
PICTURES = ((480, 640), (375, 500), (720, 1280), (1080, 1920))        # height, width of the pictures an `image` case is fed with


def _case(name, arch, dtype, batch, size, feed, instances=1, rounds=1):
    return {"name": name, "arch": arch, "dtype": dtype, "batch": batch, "size": size, "feed": feed, "instances": instances, "rounds": rounds}


def listed():
    return [
        # one picture at a time, the answer wanted at once: a camera or a request (launches and host work count)
        _case("tiny_f16_b1_image", "yolov3_tiny", "f16", 1, 416, "image"),
        _case("mobilenetv2_f16_b1_device", "mobilenetv2", "f16", 1, 224, "device"),
        _case("resnet18_f32_b1_device", "resnet18", "f32", 1, 224, "device"),          # the first benchmark configuration
        _case("yolov3_f16_b1_image", "yolov3", "f16", 1, 416, "image"),
        # the library's defaults (float32, a host float image per call): what a program written for the reference does
        _case("yolov3_f32_b1_host", "yolov3", "f32", 1, 608, "host"),
        _case("resnet50_f32_b5_host", "resnet50", "f32", 5, 224, "host"),
        # a few cameras at once, a batch and a map size that are no powers of two
        _case("yolov5s_f16_b3_device", "yolov5s", "f16", 3, 544, "device"),
        # batches of the benchmark configurations
        _case("resnet50_f16_b32_device", "resnet50", "f16", 32, 224, "device"),
        _case("mobilenetv2_f16_b64_device", "mobilenetv2", "f16", 64, 224, "device"),
        _case("yolov3_f16_b8_device", "yolov3", "f16", 8, 608, "device"),
        _case("yolov4_f16_b16_device", "yolov4", "f16", 16, 608, "device"),
        # a server: three instances of a network on the GPU, fed round-robin
        _case("yolov3_f16_b8_group", "yolov3", "f16", 8, 608, "device", instances=3, rounds=12),
    ]


_graphs = {}


def _graph(arch, batch, size):
    key = (arch, batch, size)
    if key not in _graphs:
        _graphs[key] = zoo.ARCHS[arch](batch=batch, size=size)
    return _graphs[key]


def _flops(arch, batch, size):
    g = _graph(arch, batch, size)
    return float(batch) * (g.conv_flops + g.fc_flops)


def draw(rng):
    """Any network, data type and feed; detector sizes in their steps of 32; the batch spread over its logarithm up to what costs as much
    as the largest benchmark configuration (float32 counted 16 times: the ratio of the two matrix rates)."""
    arch = rng.choice(CLASSIFIERS + DETECTORS)
    dtype = "f16" if rng.random() < 0.65 else "f32"
    feed = rng.choice(("device", "host", "image"))
    size = 224 if arch in CLASSIFIERS else 32 * rng.randint(7, 19)
    most = _flops("yolov4", 16, 608) / (16 if dtype == "f32" else 1)
    cap = max(1, min(64, int(most / _flops(arch, 1, size))))
    group = feed == "device" and rng.random() < 0.3
    rounds = rng.randint(4, 12) if group else 1
    batch = int(round(math.exp(rng.uniform(0.0, math.log(max(1, cap // rounds))))))
    c = _case("", arch, dtype, batch, size, feed, 3 if group else 1, rounds)
    del c["name"]
    return c


# ---- weights ---------------------------------------------------------------------------------------------------------------
# The seeded weights do not normalise: the channels in front of a detection head have magnitudes up to 1e6, so that every cell's score saturates
# and half of the cells are "found".  A trained detector's logits are of order one, most cells are empty and the found ones are settled.
# So the batch norm in front of a head (yolov5s, where it feeds other layers too: the head's filters) is scaled to bring the logits there,
# and the objectness comes from the biases: in the coarsest head the first two anchors of every cell are found, with boxes smaller than a cell
# and of one class, the second one a weaker copy of the first that the suppression has to remove -- 722 candidates and 361 boxes for a picture of 608.
# Positions and sizes depend on the picture, and no decision stands so close to its threshold that rounding could turn it.
HEAD_GAIN = {"yolov3_tiny": (0.8, 0.8), "yolov3": (4e-6, 3.6e-6, 3.2e-6), "yolov4": (1.6e-6, 1e-6, 9e-7), "yolov5s": (0.09, 0.066, 0.057)}
BOX_SIZE = 20.0               # pixels
BOX_SPREAD = 0.1              # of the position and size logits
CLASS = 16


def _plant_heads(arch, g, w):
    at = np.concatenate([[0], np.cumsum([s.count for s in g.slots])])
    anchors = [[int(v) for v in l.split(":")[1].split(",")] for l in g.lines if l.strip().startswith("anchors:")]
    heads = [i for i, s in enumerate(g.slots[:-1]) if s.kind == "conv_w" and g.slots[i + 1].kind == "bias" and s.count == 255 * s.fan_in]
    coarse = max(range(len(heads)), key=lambda k: anchors[k][4])
    for k, i in enumerate(heads):
        f = w[at[i]:at[i + 1]].reshape(3, 85, -1)
        b = w[at[i + 1]:at[i + 2]].reshape(3, 85)
        gain = np.float32(HEAD_GAIN[arch][k])
        if g.slots[i - 4].kind == "bn_gamma" and arch != "yolov5s":
            w[at[i - 4]:at[i - 2]] *= gain                # gamma and beta
        else:
            f *= gain
        f *= np.float32(BOX_SPREAD)
        f[:, 4] = 0.0
        b[:] = -4.0
        b[:, :2] = 0.0
        b[:, 2:4] = 0.0
        b[:, 4] = -6.0
        if k == coarse:
            f[1] = f[0]
            b[0, 4], b[1, 4] = 3.0, 2.0
            f[:2, 5 + CLASS] = 0.0
            b[:2, 5 + CLASS] = 20.0
            for a in (0, 1):
                for m in (0, 1):
                    r = BOX_SIZE / anchors[k][2 * a + m]
                    s = math.sqrt(r) / 2                  # yolov5: anchor * (2 * logistic)^2, else anchor * exp
                    b[a, 2 + m] = math.log(s / (1 - s)) if arch == "yolov5s" else math.log(r)


# ---- networks ---------------------------------------------------------------------------------------------------------------
_loaded = OrderedDict()       # a program loads a network once and keeps it; the least recently used of 16 goes


def _network(case):
    key = (case["arch"], case["dtype"], case["batch"], case["size"], case["instances"])
    if key in _loaded:
        _loaded.move_to_end(key)
        return _loaded[key], False
    g = _graph(case["arch"], case["batch"], case["size"])
    w = zoo.seeded_weights(g.slots, WEIGHT_SEED)
    if case["arch"] in DETECTORS:
        _plant_heads(case["arch"], g, w)
    with tempfile.TemporaryDirectory(prefix="msnh_perf_") as d:
        netp, binp = os.path.join(d, "net.msnhnet"), os.path.join(d, "net.msnhbin")
        with open(netp, "w") as f:
            f.write(g.text())
        w.tofile(binp)
        fp16 = case["dtype"] == "f16"
        if case["instances"] > 1:
            net = netapi.NetGroup(netp, binp, instances=case["instances"], depth=2, fp16=fp16)
        else:
            net = netapi.Net(netp, binp, fp16=fp16)
    _loaded[key] = net
    while len(_loaded) > 16:
        _loaded.popitem(last=False)[1].close()
    return net, True


def prepare(case, seed):
    net, new = _network(case)
    b, size = case["batch"], case["size"]
    state = {"net": net, "feed": case["feed"], "detect": case["arch"] in DETECTORS, "group": case["instances"] > 1}
    if case["feed"] == "image":
        rng = np.random.default_rng(seed)
        pictures = []
        for i in range(b):
            h, w = PICTURES[i % len(PICTURES)]
            coarse = rng.integers(0, 256, ((h + 7) // 8, (w + 7) // 8, 3), dtype=np.uint8)      # patches of one colour and a little noise
            p = coarse.repeat(8, axis=0).repeat(8, axis=1)[:h, :w]
            pictures.append(np.ascontiguousarray(p ^ rng.integers(0, 8, p.shape, dtype=np.uint8)))
        state["pictures"] = pictures
    elif case["feed"] == "host":
        state["x"] = np.random.default_rng(seed).random((b, 3, size, size), dtype=np.float32)
    else:
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed)
        state["x"] = [torch.rand((b, 3, size, size), generator=gen, device="cuda") for _ in range(case["rounds"])]
        if new and state["group"]:
            torch.cuda.synchronize()
            net.prime(state["x"][0].data_ptr())
    return state


def _boxes(per_image):
    return {"counts": np.array([len(p) for p in per_image]), "boxes": np.concatenate(per_image)}


def run(state):
    net, detect = state["net"], state["detect"]
    if state["group"]:
        for x in state["x"]:
            net.submit(x.data_ptr())
        net.flush()
        out = [net.fetch() for _ in state["x"]]
        return [_boxes(o) for o in out] if detect else out
    if state["feed"] == "host":
        return _boxes(net.run_yolo(state["x"])) if detect else net.run_classify(state["x"])
    if state["feed"] == "image":
        for i, p in enumerate(state["pictures"]):
            if detect:
                net.set_input_image_u8(i, p)
            else:
                net.set_input_image(i, p, PRE_TRANSFORMED, MEAN, STD)
        net.enqueue()
    else:
        net.enqueue(state["x"][0].data_ptr())
    return _boxes(net.fetch_yolo()) if detect else net.fetch_classify()


def work(case):
    """Input, weights and result once; multiply-adds of the direct convolutions."""
    g = _graph(case["arch"], case["batch"], case["size"])
    b, size, rounds = case["batch"], case["size"], case["rounds"]
    if case["feed"] == "image":
        read = sum(3 * h * w for h, w in (PICTURES[i % len(PICTURES)] for i in range(b)))
    else:
        read = 12 * b * size * size
    weights = sum(s.count * ((2 if case["dtype"] == "f16" else 4) if s.kind in ("conv_w", "fc_w") else 4) for s in g.slots)
    out = 28 * b * (size // 32) ** 2 if case["arch"] in DETECTORS else 4000 * b
    return {"bytes": float(rounds * (read + out) + weights), "flops": rounds * _flops(case["arch"], b, size)}


def tolerance(case):
    # float32: sums of up to 4608 products over up to 110 layers in another order.  float16: activations rounded to 11 bits between the layers.
    return {"rel": 2e-5, "max": 1e-3} if case["dtype"] == "f32" else {"rel": 1e-2, "max": 0.1}
