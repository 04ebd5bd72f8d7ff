"""Performance cases of the library: what an int8 inference application has it do, through the two public layers.

Two kinds of case:

* "network": a whole quantized network behind the clDNN API (cldnn_amd.api) built with optimize_data.  One pass is what an
  application does per request: set_input_data, execute, read the scores.  Small batches are requests that arrive as host
  images (the pass writes the image into the input memory as well); larger batches have their images on the device already,
  as a decoding pipeline leaves them there.
* "conv": one convolution / fused_conv_eltwise / depthwise / grouped object of the C-ABI (cldnn_amd.hip), tensors resident on
  the device in the blocked layout with the zero border the host library gives a convolution's input.  One pass is one
  enqueue: what a caller with a graph of its own does per layer.  At batch 1 or 2 the caller waits for the result, as an
  interactive program does; larger batches stay queued.

Parameters are random with the factors that keep a signal alive through a network: per-feature requantisation scaled to the
spread of the accumulators, so the int8 results use their range.
"""
import math

import numpy as np
import torch

from cldnn_amd import api, hip, mobilenet_v2_net, resnet50_net, vgg16_net, workloads

NETWORKS = {
    # definition, layers, scores, classifier layers (name, inputs, outputs)
    "resnet50": (resnet50_net, workloads.resnet50, "fc1000", (("fc1000", 2048, 1, 1000),)),
    "mobilenet_v2": (mobilenet_v2_net, workloads.mobilenet_v2, "fc1000", (("fc1000", 1280, 1, 1000),)),
    "vgg16": (vgg16_net, workloads.vgg16, "fc8", (("fc6", 512, 7, 4096), ("fc7", 4096, 1, 4096), ("fc8", 4096, 1, 1000))),
}
WAIT_BATCH = 2          # a single layer up to this batch is waited for
HOST_BATCH = 8          # requests up to this batch come as host images
LARGEST_NETWORK = 128   # images of 224 x 224


def _network(name, model, batch, hw, **more):
    return dict(name=name, kind="network", model=model, batch=batch, hw=hw, host_image=batch <= HOST_BATCH, **more)


def _conv(name, batch, ifm, ofm, h, w, k, stride=1, groups=1, in_type="u8", out_type="s8", act="relu", fused=False):
    return dict(name=name, kind="conv", batch=batch, ifm=ifm, ofm=ofm, h=h, w=w, k=k, stride=stride, groups=groups, in_type=in_type,
                out_type=out_type, act=act, fused=fused, wait=batch <= WAIT_BATCH)


def listed():
    return [
        # one image per request: the latency of an interactive classifier
        _network("resnet50_b1", "resnet50", 1, 224),
        _network("mobilenet_v2_b1", "mobilenet_v2", 1, 224),
        _network("vgg16_b1", "vgg16", 1, 224),
        # a few images of another resolution at once (sizes that fill no tile, odd planes at every level)
        _network("resnet50_b5_odd", "resnet50", 5, 201),
        # the batches of the repository's benchmark: throughput serving
        _network("resnet50_b32", "resnet50", 32, 224),
        _network("mobilenet_v2_b32", "mobilenet_v2", 32, 224),
        _network("vgg16_b16", "vgg16", 16, 224),
        # offline scoring of a data set
        _network("resnet50_b128", "resnet50", 128, 224),
        # a single layer, batch 1: the smallest call (the first configuration of the baseline)
        _conv("conv_64_b1", 1, 64, 64, 56, 56, 3),
        # a layer of a network whose widths are no multiples of 16 and whose image is not square
        _conv("conv_odd_b7", 7, 84, 108, 31, 45, 3, act="none", in_type="s8"),
        # the output layer of a detector: scores leave the int8 domain
        _conv("conv_head_f32_b8", 8, 512, 126, 19, 19, 3, act="none", in_type="s8", out_type="f32"),
        # a depthwise layer on its own
        _conv("conv_depthwise_b32", 32, 576, 576, 14, 14, 3, groups=576, act="relu6", in_type="s8"),
    ]


def _log_uniform(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    if rng.random() < 0.5:
        model = rng.choice(("resnet50", "resnet50", "mobilenet_v2", "mobilenet_v2", "vgg16"))
        # VGG-16's first classifier layer fixes its image size
        hw = 224 if model == "vgg16" or rng.random() < 0.4 else rng.randint(128, 320)
        most = {"resnet50": LARGEST_NETWORK, "mobilenet_v2": LARGEST_NETWORK, "vgg16": LARGEST_NETWORK // 5}[model]
        c = _network("", model, _log_uniform(rng, 1, max(1, int(most * 224 ** 2 / max(hw, 224) ** 2))), hw)
        del c["name"]
        return c
    while True:
        form = rng.choice(("dense", "dense", "dense", "dense", "fused", "f32", "depthwise", "depthwise", "grouped"))
        batch, h = _log_uniform(rng, 1, 64), _log_uniform(rng, 7, 112)
        w = h if rng.random() < 0.5 else _log_uniform(rng, 7, 112)
        ifm, ofm = _log_uniform(rng, 8, 1024), _log_uniform(rng, 8, 1024)
        if rng.random() < 0.5:  # widths of networks are mostly multiples of 8
            ifm, ofm = 8 * -(-ifm // 8), 8 * -(-ofm // 8)
        k, stride, groups = rng.choice((1, 1, 3, 3, 3, 5)), rng.choice((1, 1, 1, 2)), 1
        act, out_type = rng.choice(("relu", "relu", "none", "relu6")), "s8"
        if form == "fused":
            k = stride = 1
        elif form == "f32":
            act, out_type = "none", "f32"
        elif form == "depthwise":
            ofm = groups = ifm
            k = rng.choice((3, 3, 3, 5))
        elif form == "grouped":
            groups = rng.choice((2, 4, 8, 32))
            ifm, ofm, k = groups * -(-min(ifm, 512) // groups), groups * -(-min(ofm, 512) // groups), 3
        c = _conv("", batch, ifm, ofm, h, w, k, stride, groups, rng.choice(("u8", "s8")), out_type, act, form == "fused")
        del c["name"]
        n = work(c)
        # below that a queued call is all launch, which the small waited-for ones show better
        if n["flops"] <= 2e11 and n["bytes"] <= 1e8 and (c["wait"] or n["bytes"] >= 2e6 or n["flops"] >= 5e8):
            return c


_engines = {}


def _engine(kind):
    """One engine (device queue) per process and layer, as an application keeps it."""
    if kind not in _engines:
        _engines[kind] = api.engine() if kind == "network" else hip.Engine(0)
    return _engines[kind]


# --------------------------------------------------------------------------------------------------------------- networks
def _weights(r, *shape):
    return r.integers(-127, 128, shape, dtype=np.int8)


def _network_params(model, r):
    net, layers, _, fcs = NETWORKS[model]
    rms = 35.0  # of a layer's int8 input
    p = {}
    for l in layers():
        k = (l["ifm"] // l["groups"]) * l["k"] ** 2
        sigma = math.sqrt(k) * rms * 73.3
        f = r.uniform(0.7, 1.4, l["ofm"]).astype(np.float32)
        q = dict(w=_weights(r, l["ofm"], l["ifm"] // l["groups"], l["k"], l["k"]), bias=r.integers(-1000, 1001, l["ofm"]).astype(np.int32))
        if l["act"] == "relu6":  # the clamp acts on the dequantised value
            q.update(wqf=np.float32(3.0 / sigma) * f, calib=np.full(l["ofm"], 127.0 / 6.0, np.float32))
        else:
            q.update(wqf=np.ones(l["ofm"], np.float32), calib=np.float32(32.0 / sigma) * f)
        p[l["name"]] = q
    for n, ifm, plane, ofm in fcs:
        p[n] = dict(w=_weights(r, ofm, ifm, plane, plane), bias=(10 * r.standard_normal(ofm)).astype(np.float32), wqf=np.ones(ofm, np.float32),
                    calib=np.full(ofm, 40.0 / (math.sqrt(ifm * plane * plane) * 30.0 * 73.3), np.float32))
    for step in net.layer_plan():
        if step[0] == "sum":
            p[step[1]] = dict(ecal=np.full(p[step[3]]["w"].shape[0], 1.0 if model == "resnet50" else 0.75, np.float32))
    return p


def _prepare_network(case, seed):
    r = np.random.default_rng(seed)
    net_def, _, scores, _ = NETWORKS[case["model"]]
    eng = _engine("network")
    topo = net_def.topology(api, eng, _network_params(case["model"], r), case["batch"], case["hw"])
    net = api.network(eng, topo, api.build_options(optimize_data=True))
    image = r.integers(0, 256, (case["batch"], 3, case["hw"], case["hw"]), dtype=np.uint8)
    return dict(kind="network", net=net, scores=scores, input=api.make_memory(eng, image), image=image if case["host_image"] else None)


def _run_network(s):
    if s["image"] is not None:
        s["input"].write(s["image"])
    s["net"].set_input_data("input", s["input"])
    return s["net"].execute()[s["scores"]].get_memory().read()


def _planes(case):
    """Size of a plane in this case for its size at 224 x 224: every level halves, rounding up, except the 3x3 / stride 2
    pooling of ResNet-50 and the 2x2 poolings of VGG-16 (always at 224)."""
    size, out = case["hw"], {224: case["hw"]}
    for level in (112, 56, 28, 14, 7):
        if case["model"] == "resnet50" and level == 56:
            size = -(-(size - 3) // 2) + 1
        else:
            size = (size - 1) // 2 + 1
        out[level] = size
    return out


def _network_work(case):
    net, layers, _, fcs = NETWORKS[case["model"]]
    planes, macs, weights = _planes(case), 0, 0
    for l in layers():
        n = planes[l["out_hw"]]
        # only every other row and column of these is read by the stride-2 convolutions behind them
        if l["name"] in ("res2c_branch2b", "res2c_branch2c", "res3d_branch2b", "res3d_branch2c", "res4f_branch2b", "res4f_branch2c"):
            n = (n - 1) // 2 + 1
        per_output = (l["ifm"] // l["groups"]) * l["k"] ** 2
        macs += n * n * l["ofm"] * per_output
        weights += l["ofm"] * (per_output + 12)
    for _, ifm, plane, ofm in fcs:
        macs += ofm * ifm * plane * plane
        weights += ofm * (ifm * plane * plane + 12)
    return {"bytes": case["batch"] * (3 * case["hw"] ** 2 + 1000) + weights, "flops": 2 * case["batch"] * macs}


# ------------------------------------------------------------------------------------------------------------ convolutions
class _DeviceBytes:
    """The memory of a device buffer for torch, without a copy."""

    def __init__(self, buf, type_name):
        item = {"s8": ("|i1", 1), "f32": ("<f4", 4)}[type_name]
        self.buf = buf
        self.__cuda_array_interface__ = dict(shape=(buf.nbytes // item[1],), typestr=item[0], data=(buf.ptr, False), version=2)


def _out_size(case):
    return tuple((n + 2 * (case["k"] // 2) - case["k"]) // case["stride"] + 1 for n in (case["h"], case["w"]))


def _prepare_conv(case, seed):
    r = np.random.default_rng(seed)
    eng = _engine("conv")
    batch, ifm, ofm, k, groups = (case[n] for n in ("batch", "ifm", "ofm", "k", "groups"))
    shape = (batch, ifm, case["h"], case["w"])
    x = r.integers(0, 256, shape, dtype=np.uint8) if case["in_type"] == "u8" else r.integers(-128, 128, shape, dtype=np.int8)
    w = _weights(r, ofm, ifm // groups, k, k)
    sigma = math.sqrt(ifm // groups * k * k) * (147.4 if case["in_type"] == "u8" else 73.9) * 73.3
    f = r.uniform(0.5, 2.0, ofm).astype(np.float32)
    kw = dict(stride=(case["stride"],) * 2, pad=(k // 2,) * 2, groups=groups, bias_dt=hip.I32, has_wqf=True, has_calib=True)
    eltw = ecal = None
    if case["act"] == "relu6":
        wqf, calib = np.float32(3.0 / sigma) * f, np.full(ofm, 127.0 / 6.0, np.float32)
        kw.update(act="clamp", act_m=0.0, act_n=6.0)
    else:
        wqf, calib = np.ones(ofm, np.float32), np.float32(40.0 / sigma) * f
        kw.update(act=case["act"])
    if case["fused"]:
        oh, ow = _out_size(case)
        eltw = hip.upload(eng, r.integers(-128, 128, (batch, ofm, oh, ow), dtype=np.int8), "fs_b_yx_fsv16")
        ecal = r.uniform(0.25, 1.0, ofm).astype(np.float32)
        kw.update(act="none", eltw_t=eltw.tensor, eltw_act="relu", has_eltw_calib=True)
    src = hip.upload(eng, x, "fs_b_yx_fsv16", (k // 2, k // 2))
    desc = hip.conv_desc(src.tensor, w.shape, case["out_type"], **kw)
    conv = hip.Conv(eng, desc, w, r.integers(-1000, 1001, ofm).astype(np.int32), wqf, calib, ecal)
    dst = hip.Buffer(eng, desc.output)
    eng.finish()
    return dict(kind="conv", engine=eng if case["wait"] else None, conv=conv, src=src, dst=dst, eltw=eltw, out=torch.as_tensor(_DeviceBytes(dst, case["out_type"]), device="cuda"))


def _run_conv(s):
    s["conv"].enqueue(s["src"], s["dst"], s["eltw"])
    if s["engine"] is not None:
        s["engine"].finish()
    return s["out"]


def _conv_work(case):
    oh, ow = _out_size(case)
    outputs = case["batch"] * case["ofm"] * oh * ow
    per_output = case["ifm"] // case["groups"] * case["k"] ** 2
    size = {"s8": 1, "f32": 4}[case["out_type"]]
    return {"bytes": case["batch"] * case["ifm"] * case["h"] * case["w"] + outputs * (size + (1 if case["fused"] else 0))
            + case["ofm"] * (per_output + 12), "flops": 2 * outputs * per_output}


# -------------------------------------------------------------------------------------------------------------- interface
def prepare(case, seed):
    return (_prepare_network if case["kind"] == "network" else _prepare_conv)(case, seed)


def run(state):
    return (_run_network if state["kind"] == "network" else _run_conv)(state)


def work(case):
    return (_network_work if case["kind"] == "network" else _conv_work)(case)


def tolerance(case):
    """int8 results are the same bits whatever the order of the integer sums; a float result is a product of a few float
    factors with an exact integer."""
    return {"rel": 1e-6, "max": 1e-5} if case.get("out_type") == "f32" else "exact"
