"""The work whose speed counts: single layers through the C ABI and whole models through Session.

Kinds of case, each a call that a program using this framework makes:

  conv       one fused Conv (+ bias, activation, residual) through spinn_hip_conv, weights packed beforehand
  gemm       one Gemm Y = A op(B) + bias through spinn_hip_gemm
  attention  the detector's attention core: scores = scale * Q^T K, softmax, V P^T (two batched Gemms, one softmax)
  detect     the detector's post-processing: best class per anchor, TopK anchors, gather, TopK over anchor x class
  model      a whole ENNF model through Session (graph replay, input resident in HBM), its logits or decoded head out

Everything is fp32, the framework's only compute type.
"""
import ctypes as C
import math
import os
import tempfile

import numpy as np
import torch

from spinn_amd import models
from spinn_amd import native as N
from spinn_amd.runtime import Session

NONE, RELU, SILU, ADD, ADD_RELU = N.ACT_NONE, N.ACT_RELU, N.ACT_SILU, N.ACT_ADD, N.ACT_ADD_RELU
CLASSES, MAX_DET = 80, 300  # the detector's class count and detections per image


def conv(n, c, hw, oc, k=1, s=1, group=1, act=RELU):
    return {"kind": "conv", "n": n, "c": c, "hw": hw, "oc": oc, "k": k, "s": s, "group": group, "act": act}


def gemm(m, n, k, trans_b=1):
    return {"kind": "gemm", "m": m, "n": n, "k": k, "trans_b": trans_b}


def attention(batch, heads, tokens, key=32, head=64):
    return {"kind": "attention", "batch": batch, "heads": heads, "tokens": tokens, "key": key, "head": head}


def detect(batch, anchors):
    return {"kind": "detect", "batch": batch, "anchors": anchors}


def model(arch, n, hw):
    return {"kind": "model", "arch": arch, "n": n, "hw": hw}


def listed():
    named = [
        # image classification in bulk: the framework's headline workload
        ("resnet101_b32_224", model("resnet101", 32, 224)),
        # one camera frame at a time: latency, some 200 small launches
        ("yolov10n_b1_640", model("yolov10n", 1, 640)),
        # one small layer called by itself: Conv + BN + ReLU on a single image
        ("conv3x3_64_56_b1", conv(1, 64, 56, 64, 3)),
        # the most frequent layers of a bottleneck network at serving batch: reduce ...
        ("conv1x1_1024to256_14_b32", conv(32, 1024, 14, 256)),
        # ... the 3x3 between (also every layer of a 3x3 stack) ...
        ("conv3x3_256_28_b8", conv(8, 256, 28, 256, 3)),
        # ... and the strided 3x3 at a stage's start
        ("conv3x3s2_256_28_b32", conv(32, 256, 28, 256, 3, 2)),
        # a detector layer at a 416 x 416 input: planes of 13 x 13, no multiple of 4
        ("conv1x1_384to256_13_b16", conv(16, 384, 13, 256, act=SILU)),
        # a detector's depthwise layer over its largest head
        ("dw3x3_80_80_b16", conv(16, 80, 80, 80, 3, 1, 80, SILU)),
        # the classifier at batch 32
        ("gemm_32x1000x2048", gemm(32, 1000, 2048)),
        # an ordinary MLP layer over the tokens of a batch
        ("gemm_1568x2048x512", gemm(1568, 2048, 512)),
        # self-attention over a 20 x 20 map for a batch of images
        ("attention_400_b16", attention(16, 2, 400)),
        # detections of a batch of images at 640 x 640
        ("detect_8400_b16", detect(16, 8400)),
    ]
    return [dict(c, name=name) for name, c in named]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def channels(lo, hi):
        c = log_int(lo, hi)  # mostly multiples of 8, as networks have them
        return max(8, (c + 4) // 8 * 8) if rng.random() < 0.85 else c

    while True:
        kind = rng.choice(["pointwise", "pointwise", "conv3", "conv3", "conv3s2", "depthwise", "gemm", "attention",
                           "detect", "model"])
        act = rng.choice([RELU, RELU, SILU, ADD_RELU, NONE])
        if kind == "pointwise":
            case = conv(log_int(1, 32), channels(32, 2048), log_int(7, 80), channels(32, 2048), 1, 1, 1, act)
        elif kind in ("conv3", "conv3s2"):
            s = 2 if kind == "conv3s2" else 1
            case = conv(log_int(1, 32), channels(16, 512), log_int(7, 112), channels(16, 512), 3, s, 1, act)
        elif kind == "depthwise":
            c = channels(32, 512)
            k, s = rng.choice([(3, 1), (3, 1), (3, 2), (7, 1)])
            case = conv(log_int(1, 32), c, log_int(10, 112), c, k, s, c, rng.choice([SILU, RELU, NONE]))
        elif kind == "gemm":
            case = gemm(log_int(1, 4096), log_int(32, 4096), log_int(32, 4096), rng.choice([1, 1, 0]))
        elif kind == "attention":
            case = attention(log_int(1, 16), rng.choice([1, 2, 4]), rng.choice([10, 13, 15, 18, 20, 24]) ** 2)
        elif kind == "detect":
            case = detect(log_int(1, 16), sum((hw // s) ** 2 for hw in [32 * rng.randint(10, 26)] for s in (8, 16, 32)))
        elif rng.random() < 0.5:
            case = model("resnet101", log_int(1, 24), 32 * rng.randint(5, 8))
        else:
            case = model("yolov10n", log_int(1, 16), 32 * rng.randint(10, 20))
        # within the largest listed case
        if case["kind"] != "conv" or (work(case)["flops"] <= 60e9 and work(case)["bytes"] <= 600e6):
            return case


# ---- sizes ----

def _out(hw, k, s):
    return (hw + 2 * (k // 2) - k) // s + 1


def _onnx_work(g):
    """Multiply-adds of the Conv, Gemm and MatMul nodes; bytes of the input, weights and output."""
    flops = 0.0
    for nd in g.nodes:
        if nd.op_type == "Conv":
            oc, cg, kh, kw = g.dims(nd.inputs[1])
            n, _, oh, ow = g.dims(nd.outputs[0])
            flops += 2.0 * n * oc * oh * ow * cg * kh * kw
        elif nd.op_type in ("Gemm", "MatMul"):
            flops += 2.0 * float(np.prod(g.dims(nd.outputs[0]))) * g.dims(nd.inputs[0])[-1]
    elems = sum(v.size for v in g.initializers.values())
    elems += sum(float(np.prod(g.dims(t))) for t in list(g.inputs) + list(g.outputs))
    return {"bytes": 4.0 * elems, "flops": flops}


def work(case):
    kind = case["kind"]
    if kind == "conv":
        n, c, hw, oc, k, g = (case[q] for q in ("n", "c", "hw", "oc", "k", "group"))
        o = _out(hw, k, case["s"])
        y = n * oc * o * o
        res = y if case["act"] in (ADD, ADD_RELU) else 0
        return {"bytes": 4.0 * (n * c * hw * hw + oc * (c // g) * k * k + oc + y + res), "flops": 2.0 * y * (c // g) * k * k}
    if kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 4.0 * (m * k + n * k + n + m * n), "flops": 2.0 * m * n * k}
    if kind == "attention":
        bh, t, kd, hd = case["batch"] * case["heads"], case["tokens"], case["key"], case["head"]
        return {"bytes": 4.0 * bh * t * (2 * kd + 2 * hd), "flops": 2.0 * bh * t * t * (kd + hd)}
    if kind == "detect":
        b, a = case["batch"], case["anchors"]
        return {"bytes": 4.0 * b * (a * (CLASSES + 4) + MAX_DET * 6), "flops": 1.0 * b * a * CLASSES}
    return _onnx_work(_graph(case)[0].onnx)


# ---- inputs ----

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _graph(case, seed=0):
    if case["arch"] == "resnet101":
        return models.resnet(case["n"], seed, models.RESNET101_BLOCKS, case["hw"])
    return models.yolov10n(case["n"], seed, case["hw"])


class _Output:
    """A session's output in HBM as torch sees it. The tensor made from this object holds on to it,
    and so to the session whose memory it is, however long the tensor lives."""

    def __init__(self, session):
        shape, ptr = session.dims(session.output_id), session.tensor(session.output_id).data
        self.session = session
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (ptr, False), "version": 2}


def _conv_operands(case, seed):
    """Activations as the layer before leaves them (after ReLU or SiLU), Kaiming weights, BN-sized biases."""
    g = _gen(seed)
    n, c, hw, oc, k, group, act = (case[q] for q in ("n", "c", "hw", "oc", "k", "group", "act"))
    o = _out(hw, k, case["s"])
    x = torch.randn((n, c, hw, hw), generator=g, device="cuda")
    x = torch.nn.functional.silu(x) if act == SILU else torch.relu(x)
    w = torch.randn((oc, c // group, k, k), generator=g, device="cuda") * math.sqrt(2.0 / (c // group * k * k))
    b = torch.randn((oc,), generator=g, device="cuda") * 0.1
    r = torch.relu(torch.randn((n, oc, o, o), generator=g, device="cuda")) if act in (ADD, ADD_RELU) else None
    return x, w, b, r


def _gemm_operands(case, seed):
    g = _gen(seed)
    m, n, k = case["m"], case["n"], case["k"]
    a = torch.relu(torch.randn((m, k), generator=g, device="cuda"))
    b = torch.randn((n, k) if case["trans_b"] else (k, n), generator=g, device="cuda") / math.sqrt(k)
    c = torch.randn((n,), generator=g, device="cuda") * 0.01
    return a, b, c


def _attention_operands(case, seed):
    g = _gen(seed)
    bh, t = case["batch"] * case["heads"], case["tokens"]
    return [torch.randn((bh, d, t), generator=g, device="cuda") for d in (case["key"], case["key"], case["head"])]


def _detect_operands(case, seed):
    """Decoded boxes in pixels and class scores, most of them low."""
    g = _gen(seed)
    b, a = case["batch"], case["anchors"]
    boxes = torch.rand((b, a, 4), generator=g, device="cuda") * 640
    scores = torch.sigmoid(torch.randn((b, a, CLASSES), generator=g, device="cuda") * 1.5 - 5)
    return boxes, scores


def _model_input(case, seed):
    rng = np.random.default_rng(seed)
    lo = -1.0 if case["arch"] == "resnet101" else 0.0
    return rng.uniform(lo, 1.0, (case["n"], 3, case["hw"], case["hw"])).astype(np.float32)


def _workspace(nbytes):
    return torch.empty(max(nbytes // 4, 1), device="cuda") if nbytes else None


def _gemm_desc(m, n, k, trans_a, trans_b, c_mode, alpha=1.0, batch=1, sa=0, sb=0, sy=0):
    return N.GemmDesc(m, n, k, trans_a, trans_b, c_mode, alpha, 1.0, batch, 0, sa, sb, sy)


def prepare(case, seed):
    L = N.lib()
    N.check(L.spinn_hip_init(0), "spinn_hip_init")
    st = {"kind": case["kind"], "L": L}
    kind = case["kind"]
    if kind == "conv":
        k, s = case["k"], case["s"]
        o = _out(case["hw"], k, s)
        d = N.ConvDesc(case["n"], case["c"], case["hw"], case["hw"], case["oc"], o, o, k, k, s, s, k // 2, k // 2,
                       case["group"], case["act"], N.ALGO_AUTO, 0)
        x, w, b, r = _conv_operands(case, seed)
        y = torch.empty((case["n"], case["oc"], o, o), device="cuda")
        psz = L.spinn_hip_conv_packed_size(C.byref(d))
        pk = torch.empty(psz // 4, device="cuda") if psz else None
        if psz:
            N.check(L.spinn_hip_conv_pack_weights(C.byref(d), N.ptr(w), N.ptr(pk), None), "pack")
        wsz = L.spinn_hip_conv_workspace_size(C.byref(d))
        ws = _workspace(wsz)
        st["keep"] = (x, w, pk, b, r, ws)
        st["y"] = y
        st["args"] = (C.byref(d), N.ptr(x), N.ptr(w), N.ptr(pk), N.ptr(b), N.ptr(r), N.ptr(y), N.ptr(ws), wsz, None)
    elif kind == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        d = _gemm_desc(m, n, k, 0, case["trans_b"], 1)
        a, b, c = _gemm_operands(case, seed)
        y = torch.empty((m, n), device="cuda")
        wsz = L.spinn_hip_gemm_workspace_size(C.byref(d))
        ws = _workspace(wsz)
        st["keep"] = (a, b, c, ws)
        st["y"] = y
        st["args"] = (C.byref(d), N.ptr(a), N.ptr(b), N.ptr(c), N.ptr(y), N.ptr(ws), wsz, None)
    elif kind == "attention":
        bh, t, kd, hd = case["batch"] * case["heads"], case["tokens"], case["key"], case["head"]
        q, k, v = _attention_operands(case, seed)
        s = torch.empty((bh, t, t), device="cuda")
        p = torch.empty((bh, t, t), device="cuda")
        y = torch.empty((bh, hd, t), device="cuda")
        ds = _gemm_desc(t, t, kd, 1, 0, 0, kd ** -0.5, bh, kd * t, kd * t, t * t)
        dv = _gemm_desc(hd, t, t, 0, 1, 0, 1.0, bh, hd * t, t * t, hd * t)
        wsz = max(L.spinn_hip_gemm_workspace_size(C.byref(x)) for x in (ds, dv))
        ws = _workspace(wsz)
        st["keep"] = (q, k, v, s, p, ws)
        st["y"] = y
        st["scores"] = (C.byref(ds), N.ptr(q), N.ptr(k), None, N.ptr(s), N.ptr(ws), wsz, None)
        st["softmax"] = (bh * t, t, 1, N.ptr(s), N.ptr(p), None)
        st["values"] = (C.byref(dv), N.ptr(v), N.ptr(p), None, N.ptr(y), N.ptr(ws), wsz, None)
    elif kind == "detect":
        b, a = case["batch"], case["anchors"]
        boxes, scores = _detect_operands(case, seed)
        best = torch.empty((b, a), device="cuda")
        v1, i1 = torch.empty((b, MAX_DET), device="cuda"), torch.empty((b, MAX_DET), device="cuda", dtype=torch.int64)
        i1b = torch.empty((b, MAX_DET, 4), device="cuda", dtype=torch.int64)
        i1s = torch.empty((b, MAX_DET, CLASSES), device="cuda", dtype=torch.int64)
        box = torch.empty((b, MAX_DET, 4), device="cuda")
        sc = torch.empty((b, MAX_DET, CLASSES), device="cuda")
        v2, i2 = torch.empty((b, MAX_DET), device="cuda"), torch.empty((b, MAX_DET), device="cuda", dtype=torch.int64)

        def dims(*v):
            return (C.c_int64 * 8)(*v)

        def tile(src, dst, cols):
            return (3, dims(b, MAX_DET, 1), dims(b, MAX_DET, cols), 8, N.ptr(src), N.ptr(dst), None)

        def gather(cols):
            return N.GatherDesc(3, 1, 7, 0, dims(b, a, cols), dims(b, MAX_DET, cols))

        gb, gs = gather(4), gather(CLASSES)
        st["keep"] = (boxes, scores, best, v1, i1, i1b, i1s)
        st["y"] = {"boxes": box, "scores": v2, "indices": i2}
        st["steps"] = [
            (L.spinn_hip_reduce_max, (b * a, CLASSES, N.ptr(scores), N.ptr(best), None)),
            (L.spinn_hip_topk, (b, a, MAX_DET, N.ptr(best), N.ptr(v1), N.ptr(i1), None)),
            (L.spinn_hip_tile, tile(i1, i1b, 4)),
            (L.spinn_hip_gather_elements, (C.byref(gb), N.ptr(boxes), N.ptr(i1b), N.ptr(box), None)),
            (L.spinn_hip_tile, tile(i1, i1s, CLASSES)),
            (L.spinn_hip_gather_elements, (C.byref(gs), N.ptr(scores), N.ptr(i1s), N.ptr(sc), None)),
            (L.spinn_hip_topk, (b, MAX_DET * CLASSES, MAX_DET, N.ptr(sc), N.ptr(v2), N.ptr(i2), None)),
        ]
        st["keep"] += (sc,)
    else:
        g, _ = _graph(case)
        with tempfile.TemporaryDirectory() as td:
            path = g.write(os.path.join(td, "model.ennf"))
            sess = Session(path, graph=True)
        sess.upload_input(_model_input(case, seed))
        st["session"] = sess
        st["y"] = torch.as_tensor(_Output(sess), device="cuda")
    torch.cuda.synchronize()  # what is above ran on torch's and the library's own streams
    return st


def run(st):
    L, kind = st["L"], st["kind"]
    if kind == "conv":
        N.check(L.spinn_hip_conv(*st["args"]), "spinn_hip_conv")
    elif kind == "gemm":
        N.check(L.spinn_hip_gemm(*st["args"]), "spinn_hip_gemm")
    elif kind == "attention":
        N.check(L.spinn_hip_gemm(*st["scores"]), "spinn_hip_gemm")
        N.check(L.spinn_hip_softmax(*st["softmax"]), "spinn_hip_softmax")
        N.check(L.spinn_hip_gemm(*st["values"]), "spinn_hip_gemm")
    elif kind == "detect":
        for f, args in st["steps"]:
            N.check(f(*args), "detector step")
    else:
        st["session"].run_resident()
    return st["y"]


# ---- what the results are ----

def tolerance(case):
    """About four times the largest error against 64 bits that the path shows over these ranges:
    2.6e-6 for the 3x3 layers that run as Winograd, 4e-7 for other layers, 9e-7 for whole models."""
    if case["kind"] == "detect":
        return "exact"  # comparisons, sorts and copies
    return {"rel": 1e-5, "max": 4e-4}


def _conv64(x, w, b, stride, pad, group):
    n, c, h, _ = x.shape
    oc, cg, k, _ = w.shape
    ow = (x.shape[3] + 2 * pad - k) // stride + 1
    oh = (h + 2 * pad - k) // stride + 1
    out = []
    step = max(1, int(2e9 // (8 * c * k * k * oh * ow)))  # images at a time
    for i in range(0, n, step):
        u = torch.nn.functional.unfold(x[i:i + step], k, padding=pad, stride=stride)
        m = u.shape[0]
        u = u.reshape(m, group, cg * k * k, oh * ow)
        if cg * k * k <= 64 and group > 1:
            y = (w.reshape(1, group, oc // group, cg * k * k, 1) * u.unsqueeze(2)).sum(3)
        else:
            y = torch.matmul(w.reshape(1, group, oc // group, cg * k * k), u)
        out.append(y.reshape(m, oc, oh, ow))
    y = torch.cat(out)
    return y if b is None else y + b.reshape(1, -1, 1, 1)


def _onnx64(g, feeds):
    """A graph's outputs in 64 bits, node by node."""
    v = {k: torch.from_numpy(a).cuda() for k, a in g.initializers.items()}
    v.update(feeds)
    v = {k: t.double() if t.is_floating_point() else t for k, t in v.items()}
    last = {t: i for i, nd in enumerate(g.nodes) for t in nd.inputs}
    for i, nd in enumerate(g.nodes):
        x = [v.get(t) for t in nd.inputs]
        a, op = nd.attrs, nd.op_type
        if op == "Conv":
            y = _conv64(x[0], x[1], x[2] if len(x) > 2 else None, a["strides"][0], a["pads"][0], a["group"])
        elif op == "BatchNormalization":
            s, b, m, var = (t.reshape(1, -1, 1, 1) for t in x[1:5])
            y = (x[0] - m) / torch.sqrt(var + a["epsilon"]) * s + b
        elif op == "Relu":
            y = torch.relu(x[0])
        elif op == "Sigmoid":
            y = torch.sigmoid(x[0])
        elif op in ("Add", "Sub", "Mul"):
            y = {"Add": torch.add, "Sub": torch.sub, "Mul": torch.mul}[op](x[0], x[1])
        elif op == "MaxPool":
            k, p, s = a["kernel_shape"][0], a["pads"][0], a["strides"][0]
            t = torch.nn.functional.pad(x[0], (p, p, p, p), value=-math.inf)
            y = t.unfold(2, k, s).unfold(3, k, s).amax((-1, -2))
        elif op == "ReduceMean":
            y = x[0].mean(tuple(a["axes"]), keepdim=True)
        elif op == "Reshape":
            y = x[0].reshape(g.dims(nd.outputs[0]))
        elif op == "Gemm":
            y = torch.matmul(x[0], x[1].t() if a.get("transB") else x[1]) + x[2]
        elif op == "MatMul":
            y = torch.matmul(x[0].contiguous(), x[1].contiguous())
        elif op == "Softmax":
            y = torch.softmax(x[0], a["axis"])
        elif op == "Transpose":
            y = x[0].permute(a["perm"])
        elif op == "Concat":
            y = torch.cat(x, a["axis"])
        elif op == "Split":
            for t, part in zip(nd.outputs, torch.split(x[0], [g.dims(t)[a["axis"]] for t in nd.outputs], a["axis"])):
                v[t] = part
            y = None
        elif op == "Resize":
            y = x[0].repeat_interleave(2, 2).repeat_interleave(2, 3)
        else:
            raise ValueError(op)
        if y is not None:
            v[nd.outputs[0]] = y
        for t in nd.inputs:
            if last[t] == i and t not in g.outputs:
                v.pop(t, None)
    return v[next(iter(g.outputs))]


def exact(case, seed):
    kind = case["kind"]
    if kind == "conv":
        x, w, b, r = (None if t is None else t.double() for t in _conv_operands(case, seed))
        y = _conv64(x, w, b, case["s"], case["k"] // 2, case["group"])
        if r is not None:
            y = y + r
        if case["act"] in (RELU, ADD_RELU):
            y = torch.relu(y)
        elif case["act"] == SILU:
            y = torch.nn.functional.silu(y)
        return y
    if kind == "gemm":
        a, b, c = (t.double() for t in _gemm_operands(case, seed))
        return torch.matmul(a, b.t() if case["trans_b"] else b) + c
    if kind == "attention":
        q, k, v = (t.double() for t in _attention_operands(case, seed))
        s = torch.matmul(q.transpose(1, 2).contiguous(), k) * case["key"] ** -0.5
        return torch.matmul(v, torch.softmax(s, -1).transpose(1, 2).contiguous())
    if kind == "detect":
        boxes, scores = _detect_operands(case, seed)
        i1 = torch.sort(scores.amax(-1), dim=-1, descending=True, stable=True)[1][:, :MAX_DET, None]
        box = boxes.gather(1, i1.expand(-1, -1, 4))
        sc = scores.gather(1, i1.expand(-1, -1, CLASSES)).reshape(case["batch"], -1)
        v2, i2 = torch.sort(sc, dim=-1, descending=True, stable=True)
        return {"boxes": box.double(), "scores": v2[:, :MAX_DET].double(), "indices": i2[:, :MAX_DET]}
    g, _ = _graph(case)
    return _onnx64(g.onnx, {next(iter(g.onnx.inputs)): torch.from_numpy(_model_input(case, seed)).cuda()})
