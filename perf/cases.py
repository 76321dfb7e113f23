"""The work whose speed matters: what a program that uses this library has it do, through its public entry points.

A case is a plain dict.  ``model`` says what runs:

* ``cifar``, ``resnet50``, ``vgg16``, ``yolov3``, ``bert``, ``gpt2``: one network of ``aspen_amd.models`` in a ready
  pool of its own; ``pair``: ResNet-50 and VGG-16 co-scheduled in one pool.  A pass is one inference in the loop of the
  benchmark (reset queue, reset nasm, run, wait, stop) and the read-out of the network's result; with ``serve`` the pass
  also brings a new input from host memory first (``rpool_add_nasm_raw_input``), i.e. it is a whole request.
* ``sgemm``, ``sgemm_static``: the plain matrix product on device pointers (``static``: the one that allocates nothing).

A program loads a model's weights once and then builds graphs for the batches it serves, so the model handle is made at
a network's first case and shared by all later ones; the tile graph, the ready pool and the input belong to a state.
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

from aspen_amd import api, models

# tiles wanted per layer (the tile-count knob of apu_create_nasm) as the benchmark's tuned configurations have it
_TILES = {"cifar": 256, "resnet50": 1536, "vgg16": 1536, "yolov3": 1536, "bert": 192, "gpt2": 384}
_TILES_ONE_IMAGE = {"resnet50": 256, "yolov3": 768}
_STYLE = {"cifar": "he", "resnet50": "he", "vgg16": "he", "yolov3": "yolo", "bert": "gpt", "gpt2": "gpt"}
_SIZE = {"cifar": 32, "resnet50": 224, "vgg16": 224, "yolov3": 416}


def listed():
    return [
        # the smallest network for one image as a whole request: launches, waits and copies, hardly any arithmetic
        dict(name="cifar_b1_request", model="cifar", size=32, batch=1, serve=True),
        # one photograph through the classifier: the latency of some seventy dependency levels
        dict(name="resnet50_b1_request", model="resnet50", size=224, batch=1, serve=True),
        # a batch as a request queue leaves it, no power of two, with its upload
        dict(name="resnet50_b11_request", model="resnet50", size=224, batch=11, serve=True),
        # the benchmark's headline configuration, inputs resident
        dict(name="resnet50_b32", model="resnet50", size=224, batch=32, serve=False),
        # the largest: long unsplit K loops and a weight-streaming head
        dict(name="vgg16_b32", model="vgg16", size=224, batch=32, serve=False),
        # two networks in one pool, the library's co-scheduling
        dict(name="pair_b16", model="pair", size=224, batch=16, serve=False),
        # detection on one frame as a request, all three heads read out
        dict(name="yolov3_b1_request", model="yolov3", size=416, batch=1, serve=True),
        # detection on a batch: leaky convolutions over odd map sizes (13, 26, 52), large results
        dict(name="yolov3_b8", model="yolov3", size=416, batch=8, serve=False),
        # the encoder benchmark configuration
        dict(name="bert_b8_s128", model="bert", batch=8, seq=128, serve=False),
        # an encoder request of uneven length: no tile edge is met
        dict(name="bert_b3_s75_request", model="bert", batch=3, seq=75, serve=True),
        # the decoder's prefill at the benchmark's length, causal attention
        dict(name="gpt2_b4_s512", model="gpt2", batch=4, seq=512, serve=False),
        # the plain product in the shape of an im2col layer, rows and columns off every tile size
        dict(name="sgemm_1000_3137_1152", model="sgemm", M=1000, N=3137, K=1152, act=api.RELU),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any model, any batch and length of the listed range, as a request or in the loop."""
    model = rng.choice(["cifar", "resnet50", "resnet50", "vgg16", "yolov3", "bert", "bert", "gpt2", "pair", "sgemm", "sgemm_static"])
    serve = rng.random() < 0.5
    if model == "cifar":
        return dict(model=model, size=32, batch=_log_int(rng, 1, 256), serve=serve)
    if model == "resnet50":
        return dict(model=model, size=rng.choice([160, 192, 224, 256]), batch=_log_int(rng, 1, 32), serve=serve)
    if model == "vgg16":
        return dict(model=model, size=224, batch=_log_int(rng, 1, 31), serve=serve)
    if model == "yolov3":
        return dict(model=model, size=rng.choice([320, 416]), batch=_log_int(rng, 1, 8), serve=serve)
    if model == "pair":
        return dict(model=model, size=224, batch=_log_int(rng, 1, 16), serve=serve)
    if model in ("bert", "gpt2"):
        seq = _log_int(rng, 16, 512)
        return dict(model=model, batch=_log_int(rng, 1, max(1, min(16, 2048 // seq))), seq=seq, serve=serve)
    if model == "sgemm":
        return dict(model=model, M=_log_int(rng, 64, 4096), N=_log_int(rng, 64, 8192), K=32 * _log_int(rng, 2, 96),
                    act=rng.choice([api.NO_ACTIVATION, api.RELU, api.LEAKY_RELU, api.GELU]))
    # the static product's first operand, padded to whole groups of 128 rows, has to fit its 8 MiB staging array
    K = 32 * _log_int(rng, 1, 64)
    return dict(model=model, M=_log_int(rng, 32, min(2048, (8 << 20) // (4 * K) // 128 * 128)), N=_log_int(rng, 16, 4096), K=K,
                act=rng.choice([api.NO_ACTIVATION, api.RELU, api.GELU]))


def _cfg(model, size):
    if model == "cifar":
        return models.custom_cifar_cfg()
    if model == "resnet50":
        return models.resnet50_cfg(size, size)
    if model == "vgg16":
        return models.vgg16_cfg(size, size)
    if model == "yolov3":
        return models.yolov3_cfg(size)
    return models.bert_cfg() if model == "bert" else models.gpt2_cfg()


_dnns = {}


def _weights(layers, style):
    """The distributions of models.synth_weights, drawn on the GPU (VGG-16 has 138 million of them)."""
    g, out, index = torch.Generator(device="cuda"), [], 0
    g.manual_seed(20240601)

    def normal(shape, std, mean=0.0):
        return (torch.randn(shape, generator=g, device="cuda") * std + mean).cpu().numpy()

    for L in layers:
        t = L["type"]
        if t not in ("conv", "fc", "matmul", "layernorm"):
            continue
        index += 1
        if t == "layernorm":
            w, b = normal((L["M"],), 0.02, 1.0), normal((L["M"],), 0.02)
        elif t == "matmul":
            w, b = normal((L["M"], L["K"]), 0.02), normal((L["M"],), 0.02)
        else:
            shape = (L["C"], L["inC"], L["size"], L["size"]) if t == "conv" else (L["C"], L["inC"], L["inH"], L["inW"])
            gain = 1.0
            if style == "yolo":
                follows = layers[L["idx"] + 1]["type"] if L["idx"] + 1 < len(layers) else None
                gain = {"residual": 0.3, "yolo": 0.1}.get(follows, 1.0)
            w, b = normal(shape, gain * math.sqrt(2.0 / (shape[1] * shape[2] * shape[3]))), normal((shape[0],), 0.01)
        out += [(index, "WEIGHT", w), (index, "BIAS", b)]
    return out


def _dnn(model, size):
    if (model, size) not in _dnns:
        cfg = _cfg(model, size)
        layers = models.parse_cfg(cfg)
        fd, path = tempfile.mkstemp(suffix=".aspen_data", dir="/dev/shm" if os.path.isdir("/dev/shm") else None)
        os.close(fd)
        try:
            models.write_aspen_data(path, _weights(layers, _STYLE[model]))
            _dnns[model, size] = (api.Dnn(cfg, path), layers)
        finally:
            os.unlink(path)
    return _dnns[model, size]


def _input(model, layers, case, seed):
    rng = np.random.default_rng(seed)
    if model in ("bert", "gpt2"):
        x = rng.standard_normal((case["batch"], case["seq"], layers[0]["M"]), dtype=np.float32) * np.float32(0.02)
        if model == "gpt2":         # token embedding + position embedding
            x += np.random.default_rng(7).standard_normal((case["seq"], layers[0]["M"]), dtype=np.float32) * np.float32(0.02)
        return x
    x = rng.random((case["batch"], case["size"], case["size"], 3), dtype=np.float32)
    if model != "yolov3":           # classifiers take pixels normalised per channel
        x = (x - np.array([0.485, 0.456, 0.406], dtype=np.float32)) / np.array([0.229, 0.224, 0.225], dtype=np.float32)
    return np.ascontiguousarray(x, dtype=np.float32)


class _Networks:
    """One ready pool with its networks' graphs and inputs, and the engine group that runs it."""

    def __init__(self, case, seed):
        self.serve = case["serve"]
        self.pool, self.dse, self.nasms, self.inputs, self.results = api.RPool(), api.DseGroup(1), [], [], []
        self.dse.set_rpool(self.pool)
        for k, model in enumerate(["resnet50", "vgg16"] if case["model"] == "pair" else [case["model"]]):
            size = case.get("size", 0)
            dnn, layers = _dnn(model, size)
            tiles = _TILES_ONE_IMAGE.get(model, _TILES[model]) if case["batch"] == 1 else _TILES[model]
            nasm = api.Nasm(dnn, case["batch"], case.get("seq", 0), tiles)
            x = _input(model, layers, case, 2 * seed + k)
            self.pool.add_nasm_raw_input(nasm, x)
            self.nasms.append(nasm)
            self.inputs.append(x)
            heads = [L["idx"] for L in layers if L["type"] == "yolo"]
            self.results.append(heads or [nasm.num_ldata - 1])

    def __del__(self):
        if sys.is_finalizing():
            return
        self.dse.destroy()
        self.pool.destroy()
        for nasm in self.nasms:
            nasm.destroy()


class _Product:
    def __init__(self, case, seed):
        g = torch.Generator(device="cuda")
        g.manual_seed(seed)
        M, N, K = case["M"], case["N"], case["K"]
        self.M, self.N, self.K, self.act, self.static = M, N, K, case["act"], case["model"] == "sgemm_static"
        self.A = torch.randn(M, K, generator=g, device="cuda") * math.sqrt(2.0 / K)
        self.B = torch.rand(N, K, generator=g, device="cuda")
        self.bias = torch.randn(M, generator=g, device="cuda") * 0.01
        self.C = torch.zeros(N, (M + 3) // 4 * 4, device="cuda")


def prepare(case, seed):
    return _Product(case, seed) if case["model"].startswith("sgemm") else _Networks(case, seed)


def run(state):
    if isinstance(state, _Product):
        call = api.lib().aspen_hip_sgemm_static if state.static else api.lib().aspen_hip_sgemm
        rc = call(state.M, state.N, state.K, state.A.data_ptr(), state.K, state.B.data_ptr(), state.K,
                  state.C.data_ptr(), state.C.shape[1], state.bias.data_ptr(), state.act)
        if rc or (state.static and api.lib().aspen_hip_sync()):      # (C is complete after aspen_hip_sync)
            raise RuntimeError(api.lib().aspen_hip_last_error().decode())
        return state.C
    pool, dse = state.pool, state.dse
    if state.serve:
        for nasm, x in zip(state.nasms, state.inputs):
            pool.add_nasm_raw_input(nasm, x)
    else:
        pool.reset_queue()
        for nasm in state.nasms:
            pool.reset_nasm(nasm)
    dse.run()
    for nasm in state.nasms:
        dse.wait(nasm)
    dse.stop()
    return [nasm.layer_output(l) for nasm, ls in zip(state.nasms, state.results) for l in ls]


def _network_work(model, case):
    layers = models.parse_cfg(_cfg(model, case.get("size", 0)))
    B, S = case["batch"], case.get("seq", 0)
    flops = weights = 0
    for L in layers:
        t = L["type"]
        if t == "conv":
            k = L["inC"] * L["size"] ** 2
            flops += 2 * B * L["H"] * L["W"] * L["C"] * k
        elif t == "fc":
            k = L["inC"] * L["inH"] * L["inW"]
            flops += 2 * B * L["C"] * k
        elif t == "matmul":
            k = L["K"]
            flops += 2 * B * S * L["M"] * k
        elif t == "attn_k":         # scores and weighted values; the causal mask leaves half of both
            flops += 4 * B * S * S * L["n_embd"] // (2 if L["masked"] else 1)
            continue
        else:
            continue
        weights += (L["M"] or L["C"]) * (k + 1)
    last, first = layers[-1], layers[0]
    outputs = B * sum(L["C"] * L["H"] * L["W"] for L in layers if L["type"] == "yolo") or B * (S * last["M"] if S else last["C"] * last["H"] * last["W"])
    inputs = B * (S * first["M"] if S else first["C"] * first["H"] * first["W"])
    return flops, 4 * (weights + inputs + outputs)


def work(case):
    """Arithmetic of the contractions and attention; every weight, input and result moved once."""
    if case["model"].startswith("sgemm"):
        M, N, K = case["M"], case["N"], case["K"]
        return {"flops": 2.0 * M * N * K, "bytes": 4.0 * (M * K + N * K + M * N + M)}
    parts = [_network_work(m, case) for m in (["resnet50", "vgg16"] if case["model"] == "pair" else [case["model"]])]
    return {"flops": float(sum(p[0] for p in parts)), "bytes": float(sum(p[1] for p in parts))}


def tolerance(case):
    """32-bit sums through up to a hundred layers.  Graphs with other tile counts and one launch per layer (the same sums
    in another order) differ by up to 3.2e-6 (largest element: 1.3e-5) from each other over these cases, a single
    product from its 64-bit result by up to 1e-6 (8e-6)."""
    return {"rel": 1e-5, "max": 5e-5}
