"""What a user of this package has it do, as measurable cases.

The package multiplies fp16 activations with packed INT4 weights: ``Layer_2_4`` /
``mul_2_4`` on 2:4-sparse weights, its 3-bit variants ``mul_2_4_w3`` and
``mul_2_4_meta3``, the lane-native copy of ``Layer_2_4.to_native()``, and the dense
sibling ``Layer`` / ``mul``.  A case is one pass over a few linear layers:

* ``op``: "sparse" (``Layer_2_4``), "native" (the same after ``to_native()``), "w3",
  "meta3" (the function entry points) or "dense" (``Layer``);
* ``layers``: the layers of the pass in order, as "KxN" texts joined by commas;
* ``M``: activation rows of every layer (tokens in the batch);
* ``group``: quantization group along K, 128 or -1 (one scale per output column);
* ``graph``: True where a serving loop replays a captured HIP graph of the pass (how
  decode steps run, ``bench.py --workload stack``), False for plain eager calls.

The Llama-2-7B and -70B projection shapes are those of ``bench.py`` and the tests.
"""
import math

import torch

from csed499ii_amd import marlin

DEV = "cuda:0"
BLOCK_7B = "4096x12288,4096x4096,4096x22016,11008x4096"
BLOCK_70B = "8192x10240,8192x8192,8192x57344,28672x8192"


def _case(name, op, layers, M, group=128, graph=False):
    return {"name": name, "op": op, "layers": layers, "M": M, "group": group, "graph": graph}


def listed():
    return [
        # One small projection called eagerly for one token: the latency of a call.
        _case("call_o7b_m1", "sparse", "4096x4096", 1),
        # Single-stream decoding: the projections of two 7B decoder layers per replay.
        _case("decode_7b_m1", "sparse", BLOCK_7B + "," + BLOCK_7B, 1, graph=True),
        # The same decode step on the lane-native copies, speculative tokens (3 rows).
        _case("decode_7b_native_m3", "native", BLOCK_7B + "," + BLOCK_7B, 3, graph=True),
        # A small serving batch on a 7B layer with 3-bit values and per-column scales.
        _case("decode_7b_w3_m12", "w3", BLOCK_7B, 12, group=-1, graph=True),
        # Continuous batching: 24 sequences on one 70B decoder layer.
        _case("decode_70b_m24", "sparse", BLOCK_70B, 24, graph=True),
        # A full serving batch of 64 sequences on two 7B decoder layers.
        _case("decode_7b_m64", "sparse", BLOCK_7B + "," + BLOCK_7B, 64, graph=True),
        # Mixed batch (chunked prefill beside decodes, 131 tokens) with 3-bit metadata.
        _case("mixed_7b_meta3_m131", "meta3", BLOCK_7B, 131, graph=True),
        # A prompt of 777 tokens through the unfused gate and up projections of 7B.
        _case("prompt_7b_unfused_m777", "sparse", "4096x11008,4096x11008", 777),
        # A 512-token chunk through a 70B layer's attention projections.
        _case("chunk_70b_attn_m512", "sparse", "8192x10240,8192x8192", 512),
        # A full 4096-token prefill of the widest projection.
        _case("prefill_70b_gate_up_m4096", "sparse", "8192x57344", 4096),
        # The dense INT4 sibling: decoding 4 sequences on a 7B layer, per-group scales.
        _case("dense_decode_7b_m4", "dense", BLOCK_7B, 4, graph=True),
        # The dense sibling on a ragged mid-sized batch, unfused MLP shapes.
        _case("dense_mlp_7b_m200", "dense", "4096x11008,11008x4096", 200),
    ]


def _shapes(case):
    return [tuple(int(x) for x in s.split("x")) for s in case["layers"].split(",")]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["sparse", "sparse", "sparse", "native", "w3", "meta3", "dense", "dense"])
    # 1 to 4096 tokens, odd counts included; decode-sized batches run as graph replays.
    M = _log_int(rng, 1, 4096)
    layers = []
    for _ in range(rng.randint(1, 4)):
        K = 256 * _log_int(rng, 4, 112)  # 1024 .. 28672
        N = 256 * _log_int(rng, 4, 224)  # 1024 .. 57344
        while K * N > 8192 * 57344:
            N = max(1024, N // 2 // 256 * 256)
        layers.append((K, N))
    while len(layers) > 1 and sum(k * n for k, n in layers) * max(M, 256) > 8192 * 57344 * 4096 // 4:
        layers.pop()
    return {"op": op, "layers": ",".join("%dx%d" % s for s in layers), "M": M,
            "group": rng.choice([128, 128, -1]), "graph": M <= 160}


# ---- inputs: what a checkpoint and a batch hold, in plain torch ----


def _weight(K, N, op, group, gen):
    """``(w, s, mask)``: fp16 weight ~ N(0, 0.02) (pruned to the two largest of each 4
    along K unless dense), fp16 scales ``[K/group or 1, N]``."""
    w = (torch.randn((K, N), device=DEV, generator=gen) * 0.02).half()
    mask = None
    if op != "dense":
        a = w.abs().view(K // 4, 4, N)
        i = torch.arange(4, device=DEV).view(4, 1)
        rank = torch.zeros(a.shape, dtype=torch.int8, device=DEV)
        for j in range(4):  # entries that go before: larger, or equal and earlier
            o = a[:, j:j + 1]
            rank += (o > a) | ((o == a) & (i > j))
        mask = (rank < 2).view(K, N)
        w = w * mask
    g = K if group == -1 else group
    s = w.view(K // g, g, N).abs().amax(dim=1) * (2 / (7 if op == "w3" else 15))
    return w, s, mask


def _inputs(case, seed):
    """Weights and activations of the pass, layer by layer (weights made when asked for)."""
    gen = torch.Generator(device=DEV).manual_seed(int(seed) * 1000003 + 17)
    for K, N in _shapes(case):
        w = _weight(K, N, case["op"], case["group"], gen)
        A = torch.randn((case["M"], K), device=DEV, generator=gen).half()
        yield K, N, w, A


class _Linear:
    """What ``pack`` reads of a linear layer: ``weight`` as K x N."""

    def __init__(self, w):
        self.weight = torch.nn.Parameter(w, requires_grad=False)


_STREAM = None


def _capture(step):
    """The pass as a HIP graph, captured after a warm-up on the capturing stream."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    _STREAM.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(_STREAM):
        step()
    torch.cuda.current_stream().wait_stream(_STREAM)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=_STREAM):
        out = step()
    return graph, out


def _call(kind, op, A):
    """One layer's forward on activations ``A``."""
    if kind == "module":
        return op(A)
    mul, B, meta, s, ws, N = op
    C = torch.empty((A.shape[0], N), dtype=A.dtype, device=A.device)
    mul(A, B, meta, C, s, ws)
    return C


def prepare(case, seed):
    calls = []
    op, group = case["op"], case["group"]
    for K, N, (w, s, mask), A in _inputs(case, seed):
        if op == "dense":
            layer = marlin.Layer(K, N, groupsize=group).to(DEV)
            layer.pack(_Linear(w), s)
            calls.append(("module", layer, A))
        elif op in ("sparse", "native"):
            layer = marlin.Layer_2_4(K, N, groupsize=group).to(DEV)
            layer.pack(_Linear(w), s, True, mask=mask)
            calls.append(("module", layer.to_native() if op == "native" else layer, A))
        else:
            ws = torch.zeros(N // 128 * 16, dtype=torch.int32, device=DEV)
            if op == "w3":
                B, sp, meta = marlin.pack_w3(w, s, group, mask)
                mul = marlin.mul_2_4_w3
            else:
                B, sp, meta = marlin.pack_2_4(w, s, group, mask=mask)
                meta = marlin.pack_meta3(meta)
                mul = marlin.mul_2_4_meta3
            calls.append(("function", (mul, B, meta, sp, ws, N), A))
        del w, s, mask
    state = {"calls": calls}
    if case["graph"]:
        state["graph"], state["out"] = _capture(lambda: _step(calls))
    return state


def _step(calls):
    return [_call(kind, op, A) for kind, op, A in calls]


def run(state):
    if "graph" in state:
        state["graph"].replay()
        return state["out"]
    return _step(state["calls"])


def work(case):
    total, flops, M = 0, 0, case["M"]
    for K, N in _shapes(case):
        g = K if case["group"] == -1 else case["group"]
        if case["op"] == "dense":
            weight, kept = K * N // 2, K
        else:
            values = K * N // 2 * (3 if case["op"] == "w3" else 4) // 8
            weight, kept = values + K * N * (3 if case["op"] == "meta3" else 4) // 32, K // 2
        total += weight + K // g * N * 2 + 2 * M * (K + N)
        flops += 2 * M * kept * N
    return {"bytes": total, "flops": flops}


def tolerance(case):
    # fp16 operands and outputs, fp32 sums.  The kernels round code * scale to fp16
    # (group scales) or the sum to fp16 before the scale (per-column ones): 3e-4
    # against 64 bits; two orders of the sums differ by output roundings only, 2e-4.
    return {"rel": 1e-3, "max": 2e-2}


def exact(case, seed):
    outs = []
    op, group = case["op"], case["group"]
    maxq = 7 if op == "w3" else 15
    for K, N, (w, s, mask), A in _inputs(case, seed):
        g = K if group == -1 else group
        C = torch.empty((case["M"], N), dtype=torch.float64, device=DEV)
        A64 = A.double()
        step = max(256, (1 << 27) // K // 256 * 256)  # columns at a time
        for n0 in range(0, N, step):
            ws, ss = w[:, n0:n0 + step], s[:, n0:n0 + step]
            q = torch.round(ws.reshape(K // g, g, -1) / ss.unsqueeze(1)).int() + (maxq + 1) // 2
            q = torch.clamp(q, 0, maxq) - (maxq + 1) // 2
            W = (q.double() * ss.double().unsqueeze(1)).view(K, -1)
            if mask is not None:
                W *= mask[:, n0:n0 + step]
            C[:, n0:n0 + step] = A64 @ W
        outs.append(C)
        del w, s, mask
    return outs
