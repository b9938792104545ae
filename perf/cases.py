"""The work that users of this framework have it do, as measurable cases.

Three ways into the framework are in use, and all are covered:

* whole int8 models through Net / Extractor (images in, class scores out), from one image to a large batch, with the
  images in host memory, already resident on the GPU, or replayed as a recorded pass;
* the int8 Gemm of a linear layer: per-row quantisation of the fp32 activations, then the int8 product with its scales and bias;
* block-quantised weights (4, 6 or 8 bits): all projections of a decoder layer, and a whole self-attention layer with its
  key / value cache, each from one token (decoding) to many (prefill).

listed() names the cases that are always measured, draw() gives more of the same ranges."""
import ctypes as C
import math

import numpy as np
import torch

import ncnn_amd
from ncnn_amd import host, zoo
from ncnn_amd.hip import check, lib

PIXELS = 128 * 224 * 224                # the largest batch of images, in pixels
GEMM_OPS = 2 * 4096 ** 3                # the largest int8 Gemm
DECODER_OPS = 2 * 512 * (4 * 4096 ** 2 + 3 * 4096 * 11008)  # the largest decoder-layer pass
ATTENTION_OPS = 8 * 1500 * 1024 ** 2 + 4 * 1500 ** 2 * 1024  # the largest self-attention layer


def listed():
    return [
        # one camera image, classified as it arrives: latency from host memory to host memory
        {"name": "resnet50_one_image", "kind": "net", "model": "resnet50", "batch": 1, "h": 224, "w": 224, "images": "host"},
        # a few images of an odd size through the light model: crops of a detector, resolution as it comes
        {"name": "mobilenetv2_odd_images", "kind": "net", "model": "mobilenetv2", "batch": 3, "h": 193, "w": 257, "images": "host"},
        # a serving batch that lies in HBM already
        {"name": "resnet50_batch16", "kind": "net", "model": "resnet50", "batch": 16, "h": 224, "w": 224, "images": "resident"},
        {"name": "mobilenetv2_batch32", "kind": "net", "model": "mobilenetv2", "batch": 32, "h": 224, "w": 224, "images": "resident"},
        # an offline job over a large set of images in host memory
        {"name": "resnet50_batch128", "kind": "net", "model": "resnet50", "batch": 128, "h": 224, "w": 224, "images": "host"},
        # a large linear layer, every size a power of two
        {"name": "gemm_4096", "kind": "gemm", "m": 4096, "n": 4096, "k": 4096, "scales": "per_column"},
        # a linear layer over a ragged number of tokens, with sizes that fit no tile
        {"name": "gemm_ragged", "kind": "gemm", "m": 1501, "n": 1000, "k": 2008, "scales": "per_tensor"},
        # one token through the projections of a 7B-class decoder layer
        {"name": "decoder_one_token", "kind": "decoder", "rows": 1, "hidden": 4096, "inter": 11008, "bits": 8, "block": 64, "act": "fp16"},
        # a step of 48 sequences decoded together, 4-bit weights
        {"name": "decoder_48_sequences", "kind": "decoder", "rows": 48, "hidden": 4096, "inter": 11008, "bits": 4, "block": 64, "act": "fp16"},
        # a prompt of 512 tokens, fp32 activations as the Gemm layer takes them
        {"name": "decoder_prefill_512", "kind": "decoder", "rows": 512, "hidden": 4096, "inter": 11008, "bits": 8, "block": 64, "act": "fp32"},
        # self-attention layers: one token on a cache, and a whole sequence
        {"name": "attention_one_token", "kind": "attention", "heads": 32, "head_dim": 128, "src": 1, "past": 1499, "bits": 8, "block": 64},
        {"name": "attention_1500_tokens", "kind": "attention", "heads": 16, "head_dim": 64, "src": 1500, "past": 0, "bits": 8, "block": 64},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("net", "net", "gemm", "gemm", "decoder", "decoder", "attention"))
    if kind == "net":
        h, w = rng.randint(128, 320), rng.randint(128, 320)
        batch = min(_log(rng, 1, 128), PIXELS // (h * w))
        return {"kind": kind, "model": rng.choice(("resnet50", "mobilenetv2")), "batch": batch, "h": h, "w": w,
                "images": rng.choice(("host", "host", "resident", "recorded"))}
    if kind == "gemm":
        n, k = _log(rng, 256, 8192), _log(rng, 256, 8192)
        if rng.random() < 0.7:  # most layers are a multiple of something; the rest is as ragged as it comes
            n, k = n // 8 * 8, k // 64 * 64
        m = max(1, min(_log(rng, 1, 4096), GEMM_OPS // (2 * n * k)))
        return {"kind": kind, "m": m, "n": n, "k": k, "scales": rng.choice(("per_tensor", "per_column"))}
    if kind == "decoder":
        hidden = _log(rng, 1024, 5120) // 64 * 64
        inter = int(hidden * rng.uniform(2.5, 3.0)) // 16 * 16
        act = rng.choice(("fp16", "fp32"))
        rows = _log(rng, 1, 128 if act == "fp16" else 1024)
        rows = max(1, min(rows, DECODER_OPS // (2 * (4 * hidden ** 2 + 3 * hidden * inter))))
        return {"kind": kind, "rows": rows, "hidden": hidden, "inter": inter, "bits": rng.choice((4, 6, 8)), "block": rng.choice((32, 64, 128)), "act": act}
    heads, head_dim = rng.randint(4, 32), rng.choice((32, 64, 96, 128))
    embed = heads * head_dim
    src = _log(rng, 1, 1500)
    past = rng.choice((0, _log(rng, 64, 4096)))
    while 8 * src * embed ** 2 + 4 * src * (past + src) * embed > ATTENTION_OPS:
        src, past = (src + 1) // 2, past // 2
    return {"kind": "attention", "heads": heads, "head_dim": head_dim, "src": src, "past": past, "bits": rng.choice((4, 8)), "block": rng.choice((32, 64))}


# ---------------------------------------------------------------------------------------------------- what a program keeps
_models, _runtimes, _weights = {}, [], {}
SCORES = {"resnet50": "fc1000", "mobilenetv2": "fc"}  # the blob that a classifier ranks: the scores before the softmax


def _model(name):
    """The model as a program holds it: loaded once, used for every image."""
    if name not in _models:
        graph, param, blob, _ = zoo.build(name, n_calib=1)
        net = None
        if torch.cuda.is_available():
            net = host.Net()
            net.set_use_hip_compute(True)
            if net.register_int8_layers() != 0 or net.load_param_mem(param) != 0 or net.load_model_mem(blob) != 0:
                raise RuntimeError("the generated %s model does not load" % name)
        _models[name] = graph, net
    return _models[name]


def _runtime():
    if not _runtimes:
        _runtimes.append(ncnn_amd.Runtime(0))
    return _runtimes[0]


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _ptr(t):
    return None if t is None else C.c_void_p(t.data_ptr())


def _block_quantised(n, k, bits, block, seed):
    """N(0, 1/sqrt(k)) weights in the .bin layout of the block-quantised layers, repacked once for the kernels, on the GPU."""
    qmax = (1 << (bits - 1)) - 1
    blocks = -(-k // block)
    w = torch.zeros(n, blocks * block, device="cuda")
    w[:, :k] = torch.randn(n, k, generator=_generator(seed), device="cuda") / math.sqrt(k)
    w = w.view(n, blocks, block)
    scales = qmax / w.abs().amax(dim=2)
    q = (w * scales[:, :, None]).round().clamp(-qmax, qmax).to(torch.int32).view(n, -1)[:, :k] & ((1 << bits) - 1)
    if bits == 4:
        q = q[:, 0::2] | q[:, 1::2] << 4
    elif bits == 6:
        word = q[:, 0::4] | q[:, 1::4] << 6 | q[:, 2::4] << 12 | q[:, 3::4] << 18
        q = torch.stack([word & 255, word >> 8 & 255, word >> 16], dim=2).view(n, -1)
    packed, descales = _runtime().blockquant_pack(q.to(torch.uint8).cpu().numpy(), scales.cpu().numpy(), block, bits=bits, k=k)
    return torch.from_numpy(packed).cuda(), torch.from_numpy(descales).cuda()


def _matrices(key, shapes, bits, block):
    """One layer's packed weights, an own copy for every caller: a model's layers do not share theirs."""
    if key not in _weights:
        _weights.clear()
        _weights[key] = [_block_quantised(n, k, bits, block, 100 + i) for i, (n, k) in enumerate(shapes)]
    return [(w.clone(), d.clone()) for w, d in _weights[key]]


# ---------------------------------------------------------------------------------------------------- prepare
def prepare(case, seed):
    return {"net": _prepare_net, "gemm": _prepare_gemm, "decoder": _prepare_decoder, "attention": _prepare_attention}[case["kind"]](case, seed)


def _prepare_net(case, seed):
    _, net = _model(case["model"])
    x = np.random.default_rng(seed).random((case["batch"], 3, case["h"], case["w"]), dtype=np.float32)
    state = {"kind": "net", "images": case["images"], "net": net, "x": x, "scores": SCORES[case["model"]]}
    if case["images"] != "host":
        state["resident"] = net.upload(x)
    if case["images"] == "recorded":
        state["graph"] = net.record("data", state["resident"], state["scores"])
    return state


def _prepare_gemm(case, seed):
    m, n, k = case["m"], case["n"], case["k"]
    gen = _generator(seed)
    a = torch.randn(m, k, generator=gen, device="cuda")
    b = torch.randn(n, k, generator=gen, device="cuda") * 0.02
    sb = (127 / (b.abs().amax(dim=1) if case["scales"] == "per_column" else b.abs().max().view(1))).contiguous()
    bq = (b * sb[:, None]).round().clamp(-127, 127).to(torch.int8)
    bias = torch.randn(n, generator=gen, device="cuda")
    aq = torch.empty(m, k, dtype=torch.int8, device="cuda")
    sa = torch.empty(m, device="cuda")
    out = torch.empty(m, n, device="cuda")
    st = _runtime().stream
    # large layers keep B in the tiled layout, as the Gemm layer does when its weights are uploaded
    tiled = m % 256 == 0 and n % 256 == 0 and k % 64 == 0 and k <= 8192 and m * n >= 256 * 256 * 128
    if tiled:
        bt = torch.empty(n * k, dtype=torch.int8, device="cuda")
        torch.cuda.synchronize()
        check(lib().ncnnhip_gemm_int8_tile_operand(_ptr(bq), k, n, k, 1, _ptr(bt), st))
        calls = [(lib().ncnnhip_gemm_quantize_rows_tiled, (_ptr(a), k, m, k, _ptr(aq), _ptr(sa), st)),
                 (lib().ncnnhip_gemm_int8_tiled, (_ptr(aq), _ptr(bt), m, n, k, _ptr(sa), _ptr(sb), sb.numel(), _ptr(bias), 4, 1.0, 1.0, _ptr(out), n, st))]
        keep = (a, bt, sb, bias, aq, sa)
    else:
        calls = [(lib().ncnnhip_gemm_quantize_rows, (_ptr(a), k, m, k, _ptr(aq), k, _ptr(sa), st)),
                 (lib().ncnnhip_gemm_int8, (_ptr(aq), k, _ptr(bq), k, m, n, k, _ptr(sa), _ptr(sb), sb.numel(), _ptr(bias), 4, 1.0, 1.0, 0, _ptr(out), n, None, st))]
        keep = (a, bq, sb, bias, aq, sa)
    return {"kind": "calls", "calls": calls, "outputs": [out], "keep": keep}


def _decoder_shapes(case):
    h, i = case["hidden"], case["inter"]
    return [(h, h)] * 4 + [(i, h)] * 2 + [(h, i)]  # q, k, v, output; gate, up; down


def _many_rows(rows, k):
    """Whether the Gemm layer takes the entry point for many fp32 rows, which wants a workspace."""
    return rows >= 5 or (rows >= 3 and k > 4096)


def _workspace(rows, k):
    size = C.c_size_t()
    check(lib().ncnnhip_gemm_blockquant_packed_rows_workspace_bytes(rows, k, C.byref(size)))
    return torch.empty(max(size.value, 4), dtype=torch.uint8, device="cuda")


def _prepare_decoder(case, seed):
    rows, bits, block, half = case["rows"], case["bits"], case["block"], case["act"] == "fp16"
    shapes = _decoder_shapes(case)
    weights = _matrices(tuple(shapes) + (bits, block), shapes, bits, block)
    gen = _generator(seed)
    st, dt, esize = _runtime().stream, torch.float16 if half else torch.float32, 2 if half else 4
    outputs = [torch.empty(rows, n, device="cuda") for n, _ in shapes]
    calls, keep = [], [weights]
    # the matrices that read the same rows go together where one call takes them
    for group in ((0, 1, 2), (3,), (4, 5), (6,)):
        k = shapes[group[0]][1]
        a = torch.randn(rows, k, generator=gen, device="cuda").to(dt)
        keep.append(a)
        if not half and _many_rows(rows, k):
            ws = _workspace(rows, k)
            keep.append(ws)
            for g in group:
                n = shapes[g][0]
                calls.append((lib().ncnnhip_gemm_blockquant_packed_rows, (_ptr(a), k, rows, n, k, _ptr(weights[g][0]), _ptr(weights[g][1]), bits, block, None, None, -1,
                                                                          1.0, 1.0, _ptr(outputs[g]), n, _ptr(ws), ws.numel(), st)))
        elif len(group) > 1:
            count = len(group)
            pointers, ints, floats, sizes = C.c_void_p * count, C.c_int * count, C.c_float * count, C.c_size_t * count
            arrays = (ints(*[shapes[g][0] for g in group]), pointers(*[weights[g][0].data_ptr() for g in group]), pointers(*[weights[g][1].data_ptr() for g in group]))
            tail = (pointers(), ints(*[-1] * count), floats(*[1.0] * count), floats(*[1.0] * count), pointers(*[outputs[g].data_ptr() for g in group]),
                    sizes(*[shapes[g][0] for g in group]))
            calls.append((lib().ncnnhip_gemm_blockquant_packed_multi, (_ptr(a), esize, k, rows, k, count) + arrays + (bits, block, None) + tail + (st,)))
        else:
            g = group[0]
            n = shapes[g][0]
            w, d = _ptr(weights[g][0]), _ptr(weights[g][1])
            if half:
                calls.append((lib().ncnnhip_gemm_blockquant_packed_f16a, (_ptr(a), k, rows, n, k, w, d, bits, block, None, -1, 1.0, 1.0, _ptr(outputs[g]), n, st)))
            else:
                calls.append((lib().ncnnhip_gemm_blockquant_packed, (_ptr(a), k, rows, n, k, w, d, bits, block, None, None, -1, 1.0, 1.0, _ptr(outputs[g]), n, st)))
    return {"kind": "calls", "calls": calls, "outputs": outputs, "keep": keep}


def _prepare_attention(case, seed):
    heads, hd, src, past, bits, block = (case[v] for v in ("heads", "head_dim", "src", "past", "bits", "block"))
    embed, dst = heads * hd, past + src
    shapes = [(3 * embed, embed), (embed, embed)]
    weights = _matrices(tuple(shapes) + (bits, block), shapes, bits, block)
    gen = _generator(seed)
    st = _runtime().stream
    x = torch.randn(src, embed, generator=gen, device="cuda")
    biases = [(torch.rand(n, generator=gen, device="cuda") - 0.5) * 0.2 for n, _ in shapes]
    kt, vt = (torch.randn(embed, dst, generator=gen, device="cuda") for _ in range(2))
    qkv, context, out = (torch.empty(src, n, device="cuda") for n in (3 * embed, embed, embed))
    size = C.c_size_t()
    check(lib().ncnnhip_attention_workspace_bytes(heads, hd, src, dst, C.byref(size)))
    ws = torch.empty(max(size.value, 4), dtype=torch.uint8, device="cuda")
    rows_ws = _workspace(src, embed) if _many_rows(src, embed) else None

    def project(a, g, to):
        n, k = shapes[g]
        args = (_ptr(a), k, src, n, k, _ptr(weights[g][0]), _ptr(weights[g][1]), bits, block, None, _ptr(biases[g]), 4, 1.0, 1.0, _ptr(to), n)
        if rows_ws is not None:
            return lib().ncnnhip_gemm_blockquant_packed_rows, args + (_ptr(rows_ws), rows_ws.numel(), st)
        return lib().ncnnhip_gemm_blockquant_packed, args + (st,)

    calls = [project(x, 0, qkv),
             (lib().ncnnhip_attention_f32_append, (_ptr(qkv), 3 * embed, 1.0 / math.sqrt(hd), _ptr(kt), _ptr(vt), dst, past, None, 0, heads, hd, src, _ptr(context), _ptr(ws),
                                                   size.value, st)),
             project(context, 1, out)]
    return {"kind": "calls", "calls": calls, "outputs": [out, kt, vt], "keep": (weights, x, biases, qkv, context, ws, rows_ws)}


# ---------------------------------------------------------------------------------------------------- run
def run(state):
    if state["kind"] == "calls":
        for function, arguments in state["calls"]:
            check(function(*arguments))
        return state["outputs"]
    net = state["net"]
    if state["images"] == "recorded":
        graph = state["graph"]
        graph.update_input(state["x"])
        graph.launch()
        return graph.output().to_numpy()
    ex = net.create_extractor()
    if state["images"] == "host":
        ex.input("data", state["x"])
    else:
        ex.input_resident("data", state["resident"])
    return ex.extract(state["scores"])


# ---------------------------------------------------------------------------------------------------- work, tolerance
def work(case):
    if case["kind"] == "net":
        graph, _ = _model(case["model"])
        square, graph.input_shape = graph.input_shape, (3, case["h"], case["w"])
        rows = zoo.quantised_layer_table(graph)
        graph.input_shape = square
        weights = sum(layer["w"].size for layer in graph.layers if layer.get("w") is not None)
        return {"bytes": case["batch"] * (3 * case["h"] * case["w"] + 1000) * 4 + weights, "flops": 2 * case["batch"] * sum(r["macs"] for r in rows)}
    if case["kind"] == "gemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": m * k * 4 + n * k + n * 8 + m * n * 4, "flops": 2 * m * n * k}
    if case["kind"] == "decoder":
        rows, shapes = case["rows"], _decoder_shapes(case)
        size = sum(n * k * case["bits"] // 8 + n * -(-k // case["block"]) * 4 + rows * n * 4 for n, k in shapes)
        size += rows * (3 * case["hidden"] + case["inter"]) * (2 if case["act"] == "fp16" else 4)
        return {"bytes": size, "flops": 2 * rows * sum(n * k for n, k in shapes)}
    embed, src, dst = case["heads"] * case["head_dim"], case["src"], case["past"] + case["src"]
    size = 4 * embed * (embed * case["bits"] // 8 + -(-embed // case["block"]) * 4 + 4)
    size += 2 * embed * dst * 4 + 2 * embed * src * 4 + 2 * src * embed * 4
    return {"bytes": size, "flops": 8 * src * embed ** 2 + 4 * src * dst * embed}


def tolerance(case):
    # int8 sums are exact: what is left is a handful of fp32 roundings per value; in a model they may move a value that lies
    # between two int8 steps by one step of 127, rarely
    if case["kind"] in ("net", "gemm"):
        return {"rel": 1e-6 if case["kind"] == "gemm" else 1e-5}
    # exact products, fp32 sums over thousands of terms in any order
    return {"rel": 1e-5} if case["kind"] == "decoder" else {"rel": 2e-5}
