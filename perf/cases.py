"""Workloads whose time and results are followed: the calls that a program
built on this library makes, over the sizes it makes them at.

A case is a dict of plain values. ``listed()`` names the fixed ones, ``draw``
makes more of the same ranges, ``prepare`` builds what a program holds before
the call (weights, inputs, outputs, workspace, a captured graph), ``run`` is
one pass through the public entry points, ``work`` the bytes and operations it
cannot do without, ``exact`` the same results in 64 bits from plain torch.

Kinds:

  layer    `layers` mixture-of-experts layers over `tokens` tokens: one
           moe_layer call, or with `block` the stacked decoder block (RMSNorm,
           the layer, the residual). With `graph` the calls are captured once
           and a pass replays them, as a decode loop does.
  project  dense projections of a decoder layer by kernel name, `layers`
           weight matrices one after the other from a captured graph
  mixer    one prompt chunk through a gated-delta-rule layer and a causal
           attention layer over a full context

Weights belong to the model and not to a call: they are the same for every
seed, made once per shape. Inputs (and the attention context and the router
bias) come from the seed.
"""
import math

import torch

import stratacuda_amd as sm
from stratacuda_amd import workload as wl

EPS = 1e-6
GROUP = 32         # weights per scale of the dense 4- and 8-bit formats
HEADS, KV_HEADS, HEAD_DIM = 24, 2, 256
DELTA_DIM, DELTA_KEYS, DELTA_VALUES = 128, 16, 48

# (width, ff, experts, top-k): the benchmark's geometry, the real model's, and
# a small one outside the shapes that have kernels of their own
GEOMETRIES = {"bench": (2048, 512, 512, 10), "real": (2560, 640, 512, 10), "small": (1024, 256, 64, 6)}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # One token through one layer, called from the host: the smallest call.
        dict(name="token_layer", kind="layer", model="bench", tokens=1, layers=1, block=False, graph=False, skew=False),
        # A decode step of one sequence: eight layers of the real model from a graph.
        dict(name="token_stack_real", kind="layer", model="real", tokens=1, layers=8, block=True, graph=True,
             skew=False),
        # A decode step of five sequences, an odd small batch.
        dict(name="batch5_stack", kind="layer", model="bench", tokens=5, layers=4, block=True, graph=True, skew=False),
        # A decode step of 32 sequences: most experts hold a row or two.
        dict(name="batch32_stack", kind="layer", model="bench", tokens=32, layers=4, block=True, graph=True,
             skew=False),
        # A short prompt of ragged length at the real model's geometry.
        dict(name="prompt333_real", kind="layer", model="real", tokens=333, layers=1, block=False, graph=False,
             skew=False),
        # The benchmark's prompt: about ten rows for each of 512 experts.
        dict(name="prompt512", kind="layer", model="bench", tokens=512, layers=1, block=False, graph=False, skew=False),
        # A long prompt whose routing is skewed, as trained routers' is.
        dict(name="prompt2048_skewed", kind="layer", model="bench", tokens=2048, layers=1, block=False, graph=False,
             skew=True),
        # Several prompts in one batch at the real model's geometry, inside the stack.
        dict(name="prompt4096_real", kind="layer", model="real", tokens=4096, layers=1, block=True, graph=False,
             skew=True),
        # A prompt through a small model with few experts.
        dict(name="prompt200_small", kind="layer", model="small", tokens=200, layers=1, block=False, graph=False,
             skew=False),
        # A prompt chunk's bf16 projections (hidden to the delta rule's channels).
        dict(name="chunk16_bf16", kind="project", format="bf16", tokens=16, cols=2560, rows=10240, layers=4),
        # A decode step's 4-bit projections of the same shape.
        dict(name="token_s4", kind="project", format="s4", tokens=1, cols=2560, rows=10240, layers=8),
        # A prompt chunk's sequence mixers near the end of the context.
        dict(name="chunk16_mixers", kind="mixer", tokens=16, position=2032),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "layer", "project", "project", "mixer"])
    if kind == "mixer":
        tokens = rng.randint(1, 16)
        return dict(kind="mixer", tokens=tokens, position=rng.randint(0, 2048 - tokens))
    if kind == "project":
        fmt = rng.choice(["bf16", "s4", "s8"])
        return dict(kind="project", format=fmt, tokens=rng.choice([1, _log(rng, 2, 32)]), cols=64 * rng.randint(10, 48),
                    rows=_log(rng, 300, 10240), layers=rng.randint(1, 4))
    model = rng.choice(["bench", "bench", "real", "real", "small"])
    tokens = _log(rng, 1, 4096)
    step = tokens <= 64
    return dict(kind="layer", model=model, tokens=tokens, layers=rng.randint(1, 4) if step else 1, block=rng.random() < 0.5,
                graph=step and rng.random() < 0.7, skew=rng.random() < 0.5)


# ------------------------------------------------------------------ buffers
_backend = None


def backend():
    """The program's one context on the GPU."""
    global _backend
    if _backend is None:
        _backend = sm.Backend(0)
    return _backend


class _Owned:
    """A device buffer freed with its last user, readable as a torch tensor."""

    def __init__(self, nbytes, dtype, shape):
        self.buf = backend().alloc_bytes(nbytes)
        typestr = {torch.float32: "<f4", torch.int32: "<i4", torch.uint8: "|u1"}[dtype]
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (self.buf.handle, False),
                                         "version": 2, "strides": None}

    def __del__(self):
        try:
            backend().free(self.buf)
        except Exception:
            pass


def _empty(shape, dtype=torch.float32):
    """(buffer, tensor over it); the tensor keeps the buffer."""
    size = torch.empty((), dtype=dtype).element_size()
    own = _Owned(math.prod(shape) * size, dtype, shape)
    return own.buf, torch.as_tensor(own, device="cuda")


def _put(t):
    buf, view = _empty(t.shape, t.dtype)
    view.copy_(t)
    return buf, view


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _normal(shape, seed, sigma=1.0):
    return torch.randn(shape, generator=_gen(seed), device="cuda") * sigma


def _bytes(n, seed):
    return torch.randint(0, 256, (n,), generator=_gen(seed), device="cuda", dtype=torch.uint8)


# ------------------------------------------------------------ layer weights
def _scales(n, seed):
    return (_normal((n,), seed, 0.05)).abs().to(torch.float16)


def _blobs(width, ff, experts, seed):
    """(codes and scales of `experts` blobs) as the four planes of each."""
    gu, dn = 2 * ff * width // 4, width * ff // 4
    return (_bytes(experts * gu, seed).view(experts, 2 * ff, width // 4),
            _bytes(experts * dn, seed + 1).view(experts, width, ff // 4),
            _scales(experts * 2 * ff * (width // 64), seed + 2).view(experts, 2 * ff, width // 64),
            _scales(experts * width * (ff // 64), seed + 3).view(experts, width, ff // 64))


def _layer_tensors(model, layer):
    """The layer's weights as torch tensors (the same for every call)."""
    width, ff, experts, _ = GEOMETRIES[model]
    seed = 1000 * (1 + sorted(GEOMETRIES).index(model)) + 20 * layer
    return {"routed": _blobs(width, ff, experts, seed), "shared": _blobs(width, ff, 1, seed + 4),
            "Wr": _normal((experts, width), seed + 8, 0.02), "Wsg": _normal((width,), seed + 9, 0.02),
            "gamma": 1 + 0.05 * (2 * torch.rand((width,), generator=_gen(seed + 10), device="cuda") - 1)}


def _arena(planes, stride):
    """The planes as blobs, one every `stride` bytes."""
    experts = planes[0].shape[0]
    out = torch.zeros((experts, stride), dtype=torch.uint8, device="cuda")
    at = 0
    for p in planes:
        b = p.reshape(experts, -1).view(torch.uint8)
        out[:, at:at + b.shape[1]] = b
        at += b.shape[1]
    return out


_layers = {}


def _layer(model, layer):
    """The layer's weights resident in the library's buffers, kept by the program."""
    if (model, layer) not in _layers:
        width, ff, _, _ = GEOMETRIES[model]
        t = _layer_tensors(model, layer)
        stride = wl.blob_stride(width, ff)
        held = {"stride": stride, "arena": _put(_arena(t["routed"], stride)), "shared": _put(_arena(t["shared"], stride))}
        held.update({k: _put(t[k]) for k in ("Wr", "Wsg", "gamma")})
        del t
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        _layers[(model, layer)] = held
    return _layers[(model, layer)]


def _bias(case, seed):
    """A skewed router's bias: log of Zipf popularities over a seeded order."""
    experts = GEOMETRIES[case["model"]][2]
    p = torch.arange(1, experts + 1, dtype=torch.float64) ** -1.1
    order = torch.randperm(experts, generator=torch.Generator().manual_seed(seed + 77))
    bias = torch.empty(experts)
    bias[order] = (p / p.sum()).log().float()
    return bias.cuda()


def _layer_input(case, seed):
    width = GEOMETRIES[case["model"]][0]
    x = _normal((case["tokens"], width), seed)
    return x if case["block"] else x / (x.square().mean(-1, keepdim=True) + EPS).sqrt()


# -------------------------------------------------------- projection weights
def _project_tensors(case, layer):
    cols, rows = case["cols"], case["rows"]
    seed = 900000 + 10 * layer
    if case["format"] == "bf16":
        return {"Codes": _normal((rows, cols), seed, 0.05).to(torch.bfloat16)}
    bits = int(case["format"][1:])
    return {"Codes": _bytes(rows * cols * bits // 8, seed), "Scales": _normal((rows, cols // GROUP), seed + 1, 0.02),
            "Offsets": _normal((rows, cols // GROUP), seed + 2, 0.01)}


def _project_put(t):
    if t.dtype != torch.float32:
        t = t.reshape(-1).view(torch.uint8)
    return _put(t)


# ------------------------------------------------------------------ prepare
class _State:
    """A call's buffers and the pass over them."""

    def __init__(self):
        self.graph, self.keep, self.outputs, self.launch = None, [], {}, None

    def capture(self, launch):
        be = backend()
        torch.cuda.synchronize()
        be.graph_begin()
        launch()
        self.graph = be.graph_end()
        self.launch = lambda: be.graph_launch(self.graph)

    def __del__(self):
        if self.graph is not None:
            try:
                backend().graph_free(self.graph)
            except Exception:
                pass


def _prepare_layer(case, seed):
    be, s = backend(), _State()
    width, ff, experts, topk = GEOMETRIES[case["model"]]
    n = case["tokens"]
    layers = [_layer(case["model"], i) for i in range(case["layers"])]
    x = _put(_layer_input(case, seed))
    bias = _put(_bias(case, seed)) if case["skew"] else None
    size = be.moe_block_workspace_bytes if case["block"] else be.moe_workspace_bytes
    ws = _empty((size(n, width, ff, experts, topk),), torch.uint8)
    s.keep += [layers, x, bias, ws]
    steps, h = [], x
    for i, lay in enumerate(layers):
        y, ids, w = _empty((n, width)), _empty((n, topk), torch.int32), _empty((n, topk))
        s.outputs["layer%d" % i] = {"y": y[1], "ids": ids[1], "weights": w[1]}
        tail = (width, ff, experts, topk, y[0], ids[0], w[0], ws[0], bias[0] if bias else None)
        weights = (lay["Wr"][0], lay["arena"][0], lay["stride"], lay["shared"][0], lay["Wsg"][0])
        if case["block"]:
            steps.append((be.moe_block, (h[0], n, lay["gamma"][0], EPS) + weights + tail))
        else:
            steps.append((be.moe_layer, (h[0], n) + weights + tail))
        h = y

    def launch():
        for call, args in steps:
            call(*args)

    s.launch = launch
    if case["graph"]:
        s.capture(launch)
    return s


def _prepare_project(case, seed):
    be, s = backend(), _State()
    cols, rows, n, fmt = case["cols"], case["rows"], case["tokens"], case["format"]
    x = _put(_normal((n, cols), seed))
    s.keep.append(x)
    steps = []
    for i in range(case["layers"]):
        wts = {k: _project_put(v) for k, v in _project_tensors(case, i).items()}
        y = _empty((n, rows))
        s.keep.append(wts)
        s.outputs["layer%d" % i] = y[1]
        args = {k: v[0] for k, v in wts.items()}
        args.update(X=x[0], Y=y[0], cols=cols, rows=rows)
        if fmt != "bf16":
            bits = int(fmt[1:])
            args.update(bits=bits, groupSize=GROUP, bias=-(1 << (bits - 1)), codebook=0, hasOffset=1)
        if fmt == "bf16" or n > 1:
            args.update(tokens=n, outputStride=rows, outputOffset=0)
        name = "strata_bf16_project" if fmt == "bf16" else "strata_quant_gemv" if n == 1 else "strata_quant_project"
        steps.append((name, args, [rows, n, 1]))

    def launch():
        for name, args, groups in steps:
            be.run(name, args, groups)

    s.capture(launch)
    return s


def _mixer_tensors(case, seed):
    n, d = case["tokens"], DELTA_DIM
    cells = case["position"] + n
    u = torch.rand((2, n, DELTA_VALUES), generator=_gen(seed + 9), device="cuda")
    return {"State": _normal((d, DELTA_VALUES, d), seed, 0.1), "Q": _normal((n, DELTA_KEYS, d), seed + 1, d ** -0.5),
            "K": _normal((n, DELTA_KEYS, d), seed + 2, d ** -0.5), "V": _normal((n, DELTA_VALUES, d), seed + 3),
            "Decay": 0.9 + 0.09 * u[0], "Beta": 0.1 + 0.8 * u[1],
            "query": _normal((n, HEADS, HEAD_DIM), seed + 4), "keys": _normal((cells, KV_HEADS, HEAD_DIM), seed + 5),
            "values": _normal((cells, KV_HEADS, HEAD_DIM), seed + 6)}


def _prepare_mixer(case, seed):
    be, s = backend(), _State()
    n = case["tokens"]
    t = {k: _put(v) for k, v in _mixer_tensors(case, seed).items()}
    delta, attn = _empty((n, DELTA_VALUES, DELTA_DIM)), _empty((n, HEADS, HEAD_DIM))
    s.keep.append(t)
    s.outputs = {"delta": delta[1], "state": t["State"][1], "attention": attn[1]}
    gdn = {k: t[k][0] for k in ("State", "Q", "K", "V", "Decay", "Beta")}
    gdn.update(Y=delta[0], dim=DELTA_DIM, keyHeads=DELTA_KEYS, valueHeads=DELTA_VALUES, tokens=n)
    att = dict(Q=t["query"][0], Keys=t["keys"][0], Values=t["values"][0], Y=attn[0], dim=HEAD_DIM, heads=HEADS,
               kvHeads=KV_HEADS, position=case["position"], scale=HEAD_DIM ** -0.5)

    def launch():
        be.run("strata_gdn_batch", gdn, [DELTA_VALUES * DELTA_DIM // 64, 1, 1])
        be.run("strata_attention_batch", att, [HEADS, HEAD_DIM // 64, n])

    s.launch = launch
    return s


def prepare(case, seed):
    s = {"layer": _prepare_layer, "project": _prepare_project, "mixer": _prepare_mixer}[case["kind"]](case, seed)
    torch.cuda.synchronize()  # the library's stream starts from finished inputs
    return s


def run(state):
    state.launch()
    return state.outputs


# ---------------------------------------------------------------- the bound
def work(case):
    n = case["tokens"]
    if case["kind"] == "project":
        cols, rows = case["cols"], case["rows"]
        w = rows * cols * 2 if case["format"] == "bf16" else (rows * cols * int(case["format"][1:]) // 8
                                                              + 2 * 4 * rows * cols // GROUP)
        return {"bytes": case["layers"] * (w + n * rows * 4) + n * cols * 4, "flops": 2 * case["layers"] * n * rows * cols}
    if case["kind"] == "mixer":
        d, v, k, cells = DELTA_DIM, DELTA_VALUES, DELTA_KEYS, case["position"] + n
        moved = 2 * d * v * d + n * (2 * k * d + 2 * v * d + 2 * v) + 2 * cells * KV_HEADS * HEAD_DIM + 2 * n * HEADS * HEAD_DIM
        return {"bytes": 4 * moved, "flops": n * (8 * v * d * d + 4 * HEADS * HEAD_DIM * cells)}
    width, ff, experts, topk = GEOMETRIES[case["model"]]
    blob, p = wl.blob_bytes(width, ff), torch.full((experts,), 1 / experts, dtype=torch.float64)
    if case["skew"]:
        p = torch.arange(1, experts + 1, dtype=torch.float64) ** -1.1
        p = p / p.sum()
    # experts that n tokens reach, when each picks top-k of them by popularity
    touched = min(float((1 - (1 - p) ** (n * topk)).sum()), n * topk)
    moved = experts * width * 4 + (touched + 1) * blob + n * (2 * width + 2 * topk) * 4
    ops = 2 * n * ((topk + 1) * 3 * width * ff + experts * width)
    return {"bytes": case["layers"] * moved, "flops": case["layers"] * ops}


def tolerance(case):
    # Four times what the results are off from 64 bits: 1.0e-6 in the
    # attention's sums over 2,048 cells, 1.4e-7 in a projection, 2e-7 to 4e-7
    # in one layer and in a stack's (whose differences of rounding travel on,
    # and where a tie between two experts may fall the other way).
    if case["kind"] == "mixer":
        return {"rel": 4e-6}
    if case["kind"] == "project":
        return {"rel": 6e-7}
    return {"rel": 2e-6, "differ": 0.01} if case["layers"] > 1 else {"rel": 1.5e-6}


# ------------------------------------------------------------------ 64 bits
def _dequant(codes, scales):
    """[n, k/4] code bytes and [n, k/64] scales of 2-bit weights to f64 [n, k]."""
    c = torch.stack([(codes >> (2 * i)) & 3 for i in range(4)], -1).reshape(codes.shape[0], -1)
    return (c.double() - 1) * scales.double().repeat_interleave(64, 1)


def _expert(planes, e, x):
    gu = x @ _dequant(planes[0][e], planes[2][e]).T
    g, u = gu[:, 0::2], gu[:, 1::2]
    return (g / (1 + (-g).exp()) * u) @ _dequant(planes[1][e], planes[3][e]).T


def _exact_layer(case, seed):
    topk = GEOMETRIES[case["model"]][3]
    h, out = _layer_input(case, seed).double(), {}
    bias = _bias(case, seed).double() if case["skew"] else 0.0
    for i in range(case["layers"]):
        t = _layer_tensors(case["model"], i)
        x = h
        if case["block"]:
            x = h / (h.square().mean(-1, keepdim=True) + EPS).sqrt() * t["gamma"].double()
        p, ids = (x @ t["Wr"].double().T + bias).softmax(-1).topk(topk)
        w = p / p.sum(-1, keepdim=True)
        y = _expert(t["shared"], 0, x) * torch.sigmoid(x @ t["Wsg"].double())[:, None]
        for e in ids.unique().tolist():
            at, slot = (ids == e).nonzero(as_tuple=True)
            y.index_add_(0, at, _expert(t["routed"], e, x[at]) * w[at, slot][:, None])
        h = h + y if case["block"] else y
        out["layer%d" % i] = {"y": h, "ids": None, "weights": w}
        del t
    return out


def _exact_project(case, seed):
    x, out = _normal((case["tokens"], case["cols"]), seed).double(), {}
    for i in range(case["layers"]):
        t = _project_tensors(case, i)
        if case["format"] == "bf16":
            w = t["Codes"].double()
        else:
            b, bits = t["Codes"], int(case["format"][1:])
            c = b if bits == 8 else torch.stack([b & 15, b >> 4], -1).reshape(-1)
            c = c.reshape(case["rows"], case["cols"]).double() - (1 << (bits - 1))
            w = (c * t["Scales"].double().repeat_interleave(GROUP, 1) + t["Offsets"].double().repeat_interleave(GROUP, 1))
        out["layer%d" % i] = x @ w.T
    return out


def _exact_mixer(case, seed):
    t = {k: v.double() for k, v in _mixer_tensors(case, seed).items()}
    n, heads = case["tokens"], torch.arange(DELTA_VALUES, device="cuda") % DELTA_KEYS
    state, delta = t["State"].permute(1, 0, 2).clone(), []  # [value head, key, value]
    for i in range(n):
        q, k = t["Q"][i][heads], t["K"][i][heads]
        state = state * t["Decay"][i][:, None, None]
        change = (t["V"][i] - torch.einsum("hkv,hk->hv", state, k)) * t["Beta"][i][:, None]
        state = state + k[:, :, None] * change[:, None, :]
        delta.append(torch.einsum("hkv,hk->hv", state, q))
    attn, per = [], HEADS // KV_HEADS
    for i in range(n):
        cells = case["position"] + i + 1
        k = t["keys"][:cells].repeat_interleave(per, 1)
        v = t["values"][:cells].repeat_interleave(per, 1)
        p = (torch.einsum("hd,chd->hc", t["query"][i], k) * HEAD_DIM ** -0.5).softmax(-1)
        attn.append(torch.einsum("hc,chd->hd", p, v))
    return {"delta": torch.stack(delta), "state": state.permute(1, 0, 2).contiguous(), "attention": torch.stack(attn)}


def exact(case, seed):
    return {"layer": _exact_layer, "project": _exact_project, "mixer": _exact_mixer}[case["kind"]](case, seed)
