"""What the layer's speed is judged by: single forwards of a mixture-of-experts layer through the
entry points a host calls, over the shapes, storage types and batch sizes the library serves.

`listed()` names the cases, `draw()` gives further ones of the same ranges, `prepare()` builds what
a serving process has in hand before the call (the layer with its experts resident, the input rows,
the output buffer), `run()` is one forward and returns the layer's output.

A case is a dict of
  shape     layer dimensions, a key of SHAPES
  weights   storage of the expert weights: f32, bf16, int8 (one scale per output row) or int8g
            (one scale per output row and 128 input elements)
  tokens    rows of the batch
  entry     device    forward on device rows
            noalloc   the same on the library's own workspace
            block     RMSNorm, layer and residual add on an f32 residual stream on the device
            host      forward from and to host memory
  rows      type of the rows given to the device entries: bf16 or f32
"""
import math

import numpy as np
import torch

from ateniaengine_amd import capi

# The layer shapes of the benchmark and of the tests.
SHAPES = {
    # the reference's CPU-sized layer
    "tiny": dict(d=1024, E=8, k=2, f=2048),
    "mixtral": dict(d=4096, E=8, k=2, f=14336),
    "qwen": dict(d=2048, E=60, k=4, f=1408, fs=5632, gated=True, renorm=False),
    # skewed expert load: a log-Zipf(1.2) bias on the logits
    "deepseek": dict(d=2048, E=64, k=6, f=1408, fs=2816, renorm=False, zipf=True),
    # sigmoid scores, 256 experts in 8 groups, the 4 best groups, narrow experts
    "v3route": dict(d=7168, E=256, k=8, f=256, fs=256, renorm=False, v3=True),
}
W_STD = 0.02
GROUP = 128
EPS = 1e-5


def _case(shape, weights, tokens, entry="device", rows="bf16"):
    return dict(shape=shape, weights=weights, tokens=tokens, entry=entry, rows=rows)


def listed():
    cases = {
        # one user generating: two experts' weights are read for one token
        "mixtral-bf16-1": _case("mixtral", "bf16", 1),
        # sixteen users generating: every expert is read for a few rows
        "mixtral-bf16-16": _case("mixtral", "bf16", 16),
        # a short prompt, or a chunk of one beside decoding users
        "mixtral-bf16-333": _case("mixtral", "bf16", 333),
        # a long prompt: the headline batch
        "mixtral-bf16-4096": _case("mixtral", "bf16", 4096),
        # a few users on the int8 layer
        "mixtral-int8-5": _case("mixtral", "int8", 5),
        # a prompt of ragged length on the int8 layer
        "mixtral-int8-1537": _case("mixtral", "int8", 1537),
        # one user on many narrow experts with a gated shared one: launch-bound
        "qwen-bf16-1": _case("qwen", "bf16", 1),
        # a thousand-token prompt: some 66 rows for each of sixty experts
        "qwen-bf16-997": _case("qwen", "bf16", 997),
        # a full decode batch inside a decoder layer: norm, experts under skewed load, residual
        "deepseek-bf16-48-block": _case("deepseek", "bf16", 48, entry="block", rows="f32"),
        # several long prompts at once under skewed load: the largest batch
        "deepseek-bf16-16384": _case("deepseek", "bf16", 16384),
        # group-limited sigmoid routing over 256 experts
        "v3route-bf16-256": _case("v3route", "bf16", 256),
        # an f32 checkpoint behind the unchanged host-side graph op
        "tiny-f32-64-host": _case("tiny", "f32", 64, entry="host", rows="f32"),
    }
    return [dict(c, name=n) for n, c in cases.items()]


# Largest batch drawn per shape (below the listed ones: a drawn case is never the dearest) and the
# storage types a shape is drawn with.
_DRAWN = (
    ("mixtral", 3800, ("bf16", "bf16", "int8", "int8", "int8g")),
    ("qwen", 12288, ("bf16", "bf16", "int8")),
    ("deepseek", 12288, ("bf16", "bf16", "int8")),
    ("v3route", 2048, ("bf16",)),
    ("tiny", 1024, ("f32",)),
)


def draw(rng):
    shape, most, types = rng.choice(_DRAWN[:3] * 3 + _DRAWN[3:])
    weights = rng.choice(types)
    tokens = int(round(math.exp(rng.uniform(0.0, math.log(most)))))
    entries = ["device", "device", "device", "block"]
    if tokens <= 32:
        entries.append("noalloc")
    if tokens <= 256:
        entries.append("host")
    entry = rng.choice(entries)
    f32_rows = weights == "f32" or entry in ("block", "host")
    rows = "f32" if f32_rows else rng.choice(("bf16", "bf16", "bf16", "f32"))
    return _case(shape, weights, tokens, entry, rows)


def _pinned(shape, dtype):
    return torch.empty(shape, dtype=dtype, pin_memory=True)


def _to_host(t):
    return _pinned(t.shape, t.dtype).copy_(t).numpy()


def _trunc(w):
    """Truncation to bf16-valued f32, the storage convention of bf16 checkpoints."""
    return (w.view(torch.int32) & -65536).view(torch.float32)


def _projection(n, rows, cols, weights, g):
    """Host arrays (values, scales or None) of n weight matrices [rows, cols], made on the GPU a
    few matrices at a time; layers are made from host arrays."""
    values = _pinned((n, rows, cols), {"f32": torch.float32, "bf16": torch.int16}.get(weights, torch.int8))
    groups = cols // GROUP if weights == "int8g" else 1
    scales = _pinned((n, rows, groups), torch.float32)
    step = max(1, (1 << 27) // (rows * cols))
    for i in range(0, n, step):
        m = min(step, n - i)
        w = torch.randn((m * rows, cols), generator=g, device="cuda") * W_STD
        if weights == "f32":
            values[i:i + m].copy_(w.view(m, rows, cols))
            continue
        if weights == "bf16":
            values[i:i + m].copy_((w.view(torch.int32) >> 16).to(torch.int16).view(m, rows, cols))
            continue
        w = _trunc(w)
        # one row in a thousand is eight times larger
        big = torch.randint(0, m * rows, (max(1, m * rows // 1000),), generator=g, device="cuda")
        w[big] *= 8.0
        w = w.view(m * rows, groups, cols // groups)
        scale = (w.abs().amax(-1) / 127.0).clamp_min(1e-12)
        q = torch.round(w / scale[..., None]).clamp_(-127, 127).to(torch.int8)
        values[i:i + m].copy_(q.view(m, rows, cols))
        scales[i:i + m].copy_(scale.view(m, rows, groups))
    values = values.numpy()
    if weights == "bf16":
        values = values.view(np.uint16)
    if weights in ("f32", "bf16"):
        return values, None
    return values, (scales if weights == "int8g" else scales[..., 0]).numpy()


def _layer(case, g):
    s = SHAPES[case["shape"]]
    d, E, f, fs, weights = s["d"], s["E"], s["f"], s.get("fs", 0), case["weights"]

    def normal(*shape):
        return torch.randn(shape, generator=g, device="cuda") * W_STD

    router = normal(E, d)
    if case["shape"] in ("qwen", "deepseek"):  # logits of unit variance
        router *= 1.0 / (W_STD * math.sqrt(d))
    kw = dict(w_router=_to_host(router if weights == "f32" else _trunc(router)), top_k=s["k"],
              convention=capi.CONVENTION_ATENIA if s.get("renorm", True)
              else capi.CONVENTION_HUGGINGFACE_QWEN,
              weight_dtype={"f32": capi.WEIGHT_F32, "bf16": capi.WEIGHT_BF16,
                            "int8": capi.WEIGHT_INT8_W8A16,
                            "int8g": capi.WEIGHT_INT8_PER_GROUP}[weights],
              group_size=GROUP if weights == "int8g" else 0, max_tokens_hint=case["tokens"])
    for name, rows, cols in (("gate", f, d), ("up", f, d), ("down", d, f)):
        kw["w_" + name], kw["scale_" + name] = _projection(E, rows, cols, weights, g)
    if fs:
        for name, rows, cols in (("gate", fs, d), ("up", fs, d), ("down", d, fs)):
            q, scale = _projection(1, rows, cols, weights, g)
            kw["s_" + name] = q[0]
            kw["s_scale_" + name] = None if scale is None else scale[0]
        if s.get("gated"):
            kw["shared_gate"] = _to_host(_trunc(normal(d)))
    if s.get("zipf"):
        rank = torch.randperm(E, generator=g, device="cuda").cpu().numpy() + 1.0
        kw["router_bias"] = (-1.2 * np.log(rank)).astype(np.float32)
    layer = capi.Layer(**kw)
    if s.get("v3"):
        bias = 0.05 * torch.randn((E,), generator=g, device="cuda")
        layer.set_v3_router(8, 4, 2.5, True, bias.cpu().numpy())
    return layer


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    layer = _layer(case, g)
    T, d = case["tokens"], layer.d
    x = torch.randn((T, d), generator=g, device="cuda")
    state = dict(layer=layer, entry=case["entry"], tokens=T)
    if case["entry"] == "host":
        if case["weights"] != "f32":
            x = x.to(torch.bfloat16).to(torch.float32)  # what a bf16 model's host graph holds
        state.update(x=x.cpu().numpy(), out=np.empty((T, d), np.float32))
        return state
    if case["rows"] == "bf16":
        x = x.to(torch.bfloat16)
    state.update(x=x, out=torch.empty((T, d), device="cuda"),
                 rows=capi.ACT_BF16 if case["rows"] == "bf16" else capi.ACT_F32,
                 stream=torch.cuda.current_stream().cuda_stream)
    if case["entry"] == "block":
        state["gamma"] = 1.0 + 0.1 * torch.randn((d,), generator=g, device="cuda")
    return state


def run(state):
    layer, entry, T, x, out = (state[n] for n in ("layer", "entry", "tokens", "x", "out"))
    if entry == "host":
        return layer.forward(x, out)
    if entry == "block":
        layer.block_forward_device(x.data_ptr(), T, state["gamma"].data_ptr(), EPS,
                                   capi.NORM_GRAPH_F32, out.data_ptr(), state["stream"])
    elif entry == "noalloc":
        layer.forward_device_noalloc(x.data_ptr(), state["rows"], T, out.data_ptr(), state["stream"])
    else:
        layer.forward_device(x.data_ptr(), state["rows"], T, out.data_ptr(), state["stream"])
    return out


def _experts_hit(s, T):
    """Experts that some token of a batch is routed to, on a sample of the logits."""
    E, k = s["E"], s["k"]
    rng = np.random.default_rng(0)
    spread = 1.0 if s.get("renorm") is False and not s.get("v3") else W_STD * math.sqrt(s["d"])
    logits = spread * rng.standard_normal((T, E))
    if s.get("zipf"):
        logits -= 1.2 * np.log(np.arange(E) + 1.0)
    if s.get("v3"):  # corrected scores, limited to the 4 groups with the largest top-two sums
        score = 1.0 / (1.0 + np.exp(-logits)) + 0.05 * rng.standard_normal(E)
        group = np.sort(score.reshape(T, 8, E // 8), axis=-1)[..., -2:].sum(-1)
        keep = group >= np.sort(group, axis=-1)[:, -4:-3]
        logits = np.where(np.repeat(keep, E // 8, axis=1), score, -np.inf)
    return len(np.unique(np.argpartition(logits, E - k, axis=1)[:, E - k:]))


def work(case):
    """Bytes: the weights of every expert that gets a token, the router, the rows in and out.
    Flops: router and experts (2 per multiply-add)."""
    s, T = SHAPES[case["shape"]], case["tokens"]
    d, E, k, f, fs = s["d"], s["E"], s["k"], s["f"], s.get("fs", 0)
    per = {"f32": 4.0, "bf16": 2.0, "int8": 1.0, "int8g": 1.0 + 4.0 / GROUP}[case["weights"]]

    def expert(width):
        return 3.0 * d * width * per + (4.0 * (2 * width + d) if case["weights"] == "int8" else 0.0)

    row = 2.0 if case["rows"] == "bf16" else 4.0
    return dict(bytes=_experts_hit(s, T) * expert(f) + (expert(fs) if fs else 0.0) + 4.0 * E * d +
                T * d * (row + 4.0),
                flops=T * (2.0 * d * E + 6.0 * k * d * f + 6.0 * d * fs))


def tolerance(case):
    """About four times what the layer's own outputs differ by from the same arithmetic in 64 bits
    on the stored weights (2-norm, and largest difference over the rms)."""
    if case["weights"] == "f32":
        # sums in f64, results rounded to f32: 7e-8 and 5.5e-7
        return dict(rel=3e-7, max=2.2e-6)
    # rows, h and (large bf16 batches) expert outputs rounded to bf16: 1.3e-3 to 2.4e-3 on bf16
    # rows, up to 3.4e-3 on f32 rows; largest difference 2e-2 for bf16 weights, 3.7e-2 with the
    # eight times larger rows of the int8 layers
    return dict(rel=1e-2, max=8e-2 if case["weights"] == "bf16" else 0.15)
