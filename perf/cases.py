"""The work that users of this package have it do, as cases that a timing harness can run.

A model that streams video calls the package once per transformer block and
chunk: the self-attention over the ring KV cache (``RingKVPath.attend``, or
``CausalWanSelfAttention.forward`` with the projections around it), the text
cross-attention (``WanT2VCrossAttention.forward``), and, when blocks change
owner, the two ends of a hand-off (``handoff.export_block`` / ``import_block``).
One pass of a case is one chunk through a few such blocks, each with a cache of
its own, as the layers of a model follow each other on the stream.

A case is a dict of plain values:

kind      stream | module | cross | handoff
dtype     bf16 | fp32
layers    blocks per pass
rows      stream batch (one cache row per denoising stage)
heads     heads of 128 (model width = 128 * heads)
f, h, w   latent frames, height and width of a chunk in tokens
frames    latent frames that the cache holds
first     the stream's first chunk into an empty cache, once per denoising
          step, instead of a chunk into a full one
norm      q and k arrive as raw projections, their RMSNorm is folded in
sink, thr sink frames, and threshold of the adaptive refresh (-1: off)
block     block-causal mask inside the chunk, in latent frames (0: none)
scale     scale of the raw inputs
hot       share of key rows that are eight times as large
text      cached text tokens (cross)
"""
import functools
import math

import torch

from streamdiffusionv2_amd import handoff, ring, rope
from streamdiffusionv2_amd.attention import CausalWanSelfAttention, RingKVPath, WanT2VCrossAttention

EPS = 1e-6
STEPS = 2            # denoising steps of the shipped configuration: passes of a first chunk, rows of a stream batch
CUT_EVERY = 8        # a scene cut every so many chunks where the adaptive refresh watches for one
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
BASE = dict(kind="stream", dtype="bf16", layers=4, rows=1, heads=12, f=1, h=30, w=52, frames=6, first=False, norm=False, sink=1,
            thr=-1.0, block=0, scale=1.0, hot=0.0, text=0)


def listed():
    def case(name, **more):
        return dict(BASE, name=name, **more)

    return [
        # a preview at 256 x 256: the smallest chunk, where launches and host work count
        case("preview_256", layers=8, h=16, w=16, norm=True),
        # 480p with the 1.3B model, one chunk through the path itself: the benchmark's default workload
        case("stream_480p", layers=6, scale=128 ** -0.5),
        # the same through the drop-in module, projections included
        case("module_480p", kind="module", norm=True),
        # the shipped video-to-video configuration: two denoising stages, three sink frames, adaptive refresh
        case("adaptive_480p", layers=8, rows=STEPS, norm=True, sink=3, thr=0.2),
        # the 14B model's width
        case("stream_480p_14b", heads=40, norm=True),
        # four denoising stages, chunks of three latent frames
        case("batch_480p", layers=2, rows=4, f=3, frames=12),
        # 720p, a long window, outliers among the keys: the largest
        case("long_720p", layers=1, rows=2, f=3, h=45, w=80, frames=21, hot=0.01),
        # the first chunk of a session (two latent frames), submitted once per denoising step
        case("first_chunk_480p", f=2, first=True, norm=True),
        # a ragged size (432 x 752), three frames masked block by block
        case("masked_ragged", layers=3, f=3, h=27, w=47, frames=9, norm=True, block=1),
        # fp32, for runs that are compared with a CPU
        case("fp32_480p", dtype="fp32", layers=1, frames=4),
        # text cross-attention of a stream batch against the cached prompt
        case("cross_480p", kind="cross", rows=STEPS, norm=True, text=512),
        # blocks of a stream batch leave one pipeline stage and arrive at another
        case("handoff_480p", kind="handoff", rows=STEPS),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any option of the listed ones over their whole range of sizes."""
    most = 1.0e13                                  # operations of the largest listed case
    while True:
        c = dict(BASE)
        c["kind"] = rng.choices(("stream", "module", "cross", "handoff"), (10, 3, 2, 2))[0]
        c["heads"] = rng.choice((12, 12, 40, _log(rng, 4, 40)))
        c["rows"] = rng.choice((1, 1, 2, 3, 4))
        c["f"] = rng.choice((1, 1, 2, 3))
        c["h"], c["w"] = _log(rng, 9, 45), _log(rng, 16, 80)
        c["frames"] = c["f"] * max(2, _log(rng, 4, 21) // c["f"])
        c["norm"] = rng.random() < 0.6
        if c["kind"] == "cross":
            c["norm"], c["text"] = True, rng.choice((512, _log(rng, 77, 512)))
        if c["kind"] == "module":
            c["norm"] = True
        if c["kind"] == "stream":
            option = rng.choice(("", "", "", "first", "fp32", "adaptive", "block", "hot"))
            if option == "first":
                c["first"], c["rows"] = True, 1
            elif option == "fp32":
                c["dtype"] = "fp32"
            elif option == "adaptive":
                c["f"], c["sink"], c["thr"], c["frames"] = 1, rng.choice((1, 2, 3)), 0.2, rng.choice((5, 6, 8, 12))
            elif option == "block":
                c["f"], c["block"], c["frames"] = 3, rng.choice((1, 2)), rng.choice((6, 9, 12, 21))
            elif option == "hot":
                c["hot"] = 0.01
        one = dict(c, layers=1)
        w = work(one)
        # an fp32 product costs what sixteen bf16 ones do
        cost = w["flops"] * (40 if c["dtype"] == "fp32" else 1) + 300 * w["bytes"]
        c["layers"] = 8 if c["thr"] >= 0 else max(1, min(6, int(most / 8 / max(cost, 1))))
        if cost * c["layers"] <= most and c["heads"] * c["rows"] * c["frames"] * c["h"] * c["w"] * c["layers"] <= 8e6:
            return c


def _sizes(c):
    frame = c["h"] * c["w"]
    return frame, c["f"] * frame, c["frames"] * frame          # tokens of a frame, a chunk, the cache


def _pairs(c):
    """(query, key) pairs of one row and head."""
    frame, s, cap = _sizes(c)
    if c["kind"] == "cross":
        return s * c["text"]
    keys = s if c["first"] else cap
    pairs = s * keys
    if 0 < c["block"] < c["f"]:
        b = c["block"] * frame
        pairs -= sum(min(b, s - t) * (s - t - b) for t in range(0, s, b) if t + b < s)
    return pairs


def work(c):
    """What one pass cannot do without: each input read once, each output written once."""
    frame, s, cap = _sizes(c)
    e = 2 if c["dtype"] == "bf16" else 4
    width = c["heads"] * 128
    token = c["rows"] * width * e                              # one token of every row
    attention = 4.0 * c["rows"] * c["heads"] * 128 * _pairs(c)
    if c["kind"] == "handoff":
        return {"bytes": float(c["layers"]) * 8 * cap * token, "flops": 0.0}           # k and v, out and in
    if c["kind"] == "cross":
        # x, q and o weights, cached keys and values (one copy for all rows), the result
        data = 2 * s * token + 2 * width * width * e + 2 * c["text"] * width * e
        return {"bytes": float(c["layers"]) * data, "flops": c["layers"] * (attention + 4.0 * c["rows"] * s * width * width)}
    passes = STEPS if c["first"] else 1
    keys = s if c["first"] else cap
    if c["kind"] == "module":
        # x, four weights, the old keys and values, the new ones, the result
        data = (2 * s + 2 * (keys - s) + 2 * s) * token + 4 * width * width * e
        return {"bytes": float(c["layers"]) * data, "flops": c["layers"] * (attention + 8.0 * c["rows"] * s * width * width)}
    # q, k and v, the old keys and values, the new ones, the result
    data = (3 * s + 2 * (keys - s) + 2 * s + s) * token
    return {"bytes": float(passes) * c["layers"] * data, "flops": passes * c["layers"] * attention}


def tolerance(c):
    if c["kind"] == "handoff":
        return "exact"
    return {"rel": 1e-5} if c["dtype"] == "fp32" else {"rel": 1e-2}


@functools.lru_cache(maxsize=None)
def _freqs():
    """The model's RoPE table, built once per program."""
    return rope.build_freqs()


class _Random:
    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(self, shape, dtype, scale=1.0):
        return torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32).mul_(scale).to(dtype)


def _caches(c, rows):
    caches = ring.new_kv_cache(c["layers"], 1, _sizes(c)[2], c["heads"], total_steps=STEPS if c["first"] else 1,
                               dtype=DTYPES[c["dtype"]], device="cuda")
    if rows > 1:
        ring.replicate_for_stream_batch(caches, rows)
    return caches


def _steady_start(c):
    """Position of a chunk late in a stream: the drivers keep it at the cache's last frame."""
    frame, _, cap = _sizes(c)
    return [cap - frame] * c["rows"]


def _fill(c, caches, path_of, chunk_of):
    """Chunk by chunk to a full cache, as a stream gets there, and a little further."""
    _, s, cap = _sizes(c)
    for i in range(cap // s + 2):
        start = [i * s] * c["rows"] if (i + 1) * s <= cap else _steady_start(c)
        for layer, cache in enumerate(caches):
            path_of(layer, chunk_of(layer, i), cache, start)


def _qkv(c, rnd, shape, mean=None):
    """q, k and v of one chunk and block: unit normal like normalised activations (or raw projections of the same
    distribution), with rows of outliers among the keys or a scene's mean where the case has them."""
    dt = DTYPES[c["dtype"]]
    q, k, v = (rnd.normal(shape, dt, c["scale"]) for _ in range(3))
    if c["hot"]:
        hot = torch.rand((shape[0], shape[1], 1, 1), generator=rnd.gen, device="cuda") < c["hot"]
        k = torch.where(hot, k * 8, k)
    if mean is not None:
        k, v = (k.float() + mean[0]).to(dt), (v.float() + mean[1]).to(dt)
    return q, k, v


def _prepare_stream(c, rnd):
    _, s, _ = _sizes(c)
    shape = (c["rows"], s, c["heads"], 128)
    dt = DTYPES[c["dtype"]]
    width = c["heads"] * 128
    norms = [((1 + rnd.normal((width,), torch.float32, 0.1)).to(dt), (1 + rnd.normal((width,), torch.float32, 0.1)).to(dt), EPS)
             if c["norm"] else None for _ in range(c["layers"])]
    paths = [RingKVPath(sink_size=c["sink"], adapt_sink_thr=c["thr"]) for _ in range(c["layers"])]
    for p in paths:
        p.block_frames = c["block"] or None
    caches = _caches(c, c["rows"])
    adaptive = c["thr"] >= 0
    scenes = None
    if adaptive:
        # what is common to a scene's tokens, and how it drifts from chunk to chunk
        scenes = [[rnd.normal((1, 1, c["heads"], 128), torch.float32) for _ in range(4)] for _ in range(c["layers"])]

    def mean(layer, drift, cut):
        if not adaptive:
            return None
        mk, mv, dk, dv = scenes[layer]
        sign = -1.0 if cut else 1.0
        return sign * (mk + drift * dk), sign * (mv + drift * dv)

    state = {"case": c, "step": 0, "grid": torch.tensor([[c["f"], c["h"], c["w"]]] * c["rows"]), "norms": norms,
             "paths": paths, "caches": caches}
    count = CUT_EVERY if adaptive else 2
    state["inputs"] = [[_qkv(c, rnd, shape, mean(layer, 0.0, adaptive and i == count - 1)) for layer in range(c["layers"])]
                       for i in range(count)]
    if c["first"]:
        state["start"] = [0]
    else:
        state["start"] = _steady_start(c)

        def call(layer, qkv, cache, start):
            paths[layer].attend(*qkv, state["grid"], _freqs(), cache, start, qk_norm=norms[layer])

        _fill(c, caches, call, lambda layer, i: _qkv(c, rnd, shape, mean(layer, 0.5 * i, False)))
    return state


def _run_stream(state):
    c, freqs = state["case"], _freqs()
    qkv = state["inputs"][state["step"] % len(state["inputs"])]
    state["step"] += 1
    out = []
    for _ in range(STEPS if c["first"] else 1):
        out.append([state["paths"][i].attend(*qkv[i], state["grid"], freqs, state["caches"][i], state["start"],
                                             qk_norm=state["norms"][i]) for i in range(c["layers"])])
    return out[-1], _contents(state["caches"])


def _contents(caches):
    return [[e[n] for n in ("k", "v", "global_end_index", "local_end_index")] for e in caches]


def _weights(module, c, rnd):
    """A module on the GPU with weights of the usual spread."""
    module = module.to(device="cuda", dtype=DTYPES[c["dtype"]])
    width = c["heads"] * 128
    with torch.no_grad():
        for name, p in module.named_parameters():
            if name.startswith("norm"):
                p.copy_(1 + rnd.normal(p.shape, torch.float32, 0.1))
            else:
                p.copy_(rnd.normal(p.shape, torch.float32, width ** -0.5))
    return module


def _modules(cls, c, rnd):
    width = c["heads"] * 128
    with torch.device("meta"):
        made = [cls(width, c["heads"], eps=EPS) for _ in range(c["layers"])]
    return [_weights(m.to_empty(device="cuda"), c, rnd) for m in made]


def _prepare_module(c, rnd):
    _, s, _ = _sizes(c)
    shape = (c["rows"], s, c["heads"] * 128)
    modules = _modules(CausalWanSelfAttention, c, rnd)
    for m in modules:
        m.sink_size, m.adapt_sink_thr = c["sink"], c["thr"]
    caches = _caches(c, c["rows"])
    state = {"case": c, "step": 0, "grid": torch.tensor([[c["f"], c["h"], c["w"]]] * c["rows"]), "modules": modules,
             "caches": caches, "start": _steady_start(c),
             "inputs": [rnd.normal(shape, DTYPES[c["dtype"]]) for _ in range(2)]}

    def call(layer, x, cache, start):
        modules[layer](x, None, state["grid"], _freqs(), None, kv_cache=cache, current_start=start)

    with torch.no_grad():
        _fill(c, caches, call, lambda layer, i: rnd.normal(shape, DTYPES[c["dtype"]]))
    return state


def _run_module(state):
    x = state["inputs"][state["step"] % len(state["inputs"])]
    state["step"] += 1
    # (in a model each block's result joins the next one's input; here every block gets the chunk's own)
    with torch.no_grad():
        out = [module(x, None, state["grid"], _freqs(), None, kv_cache=cache, current_start=state["start"])
               for module, cache in zip(state["modules"], state["caches"])]
    return out, _contents(state["caches"])


def _prepare_cross(c, rnd):
    _, s, _ = _sizes(c)
    width, dt = c["heads"] * 128, DTYPES[c["dtype"]]
    modules = _modules(WanT2VCrossAttention, c, rnd)
    caches = ring.new_crossattn_cache(c["layers"], 1, c["heads"], dtype=dt, device="cuda", text_tokens=c["text"])
    prompt = rnd.normal((1, c["text"], width), dt)
    x = [rnd.normal((c["rows"], s, width), dt) for _ in range(2)]
    with torch.no_grad():
        for module, cache in zip(modules, caches):
            module(x[0][:1], prompt, None, crossattn_cache=cache)          # the prompt's keys and values, once
    if c["rows"] > 1:
        ring.expand_crossattn_for_stream_batch(caches, c["rows"])
    return {"case": c, "step": 0, "modules": modules, "caches": caches, "prompt": prompt, "inputs": x}


def _run_cross(state):
    x = state["inputs"][state["step"] % len(state["inputs"])]
    state["step"] += 1
    with torch.no_grad():
        return [module(x, state["prompt"], None, crossattn_cache=cache) for module, cache in zip(state["modules"], state["caches"])]


def _prepare_handoff(c, rnd):
    _, s, cap = _sizes(c)
    sides = [_caches(c, c["rows"]) for _ in range(2)]
    for entry in sides[0]:
        for name in ("k", "v"):
            entry[name].permute(0, 2, 1, 3).copy_(rnd.normal((c["rows"], c["heads"], cap, 128), DTYPES[c["dtype"]]))
        entry["global_end_index"].fill_(cap + s)
        entry["local_end_index"].fill_(cap)
    return {"case": c, "donor": sides[0], "receiver": sides[1], "wires": [handoff.new_wire_like(e) for e in sides[0]]}


def _run_handoff(state):
    frame = _sizes(state["case"])[0]
    for source, target, wire in zip(state["donor"], state["receiver"], state["wires"]):
        handoff.export_block(source, wire)
        handoff.import_block(target, wire, donor_rank=2, rank=1, frame_seq_length=frame, time_step_length=STEPS)
    return [[w.k, w.v, w.global_end_index, w.local_end_index] for w in state["wires"]], _contents(state["receiver"])


_KINDS = {
    "stream": (_prepare_stream, _run_stream),
    "module": (_prepare_module, _run_module),
    "cross": (_prepare_cross, _run_cross),
    "handoff": (_prepare_handoff, _run_handoff),
}


def prepare(case, seed):
    return _KINDS[case["kind"]][0](dict(case), _Random(seed))


def run(state):
    return _KINDS[state["case"]["kind"]][1](state)
