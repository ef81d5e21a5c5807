"""Workloads of the token loop that are timed, each through a public entry point.

A case is a dict of plain values; ``kind`` names the call:

decode   one decode step after ``rows`` cached rows (plamo_metal_forward), then
         plamo_hip_rewind, so that the same step can be taken again
stream   one decode step on full sliding windows: every step drops the oldest
         row of each window and the positions move on
prefill  a request: counters reset, the ``prefix`` rows of the prompt template
         restored (runtime/prompt_cache.c does the same copies), then the
         other ``tokens`` ids in one plamo_metal_prefill
verify   one batch of draft candidates (plamo_metal_verify), all of them
         committed, then rewound
linear   plamo_metal_linear: one projection of host rows
mlp      plamo_metal_mlp: one MLP branch with its residual on host rows

Widths are the repository's configurations (plamo_hip.CONFIGS) with fewer
layers; every ``pattern``-th layer is global (0: none), the others keep a
sliding window of 2048. Weights, ids and cached rows come from the seed.
"""

import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "plamo-3-translate.c_amd"))
import plamo_hip  # noqa: E402

WINDOW = 2048
GLOBAL_ROWS = 8192


def listed():
    return [
        # Greedy decoding with the smallest configuration, whole model with its
        # 100000-row head, shortly after a 128-token prompt.
        dict(name="decode c2 whole", kind="decode", width="c2", layers=16, pattern=8,
             vocab=100000, rows=140, pinned=True),
        # Decode layers of the headline configuration at the same context.
        dict(name="decode c4", kind="decode", width="c4", layers=4, pattern=4, vocab=1000,
             rows=140, pinned=True),
        # The same layers late in a long translation (window nearly full).
        dict(name="decode c4 long", kind="decode", width="c4", layers=4, pattern=4, vocab=1000,
             rows=1900, pinned=True),
        # Decoding past the window: a document longer than 2048 tokens.
        dict(name="stream c3", kind="stream", width="c3", layers=2, pattern=0, vocab=1000,
             pinned=True),
        # Time to first token of a 128- and a 455-token prompt whose 12-token
        # template prefix is restored.
        dict(name="prefill c4 116", kind="prefill", width="c4", layers=4, pattern=4, vocab=1000,
             prefix=12, tokens=116, pinned=True),
        dict(name="prefill c4 443", kind="prefill", width="c4", layers=4, pattern=4, vocab=1000,
             prefix=12, tokens=443, pinned=True),
        # A page of text that still fits the window.
        dict(name="prefill c4 1900", kind="prefill", width="c4", layers=2, pattern=2, vocab=1000,
             prefix=12, tokens=1900, pinned=True),
        # A document that does not (prompts may have up to 4096 tokens).
        dict(name="prefill c2 3500", kind="prefill", width="c2", layers=4, pattern=4, vocab=1000,
             prefix=0, tokens=3500, pinned=True),
        # Speculative decoding: four draft tokens and the bonus position, and a
        # long batch of a confident draft.
        dict(name="verify c5 5", kind="verify", width="c5", layers=2, pattern=2, vocab=1000,
             rows=455, candidates=5, pinned=True),
        dict(name="verify c4 12", kind="verify", width="c4", layers=2, pattern=2, vocab=1000,
             rows=300, candidates=12, pinned=True),
        # The projection and MLP hooks, which the engine calls when no fused
        # path applies: the smallest projection, and a few ragged rows.
        dict(name="linear 1", kind="linear", rows=3072, cols=2048, tokens=1),
        dict(name="mlp 37", kind="mlp", hidden=2560, intermediate=10240, tokens=37),
    ]


# ------------------------------------------------------------------ the range
MOST_PARAMETERS = 1.1e9     # projection weights of a drawn model
MOST_PRODUCTS = 0.9e12      # tokens x projection weights of a drawn prompt
MOST_WINDOW_HEADS = 3 * 16  # sliding layers x query heads of a prompt past the window


def draw(rng):
    def spread(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))

    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "verify",
                       "stream", "linear", "mlp"])
    if kind == "linear":
        step = rng.choice([512, 256, 64, 64, 8, 1])
        cols = max(step, spread(192, 8192) // step * step)
        return dict(kind=kind, rows=spread(64, 16384), cols=cols, tokens=spread(1, 600))
    if kind == "mlp":
        cfg = plamo_hip.CONFIGS[rng.choice(["c2", "c3", "c4"])]
        return dict(kind=kind, hidden=cfg["hidden"], intermediate=cfg["intermediate"],
                    tokens=spread(1, 600))
    width = rng.choice(["c2", "c3", "c4", "c5"])
    per_layer = layer_parameters(plamo_hip.CONFIGS[width])
    most = max(1, int(MOST_PARAMETERS // per_layer))
    layers = rng.randint(1, min(6, most))
    case = dict(kind=kind, width=width, layers=layers, pattern=rng.choice([2, 4]),
                vocab=rng.choice([1000, 10007]), pinned=rng.random() < 0.8)
    if kind == "decode":
        case["rows"] = spread(1, WINDOW - 1)
    elif kind == "stream":
        case["layers"], case["pattern"] = rng.randint(1, 2), 0
    elif kind == "verify":
        case["rows"], case["candidates"] = spread(16, 2000), rng.randint(1, 16)
    else:
        case["prefix"] = rng.choice([0, 12, 12, rng.randint(1, 64)])
        tokens = min(spread(1, 3500), int(MOST_PRODUCTS / (per_layer * layers)))
        sliding = layers - layers // case["pattern"]
        if case["prefix"] + tokens > WINDOW + 1 and \
                sliding * plamo_hip.CONFIGS[width]["qh"] > MOST_WINDOW_HEADS:
            tokens = WINDOW + 1 - case["prefix"]
        case["tokens"] = tokens
    return case


# ------------------------------------------------------------------ states
def layer_parameters(cfg):
    h, d, qh, kh, inter = cfg["hidden"], cfg["dim"], cfg["qh"], cfg["kh"], cfg["intermediate"]
    return (qh + 2 * kh) * d * h + h * qh * d + 3 * inter * h


def build(case, seed):
    cfg = dict(plamo_hip.CONFIGS[case["width"]])
    cfg.pop("tied", None)
    cfg.update(layers=case["layers"], vocab=case["vocab"])
    return plamo_hip.Synthetic(**cfg, window=WINDOW, global_capacity=GLOBAL_ROWS,
                               pattern=case["pattern"], seed=seed)


def generator(seed, salt):
    return np.random.Generator(np.random.PCG64([seed, salt]))


def token_ids(case, seed):
    count = {"decode": 1, "stream": 2, "verify": case.get("candidates", 1),
             "prefill": case.get("prefix", 0) + case.get("tokens", 0)}[case["kind"]]
    return generator(seed, 1).integers(0, case["vocab"], size=count).tolist()


def fill(case, inst, rows, seed):
    """Every cache holds `rows` rows of raw K and V ~ N(0,1), rotations stale."""
    rng = generator(seed, 2)
    for i in range(inst.model.count):
        for which in ("k", "v"):
            inst.kv(i, which)[:rows] = rng.standard_normal((rows, inst.cache(i).width),
                                                           dtype=np.float32)
        inst.cache(i).count = rows
        inst.rotation(i).processed_count = 0
        inst.rotation(i).scale_bits = 0


class Handles:
    """A resident model and a request's host arrays, closed with their last user."""

    def __init__(self, case, seed):
        self.backend = self.inst = None
        self.syn = build(case, seed)
        self.inst = self.syn.instance(pinned=case["pinned"])
        self.backend = plamo_hip.Backend(self.syn)

    def view(self, array):
        """The same memory as `array`, keeping these handles open."""
        memory = Memory()
        memory.handles, memory.__array_interface__ = self, dict(array.__array_interface__)
        return np.asarray(memory)

    def __del__(self):
        for part in (self.backend, self.inst, self.syn):
            if part is not None:
                part.close()


class Memory:
    pass


class ModelState:
    """A model and a request (see Handles) and the ids of the call."""

    def __init__(self, case, seed):
        handles = Handles(case, seed)
        self.case, self.backend, self.inst = case, handles.backend, handles.inst
        inst, kind, layers = self.inst, case["kind"], case["layers"]
        self.ids = token_ids(case, seed)
        self.handles = handles
        self.arrays = [handles.view(inst.kv(i, w)) for i in range(layers)
                       for w in ("k", "v", "rot")]
        self.caches = [inst.cache(i) for i in range(layers)]
        self.rotations = [inst.rotation(i) for i in range(layers)]
        self.heads = [handles.view(a) for a in (inst.logits(), inst.state(), inst.normalized())]
        if kind in ("decode", "verify"):
            rows = case["rows"]
            fill(case, inst, rows, seed)
            # One step builds the rotations; it is undone again.
            self.need(self.backend.forward(inst, self.ids[0]) == 1 and self.rewind(1))
            steps = len(self.ids)
            self.out = self.heads + [a[rows:rows + steps] for a in self.arrays]
        elif kind == "stream":
            fill(case, inst, WINDOW + 1, seed)
            self.need(self.backend.forward(inst, self.ids[0]) == 1)
            self.out = self.heads + self.arrays
        else:
            prefix = case["prefix"]
            self.need(self.backend.prepare(inst) == 1)
            if prefix:
                self.need(self.backend.prefill(inst, self.ids[:prefix]) == 1)
            self.saved = [a[:prefix].copy() for a in self.arrays]
            self.scales = [r.scale_bits for r in self.rotations]
            self.body = self.ids[prefix:]
            end = prefix + case["tokens"]
            self.out = self.heads + [a[:min(end, c.capacity)] if end > c.capacity else a[prefix:end]
                                     for i, c in enumerate(self.caches)
                                     for a in self.arrays[3 * i:3 * i + 3]]

    def need(self, ok):
        if not ok:
            raise RuntimeError(self.backend.info().note.decode() or "the call was refused")

    def rewind(self, steps):
        return self.backend.lib.plamo_hip_rewind(self.backend.handle, self.inst.model_ptr,
                                                 steps) == 1

    def restore(self):
        self.inst.reset()
        prefix = self.case["prefix"]
        if prefix:
            for a, s in zip(self.arrays, self.saved):
                a[:prefix] = s
            for c, r, scale in zip(self.caches, self.rotations, self.scales):
                c.count = r.processed_count = prefix
                r.scale_bits = scale


class RowsState:
    """Host rows and resident weights of one projection or one MLP branch."""

    def __init__(self, case, seed):
        self.case = case
        self.parts = rows_inputs(case, seed)
        self.backend = plamo_hip.Backend()
        for name in ("w", "gu", "down"):
            if name in self.parts:
                a = self.parts[name]
                if not self.backend.preload(a.ctypes.data, a.nbytes):
                    raise RuntimeError(self.backend.info().note.decode())
        if case["kind"] == "mlp":
            p = self.parts
            u16 = lambda a: ctypes.cast(a.ctypes.data, plamo_hip.u16p)  # noqa: E731
            self.mlp = plamo_hip.Mlp(None, u16(p["pre"]), u16(p["post"]), u16(p["gu"]),
                                     u16(p["down"]), None, None, None, case["hidden"],
                                     case["intermediate"])
            self.states = p["x"].copy()

    def __del__(self):
        if getattr(self, "backend", None) is not None:
            self.backend.close()


def rows_inputs(case, seed):
    """BF16 weights ~ N(0, 0.02) as bit patterns, FP32 rows ~ N(0, 1)."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    gen = torch.Generator(device=dev).manual_seed(seed)

    def weight(*shape):
        w = torch.randn(shape, generator=gen, device=dev) * 0.02
        return w.to(torch.bfloat16).view(torch.int16).cpu().numpy().view(np.uint16)

    def rows(width):
        return torch.randn((case["tokens"], width), generator=gen, device=dev).cpu().numpy()

    if case["kind"] == "linear":
        return dict(w=weight(case["rows"], case["cols"]), x=rows(case["cols"]))
    h, inter = case["hidden"], case["intermediate"]
    return dict(pre=weight(h), post=weight(h), gu=weight(2 * inter, h), down=weight(h, inter),
                x=rows(h))


def prepare(case, seed):
    if case["kind"] in ("linear", "mlp"):
        return RowsState(case, seed)
    return ModelState(case, seed)


def run(state):
    case, be = state.case, state.backend
    kind = case["kind"]
    if kind == "linear":
        ok, y = be.linear(state.parts["w"].ctypes.data, state.parts["x"], case["rows"])
        if ok != 1:
            raise RuntimeError(be.info().note.decode())
        return y
    if kind == "mlp":
        np.copyto(state.states, state.parts["x"])  # the branch is added in place
        if be.lib.plamo_metal_mlp(be.handle, ctypes.byref(state.mlp),
                                  state.states.ctypes.data_as(plamo_hip.f32p),
                                  case["tokens"]) != 1:
            raise RuntimeError(be.info().note.decode())
        return state.states
    inst = state.inst
    if kind == "decode":
        state.need(be.forward(inst, state.ids[0]) == 1 and state.rewind(1))
    elif kind == "stream":
        state.need(be.forward(inst, state.ids[1]) == 1)
    elif kind == "prefill":
        state.restore()
        state.need(be.prefill(inst, state.body) == 1)
    else:
        ok, nxt = be.verify(inst, state.ids)
        state.need(ok == 1 and all(be.commit(inst, i) == 1 for i in range(len(nxt))) and
                   state.rewind(len(nxt)))
        return state.out + [np.array(nxt, dtype=np.int64)]
    return state.out


# ------------------------------------------------------------------ work
def work(case):
    """Every weight, cached row and input read once, every output written
    once; 2 operations per product."""
    if case["kind"] == "linear":
        n, k, t = case["rows"], case["cols"], case["tokens"]
        return {"bytes": 2 * n * k + 4 * t * (n + k), "flops": 2 * n * k * t}
    if case["kind"] == "mlp":
        h, inter, t = case["hidden"], case["intermediate"], case["tokens"]
        return {"bytes": 6 * h * inter + 8 * t * h, "flops": 6 * h * inter * t}
    cfg = plamo_hip.CONFIGS[case["width"]]
    h, d, qh, kh, layers = cfg["hidden"], cfg["dim"], cfg["qh"], cfg["kh"], case["layers"]
    per_layer, head = layer_parameters(cfg), case["vocab"] * h
    cached = {"decode": case.get("rows", 0), "verify": case.get("rows", 0), "stream": WINDOW,
              "prefill": case.get("prefix", 0)}[case["kind"]]
    new = case.get("tokens", case.get("candidates", 1))
    logits_rows = new if case["kind"] == "verify" else 1
    nbytes = 2 * (per_layer * layers + head) + 4 * (case["vocab"] + 2 * h)
    flops = 2 * (per_layer * layers * new + head * logits_rows)
    for i in range(layers):
        is_global = case["pattern"] and (i + 1) % case["pattern"] == 0
        limit = GLOBAL_ROWS if is_global else WINDOW + 1
        # Rotated keys and values read, three rows written per new token; a
        # full window's rotated keys are all new.
        kept = min(cached + new, limit)
        moved = kept if cached + new > limit else new
        nbytes += 4 * kh * d * (2 * min(cached, limit) + 2 * min(new, kept) + moved)
        pairs = sum(min(cached + t + 1, limit) for t in range(new))
        flops += 4 * pairs * d * qh
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # FP32 sums in another order: about four times what the calls are off
    # exact(). Model calls are up to 2e-5 off (1900 cached rows, whose rotation
    # angles are rounded to FP32), one projection or MLP branch up to 1e-6.
    if case["kind"] == "linear":
        return {"rel": 4e-6}
    if case["kind"] == "mlp":
        return {"rel": 4e-6}
    return {"rel": 8e-5, "max": 3e-3}


# ------------------------------------------------------------------ 64 bits
def exact(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"

    def wide(bits):
        t = torch.from_numpy(np.ascontiguousarray(bits).view(np.int16)).to(dev)
        return t.view(torch.bfloat16).to(torch.float64)

    def rms(x):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)

    def branch(x, pre, gu, down):
        gate, up = ((rms(x) * (wide(pre) + 1)) @ wide(gu).T).chunk(2, -1)
        return (gate * torch.sigmoid(gate) * up) @ wide(down).T

    if case["kind"] == "linear":
        p = rows_inputs(case, seed)
        x = torch.from_numpy(p["x"]).to(dev).double()
        return (x @ wide(p["w"]).T).cpu().numpy()
    mlp_offset = 0.08944271909999159
    if case["kind"] == "mlp":
        p = rows_inputs(case, seed)
        x = torch.from_numpy(p["x"]).to(dev).double()
        out = branch(x, p["pre"], p["gu"], p["down"])
        return (x + rms(out) * (wide(p["post"]) + mlp_offset)).cpu().numpy()

    cfg = plamo_hip.CONFIGS[case["width"]]
    h, d, qh, kh, inter = (cfg[k] for k in ("hidden", "dim", "qh", "kh", "intermediate"))
    syn = build(case, seed)
    inst = syn.instance()
    try:
        m, ids, kind = inst.model, token_ids(case, seed), case["kind"]
        rows = {"decode": case.get("rows"), "verify": case.get("rows"), "stream": WINDOW + 1,
                "prefill": 0}[kind]
        if rows:
            fill(case, inst, rows, seed)

        def bits(ptr, *shape):
            return np.ctypeslib.as_array(ptr, shape=shape)

        def rotate(x, positions, freq, scale):
            angle = positions.double()[:, None] * freq
            c, s = torch.cos(angle) * scale, torch.sin(angle) * scale
            if x.dim() == 3:
                c, s = c[:, None], s[:, None]
            a, b = x.chunk(2, -1)
            return torch.cat([a * c - b * s, b * c + a * s], -1)

        emb = bits(m.embedding, m.vocab, h)
        state = wide(emb[np.array(ids)])
        new = len(ids)
        caches = []
        for i in range(m.count):
            layer = m.layers[i].contents
            mx, p = layer.mixer.contents, layer.mlp.contents
            q, c, r = mx.qkv.contents, mx.cache.contents, mx.rotation.contents
            freq = torch.from_numpy(bits(r.freq, d // 2).copy()).to(dev).double()
            scale = float(m.scales[i])
            x = rms(state) * (wide(bits(layer.pre, h)) + 1)
            y = x @ wide(bits(q.weight, (qh + 2 * kh) * d, h)).T
            qs, ks, vs = y.split([qh * d, kh * d, kh * d], -1)
            qs = rms(qs.reshape(new, qh, d)) * (wide(bits(q.qn, d)) + 1)
            ks = rms(ks.reshape(new, kh, d)) * (wide(bits(q.kn, d)) + 1)
            vs = vs.reshape(new, kh, d)
            if rows:
                old = [torch.from_numpy(inst.kv(i, w)[:rows].reshape(rows, kh, d).copy())
                       .to(dev).double() for w in ("k", "v")]
                ks, vs = torch.cat([old[0], ks]), torch.cat([old[1], vs])
            total = ks.shape[0]
            at = torch.arange(total, device=dev)
            # Scores depend on the distance alone, so absolute positions do.
            qr, kr = rotate(qs, at[total - new:], freq, scale), rotate(ks, at, freq, scale)
            gap = at[total - new:, None] - at[None, :]
            seen = (gap >= 0) & (gap < c.capacity)
            heads = []
            for head in range(qh):
                kv = head // (qh // kh)
                s = (qr[:, head] @ kr[:, kv].T) / math.sqrt(d)
                heads.append(torch.softmax(s.masked_fill(~seen, -math.inf), -1) @ vs[:, kv])
            out = torch.cat(heads, -1) @ wide(bits(mx.weight, h, qh * d)).T
            state = state + rms(out) * (wide(bits(layer.post, h)) + 0.2)
            out = branch(state, bits(p.pre, h), bits(p.gu, 2 * inter, h), bits(p.down, h, inter))
            state = state + rms(out) * (wide(bits(p.post, h)) + mlp_offset)
            kept = min(total, c.capacity)
            ks, vs = ks[total - kept:], vs[total - kept:]
            rot = rotate(ks, torch.arange(kept, device=dev), freq, scale)
            first = 0 if kind == "stream" or total > c.capacity else total - new
            if kind == "prefill" and total <= c.capacity:
                first = case["prefix"]
            caches += [t.reshape(kept, kh * d)[first:].cpu().numpy() for t in (ks, vs, rot)]
        normalized = rms(state) * (wide(bits(m.norm, h)) + 1)
        logits = normalized @ wide(bits(m.head, m.vocab, h)).T
        result = [logits[-1].cpu().numpy(), state[-1].cpu().numpy(), normalized[-1].cpu().numpy()]
        result += caches
        if kind == "verify":
            result.append(logits.argmax(-1).cpu().numpy())
        return result
    finally:
        inst.close()
        syn.close()
