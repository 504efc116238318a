"""The work that a user of this library has it do, as cases that can be timed.

Each case is one pass through the public entry points (fastgemma_amd.kernels,
or the C ABI of include/fgm_hip.h where the Python layer has no wrapper or
where a program keeps the descriptors):

* ``linear``: Gemm::run on GPU buffers, prep_rows (rotate, quantise, pack) then
  gemm_q8c / gemm_q4g;
* ``dropin``: the same on host buffers through the drop-in symbols;
* ``mlp``: the feed-forward block: rmsnorm fused with the prep, gate and up in
  one batched call, gelu_mul fused with the prep, down, post-norm, residual;
* ``attn``: one attention job per layer over the int8 KV cache;
* ``head``: final norm, int8 LM head, softcap;
* ``step``: a whole decode step of a small stack of layers, eager, to logits.

Every kernel here reproduces the reference's arithmetic bit for bit (the tests
hold it to that at tolerance 0), so outputs are compared exactly.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import fastgemma_amd as F
from fastgemma_amd import kernels as K

EPS = 1e-6
DEV = "cuda"


# ------------------------------------------------------------------- cases
def listed():
    return [
        # one token's int8 projection: launch- and latency-bound
        {"name": "linear_int8_m1", "kind": "linear", "bits": 8, "m": 1, "n": 8192, "k": 2048, "group": 0, "hsz": 0},
        # speculative / small-batch rows: a ragged M between the skinny and dense
        # kernels, wide int4 groups, rotated activations
        {"name": "linear_int4_m37_had", "kind": "linear", "bits": 4, "m": 37, "n": 6144, "k": 1536, "group": 128,
         "hsz": 128},
        # a CPU host program calling the drop-in symbols with its own buffers
        {"name": "dropin_int4_m8", "kind": "dropin", "bits": 4, "m": 8, "n": 8192, "k": 2048, "group": 64, "hsz": 0},
        # batched decode: the feed-forward blocks between attention calls, kept as
        # captured graphs by a serving loop (all weights from HBM)
        {"name": "mlp_decode_int4_m8", "kind": "mlp", "m": 8, "d": 2048, "ff": 8192, "bits": 4, "down_bits": 8,
         "group": 64, "hsz": 0, "heavy": False, "layers": 4, "graph": True},
        # a 256-token prefill chunk on the int8 twins
        {"name": "mlp_prefill_int8_m256", "kind": "mlp", "m": 256, "d": 2048, "ff": 8192, "bits": 8, "down_bits": 8,
         "group": 0, "hsz": 0, "heavy": False, "layers": 1, "graph": False},
        # a long prompt, int4 gate / up and int8 down, heavy-tailed activations
        {"name": "mlp_prefill_int4_m2048", "kind": "mlp", "m": 2048, "d": 2048, "ff": 8192, "bits": 4,
         "down_bits": 8, "group": 64, "hsz": 0, "heavy": True, "layers": 1, "graph": False},
        # batched decode over long contexts (a full-attention layer), ragged lengths
        {"name": "attn_decode_full", "kind": "attn", "seqs": 8, "rows": 1, "ctx": 8192, "window": 0, "ring": False,
         "nh": 8, "kvh": 1, "hd": 512, "layers": 2},
        # batched decode, the sliding-window layers of a step on ring caches
        {"name": "attn_decode_sliding", "kind": "attn", "seqs": 8, "rows": 1, "ctx": 20001, "window": 512,
         "ring": True, "nh": 8, "kvh": 1, "hd": 256, "layers": 4},
        # the last 256-token chunk of an 8k prompt, full attention
        {"name": "attn_prefill_full", "kind": "attn", "seqs": 1, "rows": 256, "ctx": 8192, "window": 0,
         "ring": False, "nh": 8, "kvh": 1, "hd": 512, "layers": 1},
        # a 256-token chunk through a sliding-window layer
        {"name": "attn_prefill_sliding", "kind": "attn", "seqs": 1, "rows": 256, "ctx": 20001, "window": 512,
         "ring": True, "nh": 8, "kvh": 1, "hd": 256, "layers": 1},
        # the LM head of a decode step: the largest single weight
        {"name": "head_int8_m8", "kind": "head", "m": 8, "n": 262144, "k": 2048, "cap": 30.0},
        # a whole decode step of four sequences through three sliding layers and one
        # full one, to logits
        {"name": "step_m4", "kind": "step", "m": 4, "d": 2048, "ff": 8192, "nh": 8, "kvh": 2, "hd": 256,
         "ctx": 1500, "window": 512, "layers": 4, "group": 64, "hsz": 0, "vocab": 32768},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _m64(rng, lo, hi):
    return max(64, _log(rng, lo, hi) // 64 * 64)


def _group(rng, k):
    return rng.choice([g for g in (64, 64, 128, 256, 512) if k % g == 0])


def _hsz(rng, k):
    return rng.choice([0, 0] + [h for h in (16, 128, 256, 512) if k % h == 0])


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "dropin", "mlp", "mlp", "attn", "attn", "attn", "head", "step"])
    if kind in ("linear", "dropin"):
        m = _log(rng, 1, 2048 if kind == "linear" else 64)
        n, k = _m64(rng, 512, 12288), _m64(rng, 512, 8192)
        bits = rng.choice([4, 8])
        return {"kind": kind, "bits": bits, "m": m, "n": n, "k": k, "group": _group(rng, k) if bits == 4 else 0,
                "hsz": _hsz(rng, k)}
    if kind == "mlp":
        d, ff, bits = _m64(rng, 1024, 2048), _m64(rng, 4096, 8192), rng.choice([4, 8])
        graph = rng.random() < 0.5
        return {"kind": "mlp", "m": _log(rng, 1, 32) if graph else _log(rng, 33, 2000), "d": d, "ff": ff,
                "bits": bits, "down_bits": rng.choice([bits, 8]), "group": rng.choice([64, 128]) if d % 128 == 0 and
                ff % 128 == 0 else 64, "hsz": _hsz(rng, math.gcd(d, ff)), "heavy": rng.random() < 0.3,
                "layers": rng.randint(2, 4) if graph else 1, "graph": graph}
    if kind == "attn":
        window = rng.choice([0, 0, rng.randint(128, 1024)])
        kvh, hd = rng.choice([(1, 256), (1, 512), (2, 256), (4, 128)])
        if rng.random() < 0.5:  # decode
            return {"kind": "attn", "seqs": rng.randint(1, 12), "rows": 1, "ctx": _log(rng, 100, 8192),
                    "window": window, "ring": window > 0, "nh": 8, "kvh": kvh, "hd": hd, "layers": 2}
        rows = rng.randint(24, 250)
        return {"kind": "attn", "seqs": 1, "rows": rows, "ctx": max(rows, _log(rng, 256, 8000)), "window": window,
                "ring": window > 0, "nh": 8, "kvh": kvh, "hd": hd, "layers": 1}
    if kind == "head":
        return {"kind": "head", "m": rng.randint(1, 16), "n": _m64(rng, 32768, 200000), "k": _m64(rng, 1024, 2048),
                "cap": 30.0}
    kvh, hd = rng.choice([(1, 256), (2, 256), (4, 128)])
    return {"kind": "step", "m": rng.randint(1, 6), "d": _m64(rng, 1024, 2048), "ff": _m64(rng, 3072, 8192),
            "nh": 8, "kvh": kvh, "hd": hd, "ctx": _log(rng, 64, 2000), "window": rng.choice([256, 512]),
            "layers": rng.randint(1, 4), "group": 64, "hsz": 0, "vocab": 64 * rng.randint(64, 500)}


# ------------------------------------------------------------------ inputs
class _Gen:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed & 0x7FFFFFFF)

    def normal(self, *shape):
        return torch.randn(*shape, generator=self.g, device=DEV)

    def uniform(self, lo, hi, *shape):
        return torch.rand(*shape, generator=self.g, device=DEV) * (hi - lo) + lo

    def act(self, m, k, heavy=False):
        """Activation rows; heavy: Student-t (3 degrees) with a few large channels."""
        x = self.normal(m, k)
        if heavy:
            chi = self.normal(3, m, k).square_().sum(0)
            x = x / torch.sqrt(chi / 3)
            big = torch.randint(0, k, (max(1, k // 1000),), generator=self.g, device=DEV)
            x[:, big] *= 20
        return x

    def weight(self, bits, n, k, group):
        """A quantised weight and its scales.  The entries are independent, so the
        stored order (tiles, nibbles) holds the same distribution."""
        if bits == 8:
            b = torch.empty(n * k, dtype=torch.int8, device=DEV)
            step = 1 << 26
            for i in range(0, n * k, step):
                c = min(step, n * k - i)
                b[i:i + c] = (self.normal(c) * 38).round_().clamp_(-127, 127).to(torch.int8)
            return b, self.uniform(0.5, 1.5, n) / (38 * math.sqrt(k))
        lo, hi = ((self.normal(n * k // 2) * 2.6).round_().clamp_(-8, 7).to(torch.int32) for _ in range(2))
        b = ((lo & 15) | ((hi & 15) << 4)).to(torch.uint8)
        s = self.uniform(0.5, 1.5, k // group, n) / (2.6 * math.sqrt(k))
        return b, s.to(torch.float16).view(torch.int16)


def _prep_bufs(m, k):
    return (torch.empty(m, dtype=torch.float32, device=DEV),
            torch.empty(K.packed_a_len(m, k), dtype=torch.int8, device=DEV))


def _gemm(bits, m, n, k, group, qs, pa, w, c):
    return {"bits": bits, "m": m, "n": n, "k": k, "group": group or 64, "a": pa, "a_scale": qs, "b": w[0],
            "b_scale": w[1], "c": c, "ldc": n, "n0": 0, "n1": n // 16}


def _run_gemm(bits, m, n, k, group, qs, pa, w, c):
    if bits == 8:
        K.gemm_q8c(m, n, k, pa, qs, w[0], w[1], c, n, 0, n // 16)
    else:
        K.gemm_q4g(m, n, k, pa, qs, w[0], w[1], group, c, n, 0, n // 16)


def _mlp_weights(g, c):
    d, ff, gr = c["d"], c["ff"], c["group"]
    return {"gate": g.weight(c["bits"], ff, d, gr), "up": g.weight(c["bits"], ff, d, gr),
            "down": g.weight(c["down_bits"], d, ff, gr), "pre": g.uniform(0.5, 1.5, d),
            "post": g.uniform(0.5, 1.5, d)}


def _mlp_bufs(m, d, ff):
    z = lambda *s: torch.empty(*s, dtype=torch.float32, device=DEV)  # noqa: E731
    return {"p1": _prep_bufs(m, d), "p2": _prep_bufs(m, ff), "gate": z(m, ff), "up": z(m, ff), "down": z(m, d)}


def _mlp(c, m, x, w, b, out):
    """out = x + rmsnorm(down(gelu(gate(xn)) * up(xn))), xn = rmsnorm(x)."""
    d, ff, gr = c["d"], c["ff"], c["group"]
    (qs, pa), (qs2, pa2) = b["p1"], b["p2"]
    K.prep_rmsnorm(x, d, w["pre"], EPS, qs, pa, m, d, c["hsz"])
    K.gemm_batch([_gemm(c["bits"], m, ff, d, gr, qs, pa, w["gate"], b["gate"]),
                  _gemm(c["bits"], m, ff, d, gr, qs, pa, w["up"], b["up"])])
    K.prep_gelu_mul(b["gate"], b["up"], ff, qs2, pa2, m, ff, c["hsz"])
    _run_gemm(c["down_bits"], m, d, ff, gr, qs2, pa2, w["down"], b["down"])
    K.rmsnorm_rows(out, b["down"], w["post"], m, d, EPS)
    K.add(out, x)


class _Cache:
    """One layer's int8 KV caches of `seqs` sequences: [seq][slots]..., filled
    through the cache append as a running program fills it."""

    def __init__(self, g, seqs, slots, ring, kvd, lens):
        self.slots, self.ring = slots, ring
        self.kc = torch.zeros(seqs, slots * kvd, dtype=torch.int8, device=DEV)
        self.vt = torch.zeros(seqs, (slots + 3) // 4 * 4 * kvd, dtype=torch.int8, device=DEV)
        self.ks = torch.zeros(seqs, slots, device=DEV)
        self.vs = torch.zeros(seqs, slots, device=DEV)
        for i, n in enumerate(lens):
            have = min(n, slots)
            k, v = g.normal(have, kvd), g.normal(have, kvd)
            K.kv_store(k, v, have, kvd, self.kc[i], self.ks[i], self.vt[i], self.vs[i], slots, n - have, ring)
        torch.cuda.synchronize()

    def desc(self, i, pos, rows):
        return F.AttnSeq(self.kc[i].data_ptr(), self.ks[i].data_ptr(), self.vt[i].data_ptr(),
                         self.vs[i].data_ptr(), self.slots, self.ring, pos, rows)


def _span(pos, rows, window, ring):
    return max(ring, min(window, pos + rows) if window else pos + rows)


def _scratch(m, nh, kvh, hd, span):
    nb = K.attend_scratch_bytes(m, nh, kvh, hd, span)
    raw = torch.empty(nb + 256, dtype=torch.uint8, device=DEV)
    return raw, (raw.data_ptr() + 255) & ~255, nb


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _lens(c, g_seed):
    """Ragged lengths of the decoded sequences: the longest has c["ctx"] positions."""
    r = np.random.RandomState(g_seed & 0x7FFFFFFF)
    n = [c["ctx"]] + [int(c["ctx"] * f) for f in r.uniform(0.75, 1.0, c.get("seqs", c.get("m", 1)) - 1)]
    return [max(1, x) for x in n]


def _tiles8(b, n, k):
    """int8 tiles -> [n][k]."""
    return b.view(n // 16, k // 64, 16, 16, 4).permute(0, 3, 1, 2, 4).reshape(n, k)


def _unpack4(b):
    """Nibble-packed 64-byte blocks -> the int8 stream."""
    u = b.view(-1, 32).to(torch.int16)
    s = torch.cat([u & 15, u >> 4], 1)
    return torch.where(s > 7, s - 16, s).to(torch.int8).reshape(-1)


# ----------------------------------------------------------------- prepare
def _make(case, seed):
    c, g = case, _Gen(seed)
    kind = c["kind"]
    if kind in ("linear", "dropin"):
        x = g.act(c["m"], c["k"])
        w = g.weight(c["bits"], c["n"], c["k"], c["group"])
        return g, x, w
    if kind == "mlp":
        return g, g.act(c["m"], c["d"], c["heavy"]), [_mlp_weights(g, c) for _ in range(c["layers"])]
    if kind == "head":
        return g, g.act(c["m"], c["k"]), (g.uniform(0.5, 1.5, c["k"]), g.weight(8, c["n"], c["k"], 0))
    if kind == "attn":
        m = c["seqs"] * c["rows"]
        # rms-normalised heads: scores of a few units, as after the query norm
        q = [g.normal(m, c["nh"] * c["hd"]) * (3.0 / math.sqrt(c["hd"])) for _ in range(c["layers"])]
        lens = _lens(c, seed)
        slots = c["ctx"]
        if c["ring"]:
            slots = -(-(c["window"] + c["rows"]) // 8) * 8
        caches = [_Cache(g, c["seqs"], slots, slots if c["ring"] else 0, c["kvh"] * c["hd"], lens)
                  for _ in range(c["layers"])]
        return g, q, (lens, caches)
    if kind == "step":
        d, nh, kvh, hd, gr = c["d"], c["nh"], c["kvh"], c["hd"], c["group"]
        cc = dict(c, bits=4, down_bits=8)
        lens = _lens(c, seed)
        layers = []
        for i in range(c["layers"]):
            full = i % 4 == 3
            slots = -(-(c["ctx"] + 1) // 64) * 64 if full else -(-(c["window"] + 1) // 8) * 8
            w = _mlp_weights(g, cc)
            w.update({"q": g.weight(4, nh * hd, d, gr), "k": g.weight(4, kvh * hd, d, gr),
                      "v": g.weight(4, kvh * hd, d, gr), "o": g.weight(4, d, nh * hd, gr),
                      "in": g.uniform(0.5, 1.5, d), "attn_post": g.uniform(0.5, 1.5, d),
                      "qn": g.uniform(0.5, 1.5, hd) / math.sqrt(hd), "kn": g.uniform(0.5, 1.5, hd), "full": full,
                      "cache": _Cache(g, c["m"], slots, 0 if full else slots, kvh * hd, lens)})
            layers.append(w)
        head = (g.uniform(0.5, 1.5, d), g.weight(8, c["vocab"], d, 0))
        inv = np.array([10000.0 ** (-2.0 * i / hd) for i in range(hd // 2)], np.float32)
        cs = torch.from_numpy(np.stack([K.rope_table(inv, hd, n) for n in lens])).to(DEV)
        return g, g.act(c["m"], d), (lens, layers, head, cs)
    raise ValueError(kind)


def prepare(case, seed):
    c = case
    kind = c["kind"]
    g, x, w = _make(c, seed)
    st = {"case": c, "x": x, "w": w}
    z = lambda *s: torch.empty(*s, dtype=torch.float32, device=DEV)  # noqa: E731
    if kind == "linear":
        st["p"], st["c"] = _prep_bufs(c["m"], c["k"]), z(c["m"], c["n"])
    elif kind == "dropin":
        m, n, k = c["m"], c["n"], c["k"]
        st["x"], st["w"] = x.cpu().numpy(), tuple(t.cpu().numpy() for t in w)
        st["h"] = {"rot": np.zeros((m, k), np.float32), "qa": np.zeros((m, k), np.int8),
                   "qs": np.zeros(m, np.float32), "pa": np.zeros(K.packed_a_len(m, k), np.int8),
                   "c": np.zeros((m, n), np.float32)}
    elif kind == "mlp":
        st["bufs"] = _mlp_bufs(c["m"], c["d"], c["ff"])
        st["h"] = [x] + [z(c["m"], c["d"]) for _ in range(c["layers"])]
        if c["graph"]:
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):
                _run_mlp(st)
            torch.cuda.current_stream().wait_stream(side)
            torch.cuda.synchronize()
            st["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(st["graph"]):
                _run_mlp(st)
    elif kind == "head":
        st["p"], st["c"] = _prep_bufs(c["m"], c["k"]), z(c["m"], c["n"])
    elif kind == "attn":
        lens, caches = w
        m = c["seqs"] * c["rows"]
        st["out"] = [z(m, c["nh"] * c["hd"]) for _ in range(c["layers"])]
        span = 1
        st["desc"] = []
        for l in range(c["layers"]):
            arr = (F.AttnSeq * c["seqs"])()
            for i, n in enumerate(lens):
                pos = max(n - c["rows"], 0)
                arr[i] = caches[l].desc(i, pos, c["rows"])
                span = max(span, _span(pos, c["rows"], c["window"], caches[l].ring))
            st["desc"].append(arr)
        st["scratch"] = _scratch(m, c["nh"], c["kvh"], c["hd"], span)
    else:
        lens, layers, head, cs = w
        m, d, nh, kvh, hd = c["m"], c["d"], c["nh"], c["kvh"], c["hd"]
        st["mc"] = dict(c, bits=4, down_bits=8)
        st["bufs"] = _mlp_bufs(m, d, c["ff"])
        st["p"], st["po"] = _prep_bufs(m, d), _prep_bufs(m, nh * hd)
        st["q"], st["k"], st["v"], st["ao"] = z(m, nh * hd), z(m, kvh * hd), z(m, kvh * hd), z(m, nh * hd)
        st["o"], st["mid"] = z(m, d), z(m, d)
        st["h"] = [x] + [z(m, d) for _ in layers]
        st["logits"] = z(m, c["vocab"])
        st["desc"], span = [], 1
        for l in layers:
            arr = (F.AttnSeq * m)()
            for i, n in enumerate(lens):
                arr[i] = l["cache"].desc(i, n, 1)
                span = max(span, _span(n, 1, 0 if l["full"] else c["window"], l["cache"].ring))
            st["desc"].append(arr)
        st["scratch"] = _scratch(m, nh, kvh, hd, span)
    return st


# --------------------------------------------------------------------- run
def _run_mlp(st):
    c = st["case"]
    for i, w in enumerate(st["w"]):
        _mlp(c, c["m"], st["h"][i], w, st["bufs"], st["h"][i + 1])


def _run_step(st):
    c, mc = st["case"], st["mc"]
    m, d, nh, kvh, hd, gr = c["m"], c["d"], c["nh"], c["kvh"], c["hd"], c["group"]
    lens, layers, head, cs = st["w"]
    L, stream = F.lib(), _stream()
    qs, pa = st["p"]
    qso, pao = st["po"]
    q, k, v, ao, o, mid = st["q"], st["k"], st["v"], st["ao"], st["o"], st["mid"]
    kvd = kvh * hd
    for i, w in enumerate(layers):
        x, ca = st["h"][i], w["cache"]
        K.prep_rmsnorm(x, d, w["in"], EPS, qs, pa, m, d, c["hsz"])
        K.gemm_batch([_gemm(4, m, nh * hd, d, gr, qs, pa, w["q"], q), _gemm(4, m, kvd, d, gr, qs, pa, w["k"], k),
                      _gemm(4, m, kvd, d, gr, qs, pa, w["v"], v)])
        K.rmsnorm_rows(q, q, w["qn"], m * nh, hd, EPS)
        K.rmsnorm_rows(k, k, w["kn"], m * kvh, hd, EPS)
        K.rmsnorm_rows(v, v, None, m * kvh, hd, EPS)
        F.check(L.fgm_hip_rope_dev(q.data_ptr(), m, nh, hd, cs.data_ptr(), stream))
        F.check(L.fgm_hip_rope_dev(k.data_ptr(), m, kvh, hd, cs.data_ptr(), stream))
        for s in range(m):
            K.kv_store(k[s], v[s], 1, kvd, ca.kc[s], ca.ks[s], ca.vt[s], ca.vs[s], ca.slots, lens[s], ca.ring)
        F.check(L.fgm_hip_attend_dev(ao.data_ptr(), q.data_ptr(), st["desc"][i], m, nh, kvh, hd,
                                     0 if w["full"] else c["window"], st["scratch"][1], st["scratch"][2], stream))
        K.prep_rows(ao, nh * hd, None, None, qso, pao, m, nh * hd, c["hsz"], 0, m)
        _run_gemm(4, m, d, nh * hd, gr, qso, pao, w["o"], o)
        K.rmsnorm_rows(mid, o, w["attn_post"], m, d, EPS)
        K.add(mid, x)
        _mlp(mc, m, mid, w, st["bufs"], st["h"][i + 1])
    K.prep_rmsnorm(st["h"][-1], d, head[0], EPS, qs, pa, m, d, 0)
    _run_gemm(8, m, c["vocab"], d, 0, qs, pa, head[1], st["logits"])
    K.softcap(st["logits"], 30.0)
    return {"logits": st["logits"], "hidden": st["h"][-1], "ks": [w["cache"].ks for w in layers],
            "kc": [w["cache"].kc for w in layers], "vs": [w["cache"].vs for w in layers],
            "vt": [w["cache"].vt for w in layers]}


def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "linear":
        qs, pa = st["p"]
        K.prep_rows(st["x"], c["k"], None, None, qs, pa, c["m"], c["k"], c["hsz"], 0, c["m"])
        _run_gemm(c["bits"], c["m"], c["n"], c["k"], c["group"], qs, pa, st["w"], st["c"])
        return {"c": st["c"], "qs": qs, "pa": pa}
    if kind == "dropin":
        h, m, n, k = st["h"], c["m"], c["n"], c["k"]
        K.prep_rows(st["x"], k, h["rot"], h["qa"], h["qs"], h["pa"], m, k, c["hsz"], 0, m)
        if c["bits"] == 8:
            K.gemm_q8c(m, n, k, h["pa"], h["qs"], st["w"][0], st["w"][1], h["c"], n, 0, n // 16)
        else:
            K.gemm_q4g(m, n, k, h["pa"], h["qs"], st["w"][0], st["w"][1], c["group"], h["c"], n, 0, n // 16)
        return {"c": h["c"], "qs": h["qs"], "pa": h["pa"], "qa": h["qa"], "rot": h["rot"]}
    if kind == "mlp":
        if c["graph"]:
            st["graph"].replay()
        else:
            _run_mlp(st)
        return {"out": st["h"][1:], "gate": st["bufs"]["gate"], "up": st["bufs"]["up"], "down": st["bufs"]["down"]}
    if kind == "head":
        qs, pa = st["p"]
        K.prep_rmsnorm(st["x"], c["k"], st["w"][0], EPS, qs, pa, c["m"], c["k"], 0)
        _run_gemm(8, c["m"], c["n"], c["k"], 0, qs, pa, st["w"][1], st["c"])
        K.softcap(st["c"], c["cap"])
        return {"logits": st["c"], "qs": qs}
    if kind == "attn":
        L, stream, (_, sc, nb) = F.lib(), _stream(), st["scratch"]
        for q, out, desc in zip(st["x"], st["out"], st["desc"]):
            F.check(L.fgm_hip_attend_dev(out.data_ptr(), q.data_ptr(), desc, c["seqs"], c["nh"], c["kvh"], c["hd"],
                                         c["window"], sc, nb, stream))
        return {"out": st["out"]}
    return _run_step(st)


# -------------------------------------------------------------------- work
def _gemm_work(bits, m, n, k, group):
    """Weights and scales, packed A and its scales, f32 C: each once."""
    w = n * k + 4 * n if bits == 8 else n * k // 2 + (k // group) * n * 2
    return w + m * k + 4 * m + 4 * m * n, 2.0 * m * n * k


def _prep_work(m, k):
    return 5 * m * k + 4 * m


def _attn_work(lens_rows, nh, kvh, hd):
    """lens_rows: (cache slots read, positions attended by each row) per sequence;
    each sequence's K and V are read once."""
    by, fl = 0, 0.0
    for slots, ns in lens_rows:
        by += slots * (2 * kvh * hd + 8) + 8 * len(ns) * nh * hd
        fl += sum(4.0 * n * nh * hd for n in ns)
    return by, fl


def _mlp_work(c, m):
    d, ff = c["d"], c["ff"]
    b, f = 0, 0.0
    for bits, n, k in ((c["bits"], ff, d), (c["bits"], ff, d), (c["down_bits"], d, ff)):
        gb, gf = _gemm_work(bits, m, n, k, c["group"])
        b, f = b + gb, f + gf
    # norm + prep of x; gelu * up + prep; post-norm and residual
    return b + _prep_work(m, d) + 4 * d + 9 * m * ff + 4 * m + 20 * m * d + 4 * d, f


def work(case):
    c = case
    kind = c["kind"]
    if kind in ("linear", "dropin"):
        b, f = _gemm_work(c["bits"], c["m"], c["n"], c["k"], c["group"])
        return {"bytes": b + _prep_work(c["m"], c["k"]), "flops": f}
    if kind == "mlp":
        b, f = _mlp_work(c, c["m"])
        return {"bytes": b * c["layers"], "flops": f * c["layers"]}
    if kind == "head":
        b, f = _gemm_work(8, c["m"], c["n"], c["k"], 0)
        return {"bytes": b + _prep_work(c["m"], c["k"]) + 4 * c["k"] + 8 * c["m"] * c["n"], "flops": f}
    if kind == "attn":
        rows = []
        for n in [c["ctx"]] + [int(c["ctx"] * 0.875)] * (c["seqs"] - 1):
            pos = max(n - c["rows"], 0)
            ns = [min(pos + r + 1, c["window"] or 1 << 30) for r in range(c["rows"])]
            rows.append((min(pos + c["rows"], (c["window"] or 1 << 30) + c["rows"] - 1), ns))
        b, f = _attn_work(rows, c["nh"], c["kvh"], c["hd"])
        return {"bytes": b * c["layers"], "flops": f * c["layers"]}
    m, d, nh, kvh, hd, gr = c["m"], c["d"], c["nh"], c["kvh"], c["hd"], c["group"]
    b, f = _gemm_work(8, m, c["vocab"], d, 0)
    b += _prep_work(m, d) + 8 * m * c["vocab"]
    for i in range(c["layers"]):
        gb, gf = _mlp_work(dict(c, bits=4, down_bits=8), m)
        b, f = b + gb + 3 * _prep_work(m, d) + 8 * m * (nh + 2 * kvh) * hd, f + gf
        for n, k in ((nh * hd, d), (kvh * hd, d), (kvh * hd, d), (d, nh * hd)):
            gb, gf = _gemm_work(4, m, n, k, gr)
            b, f = b + gb, f + gf
        n = c["ctx"] if i % 4 == 3 else min(c["ctx"], c["window"])
        ab, af = _attn_work([(n, [n])] * m, nh, kvh, hd)
        b, f = b + ab, f + af
    return {"bytes": b, "flops": f}


def tolerance(case):
    """The library's contract is the reference's bytes: integers are exact, and
    the float operations are the reference's in the reference's order."""
    return "exact"


# ------------------------------------------------------------------- exact
def _x_quant(x):
    s = x.abs().amax(-1, keepdim=True) / 127.0
    s = torch.where(s == 0, torch.ones_like(s), s)
    return torch.clamp(torch.round(x / s), -128, 127), s


def _x_had(x, hsz):
    if hsz <= 1:
        return x
    h = torch.ones(1, 1, dtype=torch.float64, device=x.device)
    while h.shape[0] < hsz:
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return ((x.reshape(-1, hsz) @ h) / math.sqrt(hsz)).reshape(x.shape)


def _x_linear(x, w, bits, n, k, group, hsz=0):
    q, s = _x_quant(_x_had(x, hsz))
    if bits == 8:
        out = torch.empty(x.shape[0], n, dtype=torch.float64, device=x.device)
        step = 1 << 14
        for i in range(0, n, step):
            c = min(step, n - i)
            t = _tiles8(w[0][i * k:(i + c) * k], c, k).double()
            out[:, i:i + c] = (q @ t.t()) * w[1][i:i + c].double()
        return out * s, s[:, 0]
    t = _tiles8(_unpack4(w[0]), n, k).double()
    sc = w[1].view(torch.float16).double().view(k // group, n)
    t = (t.view(n, k // group, group) * sc.t().unsqueeze(-1)).reshape(n, k)
    return (q @ t.t()) * s, s[:, 0]


def _x_rms(x, w, n):
    y = x.reshape(-1, n)
    y = y / torch.sqrt(y.square().mean(-1, keepdim=True) + EPS)
    return (y if w is None else y * w.double()).reshape(x.shape)


def _x_mlp(c, x, w):
    xn = _x_rms(x, w["pre"], c["d"])
    gate, _ = _x_linear(xn, w["gate"], c["bits"], c["ff"], c["d"], c["group"], c["hsz"])
    up, _ = _x_linear(xn, w["up"], c["bits"], c["ff"], c["d"], c["group"], c["hsz"])
    act = 0.5 * gate * (1 + torch.tanh(math.sqrt(2 / math.pi) * (gate + 0.044715 * gate ** 3))) * up
    down, _ = _x_linear(act, w["down"], c["down_bits"], c["d"], c["ff"], c["group"], c["hsz"])
    return x + _x_rms(down, w["post"], c["d"]), gate, up, down


def _x_attn(q, ca, i, pos, rows, window, nh, kvh, hd):
    """Rows pos .. pos + rows - 1 of one sequence; q [rows, nh * hd] float64."""
    kvd = kvh * hd
    first = max(0, pos + 1 - window) if window else 0
    t = torch.arange(first, pos + rows, device=DEV)
    slot = t % ca.ring if ca.ring else t
    kf = ca.kc[i].view(-1, kvd)[slot].double()
    vf = ca.vt[i].view(-1, kvd, 4).permute(0, 2, 1).reshape(-1, kvd)[slot].double()
    ks, vs = ca.ks[i][slot].double(), ca.vs[i][slot].double()
    p = torch.arange(pos, pos + rows, device=DEV).view(-1, 1, 1)
    live = (t <= p) & ((t > p - window) if window else (t >= 0))  # [rows, 1, T]
    out = torch.empty(rows, nh, hd, dtype=torch.float64, device=DEV)
    grp = nh // kvh
    for h in range(kvh):
        qq, qsc = _x_quant(q.view(rows, nh, hd)[:, h * grp:(h + 1) * grp])
        s = (qq @ kf[:, h * hd:(h + 1) * hd].t()) * qsc * ks
        s = torch.where(live, s, torch.full_like(s, -math.inf))
        w = torch.softmax(s, -1) * vs
        step = w.amax(-1, keepdim=True) / 65535.0
        iw = torch.floor(w / step + 0.5)
        out[:, h * grp:(h + 1) * grp] = (iw @ vf[:, h * hd:(h + 1) * hd]) * step
    return out.view(rows, nh * hd)


def _x_rope(x, m, heads, hd, cs):
    y = x.view(m, heads, 2, hd // 2)
    co, si = cs[:, None, :, 0].double(), cs[:, None, :, 1].double()
    lo, hi = y[:, :, 0], y[:, :, 1]
    return torch.stack([lo * co - hi * si, hi * co + lo * si], 2).reshape(m, heads * hd)


def _x_step(c, x, w):
    m, d, nh, kvh, hd, gr = c["m"], c["d"], c["nh"], c["kvh"], c["hd"], c["group"]
    lens, layers, head, cs = w
    mc = dict(c, bits=4, down_bits=8)
    for l in layers:
        ca = l["cache"]
        xn = _x_rms(x, l["in"], d)
        q = _x_rms(_x_linear(xn, l["q"], 4, nh * hd, d, gr, c["hsz"])[0], l["qn"].repeat(1), hd)
        k = _x_rms(_x_linear(xn, l["k"], 4, kvh * hd, d, gr, c["hsz"])[0], l["kn"], hd)
        v = _x_rms(_x_linear(xn, l["v"], 4, kvh * hd, d, gr, c["hsz"])[0], None, hd)
        q, k = _x_rope(q, m, nh, hd, cs), _x_rope(k, m, kvh, hd, cs)
        (kq, ksc), (vq, vsc) = _x_quant(k), _x_quant(v)
        ao = torch.empty(m, nh * hd, dtype=torch.float64, device=DEV)
        for i, n in enumerate(lens):
            s = n % ca.ring if ca.ring else n
            ca.kc[i].view(-1, kvh * hd)[s] = kq[i].to(torch.int8)
            ca.vt[i].view(-1, kvh * hd, 4)[s // 4, :, s % 4] = vq[i].to(torch.int8)
            ca.ks[i][s], ca.vs[i][s] = ksc[i, 0].float(), vsc[i, 0].float()
            ao[i] = _x_attn(q[i:i + 1], ca, i, n, 1, 0 if l["full"] else c["window"], nh, kvh, hd)[0]
        o, _ = _x_linear(ao, l["o"], 4, d, nh * hd, gr, c["hsz"])
        x = _x_mlp(mc, x + _x_rms(o, l["attn_post"], d), l)[0]
    logits, _ = _x_linear(_x_rms(x, head[0], d), head[1], 8, c["vocab"], d, 0)
    none = [None] * len(layers)
    return {"logits": 30.0 * torch.tanh(logits / 30.0), "hidden": x, "ks": none, "kc": none, "vs": none, "vt": none}


def exact(case, seed):
    """What run returns, from the same inputs in float64 (values are quantised
    where the library quantises them)."""
    c = case
    kind = c["kind"]
    _, x, w = _make(c, seed)
    if kind == "attn":
        lens, caches = w
        r, nh, hd = c["rows"], c["nh"], c["hd"]
        return {"out": [torch.cat([_x_attn(q.double()[i * r:(i + 1) * r], ca, i, max(n - r, 0), r, c["window"], nh,
                                           c["kvh"], hd) for i, n in enumerate(lens)])
                        for q, ca in zip(x, caches)]}
    x = x.double()
    if kind in ("linear", "dropin"):
        y, s = _x_linear(x, w, c["bits"], c["n"], c["k"], c["group"], c["hsz"])
        out = {"c": y, "qs": s, "pa": None}
        if kind == "dropin":
            out["qa"], out["rot"] = None, _x_had(x, c["hsz"])
        return out
    if kind == "mlp":
        outs = []
        for l in w:
            x, gate, up, down = _x_mlp(c, x, l)
            outs.append(x)
        return {"out": outs, "gate": gate, "up": up, "down": down}
    if kind == "head":
        y, s = _x_linear(_x_rms(x, w[0], c["k"]), w[1], 8, c["n"], c["k"], 0)
        return {"logits": c["cap"] * torch.tanh(y / c["cap"]), "qs": s}
    return _x_step(c, x, w)
