"""GPU parity of the int8-KV attention (fgm_attn.hip) against the reference's
bytes (golden digests) and the oracle restatement (pinned in
tests/test_attn_oracle.py).

Bar: bit-exact.  The only operation evaluated differently from the reference
is exp on the n % 16 tail of the softmax (glibc's expf there, correctly
rounded here); the oracle counts tail values where glibc's expf is not
correctly rounded, and only such a case may differ -- then within 1e-6
relative of the largest output.  None of the fixtures has one.
"""
from __future__ import annotations

import hashlib
import json
import os

import numpy as np
import pytest

import oracle
from fastgemma_amd import kernels as K
from tests.golden import cases
from tests import hip_util as H

pytestmark = pytest.mark.gpu

GOLD = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "ref_outputs.json")))


def sha(a) -> str:
    return hashlib.sha256(np.ascontiguousarray(a).tobytes()).hexdigest()


def same_or_tail_close(got, want, noncr):
    if noncr == 0:
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    else:
        scale = max(float(np.max(np.abs(want))), 1e-30)
        assert np.max(np.abs(got - want)) <= 1e-6 * scale


def dev_kv(kv):
    return H.dev(kv.kc), H.dev(kv.ks), H.dev(kv.vt), H.dev(kv.vs)


def run_device(path, q, kv, nh, st, en, h0, h1, ring, fill=7.0):
    t = H.torch()
    out = t.full((nh * kv.hd,), fill, dtype=t.float32, device="cuda")
    dq = H.dev(q)
    kc, ks, vc, vs = dev_kv(kv)
    if path == "row":
        K.attend_q8_row(out, dq, kc, ks, vc, vs, nh, kv.kvh, kv.hd, st, en, None, ring, kv.cap)
    elif path == "q8":
        K.attend_q8(out, dq, kc, ks, vc, vs, nh, kv.kvh, kv.hd, st, en)
    else:
        K.attend_q8_heads(out, dq, kc, ks, vc, vs, nh, kv.kvh, kv.hd, st, en, None, h0, h1, ring,
                          kv.cap)
    return H.host(out)


def oracle_out(path, q, kv, nh, st, en, h0, h1, ring, fill=7.0):
    o = np.full(nh * kv.hd, fill, np.float32)
    oracle.reset_tail_noncr()
    if path == "row":
        oracle.attend_row(q, kv, nh, st, en, ring, out=o)
    elif path == "q8":
        oracle.attend_heads(q, kv, nh, st, en, 0, nh, 0, out=o)
    else:
        oracle.attend_heads(q, kv, nh, st, en, h0, h1, ring, out=o)
    return o, oracle.tail_noncr()


@pytest.fixture(params=["auto", "split"])
def attn_path(request, monkeypatch):
    """Rows of at most 1024 positions take the single-launch kernel unless
    FGM_ATTN_FUSED=0 (read per call): run every case both ways."""
    if request.param == "split":
        monkeypatch.setenv("FGM_ATTN_FUSED", "0")
    else:
        monkeypatch.delenv("FGM_ATTN_FUSED", raising=False)
    return request.param


@pytest.mark.parametrize("case", cases.ATTN_CASES, ids=[c[0] for c in cases.ATTN_CASES])
def test_attention_device_matches_reference(case, attn_path):
    name, nh, kvh, hd, cap, ring, st, en, h0, h1, qmul, path = case
    print(f"attn case {name} ({attn_path})", flush=True)
    q, kv = cases.attn_inputs(name, nh, kvh, hd, cap, qmul)
    want, noncr = oracle_out(path, q, kv, nh, st, en, h0, h1, ring)
    got = run_device(path, q, kv, nh, st, en, h0, h1, ring)
    same_or_tail_close(got, want, noncr)
    if noncr == 0:
        assert sha(got) == GOLD["attn"][name]["sha256"]


@pytest.mark.parametrize("name", ["dec256_n1000", "ring_wrap", "gqa_kv2_row", "heads_sub", "empty_row"])
def test_attention_dropins_host_pointers(name):
    """The host-pointer drop-ins with the reference's parameter lists."""
    case = next(c for c in cases.ATTN_CASES if c[0] == name)
    _, nh, kvh, hd, cap, ring, st, en, h0, h1, qmul, path = case
    q, kv = cases.attn_inputs(name, nh, kvh, hd, cap, qmul)
    out = np.full(nh * hd, 7.0, np.float32)
    if path == "row":
        K.attend_q8_row(out, q, kv.kc, kv.ks, kv.vt, kv.vs, nh, kvh, hd, st, en, None, ring, cap)
    else:
        K.attend_q8_heads(out, q, kv.kc, kv.ks, kv.vt, kv.vs, nh, kvh, hd, st, en, None, h0, h1,
                          ring, cap)
    assert sha(out) == GOLD["attn"][name]["sha256"]


def test_long_context_decode(attn_path):
    """A full-attention decode row at head_dim 512 over 8192 positions, and a
    sliding row at head_dim 256 in a ring that has wrapped many times."""
    for name, nh, hd, cap, ring, st, en in (("long512", 8, 512, 8192, 0, 0, 8192),
                                            ("slide256", 8, 256, 1040, 1040, 20000 - 1024, 20000)):
        q, kv = cases.attn_inputs(name, nh, 1, hd, cap, 1.0)
        want, noncr = oracle_out("heads", q, kv, nh, st, en, 0, nh, ring, 0.0)
        got = run_device("heads", q, kv, nh, st, en, 0, nh, ring, 0.0)
        same_or_tail_close(got, want, noncr)


def test_job_api_batched_decode_and_prefill(attn_path):
    """fgm_hip_attend_dev: three decode sequences (linear, ring, and a short
    one) plus a 40-row prefill chunk with a sliding window in a ring, one
    launch sequence; every row equals the per-row reference computation."""
    t = H.torch()
    nh, hd, window = 8, 256, 300
    seqs, qs, want = [], [], []
    specs = [("bd0", 700, 0, 699, 1), ("bd1", 340, 340, 5000, 1), ("bd2", 64, 0, 2, 1),
             ("pf", 360, 360, 1000, 40)]
    keep = []
    for name, cap, ring, pos, rows in specs:
        q, kv = cases.attn_inputs(name, nh, 1, hd, cap, 1.0)
        qrows = np.stack([np.roll(q, 17 * r) for r in range(rows)])
        kc, ks, vc, vs = dev_kv(kv)
        keep += [kc, ks, vc, vs]
        seqs.append((kc, ks, vc, vs, cap, ring, pos, rows))
        qs.append(qrows)
        for r in range(rows):
            en = pos + r + 1
            st = max(en - window, 0)
            want.append(oracle_out("heads", qrows[r], kv, nh, st, en, 0, nh, ring, 0.0))
    q_all = H.dev(np.concatenate([x.reshape(-1) for x in qs]))
    out = t.zeros(len(want) * nh * hd, dtype=t.float32, device="cuda")
    K.attend(out, q_all, seqs, nh, 1, hd, window)
    got = H.host(out).reshape(len(want), nh * hd)
    exact = 0
    for r, (w, noncr) in enumerate(want):
        same_or_tail_close(got[r], w, noncr)
        exact += noncr == 0
    assert exact >= len(want) - 4          # glibc's expf is rarely off by an ulp


@pytest.mark.parametrize("nh,kvh,hd,cap,ring,window,pos,rows", [
    (8, 1, 64, 700, 700, 100, 1440, 3),      # a wrapped range whose ring is mostly unused
    (8, 1, 64, 701, 699, 5, 1400, 1),        # both spans of the wrap in one slot group
    (6, 2, 128, 1200, 1200, 1024, 1300, 2),  # the longest single-launch row, three heads per kv head
    (5, 1, 320, 90, 0, 0, 60, 30),           # five heads, eight waves
    (8, 1, 64, 64, 64, 33, 500, 32),         # one head per workgroup, the chip just filled
    (8, 1, 64, 128, 128, 33, 500, 65),       # four heads per workgroup
    (8, 1, 64, 400, 400, 33, 1000, 260),     # every head in one workgroup
    (3, 1, 64, 140, 140, 20, 700, 120),      # two of three heads, then the third
])
def test_job_heads_split_and_wrapped_rings(nh, kvh, hd, cap, ring, window, pos, rows, attn_path):
    """The head split by row count and the walk over a wrapped ring's two spans."""
    t = H.torch()
    print(f"attn rows {rows} heads {nh} hd {hd} ring {ring} ({attn_path})", flush=True)
    q, kv = cases.attn_inputs(f"split{rows}", nh, kvh, hd, cap, 1.0)
    qrows = np.stack([np.roll(q, 17 * r) for r in range(rows)])
    out = t.full((rows * nh * hd,), 7.0, dtype=t.float32, device="cuda")
    K.attend(out, H.dev(qrows.reshape(-1)), [(*dev_kv(kv), cap, ring, pos, rows)], nh, kvh, hd, window)
    got = H.host(out).reshape(rows, nh * hd)
    for r in range(rows):
        en = pos + r + 1
        st = max(en - window, 0) if window else 0
        want, noncr = oracle_out("heads", qrows[r], kv, nh, st, en, 0, nh, ring, 0.0)
        same_or_tail_close(got[r], want, noncr)


@pytest.mark.parametrize("nh,kvh,hd,cap,ring,window,pos,rows", [
    (8, 1, 64, 3000, 0, 0, 2940, 60),        # row tiles of 16, the last one partial, unaligned tails
    (3, 1, 128, 1300, 0, 0, 1100, 50),       # 42 rows a tile: 126 of its 128 pairs
    (16, 1, 64, 1500, 1500, 1440, 4000, 9),  # 16 heads, a wrapped ring whose runs share a group
    (8, 2, 192, 2100, 2100, 1100, 2090, 33), # a wrapped ring with a gap, three 64-dim blocks
    (2, 2, 448, 1200, 0, 1050, 1100, 70),    # one head per kv head, window starts inside a step
    (8, 1, 64, 32768, 0, 0, 32767, 1),       # the longest row, alone
    (8, 1, 64, 20500, 0, 0, 20490, 5),       # long rows in a tile
    (16, 1, 128, 1400, 1400, 1397, 2799, 3), # single rows of 16 heads, both runs in one group
])
def test_job_row_tiles_and_long_rows(nh, kvh, hd, cap, ring, window, pos, rows):
    """Rows past the single-launch path: row tiles sharing K and V, single rows,
    the walk over their slot domain."""
    t = H.torch()
    print(f"attn long rows {rows} heads {nh} hd {hd} ring {ring}", flush=True)
    q, kv = cases.attn_inputs(f"long{rows}", nh, kvh, hd, cap, 1.0)
    qrows = np.stack([np.roll(q, 17 * r) for r in range(rows)])
    out = t.full((rows * nh * hd,), 7.0, dtype=t.float32, device="cuda")
    K.attend(out, H.dev(qrows.reshape(-1)), [(*dev_kv(kv), cap, ring, pos, rows)], nh, kvh, hd, window)
    got = H.host(out).reshape(rows, nh * hd)
    for r in range(rows):
        en = pos + r + 1
        st = max(en - window, 0) if window else 0
        want, noncr = oracle_out("heads", qrows[r], kv, nh, st, en, 0, nh, ring, 0.0)
        same_or_tail_close(got[r], want, noncr)


def check_job(specs, nh, kvh, hd, window, some=None):
    """One attend call over the sequences (cap, ring, pos, rows); every row (or, of
    a sequence of more, its first, last and `some` between) against the oracle."""
    t = H.torch()
    m = sum(s[3] for s in specs)
    out = t.full((m * nh * hd,), 7.0, dtype=t.float32, device="cuda")
    seqs, qs, rows = [], [], []
    for i, (cap, ring, pos, n) in enumerate(specs):
        q, kv = cases.attn_inputs(f"job{i % 3}", nh, kvh, hd, cap, 1.0)
        seqs.append((*dev_kv(kv), cap, ring, pos, n))
        qs.append([np.roll(q, 17 * (r + i)) for r in range(n)])
        look = set(range(n)) if some is None or n <= some + 2 else {n * j // (some + 1) for j in range(some + 1)} | {n - 1}
        rows += [(kv, ring, pos + r, qs[-1][r]) if r in look else None for r in range(n)]
    K.attend(out, H.dev(np.concatenate([x for rs in qs for x in rs])), seqs, nh, kvh, hd, window)
    got = H.host(out).reshape(m, nh * hd)
    for r, x in enumerate(rows):
        if x is None:
            continue
        kv, ring, p, q = x
        want, noncr = oracle_out("heads", q, kv, nh, max(p + 1 - window, 0) if window else 0, p + 1, 0, nh, ring, 0.0)
        same_or_tail_close(got[r], want, noncr)


@pytest.mark.parametrize("nh,kvh,hd,cap,ring,window,pos,rows", [
    (8, 8, 64, 200, 200, 64, 500, 130),      # one head per workgroup, 1040 workgroups of eight waves
    (8, 4, 128, 200, 0, 0, 0, 200),          # a prompt from its first row, two heads
    (4, 2, 192, 300, 300, 170, 700, 120),    # three 64-dim blocks on eight waves
    (8, 1, 64, 1100, 1100, 1024, 3000, 40),  # two heads of 1024 positions: eight waves
    (8, 1, 64, 1100, 1100, 1024, 3000, 70),  # four: sixteen
    (8, 1, 256, 1200, 1200, 1024, 3000, 130),
    (6, 2, 256, 600, 600, 520, 900, 90),     # three heads of 520 positions: eight waves
])
def test_job_waves_per_workgroup(nh, kvh, hd, cap, ring, window, pos, rows):
    """The single launch at both its widths, full and partly filled CUs."""
    print(f"attn waves rows {rows} heads {nh}/{kvh} hd {hd} window {window}", flush=True)
    check_job([(cap, ring, pos, rows)], nh, kvh, hd, window, some=20)


@pytest.mark.parametrize("name,nh,kvh,hd,window,specs", [
    # a chunk beside 15 decode rows: below and past the line from which rows go in tiles
    ("rows", 8, 1, 512, 0, [(1300, 0, 1299 - 9 * i, 1) for i in range(15)] + [(1400, 0, 1365, 30)]),
    ("tiles", 8, 1, 512, 0, [(1300, 0, 1299 - 9 * i, 1) for i in range(15)] + [(1500, 0, 1430, 61)]),
    ("tiles", 8, 4, 128, 1100, [(1204, 1204, 3000 + 301 * i, 1) for i in range(3)] + [(1204, 1204, 2500, 100)]),
    # a few rows in each sequence, one without any
    ("rows", 8, 2, 256, 0, [(1200, 0, 1100 + i, 2 + i) for i in range(5)] + [(64, 0, 0, 0)]),
    ("rows", 16, 1, 256, 0, [(700, 0, 600, 7), (100, 0, 3, 1), (90, 0, 0, 90)]),
    ("tiles", 16, 1, 256, 0, [(700, 0, 300, 400), (100, 0, 3, 1), (90, 0, 0, 90)]),
    # tiles of 42 rows: 126 of the 128 pairs; the last one partial, tails at every offset
    ("tiles", 3, 1, 128, 0, [(1400, 0, 1200, 130)]),
    ("tiles", 8, 1, 64, 0, [(3000, 0, 2860, 130)]),
    # wrapped rings: both runs in one slot group; a gap between them
    ("tiles", 16, 1, 256, 1498, [(1500, 1500, 4000, 70)]),
    ("tiles", 8, 2, 192, 1100, [(2100, 2100, 2090, 60)]),
])
def test_job_rows_or_tiles(name, nh, kvh, hd, window, specs):
    """Mixed jobs on both sides of the choice between single rows and row tiles."""
    print(f"attn {name} heads {nh}/{kvh} hd {hd} rows {[s[3] for s in specs]}", flush=True)
    check_job(specs, nh, kvh, hd, window, some=12)


@pytest.mark.parametrize("nh,kvh,hd,cap,rows", [
    (16, 1, 64, 64, 20),     # up to 1024 slots: 256 threads
    (9, 1, 64, 1000, 30),
    (12, 1, 64, 1024, 2),
    (8, 1, 64, 1500, 33),    # 256 or more (row, head) pairs, 1 .. 4 and 6 groups of slots a thread
    (8, 1, 64, 4000, 33),
    (8, 1, 64, 5200, 33),
    (8, 1, 64, 8192, 33),
    (8, 1, 64, 12200, 33),
    (8, 1, 64, 20500, 33),
    (8, 1, 64, 3000, 2),     # fewer: 1, 2, 3, 4, 6 and 9 groups, twice the threads
    (8, 1, 64, 8000, 2),
    (8, 1, 64, 12200, 2),
    (8, 1, 64, 15000, 2),
    (8, 1, 64, 24000, 2),
    (8, 1, 64, 32768, 2),
])
def test_job_softmax_widths(nh, kvh, hd, cap, rows):
    """Every width of the softmax, by row length and (row, head) pairs."""
    print(f"attn softmax rows {rows} positions {cap}", flush=True)
    check_job([(cap, 0, cap - rows, rows)], nh, kvh, hd, 0, some=2)


@pytest.mark.parametrize("nh,kvh,hd", [(8, 1, 512), (9, 1, 512), (8, 2, 512), (16, 1, 512), (8, 4, 128)])
def test_job_sixteen_decode_rows(nh, kvh, hd):
    """Sixteen sequences of one row past the single-launch path: 32 dims a
    workgroup in P.V, up to and past eight heads a kv head."""
    print(f"attn decode 16 heads {nh}/{kvh} hd {hd}", flush=True)
    check_job([(1300, 0, 1299 - 11 * i, 1) if i % 2 else (1300, 1300, 2000 + 97 * i, 1) for i in range(16)], nh, kvh, hd,
              1290)


@pytest.mark.parametrize("shift", [1, 4, 8])
@pytest.mark.parametrize("nh,kvh,hd,cap,ring,window,pos,rows", [
    (8, 1, 512, 2000, 0, 0, 1960, 40),      # row tiles where the caches are at dword addresses
    (8, 2, 128, 1300, 1300, 1200, 3000, 2), # single rows, a wrapped ring
    (16, 1, 64, 500, 0, 0, 490, 3),
    (8, 4, 64, 3000, 0, 1100, 2900, 100),   # row tiles of 64 dims
    (8, 1, 256, 540, 540, 500, 3000, 6),    # the single-launch path
])
def test_caches_at_any_address(nh, kvh, hd, cap, ring, window, pos, rows, shift):
    """K and V caches `shift` bytes past a 16-byte boundary, their scales one float."""
    t = H.torch()
    print(f"attn unaligned {shift} heads {nh}/{kvh} hd {hd} rows {rows}", flush=True)
    q, kv = cases.attn_inputs(f"shift{rows}", nh, kvh, hd, cap, 1.0)

    def moved(x, by):
        buf = t.zeros(x.size + by, dtype=H.dev(x[:1]).dtype, device="cuda")
        buf[by:] = H.dev(x)
        return buf[by:]

    kc, ks, vt, vs = moved(kv.kc, shift), moved(kv.ks, 1), moved(kv.vt, shift), moved(kv.vs, 1)
    assert kc.data_ptr() % 16 == shift and vt.data_ptr() % 16 == shift
    qrows = np.stack([np.roll(q, 17 * r) for r in range(rows)])
    out = t.full((rows * nh * hd,), 7.0, dtype=t.float32, device="cuda")
    K.attend(out, H.dev(qrows.reshape(-1)), [(kc, ks, vt, vs, cap, ring, pos, rows)], nh, kvh, hd, window)
    got = H.host(out).reshape(rows, nh * hd)
    for r in range(rows):
        en = pos + r + 1
        st = max(en - window, 0) if window else 0
        want, noncr = oracle_out("heads", qrows[r], kv, nh, st, en, 0, nh, ring, 0.0)
        same_or_tail_close(got[r], want, noncr)


@pytest.fixture(scope="module")
def big_cache():
    """K and V bytes of a layer cache past 2 GiB, and its scales: views of it with
    any kv width are valid caches."""
    t = H.torch()
    size = (1 << 31) + (1 << 26)
    g = t.Generator(device="cuda").manual_seed(5)
    kv = [t.randint(-127, 128, (size,), dtype=t.int8, device="cuda", generator=g) for _ in range(2)]
    sc = [t.rand(size // 512, device="cuda", generator=g) * 4e-4 + 1e-4 for _ in range(2)]
    yield size, kv[0], sc[0], kv[1], sc[1]
    del kv, sc
    t.cuda.empty_cache()


@pytest.mark.parametrize("nh,kvh,hd,nseq,rows,window,high", [
    (8, 4, 512, 1, 1, 1500, False),   # single rows, 16 dims a workgroup
    (8, 4, 512, 1, 1, 1500, True),    # slots past the first 2 GiB
    (8, 4, 512, 16, 1, 1100, False),  # 32 dims a workgroup
    (16, 1, 512, 1, 1, 700, False),   # more than eight heads
    (16, 1, 512, 16, 1, 700, True),
    (8, 4, 512, 1, 40, 3000, True),   # row tiles
    (8, 4, 512, 1, 2, 300, True),     # the single-launch path
])
def test_caches_past_two_gib(big_cache, nh, kvh, hd, nseq, rows, window, high):
    """Caches of 2 GiB and more hold real bytes where smaller ones read zeros."""
    print(f"attn big cache heads {nh}/{kvh} seqs {nseq} rows {rows} high {high}", flush=True)
    size, kc, ks, vt, vs = big_cache
    kvd = kvh * hd
    cap = size // kvd // 4 * 4
    m = nseq * rows
    q = oracle.gen_uniform(77 + m, m * nh * hd, -1.0, 1.0).reshape(m, nh * hd)
    out = H.torch().full((m * nh * hd,), 7.0, dtype=H.torch().float32, device="cuda")
    seqs, want = [], []
    for i in range(nseq):
        pos = (cap if high else 6000) - rows - 37 * i
        seqs.append((kc, ks, vt, vs, cap, 0, pos, rows))
        for r in range(rows):
            if r not in (0, rows // 2, rows - 1):
                want.append(None)
                continue
            en = pos + r + 1
            st = max(en - window, 0)
            base = st // 4 * 4
            kv = oracle.KvLayer((en - base + 3) // 4 * 4, kvh, hd)
            last = base + kv.cap
            kv.kc, kv.vt = (H.host(x[base * kvd:last * kvd]) for x in (kc, vt))
            kv.ks, kv.vs = (H.host(x[base:last]) for x in (ks, vs))
            want.append(oracle_out("heads", q[i * rows + r], kv, nh, st - base, en - base, 0, nh, 0, 0.0))
    K.attend(out, H.dev(q.reshape(-1)), seqs, nh, kvh, hd, window)
    got = H.host(out).reshape(m, nh * hd)
    for r, w in enumerate(want):
        if w is not None:
            same_or_tail_close(got[r], *w)


def test_kv_store_matches_reference_write_path():
    """fgm_hip_kv_store_dev equals quant_act + store_v_t per row (the forward
    pass's write, forward.rs:515-548), linear and wrapping ring."""
    t = H.torch()
    hd = 512
    for cap, ring, pos, m in ((96, 0, 37, 21), (40, 40, 77, 13)):
        kv = oracle.KvLayer(cap, 1, hd)
        kf = oracle.gen_uniform(11 + pos, m * hd, -3.0, 3.0).reshape(m, hd)
        vf = oracle.gen_normal(12 + pos, m * hd).reshape(m, hd)
        kf[3] = 0.0                                    # amax 0: scale 1
        for r in range(m):
            kv.store((pos + r) % ring if ring else pos + r, kf[r], vf[r])
        kc = t.zeros(cap * hd, dtype=t.int8, device="cuda")
        ks = t.zeros(cap, dtype=t.float32, device="cuda")
        vt = t.zeros((cap + 3) // 4 * 4 * hd, dtype=t.int8, device="cuda")
        vs = t.zeros(cap, dtype=t.float32, device="cuda")
        K.kv_store(H.dev(kf), H.dev(vf), m, hd, kc, ks, vt, vs, cap, pos, ring)
        assert np.array_equal(H.host(kc), kv.kc)
        assert np.array_equal(H.host(ks).view(np.uint32), kv.ks.view(np.uint32))
        assert np.array_equal(H.host(vt), kv.vt)
        assert np.array_equal(H.host(vs).view(np.uint32), kv.vs.view(np.uint32))


def test_store_v_t_device_and_dropin():
    n, cap = 256, 9
    rows = oracle.gen_i8(3, cap * n, -127, 127).reshape(cap, n)
    want = np.zeros((cap + 3) // 4 * 4 * n, np.int8)
    for s in range(cap):
        oracle.store_v_t(want, rows[s], s)
    t = H.torch()
    vt = t.zeros(want.size, dtype=t.int8, device="cuda")
    for s in range(cap):
        K.store_v_t(vt, H.dev(rows[s]), n, s)
    assert np.array_equal(H.host(vt), want)
    host_vt = np.zeros_like(want)
    for s in range(cap):
        K.store_v_t(host_vt, np.ascontiguousarray(rows[s]), n, s)
    assert np.array_equal(host_vt, want)


def test_rowbatch_scratch_and_flag():
    assert K.rowbatch_scratch(8, 1024, 256) == 8 * 1024 + (1024 + 3) // 2 + 2 * 256 + 64
    K.set_scalar_wfill(True)
    K.set_scalar_wfill(False)
