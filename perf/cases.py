"""The calls whose speed matters: what users of the library have it do, over the
sizes they do it at, each through the package's public entry points.

A case is a dict:
  call      score | counts | rows | local_rows | banded_score | banded_rows
  residues  dna | protein
  pairs     number of pairs in the call
  lengths   fixed (every |H| = length), lognormal (median `length`, sigma 1,
            clipped to 100..10,000) or uniform (|H| in 50..length, |V| in
            50..2 * length)
  sub, indel, geom   mutation rates of V against H (DNA): substitutions,
            indels and the parameter of their geometric lengths (1: single
            bases)
  mode      global, overlap (AlignConfig<1,0,0,1>), free (AlignConfig<1,1,1,1>)
            or local
  band      half width of the band, 0 without one
  match, mismatch, extend, open   Score<int, Simple> (DNA); proteins take
            Blosum62 with extend and open
  resident  residues and outputs in device memory; otherwise host buffers,
            whose copies belong to the call

The rows calls go through the C ABI into buffers that the program keeps (a
call leaves the bytes of `ops` past the last row as they were); the others
through the Python package.
"""
import ctypes
import math

import numpy as np
import torch

import seqan_amd as sa

MODES = {"global": 0, "overlap": sa.FREE_TOP | sa.FREE_BOTTOM,
         "free": sa.FREE_TOP | sa.FREE_LEFT | sa.FREE_RIGHT | sa.FREE_BOTTOM, "local": sa.LOCAL}


def _case(call, pairs, length, name=None, residues="dna", lengths="fixed", sub=0.05, indel=0.01, geom=1.0,
          mode="global", band=0, match=2, mismatch=-3, extend=-1, open=-5, resident=True):
    c = {"call": call, "residues": residues, "pairs": pairs, "lengths": lengths, "length": length, "sub": sub,
         "indel": indel, "geom": geom, "mode": mode, "band": band, "match": match, "mismatch": mismatch,
         "extend": extend, "open": open, "resident": resident}
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # A handful of reads scored from host buffers: an interactive call or
        # one step of a host loop, where the latency of a call is what counts.
        _case("score", 64, 150, "score_few_reads", resident=False),
        # A batch of short reads resident on the device (read mapping's
        # verification step): a full call that is still launch bound.
        _case("score", 4096, 150, "score_reads"),
        # A batch of a few thousand uneven reads: too few pairs to hide the
        # longest ones behind the rest.
        _case("score", 3001, 300, "score_uneven_batch", lengths="lognormal", sub=0.08, indel=0.02, geom=0.5,
              mode="overlap"),
        # The headline workload: a million uneven DNA pairs, semi-global.
        _case("score", 1 << 20, 300, "score_uneven", lengths="lognormal", sub=0.08, indel=0.02, geom=0.5,
              mode="overlap"),
        # Protein homology search: Smith-Waterman scores with Blosum62.
        _case("score", 1 << 18, 1000, "score_protein_local", residues="protein", lengths="uniform", mode="local",
              open=-11),
        # Training a scoring scheme: scores and their gradient (counts).
        _case("counts", 1 << 16, 1000, "counts_1k", sub=0.10, indel=0.02),
        # Alignments (rows) of a batch of uneven reads from host buffers.
        _case("rows", 8191, 300, "rows_uneven", lengths="lognormal", sub=0.08, indel=0.02, geom=0.5, mode="overlap",
              resident=False),
        # Local protein alignments with their rows, from host buffers: the
        # hits of a search shown to a user.
        _case("local_rows", 8192, 1000, "rows_protein_local", residues="protein", lengths="uniform", mode="local",
              open=-11, resident=False),
        # Whole genomic segments: scores and counts of 100 kbp pairs.
        _case("counts", 64, 100000, "counts_long", sub=0.12, indel=0.03, geom=0.3),
        # Banded verification of a million mapped reads.
        _case("banded_score", 1 << 20, 150, "banded_reads", sub=0.08, indel=0.0, band=16),
        # Banded overlaps of 1 kbp reads with all ends free.
        _case("banded_score", 1 << 16, 1000, "banded_overlap", sub=0.10, indel=0.02, mode="free", band=100),
        # Banded alignments (rows) of mapped reads from host buffers: what a
        # mapper writes to its output.
        _case("banded_rows", 1 << 16, 150, "banded_rows_reads", sub=0.08, indel=0.01, band=16, resident=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["reads", "uneven", "protein", "counts", "rows", "local_rows", "long", "banded", "banded_rows"])
    scheme = rng.choice([(2, -3, -1, -5), (2, -3, -1, -5), (1, -1, -1, -2), (5, -4, -2, -10), (1, -2, -2, -2)])
    if kind in ("uneven", "rows"):      # lengths up to 10,000: the schemes whose scores of such pairs fit int16
        scheme = rng.choice([(2, -3, -1, -5), (1, -1, -1, -2)])
    s = dict(zip(("match", "mismatch", "extend", "open"), scheme))
    if kind == "reads":
        length = _log_int(rng, 50, 2000)
        pairs = _log_int(rng, 16, max(32, min(1 << 18, 6e10 / length ** 2)))
        return _case("score", pairs, length, sub=rng.choice([0.05, 0.10]), indel=rng.choice([0.01, 0.02]),
                     mode=rng.choice(["global", "overlap", "local"]), resident=rng.random() < 0.7, **s)
    if kind == "uneven":
        return _case("score", _log_int(rng, 512, 1 << 18), _log_int(rng, 200, 600), lengths="lognormal", sub=0.08,
                     indel=0.02, geom=0.5, mode=rng.choice(["global", "overlap", "local"]), **s)
    if kind == "protein":
        return _case("score", _log_int(rng, 256, 1 << 17), _log_int(rng, 200, 1000), residues="protein",
                     lengths="uniform", mode="local", open=rng.choice([-11, -10, -13]), resident=rng.random() < 0.7)
    if kind == "counts":
        length = _log_int(rng, 100, 3000)
        return _case("counts", _log_int(rng, 64, min(1 << 16, 3e10 / length ** 2)), length, sub=0.10, indel=0.02,
                     mode=rng.choice(["global", "overlap", "local"]), **s)
    if kind == "rows":
        return _case("rows", _log_int(rng, 64, 1 << 14), _log_int(rng, 200, 500), lengths="lognormal", sub=0.08,
                     indel=0.02, geom=0.5, mode=rng.choice(["global", "overlap"]), resident=False, **s)
    if kind == "local_rows":
        return _case("local_rows", _log_int(rng, 64, 1 << 13), _log_int(rng, 200, 1000), residues="protein",
                     lengths="uniform", mode="local", open=rng.choice([-11, -10, -13]), resident=False)
    if kind == "long":
        length = _log_int(rng, 16000, 64000)
        return _case("counts", _log_int(rng, 4, min(64, 1.5e11 / length ** 2 + 5)), length, sub=0.12, indel=0.03,
                     geom=0.3)
    length = _log_int(rng, 80, 2000)
    indel = rng.choice([0.0, 0.01, 0.02])
    least = 8 + int(8 * math.sqrt(length * indel))    # both corner diagonals lie inside the band
    band = _log_int(rng, least, max(least + 4, min(150, length // 4)))
    if kind == "banded":
        return _case("banded_score", _log_int(rng, 1000, min(1 << 20, 1.5e10 / (length * band))), length, sub=0.08,
                     indel=indel, mode=rng.choice(["global", "free", "local"]), band=band,
                     resident=rng.random() < 0.7, **s)
    return _case("banded_rows", _log_int(rng, 500, min(1 << 16, 1.5e9 / (length * band))), length, sub=0.08,
                 indel=indel, mode=rng.choice(["global", "free"]), band=band, resident=False, **s)


def _offsets(lengths):
    off = np.zeros(len(lengths) + 1, np.int64)
    np.cumsum(lengths, out=off[1:])
    return off


def _dna(case, rng, gen):
    """H uniform over ACGT, V a mutated copy: (h, h offsets, v, v offsets), residues on the device."""
    n = case["pairs"]
    if case["lengths"] == "lognormal":
        hl = np.clip(np.rint(np.exp(rng.normal(math.log(case["length"]), 1.0, n))), 100, 10000).astype(np.int64)
    else:
        hl = np.full(n, case["length"], np.int64)
    hoff = _offsets(hl)
    total = int(hoff[-1])
    dev = "cuda"

    def uniform():
        return torch.rand(total, device=dev, generator=gen)

    h = torch.randint(0, 4, (total,), device=dev, generator=gen, dtype=torch.uint8)
    base = torch.where(uniform() < case["sub"],
                       (h + 1 + torch.randint(0, 3, (total,), device=dev, generator=gen, dtype=torch.uint8)) & 3, h)
    if case["indel"] <= 0:
        return h, hoff, base, hoff.copy()
    event = uniform()
    size = torch.ones(total, device=dev, dtype=torch.int32)
    if case["geom"] < 1:
        size += torch.floor(torch.log(uniform().clamp_min(1e-9)) / math.log(1 - case["geom"])).to(torch.int32)
    at = torch.arange(total, device=dev, dtype=torch.int32)
    ends = torch.from_numpy(hoff[1:].astype(np.int32)).to(dev)
    last = torch.repeat_interleave(ends, torch.from_numpy(hl).to(dev), output_size=total)
    zero = torch.zeros((), device=dev, dtype=torch.int32)
    # A deletion drops `size` bases from its position on, up to its pair's end.
    cut = torch.where(event < case["indel"] / 2, torch.minimum(at + size, last), zero)
    kept = torch.cummax(cut, 0).values <= at
    # An insertion puts `size` random bases before its position.
    inserted = torch.where((event >= case["indel"] / 2) & (event < case["indel"]), size, zero)
    upto = torch.cumsum(kept.to(torch.int32) + inserted, 0, dtype=torch.int32)
    voff = np.zeros(n + 1, np.int64)
    voff[1:] = upto[torch.from_numpy(hoff[1:] - 1).to(dev)].cpu().numpy()
    v = torch.randint(0, 4, (int(voff[-1]),), device=dev, generator=gen, dtype=torch.uint8)
    v[(upto - 1)[kept].long()] = base[kept]
    return h, hoff, v, voff


# Robinson & Robinson (1991) background frequencies, per 1000.
_AMINO = "ACDEFGHIKLMNPQRSTVWY"
_FREQ = np.array([78.05, 19.25, 53.64, 62.95, 38.56, 73.77, 21.99, 51.42, 57.44, 90.19, 22.43, 44.87, 52.03, 42.64,
                  51.29, 71.20, 58.41, 64.41, 13.30, 32.16])


def _protein(case, rng, gen):
    """Random proteins; 30% of the pairs hold a homolog of a piece of H in V at about 40% identity."""
    n, dev = case["pairs"], "cuda"
    hl = rng.integers(50, case["length"] + 1, n)
    vl = rng.integers(50, 2 * case["length"] + 1, n)
    hoff, voff = _offsets(hl), _offsets(vl)
    codes = np.array([sa.AMINO_ACIDS.index(c) for c in _AMINO])
    code = torch.from_numpy(codes.astype(np.uint8)).to(dev)
    p = _FREQ / _FREQ.sum()

    def residues(total):
        u = torch.rand(total, device=dev, generator=gen)
        return torch.searchsorted(torch.from_numpy(np.cumsum(p)[:-1].astype(np.float32)).to(dev), u)

    h, v = residues(int(hoff[-1])), residues(int(voff[-1]))
    # Segments: length, start in H and in V of the pairs that hold a homolog.
    pick = np.nonzero(rng.random(n) < 0.30)[0]
    most = np.minimum(hl, vl)[pick]
    seg = rng.integers(np.minimum(30, most), most + 1)
    hs = hoff[pick] + rng.integers(0, hl[pick] - seg + 1)
    vs = voff[pick] + rng.integers(0, vl[pick] - seg + 1)
    if len(pick):
        seg_d = torch.from_numpy(seg).to(dev)
        first = torch.from_numpy(_offsets(seg)[:-1]).to(dev)
        k = torch.arange(int(seg.sum()), device=dev) - torch.repeat_interleave(first, seg_d)
        src = h[torch.repeat_interleave(torch.from_numpy(hs).to(dev), seg_d) + k]
        # Substitutions weighted by background * exp(lambda * Blosum62).
        table = sa.blosum62().table[np.ix_(codes, codes)]
        w = p[None, :] * np.exp(0.3176 * table)
        np.fill_diagonal(w, 0)
        cum = torch.from_numpy(np.cumsum(w / w.sum(1, keepdims=True), 1).astype(np.float32)).to(dev)
        other = torch.empty_like(src)
        for a in range(20):
            here = (src == a).nonzero().squeeze(1)
            u = torch.rand(len(here), device=dev, generator=gen)
            other[here] = torch.searchsorted(cum[a], u).clamp_max(19)
        same = torch.rand(len(k), device=dev, generator=gen) < 0.40
        v[torch.repeat_interleave(torch.from_numpy(vs).to(dev), seg_d) + k] = torch.where(same, src, other)
    return code[h], hoff, code[v], voff


def _scoring(case):
    if case["residues"] == "protein":
        return sa.blosum62(case["extend"], case["open"])
    return sa.simple_score(case["match"], case["mismatch"], case["extend"], case["open"])


def _inputs(case, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return (_protein if case["residues"] == "protein" else _dna)(case, rng, gen)


class _Set(ctypes.Structure):       # sqmi_sequences
    _fields_ = [("residues", ctypes.c_void_p), ("offsets", ctypes.c_void_p), ("count", ctypes.c_int64)]


class _Scheme(ctypes.Structure):    # sqmi_scoring
    _fields_ = [("alphabet_size", ctypes.c_int32), ("gap_open", ctypes.c_int32), ("gap_extend", ctypes.c_int32),
                ("table", ctypes.c_void_p)]


_native = []


def _library():
    """The library and one context for the rows calls, made on first use."""
    if not _native:
        lib = ctypes.CDLL(sa.LIB_PATH)
        ctx = ctypes.c_void_p()
        if lib.sqmi_create(0, ctypes.byref(ctx)):
            raise RuntimeError("sqmi_create failed")
        _native.extend([lib, ctx])
    return _native


def _rows_call(case, st):
    """The arguments of a rows call, with its output buffers (of one size for all inputs of a case)."""
    H, V, score, n = st["H"], st["V"], st["score"], case["pairs"]
    lib, ctx = _library()
    seg = _offsets(H.lengths() + V.lengths())
    room = max(int(n * 2 * _mean_cells(case)[1]) + 60000, int(seg[-1]))
    table = np.ascontiguousarray(score.table, np.int32)
    scheme = _Scheme(score.alphabet_size, score.gap_open, score.gap_extend, table.ctypes.data)
    sets = [_Set(s.residues.ctypes.data, s.offsets.ctypes.data, n) for s in (H, V)]
    out = [np.zeros(n, np.int32), np.zeros((n, score.alphabet_size ** 2 + 2), np.int32), np.zeros(room, np.uint8),
           np.zeros(n, np.int64)]
    scores, counts, ops, lens = (ctypes.c_void_p(a.ctypes.data) for a in out)
    head = [ctx, ctypes.byref(sets[0]), ctypes.byref(sets[1]), ctypes.byref(scheme)]
    tail = [scores, counts, ops, ctypes.c_void_p(seg.ctypes.data), lens]
    packed = ctypes.c_uint32(sa.ROWS_PACKED)
    if case["call"] == "rows":
        fn, args = lib.sqmi_align_rows, head + [ctypes.c_uint32(st["mode"])] + tail + [packed]
    elif case["call"] == "local_rows":
        out.append(np.zeros((n, 2), np.int64))
        fn, args = lib.sqmi_align_local_rows, head + tail + [ctypes.c_void_p(out[4].ctypes.data), packed]
    else:
        band = [ctypes.c_int64(-case["band"]), ctypes.c_int64(case["band"])]
        fn, args = lib.sqmi_align_rows_banded, head + [ctypes.c_uint32(st["mode"])] + band + tail + [None, packed]
    st.update(fn=fn, args=args, out=out, keep=(table, scheme, sets, seg))


def prepare(case, seed):
    h, hoff, v, voff = _inputs(case, seed)
    st = {"call": case["call"], "mode": MODES[case["mode"]], "band": case["band"], "score": _scoring(case),
          "ctx": sa.default_context(), "dev": {}}
    if case["resident"]:
        n, alpha = case["pairs"], st["score"].alphabet_size
        none = np.zeros(0, np.uint8)
        st["H"], st["V"] = sa.SeqSet(none, hoff), sa.SeqSet(none, voff)
        st["residues"] = (h, v)     # keeps them alive
        st["out"] = [torch.zeros(n, device="cuda", dtype=torch.int32)]
        st["dev"] = {"h_dev": h.data_ptr(), "v_dev": v.data_ptr(), "scores_dev": st["out"][0].data_ptr()}
        if case["call"] == "counts":
            st["out"].append(torch.zeros((n, alpha * alpha + 2), device="cuda", dtype=torch.int32))
            st["dev"]["counts_dev"] = st["out"][1].data_ptr()
    else:
        st["H"], st["V"] = sa.SeqSet(h.cpu().numpy(), hoff), sa.SeqSet(v.cpu().numpy(), voff)
    if "rows" in case["call"]:
        _rows_call(case, st)
    torch.cuda.synchronize()
    return st


def run(st):
    if "fn" in st:
        status = st["fn"](*st["args"])
        if status:
            raise RuntimeError("rows call: status %d" % status)
        return st["out"]
    ctx, H, V, score, mode, b = st["ctx"], st["H"], st["V"], st["score"], st["mode"], st["band"]
    if st["call"] == "counts":
        got = ctx.align_counts(H, V, score, mode, **st["dev"])
    elif st["call"] == "banded_score":
        got = ctx.align_score_banded(H, V, score, -b, b, mode, **st["dev"])
    else:
        got = ctx.align_score(H, V, score, mode, **st["dev"])
    return st["out"] if got is None else got


def _mean_cells(case):
    """Mean cells and mean residues of a pair."""
    L = case["length"]
    if case["lengths"] == "uniform":
        return (50 + L) / 2 * (50 + 2 * L) / 2, (100 + 3 * L) / 2
    if case["lengths"] == "lognormal":
        x = np.clip(np.exp(np.random.default_rng(0).normal(math.log(L), 1.0, 100000)), 100, 10000)
        return float((x ** 2).mean()), 2 * float(x.mean())
    if case["band"]:
        return min(L * (2 * case["band"] + 1), L * L), 2 * L
    return L * L, 2 * L


def work(case):
    """Residues in, results out; eight operations a cell (two sums and a
    maximum for each gap state's recurrence, shared terms once, two maxima
    for the cell), nine with the local floor."""
    cells, residues = _mean_cells(case)
    alpha = 27 if case["residues"] == "protein" else 4
    out = 4
    if case["call"] != "score" and case["call"] != "banded_score":
        out += 4 * (alpha * alpha + 2)
    if "rows" in case["call"]:
        out += residues / 2 + 8
    return {"bytes": case["pairs"] * (residues + 16 + out),
            "flops": case["pairs"] * cells * (9 if case["mode"] == "local" else 8)}


def exact(case, seed):
    """The scores by the textbook recurrence (Gotoh) in 64 bits over the
    anti-diagonals of all pairs at once; the path outputs have no such value
    (which of several best alignments is returned is a rule, not a number)."""
    h, hoff, v, voff = _inputs(case, seed)
    hl, vl = np.diff(hoff), np.diff(voff)
    n, m = int(hl.max()), int(vl.max())
    if case["pairs"] * (m + 1) * (n + m) > 6e9 or case["pairs"] * max(n, m) > 2e8:
        return None
    dev, LOW = h.device, -(1 << 40)
    hl, vl = (torch.from_numpy(x).to(dev)[:, None] for x in (hl, vl))

    def padded(res, off, width, reverse):
        at = torch.arange(width, device=dev)[None, :]
        at = width - 1 - at if reverse else at
        start = torch.from_numpy(off[:-1]).to(dev)[:, None]
        return res[(start + at).clamp_max(len(res) - 1)].long()

    hr, vp = padded(h, hoff, n, True), padded(v, voff, m, False)
    score, mode, band = _scoring(case), case["mode"], case["band"]
    table = torch.from_numpy(score.table.astype(np.int64)).to(dev).reshape(-1)
    alpha, op, ext = score.alphabet_size, score.gap_open, score.gap_extend
    local = mode == "local"
    top, left = local or mode in ("overlap", "free"), local or mode == "free"
    bottom, right = mode in ("overlap", "free"), mode == "free"
    P = case["pairs"]
    i = torch.arange(m + 1, device=dev)[None, :]
    low = torch.full((P, m + 1), LOW, device=dev, dtype=torch.int64)
    H1, H2, E1, F1 = low.clone(), low.clone(), low.clone(), low.clone()
    best = torch.full((P,), 0 if local else LOW, device=dev, dtype=torch.int64)

    def down(x):     # the value of row i - 1
        return torch.cat([low[:, :1], x[:, :-1]], 1)

    for d in range(n + m + 1):
        j = d - i
        E = torch.maximum(E1 + ext, H1 + op)
        F = torch.maximum(down(F1) + ext, down(H1) + op)
        # Rows 1.. of this diagonal: V[i - 1] against H[d - i - 1] = hr[n - d + i].
        s = torch.zeros((P, m + 1), device=dev, dtype=torch.int64)
        lo, hi = max(1, d - n), min(m, d - 1)
        if lo <= hi:
            s[:, lo:hi + 1] = table[hr[:, n - d + lo:n - d + hi + 1] * alpha + vp[:, lo - 1:hi]]
        G = torch.maximum(torch.maximum(E, F), down(H2) + s)
        if d == 0:
            G[:, 0] = 0
        if top and d <= n:
            G[:, 0] = torch.clamp_min(G[:, 0], 0)
        if left and d <= m:
            G[:, d] = torch.clamp_min(G[:, d], 0)
        if local:
            G = G.clamp_min(0)
        out = (j < 0) | (j > hl) | (i > vl)
        if band:
            out = out | (j - i < -band) | (j - i > band)
        E, F, G = (torch.where(out, LOW, x) for x in (E, F, G))
        end = (i == vl) & (j == hl)
        if local:
            end = ~out
        if bottom:
            end = end | (i == vl)
        if right:
            end = end | (j == hl)
        best = torch.maximum(best, torch.where(end & ~out, G, LOW).max(1).values)
        H1, H2, E1, F1 = G, H1, E, F
    scores = best.to(torch.int32)
    others = {"score": 0, "banded_score": 0, "counts": 1, "rows": 3, "banded_rows": 3, "local_rows": 4}[case["call"]]
    if case["call"] in ("score", "banded_score"):
        return [scores] if case["resident"] else scores
    return [scores] + [None] * others
