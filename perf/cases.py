"""The measured cases: the operators and queries a user of this framework runs, over its own ranges.

Every input is made from the seed with torch on the device.  Numbers of matches, joined rows and
corrupt codes are exact (the same for every seed), so output shapes depend on the case alone: the
positions and values are what the seed chooses.  Corrupt codes carry one flipped bit each, at the
rates of the star-schema workloads (1e-7 to 1e-4 of the codes).

The single operators are called through the C ABI on output buffers the caller owns, as a program
linked against libahead_hip.so does; the operator sequences and whole queries go through the device
BATs (ahead_amd.bat) and ahead_amd.ssb.  All results are whole numbers.
"""
from __future__ import annotations

import ctypes
import math

import torch

from ahead_amd import an, bat as B, capi, ssb

A_OID, A_ERR = an.A_OID, an.A_OID_ERR
RESOID = an.an_meta(an.RESOID, A_OID)
DTYPE = {2: torch.int16, 4: torch.int32, 8: torch.int64}
SIGN = -(1 << 63)

# code width in bits -> (column type, A, largest value): 8-bit values in 16-bit codes, 16-bit values
# in 32-bit codes, 32-bit values in 64-bit codes (the reference's default A per type)
WIDTHS = {16: (an.RESTINY, 233, 0xFF), 32: (an.RESSHORT, 233, 0xFFFF), 64: (an.RESINT, 65117, 0xFFFFFFFF)}

QUERIES = {"Q1.1": ("P1", 20), "Q2.1": ("P2", 32), "Q3.1": ("P3", 32), "Q4.1": ("P4", 48)}  # shape, bytes per row


def listed():
    return [
        # a filtered date dimension (7 years of days): the smallest selection + key fetch of a query
        dict(name="date_keys", kind="dimkeys", rows=2556, matches=365, flips=1),
        # range select + sum of decoded values over a 6M-row fact column (scale factor 1)
        dict(name="select_sum_6m", kind="select", rows=6_000_000, width=32, share=0.5, pred="range", sum=True,
             flips=6),
        # selection on a 60M-row fact measure (scale factor 10), one predicate
        dict(name="select_60m", kind="select", rows=60_000_000, width=64, share=0.5, pred="below", sum=False,
             flips=6),
        # a fact column checked and decoded before a plain operator sees it ("early" detection)
        dict(name="decode_60m", kind="decode", rows=60_000_000, width=64, mode="check_and_decode", flips=6),
        # a dimension attribute fetched for every joined fact row
        dict(name="fetch_60m", kind="fetch", rows=60_000_000, table=200_000, width=16, order="random", flips=6),
        # foreign keys against a whole dimension
        dict(name="hashjoin_60m", kind="hashjoin", rows=60_000_000, table=200_000, build=200_000, share=1.0,
             reenc=False, flips=6),
        # foreign keys against a fifth of a dimension (one region's suppliers), pairs re-encoded as Q2.1 does
        dict(name="hashjoin_region_60m", kind="hashjoin", rows=60_000_000, table=200_000, build=40_000, share=0.2,
             reenc=True, flips=6),
        # the tail of Q4.1 on its joined rows: profit, grouping by year and nation, grouped sum
        dict(name="group_profit_12m", kind="group", rows=12_000_000, years=7, nations=5, flips=12),
        # two selections of one fact table intersected (Q1.1)
        dict(name="merge_60m", kind="merge", rows=60_000_000, left=30_000_000, right=16_400_000, both=8_200_000),
        # a whole query, operator by operator
        dict(name="chain_q21_60m", kind="chain", query="Q2.1", rows=60_000_000, dims=10, flips=6),
        # a whole query with one fact scan
        dict(name="star_q41_240m", kind="star", query="Q4.1", rows=240_000_000, dims=1, flips=24),
        # many selections of uneven length and mixed width in one launch
        dict(name="batch_256", kind="batch", count=256, median=700_000, top=50_000_000, flips=2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _flips(rng, rows):
    return min(rows // 8, int(rows * 10 ** rng.uniform(-7, -4)) + rng.randrange(2))


def draw(rng):
    kind = rng.choice(["dimkeys", "select", "select", "decode", "decode", "fetch", "fetch", "hashjoin", "hashjoin",
                       "group", "sums", "merge", "chain", "star", "batch"])
    if kind == "dimkeys":
        n = _log(rng, 300, 1_500_000)
        return dict(kind=kind, rows=n, matches=max(1, int(n * rng.uniform(0.02, 0.5))), flips=_flips(rng, n))
    if kind == "select":
        n = _log(rng, 2_000, 200_000_000)
        return dict(kind=kind, rows=n, width=rng.choice([16, 32, 64]), share=round(rng.uniform(0.01, 0.9), 3),
                    pred=rng.choice(["range", "below", "outside"]), sum=rng.random() < 0.5, flips=_flips(rng, n))
    if kind == "decode":
        n = _log(rng, 2_000, 200_000_000)
        return dict(kind=kind, rows=n, width=rng.choice([16, 32, 64]),
                    mode=rng.choice(["check", "decode", "check_and_decode"]), flips=_flips(rng, n))
    if kind == "fetch":
        n = _log(rng, 2_000, 150_000_000)
        if rng.random() < 0.5:  # dimension rows in fact order, or a selection's ascending rows of a fact column
            return dict(kind=kind, rows=n, table=_log(rng, 2_556, 3_000_000), width=rng.choice([16, 32]),
                        order="random", flips=_flips(rng, n))
        return dict(kind=kind, rows=n, table=int(n * rng.uniform(1.2, 4)), width=rng.choice([16, 64]),
                    order="ascending", flips=_flips(rng, n))
    if kind == "hashjoin":
        n, t = _log(rng, 2_000, 150_000_000), _log(rng, 2_556, 3_000_000)
        share = 1.0 if rng.random() < 0.4 else round(rng.uniform(0.02, 0.6), 3)
        return dict(kind=kind, rows=n, table=t, build=max(1, int(t * share)), share=share,
                    reenc=rng.random() < 0.5, flips=min(_flips(rng, n), n // 100))
    if kind == "group":
        n = _log(rng, 20_000, 60_000_000)
        return dict(kind=kind, rows=n, years=rng.randrange(1, 8), nations=rng.choice([5, 25, 40]),
                    flips=_flips(rng, n))
    if kind == "sums":
        n = _log(rng, 2_000, 150_000_000)
        return dict(kind=kind, rows=n, width=rng.choice([16, 64]), flips=_flips(rng, n))
    if kind == "merge":
        n = _log(rng, 10_000, 150_000_000)
        l, r = int(n * rng.uniform(0.05, 0.7)), int(n * rng.uniform(0.05, 0.7))
        lo = max(0, l + r - n)
        return dict(kind=kind, rows=n, left=l, right=r, both=lo + int((min(l, r) - lo) * rng.uniform(0.1, 0.9)))
    if kind == "chain":
        n = _log(rng, 2_000_000, 100_000_000)
        return dict(kind=kind, query=rng.choice(list(QUERIES)), rows=n, dims=rng.choice([10, 30]),
                    flips=_flips(rng, n))
    if kind == "star":
        n = _log(rng, 2_000_000, 200_000_000)
        return dict(kind=kind, query=rng.choice(list(QUERIES)), rows=n, dims=rng.choice([1, 3, 10]),
                    flips=min(200, _flips(rng, n)))
    return dict(kind="batch", count=rng.randrange(8, 257), median=_log(rng, 20_000, 700_000), top=20_000_000,
                flips=rng.randrange(0, 4))


# ---- inputs ------------------------------------------------------------------------------------------------

def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 64 + salt)
    return g


def _ints(g, n, lo, hi):
    """n int64 values uniform in [lo, hi]."""
    return torch.randint(lo, hi + 1, (n,), generator=g, device="cuda", dtype=torch.int64)


def _mask(g, n, m):
    """n booleans, exactly m of them true, at random places."""
    mask = torch.rand(n, generator=g, device="cuda") < m / max(1, n)
    d = int(mask.sum()) - m
    if d:
        at = torch.nonzero(mask if d > 0 else ~mask).reshape(-1)
        mask[at[torch.randperm(at.numel(), generator=g, device="cuda")[:abs(d)]]] = d < 0
    return mask


def _fold(x, width):
    """int64 values modulo 2^width (64-bit values wrap by themselves)."""
    return x if width == 64 else x & ((1 << width) - 1)


def _column(codes, meta):
    """A device column over int64 codes, stored at the column's width."""
    n = codes.numel()
    buf = capi.DeviceBuffer(meta.width * n)
    if n:
        buf.t.view(DTYPE[meta.width]).copy_(codes)
    return capi.Column(buf, n, meta)


def _some(g, n, k):
    """k distinct positions below n, ascending."""
    return torch.nonzero(_mask(g, n, k)).reshape(-1)


def _hit(codes, lo, hi, inside):
    """Unsigned lo <= code <= hi over int64 bit patterns."""
    return (((codes - lo) ^ SIGN) <= ((hi - lo) ^ SIGN)) == inside


def _flip(g, codes, at, bits):
    """One random bit of `bits` flipped in the codes at positions `at`."""
    if at.numel():
        b = torch.tensor(bits, device="cuda")[_ints(g, at.numel(), 0, len(bits) - 1)]
        codes[at] = codes[at] ^ (torch.ones_like(b) << b)


def _selection(case, g):
    """Values and codes of a column of which exactly share * rows codes (flipped ones among them)
    satisfy the predicate: (values, codes, flipped rows, lo, hi of the interval, matches)."""
    n, width = case["rows"], case["width"]
    _, a, top = WIDTHS[width]
    m = int(n * case["share"])
    part = max(1, int((top + 1) * (1 - case["share"] if case["pred"] == "outside" else case["share"])))
    lo = 0 if case["pred"] == "below" else (top + 1 - part) // 2
    hi = min(top, lo + part - 1)
    inside = case["pred"] != "outside"
    mask = _mask(g, n, m if inside else n - m)  # rows in the interval
    span = hi - lo + 1
    if span > top:
        mask[:] = True
        m = n if inside else 0
    v = torch.where(mask, _ints(g, n, lo, hi), _ints(g, n, 0, max(0, top - span)))
    v += torch.where(~mask & (v >= lo), span, 0)
    codes = v * a
    at = _some(g, n, case["flips"])
    if at.numel():  # a bit whose flip leaves the row's side of the predicate
        one = torch.ones(width, dtype=torch.int64, device="cuda") << torch.arange(width, device="cuda")
        near = _fold(codes[at][:, None] ^ one[None, :], width)
        same = _hit(near, lo * a, hi * a, True) == mask[at][:, None]
        pick = (torch.rand(near.shape, generator=g, device="cuda") * same).argmax(1)
        codes[at] = near[torch.arange(at.numel(), device="cuda"), pick]
    return v, codes, at, lo, hi, mask if inside else ~mask, m


def _table(seed, case):
    """The star-schema columns of a query: name -> (values, codes, meta), the selected attributes of
    each dimension and lo_quantity with `flips` corrupt codes."""
    g = _gen(seed)
    spec = ssb.SsbSpec(n_fact=case["rows"], n_cust=3_000_000 // case["dims"], n_supp=200_000 // case["dims"],
                       n_part=1_400_000 // case["dims"])
    rows = {"date": spec.n_date, "cust": spec.n_cust, "supp": spec.n_supp, "part": spec.n_part, "fact": spec.n_fact}
    q = ssb.QUERIES[case["query"]]
    want = set(q.meas) | {c for c, _ in q.preds}
    for d in q.dims:
        want |= set(ssb.DIM_KEYS[d.name]) | {c for c, _ in d.sels} | ({d.attr} if d.attr else set())
    want |= {c for c in ("d_year",) if any(d.name == "date" for d in q.dims)}
    made = {}

    def values(name):
        if name not in made:
            table, _, _, vs, _ = ssb.COLUMNS[name]
            n = rows[table]
            if vs[0] == "rowid":
                v = torch.arange(n, device="cuda")
            elif vs[0] == "cal":
                v = 1992 + torch.arange(n, device="cuda") * 7 // n
            elif vs[0] == "fk":
                v = _ints(g, n, 0, rows[vs[1]] - 1)
            elif vs[0] == "uniform":
                v = _ints(g, n, vs[1], vs[2])
            else:
                v = values(vs[1]) * vs[2] + _ints(g, n, 0, vs[3] - 1)
            made[name] = v
        return made[name]

    out = {}
    for name in sorted(want):
        table, kind, _, _, flipped = ssb.COLUMNS[name]
        v, meta = values(name), ssb.META[kind]
        codes = v * meta.a
        if flipped:
            k = case["flips"] if table == "fact" else 1
            _flip(g, codes, _some(g, v.numel(), k), range(8 * meta.width))
        out[name] = (v, codes, meta)
    return q, out


def _inputs(case, seed):
    g = _gen(seed)
    n = case.get("rows", 0)
    kind = case["kind"]
    if kind == "select":
        return _selection(case, g)
    if kind == "dimkeys":
        mask = _mask(g, n, case["matches"])
        attr = torch.where(mask, 1994, 1992 + _ints(g, n, 0, 1))
        codes = attr * ssb.A_SHORT
        at = torch.nonzero(~mask).reshape(-1)
        at = at[torch.randperm(at.numel(), generator=g, device="cuda")[:case["flips"]]]
        _flip(g, codes, at, (0, 1, 2))  # (1992 or 1993) * A and 1994 * A differ in higher bits too
        return mask, codes, at.sort().values
    if kind == "decode":
        _, a, top = WIDTHS[case["width"]]
        v = _ints(g, n, 0, top)
        codes, at = v * a, _some(g, n, case["flips"])
        _flip(g, codes, at, range(case["width"]))
        return v, codes, at
    if kind == "fetch":
        _, a, top = WIDTHS[case["width"]]
        t = _ints(g, case["table"], 0, top)
        o = (_some(g, case["table"], n) if case["order"] == "ascending" else _ints(g, n, 0, case["table"] - 1))
        codes, at = o * A_OID, _some(g, n, case["flips"])
        _flip(g, codes, at, range(64))
        return t, t * a, o, codes, at
    if kind == "hashjoin":
        keys = torch.arange(case["table"], device="cuda")
        sel = _mask(g, case["table"], case["build"])
        in_, out = keys[sel], keys[~sel]
        joins = _mask(g, n, int(n * case["share"])) if out.numel() else torch.ones(n, dtype=torch.bool, device="cuda")
        fk = in_[_ints(g, n, 0, in_.numel() - 1)]
        if out.numel():
            fk = torch.where(joins, fk, out[_ints(g, n, 0, out.numel() - 1)])
        codes = fk * ssb.A_KEY
        at = _some(g, n, case["flips"])
        # a flip in the upper half leaves the 32-bit key (the row still joins), one in the lower does not
        low = joins[at] & (torch.arange(at.numel(), device="cuda") % 2 == 0)
        _flip(g, codes, at[low], range(32))
        _flip(g, codes, at[~low], range(32, 64))
        kept = joins.clone()
        kept[at[low]] = False
        # rows that join: fixed, so as many rows that do not join as flips took out of the join do now
        want = int(n * case["share"]) - (at.numel() + 1) // 2
        more = torch.nonzero(kept).reshape(-1)
        for_out = more[~torch.isin(more, at)][:max(0, int(kept.sum()) - want)]
        codes[for_out] = (case["table"] + 5) * ssb.A_KEY
        kept[for_out] = False
        return in_, fk, codes, at, kept
    if kind == "group":
        y, k = _ints(g, n, 0, case["years"] - 1), _ints(g, n, 0, case["nations"] - 1)
        rev, cost = _ints(g, n, 90_000, 10_500_000), _ints(g, n, 1_000, 80_000)
        rc, cc = rev * ssb.A_MEAS, cost * ssb.A_MEAS
        at = _some(g, n, case["flips"])
        _flip(g, rc, at, range(64))
        return y, k, rev, cost, rc, cc, at
    if kind == "sums":
        p, d = _ints(g, n, 90_000, 10_500_000), _ints(g, n, 0, 10)
        pc, at = p * ssb.A_MEAS, _some(g, n, case["flips"])
        _flip(g, pc, at, range(64))
        return p, d, pc, at
    if kind == "merge":
        l, r, both = case["left"], case["right"], case["both"]
        left = _mask(g, n, l)
        lrows, rest = torch.nonzero(left).reshape(-1), torch.nonzero(~left).reshape(-1)
        hit, miss = lrows[_some(g, l, both)], rest[_some(g, n - l, r - both)]
        return lrows, torch.cat([hit, miss]).sort().values, hit
    if kind == "batch":
        lens = torch.exp(torch.randn(case["count"], generator=torch.Generator().manual_seed(4242)) * 1.42)
        jobs = []
        for i, x in enumerate(lens.tolist()):  # lengths are the case's own; values and flips the seed's
            rows = int(min(case["top"], max(10_000, x * case["median"])))
            c = dict(rows=rows, width=(16, 32, 64)[i % 3], share=0.01 + 0.49 * ((i * 37) % 100) / 100, pred="range",
                     flips=case["flips"])
            jobs.append((c, _selection(c, _gen(seed, 0) if i == 0 else g)))
        return jobs
    raise ValueError(kind)


# ---- calls -------------------------------------------------------------------------------------------------

def _bytes(n):
    return capi.DeviceBuffer(max(8, n))


def _u64(buf, n):
    return buf.t[:8 * n].view(torch.int64)


class _Call:
    """An entry point of the C ABI with its arguments and the caller's output buffers."""

    def __init__(self, name, args, outs, keep):
        self.fn, self.args, self.outs, self.keep = getattr(capi.load(), name), args, outs, keep

    def __call__(self):
        st = self.fn(*self.args, capi.current_stream())
        if st:
            capi.check(st)
        return self.outs


def _errs(k, cap):
    return [_bytes(8 * cap) for _ in range(k)]


def prepare(case, seed):
    kind, n = case["kind"], case.get("rows", 0)
    ws = capi.workspace().h
    ref = ctypes.byref
    cnt = capi.DeviceBuffer(64, zero=True)
    if kind == "select":
        _, codes, at, lo, hi, _, m = _inputs(case, seed)
        t, a, _ = WIDTHS[case["width"]]
        col, oids, (err,) = _column(codes, an.an_meta(t, a)), _bytes(8 * n), _errs(1, 4096 + at.numel())
        pred = {"range": (capi.GE, lo * a, capi.LE, hi * a, capi.COMB_AND), "below": (capi.LE, hi * a, 0, 0, 0),
                "outside": (capi.LT, lo * a, capi.GT, hi * a, capi.COMB_OR)}[case["pred"]]
        total = _bytes(8) if case["sum"] else None
        outs = [_u64(oids, m), _u64(err, at.numel()), _u64(cnt, 2)] + ([_u64(total, 1)] if total else [])
        return _Call("ahead_hip_select_an",
                     (ref(col.desc()), *pred, A_OID, A_ERR, oids.ptr, n, err.ptr, 4096 + at.numel(), cnt.ptr,
                      total.ptr if total else None, ws), outs, (col, oids, err, total, cnt))
    if kind == "decode":
        _, codes, at = _inputs(case, seed)
        t, a, _ = WIDTHS[case["width"]]
        col, (err,) = _column(codes, an.an_meta(t, a)), _errs(1, 4096 + at.numel())
        w, ecap, k = t.unenc_bits // 8, 4096 + at.numel(), at.numel()
        dec = _bytes(w * n)
        d = ref(col.desc())
        keep = (col, dec, err, cnt)
        if case["mode"] == "check":
            return _Call("ahead_hip_check_an", (d, A_ERR, err.ptr, ecap, cnt.ptr, ws), [_u64(err, k), _u64(cnt, 1)],
                         keep)
        left = n - k if case["mode"] == "check_and_decode" else n
        outs = [dec.t[:w * left], _u64(err, k), _u64(cnt, 2)]
        if case["mode"] == "decode":
            return _Call("ahead_hip_decode_an", (d, A_ERR, dec.ptr, err.ptr, ecap, cnt.ptr, ws), outs, keep)
        return _Call("ahead_hip_check_and_decode_an", (d, A_ERR, dec.ptr, n, err.ptr, ecap, cnt.ptr, ws), outs, keep)
    if kind == "fetch":
        _, tc, _, oc, at = _inputs(case, seed)
        t, a, _ = WIDTHS[case["width"]]
        col, oids = _column(tc, an.an_meta(t, a)), _column(oc, RESOID)
        out, errs, k = _bytes(t.width * n), _errs(2, 4096 + at.numel()), at.numel()
        return _Call("ahead_hip_fetchjoin_an",
                     (ref(oids.desc()), ref(col.desc()), 0, 0, A_ERR, capi.Buf(out.ptr, n),
                      *[capi.Buf(e.ptr, 4096 + k) for e in errs], cnt.ptr, ws),
                     [out.t[:t.width * (n - k)], _u64(errs[0], k), _u64(cnt, 3)], (col, oids, out, errs, cnt))
    if kind == "hashjoin":
        keys, _, codes, at, kept = _inputs(case, seed)
        meta = ssb.META["key"]
        fk, key = _column(codes, meta), _column(keys * ssb.A_KEY, meta)
        pairs, w = int(n * case["share"]) - (at.numel() + 1) // 2, 8 if case["reenc"] else 4
        out_h, out_t, errs = _bytes(w * n), _bytes(w * n), _errs(4, 4096 + at.numel())
        # the dimension's row ids beside its keys, as a selection's OIDs (re-encoded) or void
        if case["reenc"]:
            dim = _column(keys * A_OID, RESOID)
            tail = (1, A_OID * an.inverse(A_OID, 64) & an.MASK64, w)
        else:
            dim, tail = capi.Column.void(keys.numel()), (0, 0, w)
        head = (1, A_OID, w) if case["reenc"] else (0, 0, w)
        return _Call("ahead_hip_hashjoin_an",
                     (ref(capi.Column.void(n).desc()), ref(fk.desc()), ref(key.desc()), ref(dim.desc()), 1, *head, *tail,
                      A_ERR, capi.Buf(out_h.ptr, n), capi.Buf(out_t.ptr, n),
                      *[capi.Buf(e.ptr, 4096 + at.numel()) for e in errs], cnt.ptr, ws),
                     [out_h.t[:w * pairs], out_t.t[:w * pairs], _u64(errs[1], at.numel()), _u64(cnt, 6)],
                     (fk, key, dim, out_h, out_t, errs, cnt))
    if kind == "sums":
        _, d, pc, at = _inputs(case, seed)
        p = _column(pc, ssb.META["meas"])
        x = _column(d * (ssb.A_TINY if case["width"] == 16 else ssb.A_MEAS),
                    ssb.META["tiny" if case["width"] == 16 else "meas"])
        total, errs, k = _bytes(8), _errs(2, 4096 + at.numel()), at.numel()
        return _Call("ahead_hip_aggregate_mul_sum_an",
                     (ref(p.desc()), ref(x.desc()), 0, 1, an.A_RESULT, A_ERR, total.ptr,
                      *[capi.Buf(e.ptr, 4096 + k) for e in errs], cnt.ptr, ws),
                     [_u64(total, 1), _u64(errs[0], k), _u64(cnt, 3)], (p, x, total, errs, cnt))
    if kind == "merge":
        left, right, hit = _inputs(case, seed)
        l, r = _column(left * A_OID, RESOID), _column(right * A_OID, RESOID)
        cap = max(1, min(l.n, r.n))
        out_h, out_t, errs = _bytes(8 * cap), _bytes(8 * cap), _errs(4, 1024)
        dl, dr = l.desc(), r.desc()
        return _Call("ahead_hip_matchjoin_merge_an",
                     (ref(dl), ref(dl), ref(dr), ref(dr), 0, 0, 8, 0, 0, 8, A_ERR, capi.Buf(out_h.ptr, cap),
                      capi.Buf(out_t.ptr, cap), *[capi.Buf(e.ptr, 1024) for e in errs], cnt.ptr, ws),
                     [_u64(out_h, hit.numel()), _u64(out_t, hit.numel()), _u64(cnt, 5)],
                     (l, r, out_h, out_t, errs, cnt))
    if kind == "batch":
        jobs = _inputs(case, seed)
        arr, keep, k = (capi.SelectJob * len(jobs))(), [], case["flips"]
        total = sum(x[-1] for _, x in jobs)
        # the instances' outputs one after another, each exactly as long as its result
        oids, errs, sums, counts = (_bytes(8 * c) for c in (total, k * len(jobs), len(jobs), 2 * len(jobs)))
        at = 0
        for i, (c, (_, codes, _, lo, hi, _, m)) in enumerate(jobs):
            t, a, _ = WIDTHS[c["width"]]
            col = _column(codes, an.an_meta(t, a))
            keep.append(col)
            arr[i] = capi.SelectJob(col.desc(), capi.GE, capi.LE, capi.COMB_AND, 0, lo * a, hi * a, A_OID, A_ERR,
                                    oids.ptr + 8 * at, m, errs.ptr + 8 * k * i, k, counts.ptr + 16 * i, sums.ptr + 8 * i)
            at += m
        h = ctypes.c_void_p()
        capi.check(capi.load().ahead_hip_select_batch_create(arr, len(jobs), 16, 0, ctypes.byref(h)))
        return _Batch(h, [_u64(oids, total), _u64(errs, k * len(jobs)), _u64(sums, len(jobs)),
                          _u64(counts, 2 * len(jobs))], (keep, oids, errs, sums, counts))
    if kind == "dimkeys":
        _, codes, _ = _inputs(case, seed)
        return {"kind": kind, "attr": B.BAT(capi.Column.void(n), _column(codes, ssb.META["short"])),
                "key": B.BAT(capi.Column.void(n), _column(torch.arange(n, device="cuda") * ssb.A_KEY, ssb.META["key"]))}
    if kind == "group":
        y, k, _, _, rc, cc, _ = _inputs(case, seed)

        def side(codes, meta):
            return B.BAT(capi.Column.void(n), _column(codes, meta))
        return {"kind": kind, "year": side((1992 + y) * ssb.A_SHORT, ssb.META["short"]),
                "nation": side(k * ssb.A_TINY, ssb.META["tiny"]), "revenue": side(rc, ssb.META["meas"]),
                "cost": side(cc, ssb.META["meas"])}
    q, cols = _table(seed, case)
    t = {}
    for name in list(cols):
        _, codes, meta = cols.pop(name)
        t[name] = B.BAT(capi.Column.void(codes.numel()), _column(codes, meta))
    if kind == "star":  # a program keeps the key index with a resident dimension
        for d in q.dims:
            B.key_index(t[ssb.DIM_KEYS[d.name][1]].tail)
    return {"kind": kind, "q": q, "t": t}


class _Batch:
    """A batch of selections: its handle, kept as long as its columns."""

    def __init__(self, h, outs, keep):
        self.h, self.outs, self.keep, self.lib = h, outs, keep, capi.load()

    def __call__(self):
        capi.check(self.lib.ahead_hip_select_batch_launch(self.h, capi.current_stream()))
        return self.outs

    def __del__(self):
        self.lib.ahead_hip_select_batch_destroy(self.h)


def _codes(col):
    return col.buf.t[:col.meta.width * col.n]


def run(state):
    if not isinstance(state, dict):
        return state()
    if state["kind"] == "dimkeys":
        sel, err = B.selectAN(state["attr"], capi.EQ, 1994 * ssb.A_SHORT)
        r = B.matchjoinAN(state["key"].reverse(), sel.mirror_head())
        return [_codes(r[0].head), _codes(r[0].tail), err]
    if state["kind"] == "group":
        profit = B.arithmeticAN(B.SUB, state["revenue"], state["cost"])
        g1 = B.groupbyAN(state["year"])
        g2 = B.groupbyAN(state["nation"], g1[0], g1[1].size())
        s = B.aggregate_sum_groupedAN(profit[0], g2[0], g2[1].size())
        return [_codes(profit[0].tail), _codes(g2[0].tail), _codes(g2[1].tail), _codes(s[0].tail), profit[2], s[2]]
    r = (ssb.chain if state["kind"] == "chain" else ssb.fused)(state["t"], state["q"])
    out = [r["rows"], [v for _, v in r["errors"].items]]
    return out + ([r["result"] & (2 ** 63 - 1)] if "result" in r else [r["sums"], r["keys"]])


# ---- what a pass cannot do without ---------------------------------------------------------------------------

def work(case):
    kind, n = case["kind"], case.get("rows", 0)
    k = case.get("flips", 0)
    if kind == "select":
        b = n * case["width"] // 8 + 8 * int(n * case["share"]) + 8 * k
    elif kind == "decode":
        b = n * case["width"] // 8 + (0 if case["mode"] == "check" else n * case["width"] // 16) + 8 * k
    elif kind == "fetch":
        t = min(case["table"], n) if case["order"] == "ascending" else case["table"]
        b = 8 * n + (n + t) * case["width"] // 8 + 8 * k
    elif kind == "hashjoin":
        b = 8 * n + 8 * case["build"] + int(n * case["share"]) * (16 if case["reenc"] else 8) + 8 * k
    elif kind == "sums":
        b = (8 + case["width"] // 8) * n + 8 * k
    elif kind == "merge":
        b = 8 * (case["left"] + case["right"]) + 16 * case["both"]
    elif kind == "dimkeys":
        b = 4 * n + 8 * case["matches"] * 4 + 8 * k  # attribute, OIDs, the selected keys, both outputs
    elif kind == "group":
        b = n * (4 + 2 + 8 + 8 + 8 + 8) + 16 * k     # the four columns, the profits and the group ids
    elif kind == "batch":
        b = 0
        lens = torch.exp(torch.randn(case["count"], generator=torch.Generator().manual_seed(4242)) * 1.42)
        for i, x in enumerate(lens.tolist()):
            rows = int(min(case["top"], max(10_000, x * case["median"])))
            b += rows * (2, 4, 8)[i % 3] + 8 * int(rows * (0.01 + 0.49 * ((i * 37) % 100) / 100)) + 8 * k
    else:
        b = n * QUERIES[case["query"]][1]            # every fact column the query names, once
    return {"bytes": int(b), "flops": 0}


def tolerance(case):
    return "exact"


# ---- the same in plain torch -----------------------------------------------------------------------------------

def _sgn(x):
    """A whole number modulo 2^64 as an int64 value."""
    x &= an.MASK64
    return x - (1 << 64) if x >> 63 else x


def exact(case, seed):
    kind, n = case["kind"], case.get("rows", 0)
    if kind in ("chain", "star"):
        return _exact_query(case, seed)
    if kind == "batch":
        jobs = _inputs(case, seed)
        oids = torch.cat([torch.nonzero(x[5]).reshape(-1) * A_OID for _, x in jobs])
        errs = torch.cat([x[2] * A_ERR for _, x in jobs])
        sums = torch.stack([_clean(x[5], x[2], x[0]).sum() for _, x in jobs])
        counts = torch.tensor([c for _, x in jobs for c in (x[-1], x[2].numel())], device="cuda")
        return [oids, errs, sums, counts]
    x = _inputs(case, seed)

    def count(*v):
        return torch.tensor(v, device="cuda")

    def stored(v, width):
        return v.to(DTYPE[width]).view(torch.uint8) if width > 1 else (v & 255).to(torch.uint8)

    if kind == "select":
        v, _, at, _, _, hit, m = x
        out = [torch.nonzero(hit).reshape(-1) * A_OID, at * A_ERR, count(m, at.numel())]
        return out + ([_clean(hit, at, v).sum().reshape(1)] if case["sum"] else [])
    if kind == "decode":
        v, codes, at = x
        if case["mode"] == "check":
            return [at * A_ERR, count(at.numel())]
        t, a, _ = WIDTHS[case["width"]]
        keep = torch.ones(n, dtype=torch.bool, device="cuda")
        if case["mode"] == "decode":  # a corrupt code decodes to the low half of code * A^-1
            v[at] = codes[at] * _sgn(an.inverse(a, case["width"]))
        else:
            keep[at] = False
        return [stored(v[keep], t.unenc_bits // 8), at * A_ERR, count(int(keep.sum()), at.numel())]
    if kind == "fetch":
        _, tc, o, _, at = x
        keep = torch.ones(n, dtype=torch.bool, device="cuda")
        keep[at] = False
        return [stored(tc[o[keep]], case["width"] // 8), at * A_ERR, count(n - at.numel(), at.numel(), 0)]
    if kind == "hashjoin":
        keys, fk, _, at, kept = x
        rows = torch.nonzero(kept).reshape(-1)
        at_row = torch.searchsorted(keys, fk[rows])
        if case["reenc"]:
            h, t = stored(rows * A_OID, 8), stored(keys[at_row] * A_OID, 8)
        else:
            h, t = stored(rows, 4), stored(at_row, 4)
        return [h, t, at * A_ERR, count(rows.numel(), 0, at.numel(), 0, 0, 0)]
    if kind == "sums":
        p, d, pc, at = x
        total = (pc * _sgn(an.inverse(ssb.A_MEAS, 64)) * d).sum() * an.A_RESULT
        return [total.reshape(1), at * A_ERR, count(1, at.numel(), 0)]
    if kind == "merge":
        codes = x[2] * A_OID
        return [codes, codes, count(codes.numel(), 0, 0, 0, 0)]
    if kind == "dimkeys":
        mask, _, at = x
        rows = torch.nonzero(mask).reshape(-1)
        return [stored(rows * ssb.A_KEY, 8), stored(rows * A_OID, 8), at * A_ERR]
    if kind == "group":
        y, k, _, _, rc, cc, at = x
        profit = (rc * _sgn(an.inverse(ssb.A_MEAS, 64)) - cc * _sgn(an.inverse(ssb.A_MEAS, 64))) * an.A_RESULT
        gid, first = _first_groups(y * 64 + k)
        sums = torch.zeros(first.numel(), dtype=torch.int64, device="cuda").index_add_(0, gid, profit)
        return [stored(profit, 8), stored(gid * A_OID, 8), stored(first * A_OID, 8), stored(sums, 8), at * A_ERR, None]
    return None


def _clean(hit, at, v):
    """The decoded values of matching rows whose code is not corrupt."""
    hit = hit.clone()
    hit[at] = False
    return v[hit]


def _first_groups(key):
    """Group number of every row in order of first occurrence, and each group's first row."""
    _, inv = torch.unique(key, return_inverse=True)
    k = int(inv.max()) + 1
    first = torch.full((k,), key.numel(), dtype=torch.int64, device="cuda")
    first.scatter_reduce_(0, inv, torch.arange(key.numel(), device="cuda"), "amin")
    order = torch.argsort(first)
    rank = torch.empty_like(order)
    rank[order] = torch.arange(k, device="cuda")
    return rank[inv], first[order]


def _holds(col, p):
    codes, meta = _fold(col[1], 8 * col[2].width), col[2]
    ops = {B.LT: lambda a, b: a < b, B.LE: lambda a, b: a <= b, B.GT: lambda a, b: a > b, B.GE: lambda a, b: a >= b,
           B.EQ: lambda a, b: a == b}
    r = ops[p[0]](codes, p[1] * meta.a)
    if len(p) > 2:
        s = ops[p[2]](codes, p[3] * meta.a)
        r = r & s if p[4] == B.AND else r | s
    return r


def _exact_query(case, seed):
    q, cols = _table(seed, case)
    keep = torch.ones(case["rows"], dtype=torch.bool, device="cuda")
    for c, p in q.preds:
        keep &= _holds(cols[c], p)
    for d in q.dims:
        for c, p in d.sels:
            keep &= _holds(cols[c], p)[cols[ssb.DIM_KEYS[d.name][0]][0]]
    rows = torch.nonzero(keep).reshape(-1)
    m = [cols[c][0][rows] for c in q.meas]
    value = m[0] * m[1] if q.kind == ssb.MULSUM else m[0] - m[1] if q.kind == ssb.SUBTRACT else m[0]
    if not q.groups:
        return [rows.numel(), None, int(value.sum())]
    attrs = [cols[q.dims[i].attr][0][cols[ssb.DIM_KEYS[q.dims[i].name][0]][0][rows]] for i in q.groups]
    key = torch.zeros_like(rows)
    for a in attrs:
        key = key * 4096 + a
    gid, first = _first_groups(key)
    sums = torch.zeros(first.numel(), dtype=torch.int64, device="cuda").index_add_(0, gid, value)
    return [rows.numel(), None, sums, [a[first] for a in attrs]]
