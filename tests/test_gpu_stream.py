"""The single-pass engine (stream.hpp) at the edges of its tiles (1024 threads x 4, 8, 16 or 32 rows, by the size
of the call) and of its 512-tile window, against the oracle: outputs, counts and error positions."""
import ctypes

import numpy as np
import pytest

import oracle_lib as O
from ahead_amd import an, capi, datagen

pytestmark = pytest.mark.gpu

KINDS = {2: (an.RESTINY, 233, 0xFF), 4: (an.RESSHORT, 63877, 0xFFFF), 8: (an.RESINT, 65117, 0xFFFFFFFF)}
TILE = 1024 * 16


def codes_of(n, width, bad, seed):
    t, a, top = KINDS[width]
    rng = np.random.default_rng(seed)
    c = datagen.encode(rng.integers(0, top + 1, n).astype(np.uint64), a, width)
    hit = rng.choice(n, min(bad, n), replace=False)
    c[hit] ^= (np.ones(hit.size, np.uint64) << rng.integers(0, 8 * width, hit.size).astype(np.uint64)).astype(c.dtype)
    return c, an.an_meta(t, a)


def decode_call(col, cap, ecap, stream=None):
    lib, ws = capi.load(), capi.workspace()
    w = col.meta.type.unenc_bits // 8
    dec, err, cnt = capi.DeviceBuffer(max(8, w * cap)), capi.DeviceBuffer(8 * ecap), capi.DeviceBuffer(16)
    d = col.desc()

    def launch(s=None):
        capi.check(lib.ahead_hip_check_and_decode_an(ctypes.byref(d), an.A_OID_ERR, dec.ptr, cap, err.ptr, ecap,
                                                     cnt.ptr, ws.h, capi.current_stream() if s is None else s))
    return launch, dec, err, cnt


@pytest.mark.parametrize("width", [2, 4, 8])
@pytest.mark.parametrize("n,bad", [
    (0, 0), (1, 0), (1, 1), (63, 2), (TILE - 1, 0), (TILE, 1), (TILE + 1, 3), (2 * TILE + 64, 40),
    (40 * TILE + 777, 0), (40 * TILE + 777, 5000), (511 * TILE + 5, 3), (513 * TILE + 9, 700),
    (1100 * TILE + 31, 2),
])
def test_check_and_decode_tiles(width, n, bad):
    codes, meta = codes_of(n, width, bad, seed=n + bad + width)
    col = capi.Column.from_numpy(codes, meta)
    ref = O.check_and_decode_an(O.Col(codes, meta))
    print(f"check_and_decode width={width} n={n} bad={bad}", flush=True)
    launch, dec, err, cnt = decode_call(col, n, max(1, bad))
    launch()
    capi.synchronize()
    c = [int(x) for x in cnt.to_numpy(np.uint64, 2)]
    assert c == [len(ref[0]), len(ref[1])]
    assert np.array_equal(dec.to_numpy(f"u{meta.type.unenc_bits // 8}", c[0]), ref[0])
    assert np.array_equal(err.to_numpy(np.uint64, c[1]), ref[1])


@pytest.mark.parametrize("width", [2, 4, 8])
@pytest.mark.parametrize("tiles,past", [(1, 1), (96, -1), (96, 0), (384, -1), (384, 0), (384, 1)])
def test_check_and_decode_where_the_tile_changes(width, tiles, past):
    """Rows per lane follow the size of a call: 4, 8 or the operator's own (launch_stream)."""
    import torch

    per_cu = torch.cuda.get_device_properties(0).multi_processor_count / 256
    rows = 8 if tiles <= 96 else 32 if width == 2 else 16
    n = int(tiles * per_cu) * 1024 * rows + past
    codes, meta = codes_of(n, width, 5, seed=n)
    print(f"check_and_decode width={width} n={n}", flush=True)
    ref = O.check_and_decode_an(O.Col(codes, meta))
    launch, dec, err, cnt = decode_call(capi.Column.from_numpy(codes, meta), n, 5)
    launch()
    capi.synchronize()
    assert [int(x) for x in cnt.to_numpy(np.uint64, 2)] == [len(ref[0]), len(ref[1])]
    assert np.array_equal(dec.to_numpy(f"u{meta.type.unenc_bits // 8}", len(ref[0])), ref[0])
    assert np.array_equal(err.to_numpy(np.uint64, len(ref[1])), ref[1])


@pytest.mark.parametrize("cap,ecap", [(0, 1), (1, 0), (TILE - 3, 7), (2 * TILE + 100, 900)])
def test_check_and_decode_capacities(cap, ecap):
    n, bad = 3 * TILE + 11, 800
    codes, meta = codes_of(n, 8, bad, seed=9)
    ref = O.check_and_decode_an(O.Col(codes, meta))
    launch, dec, err, cnt = decode_call(capi.Column.from_numpy(codes, meta), n, bad)
    guard = 0xAB
    dec.t.fill_(guard)
    err.t.fill_(guard)
    lib, ws = capi.load(), capi.workspace()
    d = capi.Column.from_numpy(codes, meta)
    x = d.desc()
    capi.check(lib.ahead_hip_check_and_decode_an(ctypes.byref(x), an.A_OID_ERR, dec.ptr, cap, err.ptr, ecap, cnt.ptr,
                                                 ws.h, capi.current_stream()))
    capi.synchronize()
    assert [int(v) for v in cnt.to_numpy(np.uint64, 2)] == [len(ref[0]), len(ref[1])]
    got, e = dec.to_numpy(np.uint32, n), err.to_numpy(np.uint64, bad)
    k, j = min(cap, len(ref[0])), min(ecap, len(ref[1]))
    assert np.array_equal(got[:k], ref[0][:k]) and np.array_equal(e[:j], ref[1][:j])
    assert (got[k:].view(np.uint8) == guard).all() and (e[j:].view(np.uint8) == guard).all()


def test_check_and_decode_graph_replays():
    """The ticket and epoch live on the device: a captured launch gives the right result on every
    replay, over changed codes, with calls of other sizes between the replays."""
    import torch

    n = 20 * TILE + 5
    sets = [codes_of(n, 8, bad, seed=bad) for bad in (0, 3, 900)]
    meta = sets[0][1]
    col = capi.Column.from_numpy(sets[0][0], meta)
    launch, dec, err, cnt = decode_call(col, n, 1000)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        launch(side.cuda_stream)  # the workspace takes its size before the capture
        side.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            launch(side.cuda_stream)
        for codes, _ in sets + sets[::-1]:
            col.buf.t.copy_(torch.from_numpy(codes.view(np.uint8)))
            small, sm = codes_of(3 * TILE + 1, 8, 2, seed=1)
            got = capi.check_and_decode_an(capi.Column.from_numpy(small, sm))
            assert np.array_equal(got[0], O.check_and_decode_an(O.Col(small, sm))[0])
            g.replay()
            side.synchronize()
            ref = O.check_and_decode_an(O.Col(codes, meta))
            c = [int(v) for v in cnt.to_numpy(np.uint64, 2)]
            assert c == [len(ref[0]), len(ref[1])]
            assert np.array_equal(dec.to_numpy(np.uint32, c[0]), ref[0])
            assert np.array_equal(err.to_numpy(np.uint64, c[1]), ref[1])


@pytest.mark.parametrize("t,a,rows,n,span,bad,past", [
    # 2-byte columns: codes in LDS up to 76,800 rows; packed values beyond, by the bits they need
    (an.RESTINY, 233, 76_800, 700_001, 256, 0, 3), (an.RESTINY, 233, 76_801, 2_600_000, 256, 0, 0),
    (an.RESTINY, 29, 200_000, 6_500_003, 256, 9, 5), (an.RESTINY, 29, 200_000, 6_500_003, 25, 4, 1),
    (an.RESTINY, 29, 200_000, 6_500_003, 4, 0, 0), (an.RESTINY, 233, 1_000_001, 32_100_000, 256, 1, 2),
    (an.RESTINY, 233, 200_000, 6_400_001, 1, 200_000, 0), (an.RESTINY, 233, 200_000, 6_399_999, 256, 2, 2),
    # 4-byte columns, an offset far from zero, values too wide to pack
    (an.RESSHORT, 63877, 38_400, 620_000, 65_536, 3, 1), (an.RESSHORT, 63877, 60_000, 3_900_000, 7, 1, 0),
    (an.RESSHORT, 63877, 120_000, 7_700_000, 1000, 2, 2), (an.RESSHORT, 63877, 500_000, 32_000_001, 65_536, 2, 2),
    # 8-byte and plain columns
    (an.RESINT, 65117, 19_200, 620_000, 1 << 32, 2, 1), (an.RESINT, 65117, 19_201, 620_000, 1 << 32, 2, 1),
    (an.TINYINT, 1, 150_000, 700_000, 256, 0, 2), (an.SHORTINT, 1, 5_000, 100_000, 65_536, 0, 2),
    (an.INT, 1, 5_000, 100_000, 1 << 32, 0, 2), (an.RESTINY, 233, 1, 40_000, 256, 0, 7),
])
def test_fetch_tables(t, a, rows, n, span, bad, past):
    """fetchjoinAN with its column in LDS (codes, packed values, in part) and from the column."""
    rng = np.random.default_rng(rows + n + span)
    meta = an.an_meta(t, a) if t.encoded else an.plain_meta(t)
    lo = min(1992, (1 << t.unenc_bits) - span) if span < (1 << t.unenc_bits) else 0
    v = (lo + rng.integers(0, span, rows)).astype(np.uint64)
    col = datagen.encode(v, a, t.width) if t.encoded else v.astype(f"u{t.width}")
    hit = rng.choice(rows, min(bad, rows), replace=False)
    col[hit] ^= np.asarray(1 << 3, dtype=col.dtype)
    pos = rng.integers(0, rows, n).astype(np.uint64)
    if bad < rows:  # one fetch of each corrupt row, and few others
        clean = np.setdiff1d(np.arange(min(rows, 1000)), hit)[0]
        pos[np.isin(pos, hit)] = clean
        pos[rng.choice(n, hit.size, replace=False)] = hit
    pos[rng.choice(n, past, replace=False)] = rows + 7
    with np.errstate(over="ignore"):
        oids = pos * np.uint64(an.A_OID)
    resoid = an.an_meta(an.RESOID, an.A_OID)
    print(f"fetch {t.name} rows={rows} n={n} span={span} bad={bad}", flush=True)
    for reenc, ar in ((0, 0), (1, 13)):
        ref = O.fetchjoin_an(O.Col(oids, resoid), O.Col(col, meta), reenc, ar)
        got = capi.fetchjoin_an(capi.Column.from_numpy(oids, resoid), capi.Column.from_numpy(col, meta), reenc, ar)
        for i, (x, y) in enumerate(zip(got, ref)):
            assert np.array_equal(np.asarray(x).astype(np.uint64), np.asarray(y).astype(np.uint64)), i


RESOID = an.an_meta(an.RESOID, an.A_OID)
KEY = an.an_meta(an.RESINT, 63877)


def flipped(codes, count, rng):
    hit = rng.choice(codes.size, min(count, codes.size), replace=False)
    codes[hit] ^= np.uint64(1) << rng.integers(0, 64, hit.size).astype(np.uint64)
    return codes


def same(got, ref):
    assert len(got) == len(ref)
    for i, (x, y) in enumerate(zip(got, ref)):
        assert np.array_equal(x, np.asarray(y).astype(x.dtype)), i  # (a 4-byte output keeps the low half)


@pytest.mark.parametrize("n,build,step,share,payload,flips", [
    # payload: "v" void, "c" 8-byte codes, "n" plain 2-byte values (no lean shape): probe then build side
    (TILE - 1, 500, 1, 1.0, "vv", 0), (3 * TILE + 1, 20_000, 1, 1.0, "vv", 9), (2 * TILE + 63, 3000, 1, 0.2, "vc", 40),
    (5 * TILE + 7, 3000, 3, 0.5, "vc", 5), (8 * 1024 * 3 + 5, 3000, 1, 0.6, "cv", 5), (40_001, 900, 1, 0.9, "cc", 30),
    (70_003, 900, 5_000_011, 0.3, "cc", 9), (70_003, 5000, 700, 0.02, "vv", 3), (50_000, 800, 1, 0.7, "nc", 3),
    (50_000, 800, 1, 0.7, "nn", 3), (9 * TILE + 2, 260_000, 2, 0.4, "vv", 77), (1, 1, 1, 1.0, "cc", 0),
])
@pytest.mark.parametrize("wide", [False, True])
def test_hash_probe_shapes(n, build, step, share, payload, flips, wide):
    """The probe of unique keys: identity, direct map and hash table, exact and hashed filter."""
    rng = np.random.default_rng(n + build)
    keys = (7 + step * np.arange(build, dtype=np.uint64)) & np.uint64(0xFFFFFFFF)
    if step != 1:
        rng.shuffle(keys)
    fk = np.where(rng.random(n) < share, keys[rng.integers(0, build, n)],
                  (int(keys.max()) + 1 + rng.integers(0, 1000, n)).astype(np.uint64) & np.uint64(0xFFFFFFFF))
    with np.errstate(over="ignore"):
        fk_codes, key_codes = flipped(fk * np.uint64(KEY.a), flips, rng), keys * np.uint64(KEY.a)
        oid = lambda k: flipped(rng.integers(0, 1 << 31, k).astype(np.uint64) * np.uint64(RESOID.a), 2, rng)  # noqa: E731

    def side(kind, k):
        if kind == "v":
            return O.void(k), capi.Column.void(k)
        arr, meta = ((oid(k), RESOID) if kind == "c" else
                     (rng.integers(0, 1 << 16, k).astype(np.uint16), an.plain_meta(an.SHORTINT)))
        return O.Col(arr, meta), capi.Column.from_numpy(arr, meta)
    (oh, gh), (ot, gt) = side(payload[0], n), side(payload[1], build)
    w = 8 if wide else 4
    re = (1, 13) if wide else (0, 0)
    print(f"probe n={n} build={build} step={step} share={share} {payload} w={w}", flush=True)
    ref = O.hashjoin_an(oh, O.Col(fk_codes, KEY), O.Col(key_codes, KEY), ot, 1, *re, w, *re, w)
    for cap in (None, max(1, len(ref[0]) // 2)):
        same(capi.hashjoin_an(gh, capi.Column.from_numpy(fk_codes, KEY), capi.Column.from_numpy(key_codes, KEY), gt, 1,
                              *re, w, *re, w, out_cap=cap), ref)


@pytest.mark.parametrize("head", ["void", "same", "codes", "plain"])
@pytest.mark.parametrize("t", [an.RESTINY, an.RESSHORT, an.RESINT, an.INT])
@pytest.mark.parametrize("n,rows,flips", [(0, 5, 0), (1, 1, 0), (8191, 300, 3), (8193, 40_000, 0), (100_001, 5000, 600),
                                          (5, 0, 0)])
def test_match_positional_shapes(head, t, n, rows, flips):
    rng = np.random.default_rng(n + rows + t.width)
    meta = an.an_meta(t, 233) if t.encoded else an.plain_meta(t)
    v = rng.integers(0, 1 << t.unenc_bits, rows).astype(np.uint64)
    col = datagen.encode(v, 233, t.width) if t.encoded else v.astype(f"u{t.width}")
    if rows > 20:
        col[17] ^= np.asarray(8, dtype=col.dtype)
    with np.errstate(over="ignore"):
        oids = flipped(rng.integers(0, max(1, rows) + 3, n).astype(np.uint64) * np.uint64(RESOID.a), flips, rng)
        other = flipped(rng.integers(0, 1 << 32, n).astype(np.uint64) * np.uint64(KEY.a), flips, rng)
    g_oids, g_col = capi.Column.from_numpy(oids, RESOID), capi.Column.from_numpy(col, meta)
    plain = rng.integers(0, 1 << 16, n).astype(np.uint16)
    oh, gh, wh = {"void": (O.void(n, 3), capi.Column.void(n, 3), 4), "same": (O.Col(oids, RESOID), g_oids, 8),
                  "codes": (O.Col(other, KEY), capi.Column.from_numpy(other, KEY), 8),
                  "plain": (O.Col(plain, an.plain_meta(an.SHORTINT)),
                            capi.Column.from_numpy(plain, an.plain_meta(an.SHORTINT)), 2)}[head]
    for re in (0, 1):
        rh, rt = (re if head in ("same", "codes") else 0), (re if t.encoded else 0)
        args = (rh, 29 if rh else 0, wh, rt, 7 if rt else 0, t.width)
        same(capi.matchjoin_pos_an(gh, g_oids, g_col, *args),
             O.matchjoin_pos_an(oh, O.Col(oids, RESOID), O.Col(col, meta), *args))
