"""The operators' kernels on the CPU stand-in (tests/cpp/lockstep), whose waves progress as unevenly as the
barriers allow: what a missing barrier would only rarely show on the card fails here every time."""
import ctypes

import numpy as np
import pytest

import lockstep_lib as L
import oracle_lib as O
from ahead_amd import an, capi, datagen

pytestmark = pytest.mark.skipif(not L.available(), reason="no clang++ of ROCm to compile the kernels for the CPU")


CUS = 256  # of device 0; device 1 has 4


@pytest.fixture(params=[0, 1], ids=["ascending", "descending"])
def waves(request):
    lib = L.lib()
    lib.lockstep_set(request.param, 0, 0)
    yield request.param
    lib.lockstep_set(0, 0, 0)


@pytest.mark.parametrize("n,bad", [(5, 1), (16 * 1024 * 2 + 77, 3)])
def test_single_pass_engine_under_uneven_waves(waves, n, bad):
    """A workgroup's waves agree on every tile they take, the first one included."""
    rng = np.random.default_rng(n)
    meta = an.an_meta(an.RESINT, 65117)
    codes = datagen.encode(rng.integers(0, 1 << 32, n).astype(np.uint64), meta.a, 8)
    codes[rng.choice(n, bad, replace=False)] ^= np.uint64(1 << 40)
    ref = O.check_and_decode_an(O.Col(codes, meta))
    dec, err, cnt = np.zeros(n, np.uint32), np.zeros(bad, np.uint64), np.full(2, 77, np.uint64)
    ws, col = L.Workspace(), L.column(codes, meta)
    for _ in range(2):
        L.check(L.lib().ahead_hip_check_and_decode_an(ctypes.byref(col), an.A_OID_ERR, dec.ctypes.data, n,
                                                      err.ctypes.data, bad, cnt.ctypes.data, ws.h, None))
        assert cnt.tolist() == [n - bad, bad]
        assert np.array_equal(dec[:n - bad], ref[0]) and np.array_equal(err, ref[1])
        cnt[:] = 77



@pytest.fixture
def recorded():
    """Launches are recorded, not run."""
    lib = L.lib()
    lib.lockstep_set(0, 1, 0)
    L.launches()
    yield lib
    lib.lockstep_set(0, 0, 0)


def _somewhere(n, meta, **kw):
    return L.column(None, meta, n, data=4096 if n else None, **kw)


RESOID = an.an_meta(an.RESOID, an.A_OID)


def _calls(n, ws):
    """One call of n rows per operator of the single-pass engine: (name, rows of its streamed input, call)."""
    lib, ref, b = L.lib(), ctypes.byref, capi.Buf(4096, n)
    key, void = an.an_meta(an.RESINT, 65117), L.column(None, an.plain_meta(an.VOID), n)
    oid, short = _somewhere(n, RESOID), _somewhere(n, an.an_meta(an.RESSHORT, 233))
    out = []
    for t, a in ((an.RESTINY, 233), (an.RESSHORT, 233), (an.RESINT, 65117)):
        d = _somewhere(n, an.an_meta(t, a))
        out.append((f"decode {t.name}", lambda d=d: lib.ahead_hip_check_and_decode_an(
            ref(d), 1, 4096, n, 4096, n, 4096, ws.h, None)))
    out.append(("fetch", lambda: lib.ahead_hip_fetchjoin_an(ref(oid), ref(short), 0, 0, 1, b, b, b, 4096, ws.h, None)))
    out.append(("match", lambda: lib.ahead_hip_matchjoin_pos_an(
        ref(void), ref(oid), ref(short), 0, 0, 4, 0, 0, 4, 1, b, b, b, b, b, 4096, ws.h, None)))
    fk, bk, bv = _somewhere(n, key), _somewhere(500, key), L.column(None, an.plain_meta(an.VOID), 500)
    out.append(("probe", lambda: lib.ahead_hip_hashjoin_an(
        ref(void), ref(fk), ref(bk), ref(bv), 1, 0, 0, 4, 0, 0, 4, 1, *[b] * 6, 4096, ws.h, None)))
    out.append(("merge", lambda: lib.ahead_hip_matchjoin_merge_an(
        ref(oid), ref(oid), ref(oid), ref(oid), 0, 0, 8, 0, 0, 8, 1, *[b] * 6, 4096, ws.h, None)))
    return out


@pytest.mark.parametrize("n", [1, 4096, 4097, 20_000, 100_000, 500_000, 786_431, 786_433, 1_000_000, 2_000_000, 4_000_000,
                               6_291_455, 6_291_456, 12_582_911, 12_582_912, 60_000_000])
def test_single_pass_engine_spreads_a_call_over_the_card(recorded, n):
    """Every workgroup a call of n rows can fill with 4 rows a lane runs, up to three eighths of the CUs; from
    three eighths of the CUs x 8 rows a lane on, no fewer."""
    ws = L.Workspace()
    for name, call in _calls(n, ws):
        L.launches()
        L.check(call())
        grids = [x.grid for x in L.launches() if x.kernel.startswith("k_stream")]
        assert grids, name
        for g in grids:
            assert min(-(-n // 4096), CUS * 3 // 8) <= g <= CUS, (name, n, g)
            if n >= 60_000_000:
                assert g == CUS


def _merge(t1, h2, ws):
    """The pairs and counts of a merge of two OID lists against themselves, and the launches it made."""
    cap = max(1, min(t1.size, h2.size))
    oh, ot, cnt = np.zeros(cap, np.uint64), np.zeros(cap, np.uint64), np.zeros(5, np.uint64)
    errs = [np.zeros(4 * (t1.size + h2.size), np.uint64) for _ in range(4)]
    d1, d2 = L.column(t1, RESOID), L.column(h2, RESOID)
    L.launches()
    L.check(L.lib().ahead_hip_matchjoin_merge_an(
        *[ctypes.byref(x) for x in (d1, d1, d2, d2)], 0, 0, 8, 0, 0, 8, an.A_OID_ERR, L.buf(oh), L.buf(ot),
        *[L.buf(e) for e in errs], cnt.ctypes.data, ws.h, None))
    k = cnt.tolist()
    got = [oh[:k[0]], ot[:k[0]], *[e[:c] for e, c in zip(errs, k[1:])]]
    ref = O.matchjoin_merge_an(O.Col(t1, RESOID), O.Col(t1, RESOID), O.Col(h2, RESOID), O.Col(h2, RESOID))
    for i, (x, y) in enumerate(zip(got, ref)):
        assert np.array_equal(x, y), i
    return L.launches()


def test_merge_stops_when_list_1_fails_a_check():
    """The pass over list 1 ends soon after a row fails; the walk that writes the outputs is not its concern."""
    n = 60_000
    L.lib().lockstep_set(0, 0, 0)
    ws, keys = L.Workspace(), np.arange(n, dtype=np.uint64) * np.uint64(3)
    lists = keys * np.uint64(an.A_OID), keys[::2] * np.uint64(an.A_OID)
    steps = []
    for bad in (False, True):
        t1 = lists[0].copy()
        if bad:
            t1[700] = t1[699] - np.uint64(an.A_OID)
        steps.append(sum(x.steps for x in _merge(t1, lists[1], ws) if "k_stream" in x.kernel))
    assert steps[1] * 3 < steps[0]


def _sums(n, groups, ws, run=True):
    rng = np.random.default_rng(n + groups)
    meas = an.an_meta(an.RESINT, 65117)
    gi = rng.integers(0, groups, n).astype(np.uint64)
    t = datagen.encode(rng.integers(0, 1 << 32, n).astype(np.uint64), meas.a, 8)
    g = gi * np.uint64(an.A_OID)
    if n > 100:
        t[[3, 70]] ^= np.uint64(1 << 35)
        g[[5, n - 1]] = np.uint64(groups) * np.uint64(an.A_OID)
    sums, cnt, errs = np.full(groups, 77, np.uint64), np.zeros(4, np.uint64), [np.zeros(8, np.uint64) for _ in range(3)]
    void = L.column(None, an.plain_meta(an.VOID), n)
    ct, cg = L.column(t, meas), L.column(g, RESOID)
    L.check(L.lib().ahead_hip_aggregate_sum_grouped_an(
        ctypes.byref(void), ctypes.byref(ct), ctypes.byref(cg), groups, an.A_RESULT, an.A_OID, sums.ctypes.data,
        *[L.buf(e) for e in errs], cnt.ctypes.data, ws.h, None))
    if run:
        ref = O.aggregate_sum_grouped_an(O.void(n), O.Col(t, meas), O.Col(g, RESOID), groups)
        got = [sums, *[e[:int(c)] for e, c in zip(errs, cnt[1:])]]
        for i, (x, y) in enumerate(zip(got, ref)):
            assert np.array_equal(x, y), i


@pytest.mark.parametrize("n,groups", [(0, 7), (1, 1), (2047, 3), (2049, 5), (4097, 4096), (6000, 4097), (5000, 130)])
def test_grouped_sum_partials(n, groups):
    """Workgroups without rows leave no partials, and none of another call's are summed."""
    L.lib().lockstep_set(0, 0, 0)
    ws = L.Workspace()
    _sums(9000, min(groups, 4096), ws, run=False)
    _sums(n, groups, ws)


def test_grouped_sum_partials_follow_the_rows(recorded):
    n, groups = 250_000, 4096
    ws = L.Workspace()
    _sums(n, groups, ws, run=False)
    assert ws.bytes() < 2 * 8 * groups * (n // 2048 + 1) + (4 << 20)


def test_every_device_has_its_own_launch_geometry(recorded):
    """The LDS attribute and the CUs are the current device's, not those of the first one used."""
    n = 4_000_000
    for device, cus, first in ((0, CUS, True), (1, 4, True), (0, CUS, False)):
        recorded.lockstep_set(0, 1, device)
        ws, oid, col = L.Workspace(device), _somewhere(n, RESOID), _somewhere(5000, an.an_meta(an.RESINT, 65117))
        b = capi.Buf(4096, n)
        L.launches()
        L.check(recorded.ahead_hip_fetchjoin_an(ctypes.byref(oid), ctypes.byref(col), 0, 0, 1, b, b, b, 4096, ws.h, None))
        log = L.launches()
        assert [x.grid for x in log if x.kernel == "attribute"] == [device] * first
        assert [x.grid for x in log if x.kernel.startswith("k_stream")] == [cus]


def _group(codes, meta, ws, groups):
    n = codes.size
    out, first, cnt = np.zeros(n, np.uint64), np.zeros(groups, np.uint64), np.zeros(6, np.uint64)
    errs = [np.zeros(4, np.uint64) for _ in range(2)]
    void, col = L.column(None, an.plain_meta(an.VOID), n), L.column(codes, meta)
    L.launches()
    L.check(L.lib().ahead_hip_groupby_an(ctypes.byref(void), ctypes.byref(col), an.A_OID, 0, out.ctypes.data, L.buf(first),
                                         *[L.buf(e) for e in errs], cnt.ctypes.data, ws.h, None))
    ref = O.groupby_an(O.void(n), O.Col(codes, meta))
    assert cnt.tolist() == [n, ref[1].size, 0, 0, 0, 0]
    assert np.array_equal(out, ref[0]) and np.array_equal(first[:ref[1].size], ref[1])
    return [x for x in L.launches() if x.kernel.startswith("k_grp_first_set")]


def test_group_keys_in_order_are_inserted_once_per_lane():
    """A workgroup whose set is full inserts a key of a lane's eight rows once, not for every row."""
    meta = an.an_meta(an.RESINT, 65117)
    L.lib().lockstep_set(0, 0, 1)  # few workgroups, so that each meets more keys than its set takes
    ws = L.Workspace(1)
    n = 16 * 8192
    keys = (np.arange(n, dtype=np.uint64) // np.uint64(8)) * np.uint64(7) + np.uint64(1 << 20)
    (run,) = _group(keys * np.uint64(meta.a), meta, ws, n)
    assert n // run.grid > 8 * 1792  # more keys than the set's 1536
    assert run.swaps < 3 * (n // 8), run
    L.lib().lockstep_set(0, 0, 0)


@pytest.mark.parametrize("n", [100_000, 500_000, 2_000_000])
def test_first_sightings_spread_over_the_card(recorded, n):
    ws, void = L.Workspace(), L.column(None, an.plain_meta(an.VOID), n)
    col, b = _somewhere(n, an.an_meta(an.RESINT, 65117)), capi.Buf(4096, n)
    L.launches()
    L.check(recorded.ahead_hip_groupby_an(ctypes.byref(void), ctypes.byref(col), an.A_OID, 0, 4096, b, b, b, 4096, ws.h, None))
    (run,) = [x for x in L.launches() if x.kernel.startswith("k_grp_first_set")]
    assert run.grid >= min(2 * CUS, n // 2048) // 2


def test_reserve_sets_the_ticketed_state_apart_once():
    """A reservation sizes the scratch and the look-back state; the ticketed state is never needed beyond 32 MiB."""
    L.lib().lockstep_set(0, 0, 0)
    ws, size = L.Workspace(), 160 << 20
    L.check(L.lib().ahead_hip_ws_reserve(ws.h, size))
    assert 2 * size + (32 << 20) <= ws.bytes() < 2 * size + (33 << 20)
    small = L.Workspace()
    L.check(L.lib().ahead_hip_ws_reserve(small.h, 5 << 20))
    assert small.bytes() >= 3 * (5 << 20)
