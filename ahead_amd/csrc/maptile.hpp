// maptile.hpp -- the streaming engine of the per-operator kernels that write each row's output at its
// place, or none: check and decode, arithmetic, product sum, the grouped sum, group-id assignment.
//
// The row-tile engine (rowtile.hpp) orders its outputs with a decoupled look-back per 2048-row
// tile; at tens of millions of rows the chain of tile prefixes, not HBM, sets its pace.  This
// engine has no chain.  A persistent grid gives every wave one contiguous range of rows:
//
//  k_map      each wave streams its range (all G rows of a lane evaluated before any wave-wide
//             step, so their loads are in flight together), counts its rows per error stream,
//             records its first kErrList error rows in row order and leaves its accumulator
//             partial (kAcc);
//  k_map_scan one workgroup per stream: exclusive prefixes over the waves of every count, the totals
//             (Op::finish);
//  k_map_fix  per wave: the error positions (from the recorded rows, or by re-evaluating the range
//             when they did not fit).
//
// Op interface: that of rowtile.hpp (kMulti and kMain must be false: outputs that drop rows run on
// the single-pass engine, stream.hpp).
#pragma once

#include <type_traits>

#include "rowtile.hpp"

namespace ahead_dev {

constexpr uint32_t kMapErrList = 16;  // error rows a wave records in row order
constexpr int kMapG = 4;              // rows per lane per iteration (unless the operator sets kMapRows)

struct MapArgs {
    uint64_t rows_per_wave;
    uint32_t waves;
    uint32_t *wcnt;    // [kErr][waves] errors per stream
    uint32_t *wpre;    // same shape: exclusive prefixes over the waves
    uint32_t *werows;  // [waves] rows with any error
    uint64_t *elist;   // [waves][kMapErrList] error bits << 32 | row
    uint64_t *totals;  // [1 + kErr] per error stream from 1 on (k_map_scan; [0], a main stream's, is not written)
};

__device__ __forceinline__ uint32_t map_below(uint64_t ballot) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(ballot >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(ballot), 0u));
}

// An operator may bring a read-only table to LDS (kFilterWords 64-bit words): filter_init copies it
// at the start of k_map and k_map_fix, and eval_f (eval_n with the table) evaluates the rows.
template <class Op, class = void>
struct has_filter : std::false_type {};
template <class Op>
struct has_filter<Op, std::void_t<decltype(Op::kFilterWords)>> : std::true_type {};
template <class Op, bool = has_filter<Op>::value>
struct FilterWords {
    static constexpr int value = 1;
};
template <class Op>
struct FilterWords<Op, true> {
    static constexpr int value = Op::kFilterWords;
};

// Rows per lane and iteration: kMapG, or the operator's kMapRows (an operator whose rows bring
// few bytes keeps more loads in flight with more rows).
template <class Op, class = void>
struct MapG {
    static constexpr int value = kMapG;
};
template <class Op>
struct MapG<Op, std::void_t<decltype(Op::kMapRows)>> {
    static constexpr int value = Op::kMapRows;
};

template <class Op, int G>
__device__ __forceinline__ void map_eval(const Op &op, const uint64_t (&rows)[G], const bool (&live)[G],
                                         typename Op::State (&st)[G], uint32_t (&errs)[G],
                                         uint32_t (&cnt)[G], uint64_t &acc, const uint64_t *filt = nullptr) {
    if constexpr (has_filter<Op>::value) {
        op.template eval_f<G>(rows, live, st, errs, cnt, acc, filt);
    } else if constexpr (has_eval_n<Op>::value) {
        op.template eval_n<G>(rows, live, st, errs, cnt, acc);
    } else {
#pragma unroll
        for (int g = 0; g < G; ++g) {
            cnt[g] = 0;
            errs[g] = 0;
            if (live[g]) cnt[g] = op.eval(rows[g], st[g], errs[g], acc);
        }
    }
}

// An operator may keep per-workgroup accumulators in LDS (kSharedWords 64-bit words):
// shared_init / shared_flush bracket the scan, and eval_shared replaces eval_n.
template <class Op, class = void>
struct has_shared : std::false_type {};
template <class Op>
struct has_shared<Op, std::void_t<decltype(Op::kSharedWords)>> : std::true_type {};
template <class Op, bool = has_shared<Op>::value>
struct SharedWords {
    static constexpr int value = 1;
};
template <class Op>
struct SharedWords<Op, true> {
    static constexpr int value = Op::kSharedWords;
};

// Rows of one wave's range; lane l handles rows seg + g * 64 + l (one coalesced run per g).
template <class Op>
__global__ __launch_bounds__(kBlock) void k_map(Op op, MapArgs m) {
    static_assert(!Op::kMulti && !Op::kMain && Op::kErr > 0, "the map engine takes operators whose ordered outputs are errors");
    constexpr int G = MapG<Op>::value;
    __shared__ unsigned long long s_acc[SharedWords<Op>::value];
    __shared__ uint64_t s_filt[FilterWords<Op>::value];
    if constexpr (has_skip<Op>::value) {
        if (op.skip()) return;
    }
    if constexpr (has_shared<Op>::value) {
        op.shared_init(s_acc);
        __syncthreads();
    }
    if constexpr (has_filter<Op>::value) {
        op.filter_init(s_filt);
        __syncthreads();
    }
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t gw = blockIdx.x * kWaves + (threadIdx.x >> 6);
    const uint64_t begin = static_cast<uint64_t>(gw) * m.rows_per_wave;
    const uint64_t end = begin + m.rows_per_wave < op.n ? begin + m.rows_per_wave : op.n;
    uint32_t err_rows = 0;  // wave-uniform
    uint32_t ecnt[Op::kErr] = {};
    uint64_t acc = 0;
    for (uint64_t seg = begin; seg < end; seg += 64u * G) {
        uint64_t rows[G];
        bool live[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            rows[g] = seg + static_cast<uint64_t>(g) * 64u + lane;
            live[g] = rows[g] < end;
        }
        typename Op::State st[G];
        uint32_t errs[G], cnt[G];
        if constexpr (has_shared<Op>::value) {
            op.template eval_shared<G>(rows, live, st, errs, cnt, acc, s_acc);
        } else {
            map_eval(op, rows, live, st, errs, cnt, acc, s_filt);
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
#pragma unroll
            for (int e = 0; e < Op::kErr; ++e) ecnt[e] += (errs[g] >> e) & 1u;
            const uint64_t x = __ballot(errs[g] != 0u);
            if (x != 0ull) {  // rare: recorded in row order while the list has room
                if (errs[g] != 0u) {
                    const uint32_t i = err_rows + map_below(x);
                    if (i < kMapErrList)
                        m.elist[static_cast<size_t>(gw) * kMapErrList + i] =
                            (static_cast<uint64_t>(errs[g]) << 32) | static_cast<uint32_t>(rows[g]);
                }
                err_rows += static_cast<uint32_t>(__popcll(x));
            }
        }
    }
    if constexpr (has_shared<Op>::value) {
        __syncthreads();
        op.shared_flush(s_acc);
    }
#pragma unroll
    for (int e = 0; e < Op::kErr; ++e) ecnt[e] = wave_sum(ecnt[e]);
    if constexpr (Op::kAcc) {
        const uint64_t t = wave_sum(acc);
        if (lane == 0) op.tile_done(gw, t);
    }
    if (lane == 0) {
#pragma unroll
        for (int e = 0; e < Op::kErr; ++e) m.wcnt[static_cast<size_t>(e) * m.waves + gw] = ecnt[e];
        m.werows[gw] = err_rows;
    }
}

// One workgroup of 1024 threads per error stream: exclusive prefixes over the
// waves and the stream total.
template <class Op>
__global__ __launch_bounds__(1024) void k_map_scan(Op op, MapArgs m) {
    __shared__ uint32_t s_w[16];
    if constexpr (has_skip<Op>::value) {
        if (op.skip()) return;
    }
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    const size_t s = blockIdx.x;
    uint32_t carry = 0;
    for (uint32_t base = 0; base < m.waves; base += 8192u) {
        uint32_t v[8], t = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const uint32_t i = base + threadIdx.x * 8u + q;
            v[q] = i < m.waves ? m.wcnt[s * m.waves + i] : 0u;
            t += v[q];
        }
        const uint32_t inc = wave_incl_scan(t);
        if (lane == 63u) s_w[wv] = inc;
        __syncthreads();
        uint32_t pre = carry, tot = 0;
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            if (w < static_cast<int>(wv)) pre += s_w[w];
            tot += s_w[w];
        }
        __syncthreads();
        pre += inc - t;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const uint32_t i = base + threadIdx.x * 8u + q;
            if (i < m.waves) m.wpre[s * m.waves + i] = pre;
            pre += v[q];
        }
        carry += tot;
    }
    if (threadIdx.x == 0) m.totals[1 + s] = carry;
}

// Error positions.
template <class Op>
__global__ __launch_bounds__(kBlock) void k_map_fix(Op op, MapArgs m) {
    if constexpr (has_skip<Op>::value) {
        if (op.skip()) return;
    }
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t gw = blockIdx.x * kWaves + (threadIdx.x >> 6);
    if (gw >= m.waves) return;
    const uint64_t begin = static_cast<uint64_t>(gw) * m.rows_per_wave;
    const uint64_t end = begin + m.rows_per_wave < op.n ? begin + m.rows_per_wave : op.n;
    if (gw == 0 && lane == 0) op.finish(m.totals);

    // error positions
    const uint32_t nrows = m.werows[gw];
    if (nrows != 0u) {
        uint64_t idx[Op::kErr];
#pragma unroll
        for (int e = 0; e < Op::kErr; ++e) idx[e] = m.wpre[static_cast<size_t>(e) * m.waves + gw];
        const bool listed = nrows <= kMapErrList;
        const uint64_t span = listed ? nrows : end - begin;
        for (uint64_t j0 = 0; j0 < span; j0 += 64u) {
            const uint64_t j = j0 + lane;
            uint32_t errs = 0;
            uint64_t row = 0, acc = 0;
            typename Op::State st{};
            if (j < span) {
                if (listed) {
                    const uint64_t ent = m.elist[static_cast<size_t>(gw) * kMapErrList + j];
                    row = static_cast<uint32_t>(ent);
                    (void)op.eval(row, st, errs, acc);  // the row's state for emit_err
                } else {
                    row = begin + j;
                    (void)op.eval(row, st, errs, acc);
                }
            }
#pragma unroll
            for (int e = 0; e < Op::kErr; ++e) {
                const bool on = (errs >> e) & 1u;
                const uint64_t b = __ballot(on);
                if (on) op.emit_err(e, row, st, idx[e] + map_below(b));
                idx[e] += static_cast<uint64_t>(__popcll(b));
            }
        }
    }
}

}  // namespace ahead_dev

namespace ahead_host {

// Persistent grid of the map engine: as many workgroups as can be resident (registers decide),
// at most one wave per 64 rows.
template <class Op>
uint32_t map_grid(uint64_t n) {
    static uint32_t resident = 0;
    if (resident == 0) {
        int dev = 0, cus = 0, per_cu = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0)
            cus = 256;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu, reinterpret_cast<const void *>(ahead_dev::k_map<Op>), ahead_dev::kBlock, 0) != hipSuccess ||
            per_cu <= 0)
            per_cu = 2;
        resident = static_cast<uint32_t>(cus) * static_cast<uint32_t>(per_cu);
    }
    const uint64_t by_rows = (n + 64u * ahead_dev::kWaves - 1) / (64u * ahead_dev::kWaves);
    const uint64_t g = by_rows < resident ? by_rows : resident;
    return static_cast<uint32_t>(g == 0 ? 1 : g);
}

// Workspace bytes of the map engine's per-wave tables for n rows.
template <class Op>
size_t map_scratch_bytes(uint64_t n) {
    using namespace ahead_dev;
    constexpr int NS = Op::kErr;
    const size_t waves = static_cast<size_t>(map_grid<Op>(n)) * kWaves;
    return 2 * align_up(NS * waves * 4, 256) + align_up(waves * 4, 256) + align_up(waves * kMapErrList * 8, 256) + 256;
}

// Rows of a wave's range for n rows: whole steps.
template <class Op>
uint64_t map_rows_per_wave(uint64_t n) {
    using namespace ahead_dev;
    const uint64_t waves = static_cast<uint64_t>(map_grid<Op>(n)) * kWaves;
    constexpr uint64_t step = 64u * MapG<Op>::value;
    return ((n + waves - 1) / waves + step - 1) / step * step;
}

// Workgroups of the map engine's grid that have rows: the first ones.
template <class Op>
uint32_t map_parts(uint64_t n) {
    const uint64_t rows = map_rows_per_wave<Op>(n) * ahead_dev::kWaves;
    return n == 0 ? 1u : static_cast<uint32_t>((n + rows - 1) / rows);
}

// Launches the map engine for op over op.n rows.  Scratch: per-wave tables in the workspace region
// at `offset`.  A caller that keeps regions of its own before `offset` must have grown the
// workspace to offset + map_scratch_bytes<Op>(n) beforehand (growing moves the workspace).
template <class Op>
int launch_map(const Op &op, ahead_hip_ws *ws, size_t offset, hipStream_t s) {
    using namespace ahead_dev;
    constexpr int NS = Op::kErr;
    const uint32_t grid = map_grid<Op>(op.n);
    const uint32_t waves = grid * kWaves;
    const size_t o_cnt = offset, o_pre = o_cnt + align_up(static_cast<size_t>(NS) * waves * 4, 256),
                 o_erows = o_pre + align_up(static_cast<size_t>(NS) * waves * 4, 256),
                 o_elist = o_erows + align_up(static_cast<size_t>(waves) * 4, 256),
                 o_totals = o_elist + align_up(static_cast<size_t>(waves) * kMapErrList * 8, 256),
                 o_end = o_totals + 256;
    int st;
    if (offset > 0 && ws->bytes < kHeaderBytes + o_end)
        return fail(AHEAD_ERR_INVALID, "map engine: the workspace was not grown before its regions were placed");
    if ((st = ws_ensure(ws, o_end)) != AHEAD_OK) return st;
    MapArgs m{};
    m.rows_per_wave = map_rows_per_wave<Op>(op.n);
    m.waves = waves;
    m.wcnt = reinterpret_cast<uint32_t *>(ws_region(ws, o_cnt));
    m.wpre = reinterpret_cast<uint32_t *>(ws_region(ws, o_pre));
    m.werows = reinterpret_cast<uint32_t *>(ws_region(ws, o_erows));
    m.elist = reinterpret_cast<uint64_t *>(ws_region(ws, o_elist));
    m.totals = reinterpret_cast<uint64_t *>(ws_region(ws, o_totals));
    static_assert(8 * (1 + NS) <= 256, "totals fit their block");
    hipLaunchKernelGGL(k_map<Op>, dim3(grid), dim3(kBlock), 0, s, op, m);
    hipLaunchKernelGGL(k_map_scan<Op>, dim3(NS), dim3(1024), 0, s, op, m);
    hipLaunchKernelGGL(k_map_fix<Op>, dim3(grid), dim3(kBlock), 0, s, op, m);
    AHEAD_HIP_TRY(hipGetLastError());
    return AHEAD_OK;
}

// Waves of the map engine's grid for n rows (callers size per-wave partial tables with it).
template <class Op>
uint32_t map_waves(uint64_t n) {
    return map_grid<Op>(n) * ahead_dev::kWaves;
}

}  // namespace ahead_host
