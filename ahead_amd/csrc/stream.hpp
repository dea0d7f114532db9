// stream.hpp -- the single-pass engine of the operators that emit at most one entry per row into an
// ordered main output: check-and-decode, fetch, positional match, hash probe of unique keys.
//
// A persistent grid (one workgroup of 1024 threads per CU) takes tiles of 1024 x G rows in ticket
// order (G: the operator's kG, or fewer for smaller calls, see launch_stream).  Per tile, every lane evaluates its G rows, the tile publishes how many rows it keeps and
// reports, takes its place among all tiles from its predecessors' counts, and writes every entry
// once, at its final place.  Nothing is staged, moved or re-read: the traffic is the inputs once
// and the outputs once, whether rows are dropped or not.
//
// Bound by HBM as far as three latencies stay off the path (60M 8-byte codes checked and decoded
// to 4 bytes, 720 MB, on one MI355X; the same loads and stores without any order take 103 us):
//  - the place of a tile: a look-back that walks 64 predecessors at a time advances 128 tiles per
//    device-scope round trip, and a round trip takes several microseconds while HBM is saturated
//    (206 us).  Here one round reads the counts of all kStreamWindow predecessors, one per thread,
//    and the inclusive prefix just before them; with one workgroup per CU that prefix belongs to a
//    tile of an earlier generation and is there (170 us).  Windows of 256, 512 and 1024 tiles
//    measured alike; 512 covers two tickets per CU.
//  - the next tile's loads go out between this tile's publication and its polls (128 us).  Half of them
//    behind the polls took 150 us.  Earlier is
//    worse: a count published behind loads in flight reaches the other workgroups after them (loads
//    issued before the publication 172 us; a wave of its own for the places, with the other fifteen
//    always loading, 209 us).
//  - tickets come from one address, about 15 ns each: 7325 tiles of 8192 rows take 190 us, 3663 of
//    16384 rows 128 us.
//
// The tickets and the epoch of the status words are one 64-bit word in device memory (epoch in the
// high half, ticket in the low): one atomic hands out both, and the workgroup that takes the
// launch's last ticket (every workgroup takes one past the end) starts the next epoch.  A launch
// needs nothing from the host and can be captured in a graph and replayed.  Every ticket's holder
// is running, and a tile waits for lower tickets only, so the chain always drains.
//
// Op interface (beside eval / emit_err / finish of rowtile.hpp, which the rare error rows use):
//   static constexpr int kErr, kG;      // error streams; rows per lane, at most (even, up to 32)
//   struct Raw; using State;            // a row's streamed inputs; what its entry needs
//   uint64_t out_cap;                   // entries the outputs hold
//   struct Uniform; Uniform begin(const char *lds) const;      // read once per workgroup, after init
//   void load(uint64_t first, uint32_t k, Raw &) const;        // row first + k; or, with kLoadN, H rows at once:
//   template <int H> void load_n(uint64_t first, const uint32_t (&k)[H], Raw (&)[H]) const;
//   template <int G> void open_tile(const char *lds, const Uniform &, uint64_t first, uint32_t lane,
//            uint32_t live, const Raw (&)[G], Mid<G> &) const;
//       // rows first + 64 g + lane: decodes them and issues their lookups (bit g of live: the row
//       // exists; one past the end has the last row's inputs)
//   template <int G> void close_tile(const Uniform &, const Mid<G> &, uint32_t live, State (&)[G],
//            uint32_t &keep, uint32_t (&err)[kErr]) const;
//       // sets bit g of keep / err[e] for live rows that emit an entry / report into stream e
//   void emit(const Uniform &, const State &, uint64_t first, uint64_t pos, uint32_t row, uint32_t k) const;
//       // entry pos + k, of row first + row (first and pos are wave-uniform: scalar bases)
//   void report(uint64_t row, State &, uint32_t &errs) const;  // the error streams of one row
//   static constexpr uint32_t kPack;    // (optional) a wave that drops rows and keeps at most kPack packs
//                                       // its entries in LDS and emits them 64 at a time
//   void init(char *lds) const;         // all threads, before the first tile; a barrier follows
//   bool skip() const;                  // the whole launch stands down (from device state that no
//                                       // workgroup of this launch changes)
//   bool failed(const char *lds) const; // (optional) one thread, for a tile that reports: true if nothing that this
//                                       // launch writes will be used; the tiles still to come are then counted as empty
#pragma once

#include "rowtile.hpp"

namespace ahead_dev {

constexpr int kStreamThreads = 1024;
constexpr int kStreamWaves = kStreamThreads / 64;
constexpr uint32_t kStreamWindow = 512;

struct StreamArgs {
    unsigned long long *te;  // epoch << 32 | ticket
    WsHeader *hdr;           // fail flag
    uint64_t *agg;           // [tiles] epoch << 34 | reports << 33 | kept
    uint64_t *incl;          // [1 + kErr][tiles] epoch << 34 | inclusive count
    uint64_t *erep;          // [kErr][tiles] epoch << 34 | rows reported (tiles with reports only)
    uint32_t tiles;
    uint32_t last;           // the launch's last ticket: tiles + workgroups - 1
};

__device__ __forceinline__ uint32_t uniform(uint32_t x) { return __builtin_amdgcn_readfirstlane(x); }

// What a failed launch's ticket words carry above the ticket (at most 2^21 tiles and workgroups).
constexpr uint32_t kStreamFailed = 1u << 31;

// A ticket word's tile, and kStreamFailed; the holder of the launch's last ticket starts the next epoch.
__device__ __forceinline__ uint32_t stream_tile(const StreamArgs &m, unsigned long long v) {
    const uint32_t t = static_cast<uint32_t>(v);
    if ((t & ~kStreamFailed) == m.last)
        __hip_atomic_store(m.te, ((v >> 32) + 1ull) << 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return t;
}

__device__ __forceinline__ uint64_t stream_word(uint32_t epoch, uint64_t v) {
    return (static_cast<uint64_t>(epoch) << 34) | v;
}
// A status word of this launch (polled until its tile has published it; the spin is bounded).
__device__ __forceinline__ uint64_t stream_poll(const StreamArgs &m, const uint64_t *w, uint32_t epoch) {
    uint64_t v = lb_load(w);
    uint32_t spins = 0;
    while (static_cast<uint32_t>(v >> 34) != epoch) {
        if (++spins >= kSpinLimit) {
            atomicOr(&m.hdr->fail, 1u);
            return 0;
        }
        __builtin_amdgcn_s_sleep(1);
        v = lb_load(w);
    }
    return v;
}

__device__ __forceinline__ uint32_t wave_rank(uint64_t ballot) {
    return __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(ballot >> 32),
                                     __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(ballot), 0u));
}

template <class Op, class = void>
struct loads_halves : std::false_type {};
template <class Op>
struct loads_halves<Op, std::void_t<decltype(Op::kLoadN)>> : std::true_type {};

// The streamed inputs of a lane's G rows first + 64 g + lane, of which the wave has `left`; rows past
// the end repeat the last one (a wave past the end: row 0).
template <class Op, int H>
__device__ __forceinline__ void stream_load(const Op &op, uint64_t first, uint32_t lane, uint32_t left, int half,
                                            typename Op::Raw (&raw)[H]) {
    const uint64_t base = left != 0u ? first : 0ull;
    const uint32_t top = left != 0u ? left - 1u : 0u;
    uint32_t k[H];
#pragma unroll
    for (int g = 0; g < H; ++g) {
        k[g] = static_cast<uint32_t>((half * H + g) * 64) + lane;
        k[g] = k[g] < top ? k[g] : top;
    }
    if constexpr (loads_halves<Op>::value) {
        op.template load_n<H>(base, k, raw);
    } else {
#pragma unroll
        for (int g = 0; g < H; ++g) op.load(base, k[g], raw[g]);
    }
}

template <class Op, class = void>
struct can_fail : std::false_type {};
template <class Op>
struct can_fail<Op, std::void_t<decltype(std::declval<const Op &>().failed(nullptr))>> : std::true_type {};

// The workgroup's tiles from `tile` on, published as empty, so that no other one waits for them (thread 0).
template <int NS>
__device__ __forceinline__ void stream_drain(const StreamArgs &m, uint32_t epoch, uint32_t tile) {
    while (tile < m.tiles) {
        lb_store(&m.agg[tile], stream_word(epoch, 0));
#pragma unroll
        for (int s = 0; s < NS; ++s) lb_store(&m.incl[static_cast<size_t>(s) * m.tiles + tile], stream_word(epoch, 0));
        tile = stream_tile(m, atomicAdd(m.te, 1ull)) & ~kStreamFailed;
    }
}

template <class Op, int G, class = void>
struct pack_rows : std::integral_constant<uint32_t, 0> {};
template <class Op, int G>
struct pack_rows<Op, G, std::enable_if_t<(Op::kPack > 0)>>
    : std::integral_constant<uint32_t, (Op::kPack < 64u * G ? Op::kPack : 64u * G)> {};
template <class Op, int G>
struct StreamPack {  // a wave's packed entries
    static constexpr uint32_t kRows = pack_rows<Op, G>::value ? pack_rows<Op, G>::value : 1u;
    typename Op::State st[kRows];
    uint16_t row[kRows];
};
template <class Op, int G>
constexpr size_t stream_pack_bytes() {
    return pack_rows<Op, G>::value ? sizeof(StreamPack<Op, G>) * kStreamWaves : 0;
}

template <class Op, int G>
__global__ __launch_bounds__(kStreamThreads) void k_stream(Op op, StreamArgs m) {
    constexpr int NS = 1 + Op::kErr, NW = kStreamWaves;
    constexpr uint32_t kWaveRows = 64u * G, kAll = G == 32 ? 0xFFFFFFFFu : (1u << (G & 31)) - 1u;
    extern __shared__ __align__(16) char s_op[];
    __shared__ uint32_t s_cnt[NS][NW], s_sum[NS][NW];
    // (the first tile has a word of its own: thread 0 stores the second one before the next barrier, when
    // other waves may still have to read the first)
    __shared__ uint32_t s_begin, s_tile, s_epoch;
    constexpr uint32_t kPack = pack_rows<Op, G>::value;
    __shared__ StreamPack<Op, G> s_pack[kPack ? NW : 1];
    if (op.skip()) return;
    if (threadIdx.x == 0) {
        const unsigned long long v = atomicAdd(m.te, 1ull);
        s_begin = stream_tile(m, v);
        s_epoch = static_cast<uint32_t>(v >> 32) % ((1u << 30) - 1u) + 1u;
    }
    op.init(s_op);
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = uniform(threadIdx.x >> 6);
    const uint32_t epoch = uniform(s_epoch);
    uint32_t tile = uniform(s_begin);
    if constexpr (can_fail<Op>::value) {
        if ((tile & kStreamFailed) != 0u) {
            if (threadIdx.x == 0) stream_drain<NS>(m, epoch, tile & ~kStreamFailed);
            return;
        }
    }
    auto first_of = [&](uint32_t t) { return (static_cast<uint64_t>(t) * NW + wave) * kWaveRows; };
    auto left_of = [&](uint32_t t) {
        const uint64_t first = first_of(t);
        return first >= op.n ? 0u : op.n - first < kWaveRows ? static_cast<uint32_t>(op.n - first) : kWaveRows;
    };
    constexpr int H = G / 2;
    typename Op::Raw raw0[H], raw1[H];
    const typename Op::Uniform uni = op.begin(s_op);
    if (tile < m.tiles && op.n != 0) {
        stream_load<Op, H>(op, first_of(tile), lane, left_of(tile), 0, raw0);
        stream_load<Op, H>(op, first_of(tile), lane, left_of(tile), 1, raw1);
    }
    while (tile < m.tiles) {
        unsigned long long ticket;  // the next tile's, taken by thread 0 while the inputs arrive
        if (threadIdx.x == 0) ticket = atomicAdd(m.te, 1ull);
        const uint64_t first = first_of(tile);
        const uint32_t left = left_of(tile);
        typename Op::State st0[H], st1[H];
        uint32_t keep = 0, err[Op::kErr] = {};
        if (left != 0u) {  // (a wave past the last row has nothing to look up: its columns may be empty)
            uint32_t live = kAll;  // rows of the lane that exist
            if (left != kWaveRows) {
                live = 0;
#pragma unroll
                for (int g = 0; g < G; ++g) live |= (static_cast<uint32_t>(g * 64) + lane < left ? 1u : 0u) << g;
            }
            auto half = [&](int h, const typename Op::Raw (&raw)[H], typename Op::State (&st)[H]) {
                constexpr uint32_t kHalf = (1u << H) - 1u;
                const uint32_t on = (live >> (h * H)) & kHalf;
                typename Op::template Mid<H> mid;
                uint32_t kp = 0, er[Op::kErr] = {};
                op.template open_tile<H>(s_op, uni, first + static_cast<uint32_t>(h * H * 64), lane, on, raw, mid);
                op.template close_tile<H>(uni, mid, on, st, kp, er);
                keep |= kp << (h * H);
#pragma unroll
                for (int e = 0; e < Op::kErr; ++e) err[e] |= er[e] << (h * H);
            };
            half(0, raw0, st0);
            half(1, raw1, st1);
        }

        // what the wave keeps and reports
        const bool whole = __ballot(keep == kAll) == ~0ull;
        const uint32_t kept = whole ? kWaveRows : wave_sum(static_cast<uint32_t>(__popc(keep)));
        uint32_t any = 0;
#pragma unroll
        for (int e = 0; e < Op::kErr; ++e) any |= err[e];
        const bool reports = __ballot(any != 0u) != 0ull;
        uint32_t ecnt[Op::kErr] = {};
        if (reports) {
#pragma unroll
            for (int e = 0; e < Op::kErr; ++e) ecnt[e] = wave_sum(static_cast<uint32_t>(__popc(err[e])));
        }
        if (lane == 0) {
            s_cnt[0][wave] = kept;
#pragma unroll
            for (int e = 0; e < Op::kErr; ++e) s_cnt[1 + e][wave] = ecnt[e];
        }
        if (threadIdx.x == 0) s_tile = stream_tile(m, ticket);
        __syncthreads();
        uint32_t agg[NS], before[NS], rep = 0;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            // (every lane reads every count: independent LDS reads, where a scan over lanes is a chain of
            // twelve shuffles and cost 10 us)
            agg[s] = 0;
            before[s] = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) {
                const uint32_t c = s_cnt[s][w];
                if (w < static_cast<int>(wave)) before[s] += c;
                agg[s] += c;
            }
            agg[s] = uniform(agg[s]);
            before[s] = uniform(before[s]);
            if (s) rep |= agg[s];
        }
        if (threadIdx.x == 0) {
            if (rep != 0u) {
#pragma unroll
                for (int e = 0; e < Op::kErr; ++e)
                    lb_store(&m.erep[static_cast<size_t>(e) * m.tiles + tile], stream_word(epoch, agg[1 + e]));
            }
            lb_store(&m.agg[tile], stream_word(epoch, (rep != 0u ? 1ull << 33 : 0ull) | agg[0]));
        }
        const uint32_t drawn = uniform(s_tile), next = can_fail<Op>::value ? drawn & ~kStreamFailed : drawn;
        if constexpr (can_fail<Op>::value) {
            // (before the workgroup's last ticket, and so before the next launch's first one)
            if (rep != 0u && threadIdx.x == 0 && op.failed(s_op) && next < m.tiles)
                atomicOr(m.te, static_cast<unsigned long long>(kStreamFailed));
        }
        if (next < m.tiles) {
            stream_load<Op, H>(op, first_of(next), lane, left_of(next), 0, raw0);
            stream_load<Op, H>(op, first_of(next), lane, left_of(next), 1, raw1);
        }

        // the counts of the kStreamWindow - 1 tiles before this one, and the prefix before them
        uint32_t sum[NS] = {};
        const uint32_t back = threadIdx.x + 1u;
        if (back < kStreamWindow && back <= tile) {
            const uint64_t v = stream_poll(m, &m.agg[tile - back], epoch);
            sum[0] = static_cast<uint32_t>(v);
            if ((v >> 33) & 1ull) {
#pragma unroll
                for (int e = 0; e < Op::kErr; ++e)
                    sum[1 + e] = static_cast<uint32_t>(
                        stream_poll(m, &m.erep[static_cast<size_t>(e) * m.tiles + tile - back], epoch));
            }
        }
        if (wave == NW - 1 && tile >= kStreamWindow && lane < static_cast<uint32_t>(NS)) {
            const uint32_t v = static_cast<uint32_t>(
                stream_poll(m, &m.incl[static_cast<size_t>(lane) * m.tiles + tile - kStreamWindow], epoch));
#pragma unroll
            for (int s = 0; s < NS; ++s) sum[s] += lane == static_cast<uint32_t>(s) ? v : 0u;
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const uint32_t t = __ballot(sum[s] != 0u) != 0ull ? wave_sum(sum[s]) : 0u;
            if (lane == 0) s_sum[s][wave] = t;
        }
        __syncthreads();
        uint32_t excl[NS];
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            excl[s] = 0;
#pragma unroll
            for (int w = 0; w < NW; ++w) excl[s] += s_sum[s][w];
            excl[s] = uniform(excl[s]);
            if (threadIdx.x == static_cast<uint32_t>(s))
                lb_store(&m.incl[static_cast<size_t>(s) * m.tiles + tile], stream_word(epoch, excl[s] + agg[s]));
        }

        const uint64_t pos = static_cast<uint64_t>(excl[0]) + before[0];
        const uint32_t room = pos >= op.out_cap                   ? 0u
                              : op.out_cap - pos < kWaveRows ? static_cast<uint32_t>(op.out_cap - pos)
                                                             : kWaveRows;
        if (whole && room == kWaveRows) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const uint32_t k = static_cast<uint32_t>(g * 64) + lane;
                op.emit(uni, g < H ? st0[g % H] : st1[g % H], first, pos, k, k);
            }
        } else if (kPack != 0u && kept != 0u && kept <= kPack) {
            if constexpr (kPack != 0u) {
                // (a wave reads what its own lanes wrote: LDS operations of one wave keep their order)
                uint32_t at = 0;
#pragma unroll
                for (int g = 0; g < G; ++g) {
                    const bool on = (keep >> g) & 1u;
                    const uint64_t b = __ballot(on);
                    if (on) {
                        const uint32_t k = at + wave_rank(b);
                        s_pack[wave].st[k] = g < H ? st0[g % H] : st1[g % H];
                        s_pack[wave].row[k] = static_cast<uint16_t>(g * 64 + lane);
                    }
                    at += static_cast<uint32_t>(__popcll(b));
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                const uint32_t out = kept < room ? kept : room;
                for (uint32_t k0 = 0; k0 < out; k0 += 64u) {
                    const uint32_t k = k0 + lane;
                    if (k < out) op.emit(uni, s_pack[wave].st[k], first, pos, s_pack[wave].row[k], k);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
        } else if (kPack < kWaveRows && kept != 0u) {
            uint32_t at = 0;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const bool on = (keep >> g) & 1u;
                const uint64_t b = __ballot(on);
                const uint32_t k = at + wave_rank(b);
                if (on && k < room)
                    op.emit(uni, g < H ? st0[g % H] : st1[g % H], first, pos, static_cast<uint32_t>(g * 64) + lane, k);
                at += static_cast<uint32_t>(__popcll(b));
            }
        }
        if (reports) {  // rare: the wave's rows are evaluated again, 64 at a time
            uint64_t idx[Op::kErr];
#pragma unroll
            for (int e = 0; e < Op::kErr; ++e) idx[e] = static_cast<uint64_t>(excl[1 + e]) + before[1 + e];
            for (uint32_t k0 = 0; k0 < left; k0 += 64u) {
                const uint64_t row = first + k0 + lane;
                typename Op::State rs{};
                uint32_t errs = 0;
                if (k0 + lane < left) op.report(row, rs, errs);
#pragma unroll
                for (int e = 0; e < Op::kErr; ++e) {
                    const bool on = (errs >> e) & 1u;
                    const uint64_t b = __ballot(on);
                    if (on) op.emit_err(e, row, rs, idx[e] + wave_rank(b));
                    idx[e] += static_cast<uint64_t>(__popcll(b));
                }
            }
        }
        if (tile == m.tiles - 1u && threadIdx.x == 0) {
            uint64_t totals[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) totals[s] = static_cast<uint64_t>(excl[s]) + agg[s];
            op.finish(totals);
        }
        tile = next;
        if constexpr (can_fail<Op>::value) {
            if ((drawn & kStreamFailed) != 0u) {
                if (threadIdx.x == 0) stream_drain<NS>(m, epoch, tile);
                return;
            }
        }
    }
}

// An operator over columns of any width (at most one entry per row) on this engine.  Beside the row-tile
// interface it has two streamed columns and the evaluation of rows whose codes are there:
//   DCol first_col() const, second_col() const;
//   template <int G> void eval_codes(const bool (&live)[G], const uint64_t (&c1)[G], const uint64_t (&c2)[G], State (&)[G],
//                                    uint32_t (&errs)[G], bool (&keep)[G]) const;
template <class Op>
struct StreamRows : Op {
    static constexpr int kErr = Op::kErr, kG = 8;
    static constexpr bool kLoadN = true;
    struct Raw {
        uint64_t c1, c2;
    };
    using State = typename Op::State;
    StreamRows() = default;
    explicit StreamRows(const Op &op) : Op(op) {}
    __device__ bool skip() const {
        if constexpr (has_skip<Op>::value) return Op::skip();
        return false;
    }
    struct Uniform {};
    __device__ void init(char *) const {}
    __device__ Uniform begin(const char *) const { return Uniform{}; }
    template <int H>
    __device__ __forceinline__ void load_n(uint64_t first, const uint32_t (&k)[H], Raw (&raw)[H]) const {
        uint64_t rows[H], c1[H], c2[H];
        bool on[H];
#pragma unroll
        for (int g = 0; g < H; ++g) {
            rows[g] = first + k[g];
            on[g] = true;
        }
        Op::first_col().template raw_n<H>(rows, on, c1);
        Op::second_col().template raw_n<H>(rows, on, c2);
#pragma unroll
        for (int g = 0; g < H; ++g) raw[g] = Raw{c1[g], c2[g]};
    }
    template <int G>
    struct Mid {
        State st[G];
        uint32_t keep, err[kErr];
    };
    template <int G>
    __device__ __forceinline__ void open_tile(const char *, const Uniform &, uint64_t, uint32_t, uint32_t live, const Raw (&raw)[G],
                                              Mid<G> &mid) const {
        uint64_t c1[G], c2[G];
        bool on[G], keep[G];
        uint32_t errs[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            c1[g] = raw[g].c1;
            c2[g] = raw[g].c2;
            on[g] = (live >> g) & 1u;
        }
        Op::template eval_codes<G>(on, c1, c2, mid.st, errs, keep);
        mid.keep = 0;
#pragma unroll
        for (int e = 0; e < kErr; ++e) mid.err[e] = 0;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            mid.keep |= (keep[g] ? 1u : 0u) << g;
#pragma unroll
            for (int e = 0; e < kErr; ++e) mid.err[e] |= ((errs[g] >> e) & 1u) << g;
        }
    }
    template <int G>
    __device__ __forceinline__ void close_tile(const Uniform &, const Mid<G> &mid, uint32_t live, State (&st)[G], uint32_t &keep,
                                               uint32_t (&err)[kErr]) const {
#pragma unroll
        for (int g = 0; g < G; ++g) st[g] = mid.st[g];
        keep = live & mid.keep;
#pragma unroll
        for (int e = 0; e < kErr; ++e) err[e] = live & mid.err[e];
    }
    __device__ void report(uint64_t row, State &st, uint32_t &errs) const {
        uint64_t acc = 0;
        (void)Op::eval(row, st, errs, acc);
    }
    __device__ __forceinline__ void emit(const Uniform &, const State &st, uint64_t first, uint64_t pos, uint32_t row, uint32_t k) const {
        Op::emit_main(first + row, st, pos + k, 1u);
    }
};

}  // namespace ahead_dev

namespace ahead_host {

// Launches the engine for op over op.n rows with `lds` bytes for its tables (at most kStreamLds less the
// packed entries).
constexpr size_t kStreamLds = 152 * 1024;

// Rows per lane by the size of a call.  An operator's own kG suits tens of millions of rows, where the
// tickets (15 ns each) ask for large tiles; 16,384 rows a tile keep 256 CUs busy from 4.2M rows on only.
// One MI355X, us per call with 16 / 8 / 4 / 2 rows a lane:
//   fetch of 4-byte codes, 400,000-row column: 500,000 rows 29 / 18 / 12 / 16, 1M 31 / 20 / 20 / 21,
//   2M 33 / 27 / 26 / 33, 4M 51 / 42 / 44 / 57, 8M 68 / 67 / 75 / 100;
//   check and decode of 8-byte codes: 500,000 rows 11 / 9 / 8 / 11, 1M 11 / 9 / 12 / 15, 2M 13 / 13 / 15 / 22,
//   4M 18 / 18 / 23 / 36, 8M 25 / 28 / 38 / 63.
// So 8 rows a lane below one and a half of the operator's own tiles per CU, and 4 where tiles of 8 would
// reach fewer than three eighths of the CUs.  (2 are never better than 4 by more than 2 us.)
constexpr int kStreamMidG = 8, kStreamSmallG = 4;

template <class Op, int G>
int launch_stream_g(const Op &op, ahead_hip_ws *ws, hipStream_t s, size_t lds, uint32_t cus) {
    using namespace ahead_dev;
    constexpr uint64_t rows = static_cast<uint64_t>(kStreamThreads) * G;
    if (lds > 0) {
        static PerDevice kept;
        hipError_t e = hipSuccess;
        per_device(kept, [&] {
            e = hipFuncSetAttribute(reinterpret_cast<const void *>(k_stream<Op, G>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    static_cast<int>(kStreamLds - stream_pack_bytes<Op, G>()));
            return e == hipSuccess ? 1u : 0u;
        });
        AHEAD_HIP_TRY(e);
    }
    const uint64_t tiles = op.n == 0 ? 1 : (op.n + rows - 1) / rows;
    const uint32_t grid = static_cast<uint32_t>(tiles < cus ? tiles : cus);
    StreamArgs m{};
    m.tiles = static_cast<uint32_t>(tiles);
    m.last = m.tiles + grid - 1u;
    uint64_t *words = nullptr;
    const int st = stream_state(ws, static_cast<size_t>(tiles) * (2 + 2 * Op::kErr) * 8, s, &m.te, &words);
    if (st != AHEAD_OK) return st;
    m.hdr = ws_header(ws);
    m.agg = words;
    m.incl = words + tiles;
    m.erep = words + tiles * (2 + Op::kErr);
    hipLaunchKernelGGL((k_stream<Op, G>), dim3(grid), dim3(kStreamThreads), lds, s, op, m);
    AHEAD_HIP_TRY(hipGetLastError());
    return AHEAD_OK;
}

template <class Op>
int launch_stream(const Op &op, ahead_hip_ws *ws, hipStream_t s, size_t lds = 0) {
    using namespace ahead_dev;
    static_assert(((1ull << 32) / (kStreamThreads * Op::kG)) * (2 + 2 * Op::kErr) * 8 <= kStreamMost,
                  "the status words of the largest call");
    const uint32_t cus = device_cus();
    // Tiles of fewer rows for calls that leave CUs idle otherwise, or give them one tile each, whose loads,
    // lookups and places then follow one another (see kStreamMidG).
    if constexpr (Op::kG > kStreamSmallG) {
        constexpr int mid = Op::kG >= 2 * kStreamMidG ? kStreamMidG : Op::kG;
        if (op.n < static_cast<uint64_t>(cus) * 3 / 8 * kStreamThreads * mid)
            return launch_stream_g<Op, kStreamSmallG>(op, ws, s, lds, cus);
        if constexpr (mid < Op::kG) {
            if (op.n < static_cast<uint64_t>(cus) * 3 / 2 * kStreamThreads * Op::kG)
                return launch_stream_g<Op, mid>(op, ws, s, lds, cus);
        }
    }
    return launch_stream_g<Op, Op::kG>(op, ws, s, lds, cus);
}
}  // namespace ahead_host
