// ops_an.hip -- per-operator gfx950 kernels.  On the single-pass engine (stream.hpp):
//   fetchjoinAN                 (lib/column_operators/AN/matchjoinAN.tcc:312-353)
//   matchjoinAN, positional     (matchjoinAN.tcc:240-301)
// and on the map engine (maptile.hpp):
//   aggregate_sum_groupedAN     (aggregateAN.tcc:41-119)
//   aggregate_mul_sumAN         (aggregateAN_scalar.tcc:58-131)
//   arithmeticAN                (arithmeticAN_scalar.tcc:60-112)
// Every check applies the code-width cast (static_cast<T>(code * A^-1)).  A few reference lines
// compare the int-promoted product of 16-bit codes without it (matchjoinAN.tcc:278 and :342,
// hashjoinAN.tcc:153); no query path feeds 16-bit codes to them.
#include "maptile.hpp"
#include "stream.hpp"

using namespace ahead_dev;

namespace {

// ---------------------------------------------------------------------------------------------------
// fetchjoinAN on the single-pass engine.  The gathers bound it: a random 2-byte gather costs a 128-byte
// line between L1 and L2, so 60M of them take 270 us where the rest of the operator takes 100.  A column
// that many OIDs point into is therefore looked up in LDS:
//   kRaw     its codes, when they fit;
//   kPacked  its decoded values less the smallest, in the fewest bits that hold them, several to a word;
//            the all-ones field sends the row to the column (corrupt codes; the largest value, where the
//            bits leave no other field), whose code is checked; the other rows' values are valid.  Rows past
//            the words' capacity read the column too, so a column of 200,000 8-bit values serves three
//            quarters of its rows from LDS.
// 60M OIDs into 2-byte columns, the lookups alone with the streaming around them: 40,000 rows 220 us from
// L2, 104 from LDS; 200,000 rows 264 and 150; without any lookup 97.  The whole operator into 200,000 8-bit
// values: 408 us before (gathers 340, moving the entries behind a dropped row 67), 205 now.
enum FetchTable : uint32_t { kFetchNone = 0, kFetchRaw = 1, kFetchPacked = 2 };
constexpr uint32_t kFetchTableBytes = 150 * 1024;
struct alignas(16) FetchPack {  // in front of the packed words
    uint32_t lo, bits, per, magic, covered, full;
    uint32_t pad[2];
};
constexpr uint32_t kFetchWords = (kFetchTableBytes - sizeof(FetchPack)) / 4;
constexpr uint32_t kRangeBlocks = 64;
struct FetchRange {
    uint32_t lo, hi, bad, pad;
};

// The packed table is built once per call, by the whole card, and then copied by every workgroup (built
// by each workgroup for itself it took 100 us of a 60M-OID fetch into 200,000 rows).  First the range of the column's valid
// values, one entry per workgroup ...
template <typename T>
__global__ __launch_bounds__(kBlock) void k_fetch_range(const T *col, uint32_t n, T a_inv, T max_u, FetchRange *out) {
    __shared__ uint32_t s_lo, s_hi, s_bad;
    if (threadIdx.x == 0) {
        s_lo = 0xFFFFFFFFu;
        s_hi = 0u;
        s_bad = 0u;
    }
    __syncthreads();
    constexpr uint32_t U = 8;
    uint32_t lo = 0xFFFFFFFFu, hi = 0u;
    bool bad = false;
    for (uint32_t i0 = blockIdx.x * kBlock * U; i0 < n; i0 += kRangeBlocks * kBlock * U) {
        T c[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t i = i0 + u * kBlock + threadIdx.x;
            c[u] = col[i < n ? i : n - 1u];
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const T d = an_mul<T>(c[u], a_inv);
            const bool ok = d <= max_u;
            bad |= !ok;
            lo = ok && d < lo ? d : lo;
            hi = ok && d > hi ? d : hi;
        }
    }
    atomicMin(&s_lo, lo);
    atomicMax(&s_hi, hi);
    if (bad) s_bad = 1u;
    __syncthreads();
    if (threadIdx.x == 0) out[blockIdx.x] = FetchRange{s_lo, s_hi, s_bad, 0u};
}
// ... then, from all of them, the layout, and every thread the words it comes to.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_fetch_pack(const T *col, uint32_t n, T a_inv, T max_u,
                                                       const FetchRange *ranges, FetchPack *p) {
    __shared__ uint32_t s_r[3];
    if (threadIdx.x < 64) {
        FetchRange r = ranges[threadIdx.x];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) {
            const uint32_t l = __shfl_xor(r.lo, d, 64), h = __shfl_xor(r.hi, d, 64);
            r.lo = l < r.lo ? l : r.lo;
            r.hi = h > r.hi ? h : r.hi;
            r.bad |= __shfl_xor(r.bad, d, 64);
        }
        if (threadIdx.x == 0) {
            s_r[0] = r.lo;
            s_r[1] = r.hi;
            s_r[2] = r.bad;
        }
    }
    __syncthreads();
    const uint32_t lo = s_r[0], span = s_r[1] - lo;
    uint32_t bits = 32;  // (no valid value: lo > hi)
    if (lo <= s_r[1] && span < 0x7FFFFFFFu) {
        bits = 1;
        while ((1u << bits) - 1u < span) ++bits;
        // every field taken: a few values leave one field free, of many the largest shares its own
        if ((1u << bits) - 1u == span && bits < 6u) ++bits;
        // where as many fields fit a word, whole bytes
        if (32u / bits == 4u) bits = 8u;
        if (32u / bits == 2u) bits = 16u;
    }
    const uint32_t ones = bits == 32u ? 0xFFFFFFFFu : (1u << bits) - 1u, per = 32u / bits;
    const uint32_t cap = per * kFetchWords;
    const uint32_t covered = cap >= n ? n : (cap >= n / 4u ? cap : 0u);  // below a quarter: the column alone
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        // i / per = mulhi(i, magic) for i < 2^27
        *p = FetchPack{lo, bits, per, per > 1u ? 0xFFFFFFFFu / per + 1u : 0u, covered,
                       covered == n && s_r[2] == 0u && ones != span ? 1u : 0u, {0u, 0u}};
    }
    uint32_t *w = reinterpret_cast<uint32_t *>(p + 1);
    const uint32_t q = blockIdx.x * kBlock + threadIdx.x;
    if (static_cast<uint64_t>(q) * per >= covered || q >= kFetchWords) return;
    uint32_t v = 0;
#pragma unroll 4
    for (uint32_t r = 0; r < per; ++r) {
        const uint32_t i = q * per + r;
        const T d = an_mul<T>(col[i < n ? i : n - 1u], a_inv);
        v |= (d > max_u ? ones : static_cast<uint32_t>(d) - lo) << (r * bits);
    }
    w[q] = v;
}

template <typename T, bool ENC>
struct FetchOp {
    static constexpr int kErr = 2;
    static constexpr int kG = 16;
    struct Raw {
        uint64_t c;
    };
    using Out = std::conditional_t<ENC, T, std::conditional_t<(sizeof(T) >= 4), uint64_t,
                                                             std::conditional_t<sizeof(T) == 2, uint32_t, uint16_t>>>;
    using State = Out;
    uint64_t n;
    const uint64_t *oids;
    uint64_t o_inv;
    uint32_t o_back;  // the OIDs' A (back_factor), else 0
    const T *col;
    uint32_t col_n;
    T a, a_inv, max_u;
    uint32_t table;
    const FetchPack *pack;  // kFetchPacked: the table in the workspace
    uint32_t reenc;
    Out f;
    uint64_t a_oid;
    Out *out;
    uint64_t out_cap;
    uint64_t *e1, *e2;
    uint64_t e1_cap, e2_cap;
    uint64_t *d_counts;

    __device__ bool skip() const { return false; }
    struct Uniform {
        FetchPack p;
    };
    __device__ Uniform begin(const char *lds) const {
        Uniform u{};
        if (table == kFetchPacked) {
            const FetchPack *p = reinterpret_cast<const FetchPack *>(lds);
            u.p.lo = uniform(p->lo);
            u.p.bits = uniform(p->bits);
            u.p.per = uniform(p->per);
            u.p.magic = uniform(p->magic);
            u.p.covered = uniform(p->covered);
            u.p.full = uniform(p->full);
        }
        return u;
    }
    __device__ void init(char *lds) const {
        if (table == kFetchRaw) {
            T *t = reinterpret_cast<T *>(lds);
            for (uint32_t i = threadIdx.x; i < col_n; i += kStreamThreads) t[i] = col[i];
        }
        if (table == kFetchPacked) {
            const uint4 *src = reinterpret_cast<const uint4 *>(pack);
            uint4 *dst = reinterpret_cast<uint4 *>(lds);
            const uint32_t words = pack->covered / pack->per + 1u;  // read by 16 bytes, within the table
            const uint32_t quads = (words + sizeof(FetchPack) / 4 + 3u) / 4u;
            constexpr uint32_t most = kFetchTableBytes / 16;
            for (uint32_t i = threadIdx.x; i < (quads < most ? quads : most); i += kStreamThreads) dst[i] = src[i];
        }
    }
    __device__ __forceinline__ void load(uint64_t first, uint32_t k, Raw &r) const {
        r.c = __builtin_nontemporal_load(oids + first + k);
    }
    template <int G>
    struct Mid {
        T v[G];         // the rows' codes
        uint32_t past;  // OIDs past the column
        bool clean;     // every code is valid
    };
    template <int G>
    __device__ __forceinline__ void open_tile(const char *lds, const Uniform &u, uint64_t, uint32_t, uint32_t, const Raw (&raw)[G],
                                              Mid<G> &mid) const {
        uint32_t idx[G];
        mid.past = 0;
        mid.clean = false;
        // normative bound (the reference reads one past the end at t == |col|)
        if (o_back != 0u) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const uint32_t t = static_cast<uint32_t>(raw[g].c) * static_cast<uint32_t>(o_inv);
                const bool in = t < col_n && static_cast<uint64_t>(t) * o_back == raw[g].c;
                mid.past |= (in ? 0u : 1u) << g;
                idx[g] = in ? t : 0u;
            }
        } else {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const uint64_t t = raw[g].c * o_inv;
                const bool in = t < col_n;
                mid.past |= (in ? 0u : 1u) << g;
                idx[g] = in ? static_cast<uint32_t>(t) : 0u;
            }
        }
        if (table == kFetchRaw) {
            const T *t = reinterpret_cast<const T *>(lds);
#pragma unroll
            for (int g = 0; g < G; ++g) mid.v[g] = t[idx[g]];
            return;
        }
        if constexpr (ENC && sizeof(T) <= 4) {
            const FetchPack *p = reinterpret_cast<const FetchPack *>(lds);
            const uint32_t covered = u.p.covered;
            if (covered != 0u) {
                const uint32_t bits = u.p.bits, base = u.p.lo * a;
                const uint32_t ones = bits == 32u ? 0xFFFFFFFFu : (1u << bits) - 1u;
                mid.clean = u.p.full != 0u;
                uint32_t x[G];
                if (bits == 8u) {
                    const uint8_t *t = reinterpret_cast<const uint8_t *>(p + 1);
#pragma unroll
                    for (int g = 0; g < G; ++g) x[g] = t[idx[g] < covered ? idx[g] : 0u];
                } else if (bits == 16u) {
                    const uint16_t *t = reinterpret_cast<const uint16_t *>(p + 1);
#pragma unroll
                    for (int g = 0; g < G; ++g) x[g] = t[idx[g] < covered ? idx[g] : 0u];
                } else {
                    const uint32_t *t = reinterpret_cast<const uint32_t *>(p + 1);
                    const uint32_t per = u.p.per, magic = u.p.magic;
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        const uint32_t i = idx[g] < covered ? idx[g] : 0u;
                        const uint32_t q = per > 1u ? __umulhi(i, magic) : i;
                        x[g] = (t[q] >> (__umul24(i - q * per, bits))) & ones;
                    }
                }
#pragma unroll
                for (int g = 0; g < G; ++g) mid.v[g] = static_cast<T>(x[g] * a + base);
                if (!mid.clean) {
#pragma unroll
                    for (int g = 0; g < G; ++g) {
                        if (idx[g] >= covered || x[g] == ones) mid.v[g] = col[idx[g]];
                    }
                }
                return;
            }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) mid.v[g] = col[idx[g]];
    }
    template <int G>
    __device__ __forceinline__ void close_tile(const Uniform &, const Mid<G> &mid, uint32_t live, State (&st)[G], uint32_t &keep,
                                               uint32_t (&errs)[kErr]) const {
        uint32_t bad = 0;
#pragma unroll
        for (int g = 0; g < G; ++g) st[g] = static_cast<Out>(mid.v[g]);
        if constexpr (ENC) {
            if (!mid.clean) {
#pragma unroll
                for (int g = 0; g < G; ++g) bad |= (an_mul<T>(mid.v[g], a_inv) > max_u ? 1u : 0u) << g;
            }
        }
        if (reenc) {
#pragma unroll
            for (int g = 0; g < G; ++g) st[g] = an_mul<Out>(st[g], f);
        }
        errs[0] = live & mid.past;
        errs[1] = live & ~mid.past & bad;
        keep = live & ~mid.past & ~bad;
    }
    __device__ void report(uint64_t row, State &, uint32_t &errs) const {
        const uint64_t t = oids[row] * o_inv;
        if (t >= col_n) errs = 1u;
        else if (ENC && an_mul<T>(col[t], a_inv) > max_u) errs = 2u;
    }
    __device__ __forceinline__ void emit(const Uniform &, const State &st, uint64_t, uint64_t pos, uint32_t, uint32_t k) const {
        __builtin_nontemporal_store(st, out + pos + k);
    }
    __device__ void emit_err(int e, uint64_t row, const State &, uint64_t pos) const {
        if (e == 0) {
            if (pos < e1_cap) e1[pos] = row * a_oid;
        } else if (pos < e2_cap) {
            e2[pos] = oids[row] * o_inv * a_oid;
        }
    }
    __device__ void finish(const uint64_t *t) const {
        d_counts[0] = t[0];
        d_counts[1] = t[1];
        d_counts[2] = t[2];
    }
};

template <typename T, bool ENC>
int launch_fetch(const ahead_col *oids, const ahead_col *col, int reenc, uint64_t a_reenc, uint64_t a_oid,
                 ahead_buf out, ahead_buf err1, ahead_buf err2, uint64_t *d_counts, ahead_hip_ws *ws, hipStream_t s) {
    using Op = FetchOp<T, ENC>;
    Op op{};
    op.n = oids->n;
    op.oids = static_cast<const uint64_t *>(oids->data);
    op.o_inv = oids->a_inv;
    op.o_back = ahead_host::back_factor(oids->a_inv, 0xFFFFFFFFull);  // positions are below |col| < 2^32
    // an empty column is never read, but its row 0 is addressed: any readable element stands in
    op.col = static_cast<const T *>(col->n ? col->data : oids->data);
    op.col_n = static_cast<uint32_t>(col->n);
    op.a = static_cast<T>(col->a);
    op.a_inv = static_cast<T>(col->a_inv);
    op.max_u = static_cast<T>(col->max_u);
    op.reenc = reenc != 0;
    // matchjoinAN.tcc:323-327: re-encoding factor A_R * inv(A_col) (A_R alone for a plain column)
    op.f = static_cast<typename Op::Out>(
        reenc ? (ENC ? a_reenc * ahead_host::inverse_mod2k(col->a, 8 * sizeof(typename Op::Out)) : a_reenc) : 1);
    op.a_oid = a_oid;
    op.out = static_cast<typename Op::Out *>(out.data);
    op.out_cap = out.data ? out.cap : 0;
    op.e1 = static_cast<uint64_t *>(err1.data);
    op.e1_cap = err1.data ? err1.cap : 0;
    op.e2 = static_cast<uint64_t *>(err2.data);
    op.e2_cap = err2.data ? err2.cap : 0;
    op.d_counts = d_counts;
    // Every workgroup fills a table of its own, the packed one after two small launches, which the gathers it
    // saves have to earn.  us a call, from the column / from the table.  Codes: 40 KB, 500,000 OIDs 11 / 11,
    // 1M 16 / 14, 8M 45 / 31; 140 KB, 250,000 10 / 12, 500,000 11 / 13, 1M 17 / 16, 8M 57 / 33.  So they pay
    // from about 4 OIDs a byte on.  Packed values: 200,000 8-bit ones (400 KB of codes) 4M 40 / 38, 8M
    // 62 / 48, 60M 317 / 179; 60,000 16-bit ones (240 KB) 2M 26 / 28, 4M 40 / 35; 1M 8-bit ones 16M
    // 105 / 112, 60M 335 / 339 (below a quarter of the rows in LDS the kernel leaves it).  So from 16 OIDs
    // a byte on, and up to 2 MB.  A corrupt value re-encodes differently from its decoded form, so the packed
    // table needs A^-1 to be A's inverse.
    const uint64_t bytes = col->n * sizeof(T);
    size_t lds = 0;
    if (col->n && bytes <= kFetchTableBytes && op.n / 4 >= bytes) {
        op.table = kFetchRaw;
        lds = bytes;
    } else if (ENC && sizeof(T) <= 4 && bytes <= (2u << 20) && op.n / 16 >= bytes &&
               static_cast<T>(static_cast<uint64_t>(op.a) * op.a_inv) == 1) {
        if constexpr (ENC && sizeof(T) <= 4) {
            const int st = ahead_host::ws_ensure(ws, kFetchTableBytes + kRangeBlocks * sizeof(FetchRange));
            if (st != AHEAD_OK) return st;
            FetchPack *pack = reinterpret_cast<FetchPack *>(ahead_host::ws_region(ws, 0));
            FetchRange *ranges = reinterpret_cast<FetchRange *>(ahead_host::ws_region(ws, kFetchTableBytes));
            hipLaunchKernelGGL(k_fetch_range<T>, dim3(kRangeBlocks), dim3(kBlock), 0, s, op.col, op.col_n, op.a_inv,
                               op.max_u, ranges);
            hipLaunchKernelGGL(k_fetch_pack<T>, dim3((kFetchWords + kBlock - 1) / kBlock), dim3(kBlock), 0, s, op.col,
                               op.col_n, op.a_inv, op.max_u, ranges, pack);
            AHEAD_HIP_TRY(hipGetLastError());
            op.pack = pack;
            op.table = kFetchPacked;
            lds = kFetchTableBytes;
        }
    }
    return ahead_host::launch_stream(op, ws, s, lds);
}

// ---------------------------------------------------------------------------------------------------
struct MatchPosState {
    uint64_t h;  // head value (already re-encoded)
    uint64_t v;  // fetched value, or pos2 for an error
};

struct MatchPosOp {
    static constexpr int kErr = 3;  // e1: corrupt head, e2: position out of range, e4: corrupt fetched tail
    static constexpr bool kMulti = false, kMain = true, kAcc = false;
    using State = MatchPosState;
    uint64_t n;
    DCol h1, t1, t2;
    uint32_t reenc_h, reenc_t, wh, wt;
    uint64_t f_h1, f_t2, mh, mt, a_oid;
    void *out_h, *out_t;
    uint64_t out_cap;
    uint64_t *err[3];
    uint64_t cap[3];
    uint64_t *d_counts;

    __device__ const DCol &first_col() const { return h1; }
    __device__ const DCol &second_col() const { return t1; }
    template <int G>
    __device__ __forceinline__ void eval_codes(const bool (&live)[G], const uint64_t (&h)[G], const uint64_t (&o)[G], State (&st)[G],
                                               uint32_t (&errs)[G], bool (&keep)[G]) const {
        uint64_t p2[G], v[G];
        bool in[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            p2[g] = o[g] * t1.a_inv;
            in[g] = live[g] && p2[g] < t2.n;
        }
        t2.raw_n<G>(p2, in, v);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const bool bad = t2.bad_of(v[g]);
            errs[g] = (h1.bad_of(h[g]) ? 1u : 0u) | (!in[g] ? 2u : bad ? 4u : 0u);
            keep[g] = in[g] && !bad;
            st[g].h = reenc_h ? (h[g] * f_h1) & mh : h[g];
            st[g].v = reenc_t ? (v[g] * f_t2) & mt : v[g];
        }
    }

    __device__ uint32_t eval(uint64_t row, State &st, uint32_t &errs, uint64_t &) const {
        const uint64_t h = h1.raw(row);
        if (h1.bad_of(h)) errs |= 1u;
        st.h = reenc_h ? (h * f_h1) & mh : h;
        const uint64_t pos2 = t1.raw(row) * t1.a_inv;
        if (pos2 >= t2.n) {
            errs |= 2u;
            return 0;
        }
        const uint64_t v = t2.raw(pos2);
        if (t2.bad_of(v)) {
            errs |= 4u;
            st.v = pos2;
            return 0;
        }
        st.v = reenc_t ? (v * f_t2) & mt : v;
        return 1;
    }
    __device__ void emit_main(uint64_t, const State &st, uint64_t pos, uint32_t) const {
        if (pos < out_cap) {
            store_w(out_h, pos, wh, st.h);
            store_w(out_t, pos, wt, st.v);
        }
    }
    __device__ void emit_err(int e, uint64_t row, const State &st, uint64_t pos) const {
        if (pos >= cap[e]) return;
        err[e][pos] = (e == 2 ? st.v : row) * a_oid;
    }
    __device__ void tile_done(uint32_t, uint64_t) const {}
    __device__ void finish(const uint64_t *t) const {
        for (int i = 0; i < 4; ++i) d_counts[i] = t[i];
    }
};

enum MatchHead { kHeadVoid, kHeadSame, kHeadCol };

// The positional match for its common shapes on the single-pass engine: the left head is void, the
// left tail's own column (the chains' mirrored OID lists) or another column of 8-byte codes; fetched
// codes of T.  Same results as MatchPosOp.  12M ascending OIDs into a 60M-row column of 8-byte codes:
// 72 us before, 50 now.
template <int HEAD, typename T, typename H>
struct MatchLeanOp {
    static constexpr int kErr = 3;
    static constexpr int kG = 8;
    struct Raw1 {
        uint64_t o;
    };
    struct Raw2 {
        uint64_t o, h;
    };
    using Raw = std::conditional_t<HEAD == kHeadCol, Raw2, Raw1>;
    struct StateH {
        uint64_t h;  // (void: not used)
        T v;
    };
    struct StateV {
        T v;
    };
    using State = std::conditional_t<HEAD == kHeadVoid, StateV, StateH>;
    uint64_t n;
    const uint64_t *h1;
    uint64_t h1_inv, h1_maxu, h1_seq;
    uint32_t h1_enc;
    const uint64_t *oids;
    uint64_t o_inv;
    uint32_t o_back;  // the OIDs' A (back_factor), else 0
    const T *col;
    uint32_t col_n, col_enc;
    T col_inv, col_maxu;
    uint64_t f_h;     // re-encoding factors (1: none)
    T f_t;
    uint64_t a_oid;
    H *out_h;
    T *out_t;
    uint64_t out_cap;
    uint64_t *err[3];
    uint64_t cap[3];
    uint64_t *d_counts;

    __device__ bool skip() const { return false; }
    struct Uniform {};
    __device__ void init(char *) const {}
    __device__ Uniform begin(const char *) const { return Uniform{}; }
    __device__ __forceinline__ void load(uint64_t first, uint32_t k, Raw &r) const {
        r.o = __builtin_nontemporal_load(oids + first + k);
        if constexpr (HEAD == kHeadCol) r.h = __builtin_nontemporal_load(h1 + first + k);
    }
    __device__ __forceinline__ bool head_bad(uint64_t h) const { return h1_enc != 0u && h * h1_inv > h1_maxu; }
    template <int G>
    struct Mid {
        uint64_t h[HEAD == kHeadVoid ? 1 : G];
        T v[G];
        uint32_t hbad, past;
    };
    template <int G>
    __device__ __forceinline__ void open_tile(const char *, const Uniform &, uint64_t, uint32_t, uint32_t, const Raw (&raw)[G],
                                              Mid<G> &mid) const {
        uint32_t idx[G];
        mid.past = 0;
        mid.hbad = 0;
        if (o_back != 0u) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const uint32_t t = static_cast<uint32_t>(raw[g].o) * static_cast<uint32_t>(o_inv);
                const bool in = t < col_n && static_cast<uint64_t>(t) * o_back == raw[g].o;
                mid.past |= (in ? 0u : 1u) << g;
                idx[g] = in ? t : 0u;
            }
        } else {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const uint64_t t = raw[g].o * o_inv;
                const bool in = t < col_n;
                mid.past |= (in ? 0u : 1u) << g;
                idx[g] = in ? static_cast<uint32_t>(t) : 0u;
            }
        }
#pragma unroll
        for (int g = 0; g < G; ++g) mid.v[g] = col[idx[g]];
        if constexpr (HEAD == kHeadSame) {
#pragma unroll
            for (int g = 0; g < G; ++g) mid.h[g] = raw[g].o;
            // a position inside the column is a valid OID (h1_maxu covers 32 bits, checked by the host)
            if (__ballot(mid.past != 0u) != 0ull) {
#pragma unroll
                for (int g = 0; g < G; ++g) mid.hbad |= (head_bad(raw[g].o) ? 1u : 0u) << g;
            }
        } else if constexpr (HEAD == kHeadCol) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                mid.h[g] = raw[g].h;
                mid.hbad |= (head_bad(raw[g].h) ? 1u : 0u) << g;
            }
        }
    }
    template <int G>
    __device__ __forceinline__ void close_tile(const Uniform &, const Mid<G> &mid, uint32_t live, State (&st)[G], uint32_t &keep,
                                               uint32_t (&errs)[kErr]) const {
        uint32_t bad = 0;
        if (col_enc) {
#pragma unroll
            for (int g = 0; g < G; ++g) bad |= (an_mul<T>(mid.v[g], col_inv) > col_maxu ? 1u : 0u) << g;
        }
#pragma unroll
        for (int g = 0; g < G; ++g) {
            st[g].v = mid.v[g];
            if constexpr (HEAD != kHeadVoid) st[g].h = mid.h[g];
        }
        if (f_t != 1) {
#pragma unroll
            for (int g = 0; g < G; ++g) st[g].v = an_mul<T>(st[g].v, f_t);
        }
        if constexpr (HEAD != kHeadVoid) {
            if (f_h != 1ull) {
#pragma unroll
                for (int g = 0; g < G; ++g) st[g].h *= f_h;
            }
        }
        errs[0] = live & mid.hbad;
        errs[1] = live & mid.past;
        errs[2] = live & ~mid.past & bad;
        keep = live & ~mid.past & ~bad;
    }
    __device__ void report(uint64_t row, State &, uint32_t &errs) const {
        if (HEAD != kHeadVoid && head_bad(h1[row])) errs |= 1u;
        const uint64_t t = oids[row] * o_inv;
        if (t >= col_n) errs |= 2u;
        else if (col_enc && an_mul<T>(col[t], col_inv) > col_maxu) errs |= 4u;
    }
    __device__ __forceinline__ void emit(const Uniform &, const State &st, uint64_t first, uint64_t pos, uint32_t row, uint32_t k) const {
        H h;
        if constexpr (HEAD == kHeadVoid) h = static_cast<uint32_t>(static_cast<uint32_t>(h1_seq + first) + row);
        else h = static_cast<H>(st.h);
        __builtin_nontemporal_store(h, out_h + pos + k);
        __builtin_nontemporal_store(st.v, out_t + pos + k);
    }
    __device__ void emit_err(int e, uint64_t row, const State &, uint64_t pos) const {
        if (pos < cap[e]) err[e][pos] = (e == 2 ? oids[row] * o_inv : row) * a_oid;
    }
    __device__ void finish(const uint64_t *t) const {
        for (int i = 0; i < 4; ++i) d_counts[i] = t[i];
    }
};

template <int HEAD, typename T, typename H>
int launch_match(const MatchPosOp &p, const ahead_col *h1, const ahead_col *t1, const ahead_col *t2, ahead_hip_ws *ws,
                 hipStream_t s) {
    MatchLeanOp<HEAD, T, H> op{};
    op.n = p.n;
    op.h1 = static_cast<const uint64_t *>(h1->data);
    op.h1_inv = p.h1.a_inv;
    op.h1_maxu = p.h1.max_u;
    op.h1_seq = h1->seqbase;
    op.h1_enc = p.h1.encoded;
    op.oids = static_cast<const uint64_t *>(t1->data);
    op.o_inv = t1->a_inv;
    op.o_back = ahead_host::back_factor(t1->a_inv, 0xFFFFFFFFull);  // positions are below |t2| < 2^32
    // an empty column is never read, but its row 0 is addressed: any readable element stands in
    op.col = static_cast<const T *>(t2->n ? t2->data : t1->data);
    op.col_n = static_cast<uint32_t>(t2->n);
    op.col_enc = p.t2.encoded;
    op.col_inv = static_cast<T>(t2->a_inv);
    op.col_maxu = static_cast<T>(p.t2.max_u);
    op.f_h = p.reenc_h ? p.f_h1 : 1ull;
    op.f_t = static_cast<T>(p.reenc_t ? p.f_t2 : 1ull);
    op.a_oid = p.a_oid;
    op.out_h = static_cast<H *>(p.out_h);
    op.out_t = static_cast<T *>(p.out_t);
    op.out_cap = p.out_cap;
    for (int i = 0; i < 3; ++i) {
        op.err[i] = p.err[i];
        op.cap[i] = p.cap[i];
    }
    op.d_counts = p.d_counts;
    return ahead_host::launch_stream(op, ws, s);
}

// The lean shape of a positional match, if it has one; false: MatchPosOp runs.
bool launch_match_lean(const MatchPosOp &p, const ahead_col *h1, const ahead_col *t1, const ahead_col *t2,
                       ahead_hip_ws *ws, hipStream_t s, int *st) {
    // void heads are written as they are; fetched codes keep their width
    const int head = h1->data == nullptr ? kHeadVoid
                     : h1->width != 8    ? -1
                     : h1->data == t1->data && h1->encoded == t1->encoded && h1->a_inv == t1->a_inv &&
                               h1->max_u >= 0xFFFFFFFFull
                         ? kHeadSame
                         : kHeadCol;
    const uint32_t w = t2->data ? t2->width : 0;
    if (head < 0 || p.wt != w || (head == kHeadVoid ? p.wh != 4 || p.reenc_h : p.wh != 8)) return false;
#define AHEAD_MATCH(T)                                                                          \
    *st = head == kHeadVoid   ? launch_match<kHeadVoid, T, uint32_t>(p, h1, t1, t2, ws, s)      \
          : head == kHeadSame ? launch_match<kHeadSame, T, uint64_t>(p, h1, t1, t2, ws, s)      \
                              : launch_match<kHeadCol, T, uint64_t>(p, h1, t1, t2, ws, s);      \
    return true
    switch (w) {
        case 2: AHEAD_MATCH(uint16_t);
        case 4: AHEAD_MATCH(uint32_t);
        case 8: AHEAD_MATCH(uint64_t);
        default: return false;
    }
#undef AHEAD_MATCH
}

// ---------------------------------------------------------------------------------------------------
struct ArithOp {
    static constexpr int kErr = 4;  // head1, tail1, head2, tail2
    static constexpr bool kMulti = false, kMain = false, kAcc = false;
    static constexpr int kMapRows = 8;  // half the steps whose loads wait for the previous step's stores
    using State = uint8_t;
    uint64_t n;
    DCol h1, t1, h2, t2;
    int op;
    uint64_t a_result, rmask, a_oid;
    uint32_t rw;
    void *out;
    uint64_t *err[4];
    uint64_t cap[4];
    uint64_t *d_counts;

    __device__ uint64_t combine(uint64_t c1, uint64_t c2) const {
        const uint64_t x = (t1.dec_of(c1) * a_result) & rmask, y = (t2.dec_of(c2) * a_result) & rmask;
        uint64_t r;
        switch (op) {
            case 0: r = x + y; break;
            case 1: r = x - y; break;
            case 2: r = x * y; break;
            default: r = y ? x / y : 0; break;
        }
        return r & rmask;
    }
    static constexpr bool kBatched = true;
    template <int G>
    __device__ void eval_n(const uint64_t (&row)[G], const bool (&live)[G], State (&)[G], uint32_t (&errs)[G],
                           uint32_t (&cnt)[G], uint64_t &) const {
        uint64_t c1[G], c2[G], a1[G], a2[G];
        t1.raw_n<G>(row, live, c1);
        t2.raw_n<G>(row, live, c2);
        if (h1.encoded) h1.raw_n<G>(row, live, a1);
        if (h2.encoded) h2.raw_n<G>(row, live, a2);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            cnt[g] = 0;
            errs[g] = 0;
            if (!live[g]) continue;
            if (h1.encoded && h1.bad_of(a1[g])) errs[g] |= 1u;
            if (t1.bad_of(c1[g])) errs[g] |= 2u;
            if (h2.encoded && h2.bad_of(a2[g])) errs[g] |= 4u;
            if (t2.bad_of(c2[g])) errs[g] |= 8u;
            store_w(out, row[g], rw, combine(c1[g], c2[g]));
        }
    }
    __device__ uint32_t eval(uint64_t row, State &, uint32_t &errs, uint64_t &) const {
        if (h1.bad_of(h1.raw(row))) errs |= 1u;
        const uint64_t c1 = t1.raw(row), c2 = t2.raw(row);
        if (t1.bad_of(c1)) errs |= 2u;
        if (h2.bad_of(h2.raw(row))) errs |= 4u;
        if (t2.bad_of(c2)) errs |= 8u;
        const uint64_t x = (t1.dec_of(c1) * a_result) & rmask, y = (t2.dec_of(c2) * a_result) & rmask;
        uint64_t r;
        switch (op) {
            case 0: r = x + y; break;
            case 1: r = x - y; break;
            case 2: r = x * y; break;
            default: r = y ? x / y : 0; break;
        }
        store_w(out, row, rw, r & rmask);
        return 0;
    }
    __device__ void emit_main(uint64_t, const State &, uint64_t, uint32_t) const {}
    __device__ void emit_err(int e, uint64_t row, const State &, uint64_t pos) const {
        if (pos < cap[e]) err[e][pos] = row * a_oid;
    }
    __device__ void tile_done(uint32_t, uint64_t) const {}
    __device__ void finish(const uint64_t *t) const {
        d_counts[0] = n;
        for (int i = 1; i < 5; ++i) d_counts[i] = t[i];
    }
};

// ---------------------------------------------------------------------------------------------------
struct MulSumOp {
    static constexpr int kErr = 2;
    static constexpr bool kMulti = false, kMain = false, kAcc = true;
    using State = uint8_t;
    uint64_t n;
    DCol t1, t2;
    uint64_t a_oid;
    uint64_t *partials;
    uint64_t *err[2];
    uint64_t cap[2];
    uint64_t *d_counts;

    static constexpr bool kBatched = true;
    template <int G>
    __device__ void eval_n(const uint64_t (&row)[G], const bool (&live)[G], State (&)[G], uint32_t (&errs)[G],
                           uint32_t (&cnt)[G], uint64_t &acc) const {
        uint64_t c1[G], c2[G];
        t1.raw_n<G>(row, live, c1);
        t2.raw_n<G>(row, live, c2);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            cnt[g] = 0;
            errs[g] = (live[g] && t1.bad_of(c1[g]) ? 1u : 0u) | (live[g] && t2.bad_of(c2[g]) ? 2u : 0u);
            acc += c1[g] * c2[g];  // rows past the end load 0
        }
    }
    __device__ uint32_t eval(uint64_t row, State &, uint32_t &errs, uint64_t &acc) const {
        const uint64_t c1 = t1.raw(row), c2 = t2.raw(row);
        if (t1.bad_of(c1)) errs |= 1u;
        if (t2.bad_of(c2)) errs |= 2u;
        acc += c1 * c2;
        return 0;
    }
    __device__ void emit_main(uint64_t, const State &, uint64_t, uint32_t) const {}
    __device__ void emit_err(int e, uint64_t row, const State &, uint64_t pos) const {
        if (pos < cap[e]) err[e][pos] = row * a_oid;
    }
    __device__ void tile_done(uint32_t tile, uint64_t t) const { partials[tile] = t; }
    __device__ void finish(const uint64_t *t) const {
        d_counts[0] = 1;
        d_counts[1] = t[1];
        d_counts[2] = t[2];
    }
};

__global__ __launch_bounds__(kBlock) void k_mulsum_final(const uint64_t *partials, uint32_t n, uint64_t init,
                                                         uint64_t enc, uint64_t *out) {
    __shared__ uint64_t s_red[kWaves];
    uint64_t s = 0;
    for (uint32_t i = threadIdx.x; i < n; i += kBlock) s += partials[i];
    s = block_sum<uint64_t>(s, s_red);
    if (threadIdx.x == 0) *out = (init + s) * enc;
}

// ---------------------------------------------------------------------------------------------------
// Grouped sum: LDS-private accumulators per workgroup when the groups fit, then one partial per group and
// workgroup with rows and a reduction; otherwise straight 64-bit atomics on the output.
constexpr uint32_t kAggLds = 4096;  // 64-bit words

struct AggSumArgs {
    uint64_t n;
    DCol head, tail, grp;
    uint64_t num_groups, enc, a_oid;
    uint32_t grp_back, tail_back;  // the codes' A where 32-bit arithmetic decodes them (back_factor), else 0
    uint32_t copies;               // accumulators per group in LDS (a power of two; 0: none)
    uint32_t parts;                // workgroups with rows: those that leave partials
    uint64_t *partials;            // [parts][num_groups] (copies != 0)
    uint64_t *sums;
    uint64_t *err[3];
    uint64_t cap[3];
    uint64_t *d_counts;
};

struct AggSumOp {
    // Checks and sums in one pass.  Few groups make the lanes of a wave meet on the same LDS word, and
    // same-word atomics run one after another (12M rows into 35 groups: 71 us, 4.5 times what the two
    // columns take to read).  So a group has up to 32 accumulators side by side, each lane adding to its
    // own of them, and the workgroups leave partials: 12M rows 57 us.  The codes are summed as they
    // are and multiplied by the re-encoding factor at the end (sums mod 2^64 are linear).
    // Many groups make the partials the cost: only workgroups with rows leave them, side by side
    // (4096 groups: 250,000 rows 74 us when all 977 workgroups of the grid did, each group's in a row of
    // its own, 23 now; 4M rows 86 and 49; 30M rows 128, by atomics on the output 1230).
    static constexpr int kErr = 3;
    static constexpr int kMapRows = 8;  // twice the loads in flight
    static constexpr int kSharedWords = kAggLds;
    static constexpr bool kMulti = false, kMain = false, kAcc = false;
    using State = uint8_t;
    AggSumArgs a;
    uint64_t n;
    static constexpr bool kBatched = true;
    __device__ void shared_init(unsigned long long *s) const {
        const uint32_t nw = static_cast<uint32_t>(a.num_groups) * a.copies;
        for (uint32_t i = threadIdx.x; i < nw; i += blockDim.x) s[i] = 0ull;
    }
    __device__ void shared_flush(unsigned long long *s) const {
        if (a.copies == 0u || blockIdx.x >= a.parts) return;
        for (uint32_t i = threadIdx.x; i < a.num_groups; i += blockDim.x) {
            unsigned long long x = 0ull;
            for (uint32_t c = 0; c < a.copies; ++c) x += s[i * a.copies + ((c + i) & (a.copies - 1u))];
            a.partials[blockIdx.x * a.num_groups + i] = x;
        }
    }
    // aggregateAN.tcc:84-112: a corrupt tail is still added (and reported); a row whose group id
    // is corrupt or out of range is reported and skipped
    template <int G>
    __device__ void eval_shared(const uint64_t (&row)[G], const bool (&live)[G], State (&st)[G], uint32_t (&errs)[G],
                                uint32_t (&cnt)[G], uint64_t &acc, unsigned long long *s) const {
        uint64_t t[G], gi[G];
        eval_rows<G>(row, live, errs, t, gi);
        const uint32_t copy = threadIdx.x & (a.copies - 1u);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            cnt[g] = 0;
            if (!live[g] || (errs[g] & 4u)) continue;
            if (a.copies != 0u) atomicAdd(&s[static_cast<uint32_t>(gi[g]) * a.copies + copy], static_cast<unsigned long long>(t[g]));
            else atomicAdd(reinterpret_cast<unsigned long long *>(&a.sums[gi[g]]), static_cast<unsigned long long>(t[g] * a.enc));
        }
        (void)st;
        (void)acc;
    }
    // error bits, tail codes and group ids of G rows
    template <int G>
    __device__ void eval_rows(const uint64_t (&row)[G], const bool (&live)[G], uint32_t (&errs)[G], uint64_t (&t)[G],
                              uint64_t (&gi)[G]) const {
        uint64_t h[G], gr[G];
        if (a.head.encoded) a.head.raw_n<G>(row, live, h);
        a.tail.raw_n<G>(row, live, t);
        a.grp.raw_n<G>(row, live, gr);
#pragma unroll
        for (int g = 0; g < G; ++g) {
            bool ok, bad;
            if (a.grp_back != 0u) {
                const uint32_t x = static_cast<uint32_t>(gr[g]) * static_cast<uint32_t>(a.grp.a_inv);
                ok = x < a.num_groups && static_cast<uint64_t>(x) * a.grp_back == gr[g] && x <= a.grp.max_u;
                gi[g] = x;
            } else {
                const uint64_t x = gr[g] * a.grp.a_inv;
                ok = x <= a.grp.max_u && x < a.num_groups;
                gi[g] = x;
            }
            if (a.tail_back != 0u) {
                const uint32_t d = static_cast<uint32_t>(t[g]) * static_cast<uint32_t>(a.tail.a_inv);
                bad = static_cast<uint64_t>(d) * a.tail_back != t[g] || d > a.tail.max_u;
            } else {
                bad = a.tail.bad_of(t[g]);
            }
            errs[g] = !live[g] ? 0u
                               : (a.head.encoded && a.head.bad_of(h[g]) ? 1u : 0u) | (bad ? 2u : 0u) | (ok ? 0u : 4u);
        }
    }
    template <int G>
    __device__ void eval_n(const uint64_t (&row)[G], const bool (&live)[G], State (&)[G], uint32_t (&errs)[G],
                           uint32_t (&cnt)[G], uint64_t &) const {
        uint64_t t[G], gi[G];
        eval_rows<G>(row, live, errs, t, gi);
#pragma unroll
        for (int g = 0; g < G; ++g) cnt[g] = 0;
    }
    __device__ uint32_t eval(uint64_t row, State &, uint32_t &errs, uint64_t &) const {
        if (a.head.bad_of(a.head.raw(row))) errs |= 1u;
        if (a.tail.bad_of(a.tail.raw(row))) errs |= 2u;
        const uint64_t g = a.grp.raw(row) * a.grp.a_inv;
        if (g > a.grp.max_u || g >= a.num_groups) errs |= 4u;
        return 0;
    }
    __device__ void emit_main(uint64_t, const State &, uint64_t, uint32_t) const {}
    __device__ void emit_err(int e, uint64_t row, const State &, uint64_t pos) const {
        if (pos < a.cap[e]) a.err[e][pos] = row * a.a_oid;
    }
    __device__ void tile_done(uint32_t, uint64_t) const {}
    __device__ void finish(const uint64_t *t) const {
        a.d_counts[0] = a.num_groups;
        for (int i = 1; i < 4; ++i) a.d_counts[i] = t[i];
    }
};


// The groups' partials of all workgroups, re-encoded: kAggFinal groups per workgroup, whose threads read
// them side by side.  (Added to the output with atomics by every workgroup, 1280 of them meeting on each
// group's word cost 20 us.)
constexpr uint32_t kAggFinal = 4;
__global__ __launch_bounds__(kBlock) void k_aggsum_final(AggSumArgs a) {
    __shared__ uint64_t s_sum[kWaves][kAggFinal];
    const uint32_t lane = threadIdx.x & 63u, sub = threadIdx.x % kAggFinal;
    const uint64_t g = static_cast<uint64_t>(blockIdx.x) * kAggFinal + sub;
    uint64_t x = 0;
    if (g < a.num_groups) {
#pragma unroll 4
        for (uint32_t i = threadIdx.x / kAggFinal; i < a.parts; i += kBlock / kAggFinal) x += a.partials[i * a.num_groups + g];
    }
#pragma unroll
    for (int d = 32; d >= static_cast<int>(kAggFinal); d >>= 1) x += __shfl_xor(x, d, 64);
    if (lane < kAggFinal) s_sum[threadIdx.x >> 6][lane] = x;
    __syncthreads();
    if (threadIdx.x < kAggFinal && g < a.num_groups) {
        uint64_t t = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) t += s_sum[w][threadIdx.x];
        a.sums[g] = t * a.enc;
    }
}

__global__ void k_fill_u64(uint64_t *p, uint64_t n, uint64_t v) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < n; i += stride) p[i] = v;
}

}  // namespace

namespace ahead_host {

DCol dcol(const ahead_col &c) {
    DCol d{};
    d.data = c.data;
    d.n = c.n;
    d.width = c.data ? c.width : 4;
    d.encoded = c.encoded && c.data != nullptr;
    d.a_inv = c.a_inv;
    d.mask = width_mask(d.width);
    d.max_u = c.max_u & d.mask;
    d.seqbase = c.seqbase;
    return d;
}

}  // namespace ahead_host

using namespace ahead_host;

extern "C" int ahead_hip_fetchjoin_an(const ahead_col *oids, const ahead_col *col, int reenc, uint64_t a_reenc,
                                      uint64_t a_oid, ahead_buf out, ahead_buf err1, ahead_buf err2,
                                      uint64_t *d_counts, ahead_hip_ws *ws, void *stream) {
    int st;
    if ((st = check_col(oids, "fetchjoin.oids", false, true)) != AHEAD_OK) return st;
    if ((st = check_col(col, "fetchjoin.col", false, false)) != AHEAD_OK) return st;
    if (oids->width != 8) return fail(AHEAD_ERR_INVALID, "fetchjoin: OIDs are resoid (8-byte) codes");
    if (d_counts == nullptr) return fail(AHEAD_ERR_INVALID, "fetchjoin: d_counts is NULL");
    hipStream_t s = static_cast<hipStream_t>(stream);
#define AHEAD_FETCH(T, E) launch_fetch<T, E>(oids, col, reenc, a_reenc, a_oid, out, err1, err2, d_counts, ws, s)
    switch (col->width) {
        case 1: return AHEAD_FETCH(uint8_t, false);
        case 2: return col->encoded ? AHEAD_FETCH(uint16_t, true) : AHEAD_FETCH(uint16_t, false);
        case 4: return col->encoded ? AHEAD_FETCH(uint32_t, true) : AHEAD_FETCH(uint32_t, false);
        default: return col->encoded ? AHEAD_FETCH(uint64_t, true) : AHEAD_FETCH(uint64_t, false);
    }
#undef AHEAD_FETCH
}

extern "C" int ahead_hip_matchjoin_pos_an(const ahead_col *h1, const ahead_col *t1, const ahead_col *t2, int reenc_h,
                                          uint64_t f_h1, uint32_t wout_h, int reenc_t, uint64_t f_t2, uint32_t wout_t,
                                          uint64_t a_oid, ahead_buf out_h, ahead_buf out_t, ahead_buf err1,
                                          ahead_buf err2, ahead_buf err4, uint64_t *d_counts, ahead_hip_ws *ws,
                                          void *stream) {
    int st;
    if ((st = check_col(h1, "matchjoin.h1", true, false)) != AHEAD_OK) return st;
    if ((st = check_col(t1, "matchjoin.t1", false, true)) != AHEAD_OK) return st;
    if ((st = check_col(t2, "matchjoin.t2", false, false)) != AHEAD_OK) return st;
    if (h1->n != t1->n) return fail(AHEAD_ERR_SIZE_MISMATCH, "matchjoin: head and tail of the left BAT differ");
    if (t1->width != 8) return fail(AHEAD_ERR_INVALID, "matchjoin: the left tail holds resoid (8-byte) codes");
    if (d_counts == nullptr) return fail(AHEAD_ERR_INVALID, "matchjoin: d_counts is NULL");
    if ((wout_h != 1 && wout_h != 2 && wout_h != 4 && wout_h != 8) || (wout_t != 1 && wout_t != 2 && wout_t != 4 && wout_t != 8))
        return fail(AHEAD_ERR_INVALID, "matchjoin: output widths must be 1, 2, 4 or 8");
    MatchPosOp op{};
    op.n = t1->n;
    op.h1 = dcol(*h1);
    op.t1 = dcol(*t1);
    op.t2 = dcol(*t2);
    op.reenc_h = reenc_h != 0;
    op.reenc_t = reenc_t != 0;
    op.wh = wout_h;
    op.wt = wout_t;
    op.f_h1 = f_h1;
    op.f_t2 = f_t2;
    op.mh = width_mask(wout_h);
    op.mt = width_mask(wout_t);
    op.a_oid = a_oid;
    op.out_h = out_h.data;
    op.out_t = out_t.data;
    op.out_cap = (out_h.data && out_t.data) ? (out_h.cap < out_t.cap ? out_h.cap : out_t.cap) : 0;
    const ahead_buf e[3] = {err1, err2, err4};
    for (int i = 0; i < 3; ++i) {
        op.err[i] = static_cast<uint64_t *>(e[i].data);
        op.cap[i] = e[i].data ? e[i].cap : 0;
    }
    op.d_counts = d_counts;
    if (launch_match_lean(op, h1, t1, t2, ws, static_cast<hipStream_t>(stream), &st)) return st;
    return launch_stream(StreamRows<MatchPosOp>(op), ws, static_cast<hipStream_t>(stream));
}

extern "C" int ahead_hip_arithmetic_an(const ahead_col *h1, const ahead_col *t1, const ahead_col *h2, const ahead_col *t2,
                                       int op_code, uint64_t a_result, uint32_t result_width, uint64_t a_oid, void *out,
                                       ahead_buf eh1, ahead_buf et1, ahead_buf eh2, ahead_buf et2, uint64_t *d_counts,
                                       ahead_hip_ws *ws, void *stream) {
    int st;
    if ((st = check_col(h1, "arithmetic.h1", true, false)) != AHEAD_OK) return st;
    if ((st = check_col(t1, "arithmetic.t1", false, true)) != AHEAD_OK) return st;
    if ((st = check_col(h2, "arithmetic.h2", true, false)) != AHEAD_OK) return st;
    if ((st = check_col(t2, "arithmetic.t2", false, true)) != AHEAD_OK) return st;
    if (t1->n != t2->n) return fail(AHEAD_ERR_SIZE_MISMATCH, "arithmetic: bat1->size() != bat2->size()");
    if (op_code < 0 || op_code > 3) return fail(AHEAD_ERR_INVALID, "arithmetic: op must be 0..3 (add sub mul div)");
    if (result_width != 2 && result_width != 4 && result_width != 8)
        return fail(AHEAD_ERR_INVALID, "arithmetic: result width must be 2, 4 or 8");
    if (d_counts == nullptr || (out == nullptr && t1->n)) return fail(AHEAD_ERR_INVALID, "arithmetic: NULL output");
    ArithOp op{};
    op.n = t1->n;
    op.h1 = dcol(*h1);
    op.t1 = dcol(*t1);
    op.h2 = dcol(*h2);
    op.t2 = dcol(*t2);
    op.op = op_code;
    op.a_result = a_result;
    op.rw = result_width;
    op.rmask = width_mask(result_width);
    op.a_oid = a_oid;
    op.out = out;
    const ahead_buf e[4] = {eh1, et1, eh2, et2};
    for (int i = 0; i < 4; ++i) {
        op.err[i] = static_cast<uint64_t *>(e[i].data);
        op.cap[i] = e[i].data ? e[i].cap : 0;
    }
    op.d_counts = d_counts;
    return launch_map(op, ws, 0, static_cast<hipStream_t>(stream));
}

extern "C" int ahead_hip_aggregate_mul_sum_an(const ahead_col *t1, const ahead_col *t2, uint64_t init,
                                              int result_encoded, uint64_t ra, uint64_t a_oid, uint64_t *d_total,
                                              ahead_buf err1, ahead_buf err2, uint64_t *d_counts, ahead_hip_ws *ws,
                                              void *stream) {
    int st;
    if ((st = check_col(t1, "mul_sum.t1", false, false)) != AHEAD_OK) return st;
    if ((st = check_col(t2, "mul_sum.t2", false, false)) != AHEAD_OK) return st;
    if (d_total == nullptr || d_counts == nullptr) return fail(AHEAD_ERR_INVALID, "mul_sum: NULL output");
    MulSumOp op{};
    op.n = t1->n < t2->n ? t1->n : t2->n;  // aggregateAN_scalar.tcc:91 stops at the shorter input
    op.t1 = dcol(*t1);
    op.t2 = dcol(*t2);
    op.a_oid = a_oid;
    const uint32_t waves = map_waves<MulSumOp>(op.n);  // one partial per wave of the streaming engine
    const size_t o_map = align_up(waves * 8ull, 256);
    if ((st = ws_ensure(ws, o_map + map_scratch_bytes<MulSumOp>(op.n))) != AHEAD_OK) return st;
    op.partials = reinterpret_cast<uint64_t *>(ws_region(ws, 0));
    const ahead_buf e[2] = {err1, err2};
    for (int i = 0; i < 2; ++i) {
        op.err[i] = static_cast<uint64_t *>(e[i].data);
        op.cap[i] = e[i].data ? e[i].cap : 0;
    }
    op.d_counts = d_counts;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if ((st = launch_map(op, ws, o_map, s)) != AHEAD_OK) return st;
    // aggregateAN_scalar.tcc:83-85: RA * inv(A_T1) * inv(A_T2) over 64 bits
    const uint64_t enc = (result_encoded ? ra : 1ull) * (t1->encoded ? inverse_mod2k(t1->a, 64) : 1ull) *
                         (t2->encoded ? inverse_mod2k(t2->a, 64) : 1ull);
    hipLaunchKernelGGL(k_mulsum_final, dim3(1), dim3(kBlock), 0, s, op.partials, waves, init, enc, d_total);
    AHEAD_HIP_TRY(hipGetLastError());
    return AHEAD_OK;
}

extern "C" int ahead_hip_aggregate_sum_grouped_an(const ahead_col *head, const ahead_col *tail, const ahead_col *grouping,
                                                  uint64_t num_groups, uint64_t a_result, uint64_t a_oid, uint64_t *sums,
                                                  ahead_buf e_head, ahead_buf e_tail, ahead_buf e_group,
                                                  uint64_t *d_counts, ahead_hip_ws *ws, void *stream) {
    int st;
    if ((st = check_col(head, "sum_grouped.head", true, false)) != AHEAD_OK) return st;
    if ((st = check_col(tail, "sum_grouped.tail", false, false)) != AHEAD_OK) return st;
    if ((st = check_col(grouping, "sum_grouped.grouping", false, true)) != AHEAD_OK) return st;
    if (tail->n != grouping->n) return fail(AHEAD_ERR_SIZE_MISMATCH, "bat and grouping must have the same size!");
    if (grouping->width != 8) return fail(AHEAD_ERR_INVALID, "sum_grouped: group ids are resoid (8-byte) codes");
    if (d_counts == nullptr || (sums == nullptr && num_groups)) return fail(AHEAD_ERR_INVALID, "sum_grouped: NULL output");
    AggSumArgs a{};
    a.n = tail->n;
    a.head = dcol(*head);
    a.tail = dcol(*tail);
    a.grp = dcol(*grouping);
    a.grp.max_u = grouping->max_u;
    a.num_groups = num_groups;
    // aggregateAN.tcc:74-75: A_result * inv(A_tail) mod 2^64
    a.enc = a_result * (tail->encoded ? inverse_mod2k(tail->a, 64) : 1ull);
    a.a_oid = a_oid;
    // (a group id in range is below 2^32 unless there are more groups than that)
    a.grp_back = num_groups <= 0xFFFFFFFFull ? back_factor(grouping->a_inv, 0xFFFFFFFFull) : 0u;
    a.tail_back = a.tail.encoded && a.tail.width == 8 ? back_factor(a.tail.a_inv, a.tail.max_u) : 0u;
    a.sums = sums;
    const ahead_buf e[3] = {e_head, e_tail, e_group};
    for (int i = 0; i < 3; ++i) {
        a.err[i] = static_cast<uint64_t *>(e[i].data);
        a.cap[i] = e[i].data ? e[i].cap : 0;
    }
    a.d_counts = d_counts;
    hipStream_t s = static_cast<hipStream_t>(stream);
    AggSumOp op{};
    op.n = a.n;
    size_t o_map = 0;
    if (num_groups && num_groups <= kAggLds) {
        a.copies = 1;
        while (a.copies < 32u && 2ull * a.copies * num_groups <= kAggLds) a.copies *= 2;
        a.parts = map_parts<AggSumOp>(op.n);
        o_map = align_up(num_groups * a.parts * 8ull, 256);
        if ((st = ws_ensure(ws, o_map + map_scratch_bytes<AggSumOp>(op.n))) != AHEAD_OK) return st;
        a.partials = reinterpret_cast<uint64_t *>(ws_region(ws, 0));
    } else if (num_groups) {
        hipLaunchKernelGGL(k_fill_u64, dim3(64), dim3(256), 0, s, sums, num_groups, 0ull);
        AHEAD_HIP_TRY(hipGetLastError());
    }
    op.a = a;
    if ((st = launch_map(op, ws, o_map, s)) != AHEAD_OK) return st;
    if (a.copies != 0u) {
        hipLaunchKernelGGL(k_aggsum_final, dim3(static_cast<uint32_t>((num_groups + kAggFinal - 1) / kAggFinal)), dim3(kBlock), 0,
                           s, a);
        AHEAD_HIP_TRY(hipGetLastError());
    }
    return AHEAD_OK;
}
