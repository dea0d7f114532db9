// decode_an.hip -- encodeAN, checkAN, decodeAN and checkAndDecodeAN<void,Tail> for gfx950.
//
// Semantics (lib/column_operators/AN/encdecAN_scalar.tcc):
//   encodeAN          :44-67   out[i] = (code_t)v_i * A
//   checkAN           :69-94   err += i*A_OID for every i with (c_i * A^-1 mod 2^k) > maxU
//   decodeAN          :96-126  every row decoded (truncated to the unencoded width), err as above
//   checkAndDecodeAN  :185-210 corrupt rows are dropped from the decoded output, err as above
// checkAN and decodeAN, whose outputs stay at their row, run on the streaming engine of maptile.hpp
// (DecodeMapOp); checkAndDecodeAN on the single-pass engine of stream.hpp (CheckDecodeOp).
#include "maptile.hpp"
#include "stream.hpp"

using namespace ahead_dev;

namespace {

enum Mode { kCheck = 0, kDecode = 1, kCheckDecode = 2 };

// One row of checkAN / decodeAN for the streaming engine: codes of CodeT, decoded values stored at
// the runtime width ow (the unencoded width).
template <typename CodeT, int MODE>
struct DecodeMapOp {
    static constexpr int kErr = 1;
    static constexpr bool kMulti = false, kMain = false, kAcc = false;
    static constexpr bool kBatched = true;
    using State = uint64_t;  // the decoded value
    uint64_t n;
    const CodeT *codes;
    CodeT a_inv, max_u;
    uint32_t ow;
    uint64_t a_oid;
    void *dec;
    uint64_t *err;
    uint64_t err_cap;
    uint64_t *d_counts;

    template <int G>
    __device__ void eval_n(const uint64_t (&row)[G], const bool (&live)[G], State (&st)[G], uint32_t (&errs)[G],
                           uint32_t (&cnt)[G], uint64_t &) const {
        CodeT c[G];
#pragma unroll
        for (int g = 0; g < G; ++g) c[g] = codes[live[g] ? row[g] : 0ull];  // n > 0 whenever a row is live
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const CodeT d = an_mul<CodeT>(c[g], a_inv);
            errs[g] = live[g] && d > max_u ? 1u : 0u;
            st[g] = d;
            cnt[g] = 0u;
            if (MODE == kDecode && live[g]) store_w(dec, row[g], ow, d);
        }
    }
    __device__ uint32_t eval(uint64_t row, State &st, uint32_t &errs, uint64_t &) const {
        const CodeT d = an_mul<CodeT>(codes[row], a_inv);
        errs = d > max_u ? 1u : 0u;
        st = d;
        if (MODE == kDecode) store_w(dec, row, ow, d);
        return 0u;
    }
    __device__ void emit_main(uint64_t, const State &, uint64_t, uint32_t) const {}
    __device__ void emit_err(int, uint64_t row, const State &, uint64_t pos) const {
        if (pos < err_cap) err[pos] = row * a_oid;
    }
    __device__ void tile_done(uint32_t, uint64_t) const {}
    __device__ void finish(const uint64_t *t) const {
        if (MODE == kDecode) {
            d_counts[0] = n;
            d_counts[1] = t[1];
        } else {
            d_counts[0] = t[1];
        }
    }
};

// checkAndDecodeAN on the single-pass engine.
template <typename CodeT, typename OutT>
struct CheckDecodeOp {
    static constexpr int kErr = 1;
    static constexpr int kG = sizeof(CodeT) == 2 ? 32 : 16;  // 64 bytes of codes per lane at least
    struct Raw {
        CodeT c;
    };
    using State = OutT;  // the decoded value
    uint64_t n;
    const CodeT *codes;
    CodeT a_inv, max_u;
    uint32_t back;  // 8-byte codes of values below 2^32: A (back_factor), else 0
    uint64_t a_oid;
    OutT *dec;
    uint64_t out_cap;
    uint64_t *err;
    uint64_t err_cap;
    uint64_t *d_counts;

    __device__ bool skip() const { return false; }
    struct Uniform {};
    __device__ void init(char *) const {}
    __device__ Uniform begin(const char *) const { return Uniform{}; }
    __device__ __forceinline__ void load(uint64_t first, uint32_t k, Raw &r) const {
        r.c = __builtin_nontemporal_load(codes + first + k);
    }
    template <int G>
    struct Mid {
        OutT d[G];
        uint32_t bad;
    };
    template <int G>
    __device__ __forceinline__ void open_tile(const char *, const Uniform &, uint64_t, uint32_t, uint32_t, const Raw (&raw)[G],
                                              Mid<G> &mid) const {
        mid.bad = 0;
        if (sizeof(CodeT) == 8 && back != 0u) {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const uint32_t d = static_cast<uint32_t>(raw[g].c) * static_cast<uint32_t>(a_inv);
                mid.d[g] = static_cast<OutT>(d);
                mid.bad |= (static_cast<uint64_t>(d) * back != raw[g].c || d > max_u ? 1u : 0u) << g;
            }
        } else {
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const CodeT d = an_mul<CodeT>(raw[g].c, a_inv);
                mid.d[g] = static_cast<OutT>(d);
                mid.bad |= (d > max_u ? 1u : 0u) << g;
            }
        }
    }
    template <int G>
    __device__ __forceinline__ void close_tile(const Uniform &, const Mid<G> &mid, uint32_t live, State (&st)[G], uint32_t &keep,
                                               uint32_t (&errs)[kErr]) const {
#pragma unroll
        for (int g = 0; g < G; ++g) st[g] = mid.d[g];
        keep = live & ~mid.bad;
        errs[0] = live & mid.bad;
    }
    __device__ void report(uint64_t row, State &, uint32_t &errs) const {
        errs = an_mul<CodeT>(codes[row], a_inv) > max_u ? 1u : 0u;
    }
    __device__ __forceinline__ void emit(const Uniform &, const State &st, uint64_t, uint64_t pos, uint32_t, uint32_t k) const {
        __builtin_nontemporal_store(st, dec + pos + k);
    }
    __device__ void emit_err(int, uint64_t row, const State &, uint64_t pos) const {
        if (pos < err_cap) err[pos] = row * a_oid;
    }
    __device__ void finish(const uint64_t *t) const {
        d_counts[0] = t[0];
        d_counts[1] = t[1];
    }
};

template <typename CodeT, int MODE>
int launch_map_mode(const ahead_col *col, uint64_t a_oid, void *dec, uint64_t *err, uint64_t err_cap,
                    uint64_t *d_counts, ahead_hip_ws *ws, hipStream_t s, size_t offset) {
    DecodeMapOp<CodeT, MODE> op{};
    op.n = col->n;
    op.codes = static_cast<const CodeT *>(col->data);
    op.a_inv = static_cast<CodeT>(col->a_inv);
    op.max_u = static_cast<CodeT>(col->max_u);
    op.ow = col->unenc_bits / 8;
    op.a_oid = a_oid;
    op.dec = dec;
    op.err = err;
    op.err_cap = err == nullptr ? 0 : err_cap;
    op.d_counts = d_counts;
    return ahead_host::launch_map(op, ws, offset, s);
}

template <int MODE>
int launch_map_width(const ahead_col *col, uint64_t a_oid, void *dec, uint64_t *err, uint64_t err_cap,
                     uint64_t *d_counts, ahead_hip_ws *ws, hipStream_t s, size_t offset = 0) {
    switch (col->width) {
        case 2: return launch_map_mode<uint16_t, MODE>(col, a_oid, dec, err, err_cap, d_counts, ws, s, offset);
        case 4: return launch_map_mode<uint32_t, MODE>(col, a_oid, dec, err, err_cap, d_counts, ws, s, offset);
        default: return launch_map_mode<uint64_t, MODE>(col, a_oid, dec, err, err_cap, d_counts, ws, s, offset);
    }
}

template <typename CodeT, typename OutT>
int launch_check_decode(const ahead_col *col, uint64_t a_oid, void *dec, uint64_t dec_cap, uint64_t *err,
                        uint64_t err_cap, uint64_t *d_counts, ahead_hip_ws *ws, hipStream_t s) {
    CheckDecodeOp<CodeT, OutT> op{};
    op.n = col->n;
    op.codes = static_cast<const CodeT *>(col->data);
    op.a_inv = static_cast<CodeT>(col->a_inv);
    op.max_u = static_cast<CodeT>(col->max_u);
    op.back = sizeof(CodeT) == 8 ? ahead_host::back_factor(col->a_inv, col->max_u) : 0u;
    op.a_oid = a_oid;
    op.dec = static_cast<OutT *>(dec);
    op.out_cap = dec == nullptr ? 0 : dec_cap;
    op.err = err;
    op.err_cap = err == nullptr ? 0 : err_cap;
    op.d_counts = d_counts;
    return ahead_host::launch_stream(op, ws, s);
}

template <typename CodeT>
int launch_check_decode_width(const ahead_col *col, uint64_t a_oid, void *dec, uint64_t dec_cap, uint64_t *err,
                              uint64_t err_cap, uint64_t *d_counts, ahead_hip_ws *ws, hipStream_t s) {
    switch (col->unenc_bits) {  // at most 8 * sizeof(CodeT)
        case 8: return launch_check_decode<CodeT, uint8_t>(col, a_oid, dec, dec_cap, err, err_cap, d_counts, ws, s);
        case 16: return launch_check_decode<CodeT, uint16_t>(col, a_oid, dec, dec_cap, err, err_cap, d_counts, ws, s);
        case 32:
            if constexpr (sizeof(CodeT) >= 4)
                return launch_check_decode<CodeT, uint32_t>(col, a_oid, dec, dec_cap, err, err_cap, d_counts, ws, s);
            break;
        default:
            if constexpr (sizeof(CodeT) >= 8)
                return launch_check_decode<CodeT, uint64_t>(col, a_oid, dec, dec_cap, err, err_cap, d_counts, ws, s);
            break;
    }
    return ahead_host::fail(AHEAD_ERR_INVALID, "decode: unenc_bits wider than the code");
}

int run(int mode, const ahead_col *col, uint64_t a_oid, void *dec, uint64_t dec_cap, uint64_t *err,
        uint64_t err_cap, uint64_t *d_counts, ahead_hip_ws *ws, void *stream) {
    using namespace ahead_host;
    int st = check_col(col, "decode.col", false, true);
    if (st != AHEAD_OK) return st;
    if (d_counts == nullptr) return fail(AHEAD_ERR_INVALID, "decode: d_counts is NULL");
    if (mode != kCheck && dec == nullptr && col->n) return fail(AHEAD_ERR_INVALID, "decode: NULL output");
    if (err == nullptr && err_cap) return fail(AHEAD_ERR_INVALID, "decode: NULL err with capacity");
    if (col->unenc_bits > 8 * col->width) return fail(AHEAD_ERR_INVALID, "decode: unenc_bits wider than the code");
    if (col->unenc_bits != 8 && col->unenc_bits != 16 && col->unenc_bits != 32 && col->unenc_bits != 64)
        return fail(AHEAD_ERR_INVALID, "decode: unenc_bits must be 8, 16, 32 or 64");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (mode == kCheck) return launch_map_width<kCheck>(col, a_oid, nullptr, err, err_cap, d_counts, ws, s);
    if (mode == kDecode) return launch_map_width<kDecode>(col, a_oid, dec, err, err_cap, d_counts, ws, s);
    switch (col->width) {
        case 2: return launch_check_decode_width<uint16_t>(col, a_oid, dec, dec_cap, err, err_cap, d_counts, ws, s);
        case 4: return launch_check_decode_width<uint32_t>(col, a_oid, dec, dec_cap, err, err_cap, d_counts, ws, s);
        default: return launch_check_decode_width<uint64_t>(col, a_oid, dec, dec_cap, err, err_cap, d_counts, ws, s);
    }
}

template <typename InT, typename OutT>
__global__ __launch_bounds__(256) void k_encode(const InT *in, uint64_t n, uint64_t seqbase, OutT *out, OutT a) {
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * blockDim.x;
    for (uint64_t i = blockIdx.x * static_cast<uint64_t>(blockDim.x) + threadIdx.x; i < n; i += stride) {
        const OutT v = in ? static_cast<OutT>(in[i]) : static_cast<OutT>(static_cast<uint32_t>(seqbase + i));
        out[i] = an_mul<OutT>(v, a);
    }
}

template <typename InT>
int launch_encode(const ahead_col *col, uint64_t a, uint32_t ow, void *out, hipStream_t s) {
    const uint64_t blocks = (col->n + 255) / 256;
    const dim3 g(static_cast<uint32_t>(blocks < 8192 ? blocks : 8192)), b(256);
    const InT *in = static_cast<const InT *>(col->data);
    switch (ow) {
        case 2: hipLaunchKernelGGL((k_encode<InT, uint16_t>), g, b, 0, s, in, col->n, col->seqbase, static_cast<uint16_t *>(out), static_cast<uint16_t>(a)); break;
        case 4: hipLaunchKernelGGL((k_encode<InT, uint32_t>), g, b, 0, s, in, col->n, col->seqbase, static_cast<uint32_t *>(out), static_cast<uint32_t>(a)); break;
        case 8: hipLaunchKernelGGL((k_encode<InT, uint64_t>), g, b, 0, s, in, col->n, col->seqbase, static_cast<uint64_t *>(out), a); break;
        default: return ahead_host::fail(AHEAD_ERR_INVALID, "encode: out_width must be 2, 4 or 8");
    }
    return AHEAD_OK;
}

}  // namespace

using namespace ahead_host;

namespace ahead_host {
int check_an_ws(const ahead_col *col, uint64_t a_oid, uint64_t *err, uint64_t err_cap, uint64_t *d_counts,
                ahead_hip_ws *ws, void *stream, size_t offset) {
    int st = check_col(col, "check.col", false, true);
    if (st != AHEAD_OK) return st;
    if (d_counts == nullptr) return fail(AHEAD_ERR_INVALID, "check: d_counts is NULL");
    if (err == nullptr && err_cap) return fail(AHEAD_ERR_INVALID, "check: NULL err with capacity");
    return launch_map_width<kCheck>(col, a_oid, nullptr, err, err_cap, d_counts, ws, static_cast<hipStream_t>(stream),
                                    offset);
}
size_t check_an_status_bytes(uint64_t n, uint32_t width) {
    return lb_plan(n, 4u * kBlock * (16u / width), 2).status_bytes;
}
size_t check_an_scratch_bytes(uint64_t n, uint32_t width) {
    switch (width) {
        case 2: return map_scratch_bytes<DecodeMapOp<uint16_t, kCheck>>(n);
        case 4: return map_scratch_bytes<DecodeMapOp<uint32_t, kCheck>>(n);
        default: return map_scratch_bytes<DecodeMapOp<uint64_t, kCheck>>(n);
    }
}
}  // namespace ahead_host

extern "C" int ahead_hip_check_an(const ahead_col *col, uint64_t a_oid, uint64_t *err, uint64_t err_cap,
                                  uint64_t *d_counts, ahead_hip_ws *ws, void *stream) {
    return run(kCheck, col, a_oid, nullptr, 0, err, err_cap, d_counts, ws, stream);
}

extern "C" int ahead_hip_decode_an(const ahead_col *col, uint64_t a_oid, void *dec, uint64_t *err,
                                   uint64_t err_cap, uint64_t *d_counts, ahead_hip_ws *ws, void *stream) {
    return run(kDecode, col, a_oid, dec, col ? col->n : 0, err, err_cap, d_counts, ws, stream);
}

extern "C" int ahead_hip_check_and_decode_an(const ahead_col *col, uint64_t a_oid, void *dec,
                                             uint64_t dec_cap, uint64_t *err, uint64_t err_cap,
                                             uint64_t *d_counts, ahead_hip_ws *ws, void *stream) {
    return run(kCheckDecode, col, a_oid, dec, dec_cap, err, err_cap, d_counts, ws, stream);
}

extern "C" int ahead_hip_encode_an(const ahead_col *col, uint64_t a, uint32_t out_width, void *out,
                                   void *stream) {
    int st = check_col(col, "encode.col", true, false);
    if (st != AHEAD_OK) return st;
    if (col->n == 0) return AHEAD_OK;
    if (out == nullptr) return fail(AHEAD_ERR_INVALID, "encode: NULL output");
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (col->data == nullptr) st = launch_encode<uint32_t>(col, a, out_width, out, s);
    else if (col->width == 1) st = launch_encode<uint8_t>(col, a, out_width, out, s);
    else if (col->width == 2) st = launch_encode<uint16_t>(col, a, out_width, out, s);
    else if (col->width == 4) st = launch_encode<uint32_t>(col, a, out_width, out, s);
    else st = launch_encode<uint64_t>(col, a, out_width, out, s);
    if (st != AHEAD_OK) return st;
    AHEAD_HIP_TRY(hipGetLastError());
    return AHEAD_OK;
}
