// fp32 attention (forward, dQ, dK/dV) on the bf16 matrix instruction: every fp32 operand as three bf16 parts.
//
// A value is split into the bf16 next to it, the bf16 next to what that leaves, and the rest, which is a bf16 exactly: 8
// significant bits each with signs of their own hold the 24 of an fp32 value. A product of two such values is nine products
// of parts, of which the three smallest are at most 2^-24 of the whole (2^-8 times 2^-17, twice; 5e-9 in the mean square) and are
// left out; the other six are exact in fp32 and are added in fp32 by the matrix unit, small ones first. Error of scores against
// float64, of the result's norm (in brackets v_mfma_f32_32x32x2_f32, which rounds its sum every second column): 1 column
// 3.5e-8 (4.0e-8), 4 3.2e-8 (4.9e-8), 16 3.4e-8 (8.2e-8), 64 4.6e-8 (1.4e-7). A single product is off by 1.44e-7 at most, where
// both factors are just above a power of two, and by 1.3e-7 elsewhere and on the fp32 instruction. Parts below 2^-133, the smallest bf16,
// are lost, and with them bits of values below 2^-109: rows_to_redo, UP.
//
// What bounds it: the fp32 instruction does 157 TFLOP/s, and the kernels on it (attn_f32_split.hip) stood at 105 to 130; six
// bf16 products for one take 3/8 of its clocks. Beside them stands the splitting, 5.5 vector instructions an element: a tile
// is split once, on its way into LDS, for all wavefronts of a workgroup, so a workgroup is QW x 32 rows that share tiles
// (times KW groups that take every KW-th tile, for launches with few blocks).
#include <type_traits>

#include "attn_split.h"

namespace pk {
namespace {

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LAZY_T = 6.0f;  // as in attn_split.hip: the running maximum moves when it is outgrown by 2^6

// Bits of values below 2^-109 do not count beside ordinary ones, but they show in a column that is all as small and where a large partner
// makes the product ordinary (a column of K at 2^-120 under one of Q at 2^120: dQ off by 3.6e-5). Launches that hold what the fp32
// instruction does (ALL: f32x3_takes_bwd) split everything at 2^24 times its size, at which the last bit of the smallest fp32 value is a part that
// is kept. Powers of two change no other bit and leave with factors that are there anyway: scores (2^48) with the exponent's, dP with the
// subtraction of delta, gradients (2^48) when they are stored. What leaves fp32 at that size (values from 2^104 on, products and gradients from
// 2^80) ends in results that are not finite. A multiplication an element moved and one for each of P: T 313 x 4, 16 heads of 64, backward
// 35.1 -> 36.4 us (71 on the fp32 instruction); T 2132, 8 heads of 128 278 -> 291 (394); T 241 x 10, 4 heads of 96 33.0 -> 34.1 (52); T 1037 x
// 2, 8 heads of 32 49.7 -> 51.4 (62).
template <bool ALL>
constexpr float UP = ALL ? 0x1p24f : 1.0f;
template <bool ALL>
constexpr float DOWN = 1.0f / UP<ALL>;

// A product that is not fused into the sum it enters.
__device__ inline float mul_rounded(float x, float y) {
#pragma clang fp contract(off)
    return x * y;
}

// Two fp32 values as three packed bf16 pairs, each part rounded: a part cut off leaves a rest of up to 2^-7 of the value instead of
// 2^-8, and the products left out are then up to 2^-22 of the whole (measured: 2.0e-7, rounded 5.0e-8), for as many instructions.
__device__ inline void split2(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = pack_bf16(x0, x1);
    x0 -= __uint_as_float(h << 16), x1 -= __uint_as_float(h & 0xffff0000u);
    m = pack_bf16(x0, x1);
    x0 -= __uint_as_float(m << 16), x1 -= __uint_as_float(m & 0xffff0000u);
    l = pack_bf16(x0, x1);
}

// Columns and rows as in mfma_common.h (TrMap, lds_row), so that row reads and transposing reads of one plane are both free
// of bank conflicts at 64 and 128 columns; at 32 and 96 both are in natural order.
template <int D>
__device__ constexpr int tr_src_col(int db, int u, int a) {
    if constexpr (D == 128)
        return TrMap<128>::src_col(db, u, a);
    else
        return 32 * db + 16 * u + 4 * a;
}
template <int D>
__device__ constexpr int tr_col0(int db, int qd, int g) {
    if constexpr (D == 128)
        return TrMap<128>::col0(db, qd, g);
    else
        return 32 * db + 8 * qd + 4 * g;
}
// operand of the 16 rows from row0 on (a multiple of 16), the 32 columns of block db
template <int D>
__device__ inline bf16x8 tr_operand(const uint16_t* plane, int row0, int db, int lane) {
    const int g = lane >> 5, u = (lane >> 4) & 1, j = lane & 15;
    const uint16_t* p = plane + (row0 + lds_row<D>(4 * g + (j >> 2))) * (D + 8) + tr_src_col<D>(db, u, j & 3);
    const s16x4 lo = lds_read_tr4(p), hi = lds_read_tr4(p + TR_HI_ROWS<D> * (D + 8));
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    s16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return *reinterpret_cast<bf16x8*>(&v);
}
// store_block of attn_split.h in this column order, fp32
template <int D>
__device__ inline void store_block32(void* base, int64_t row_off, int db, int g, const f32x16& acc, float sc, int dk, const TurnRow& turn = {}) {
    float* row = static_cast<float*>(base) + row_off;
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
        const int col = tr_col0<D>(db, qd, g);
        const f32x4 v = {acc[qd * 4] * sc, acc[qd * 4 + 1] * sc, acc[qd * 4 + 2] * sc, acc[qd * 4 + 3] * sc};
        if (col < dk) *reinterpret_cast<f32x4*>(row + col) = turn.quad(v, col, dk);
    }
}

// A 32-row tile of a [T, dk] fp32 matrix, moved by G threads (rows past T and chunks past dk read as zero) into three
// planes of 32 rows of pitch D + 8: 16-byte row reads then touch all banks once.
template <int D, int G, bool ALL = false>
struct Mover3 {
    static constexpr int NCH = D / 4, CPT = 32 * NCH / G, P = D + 8, PLANE = 32 * P;
    static_assert(CPT >= 1 && 32 * NCH % G == 0, "every thread moves the same number of chunks");
    int off[CPT];
    u32x4 r[CPT];
    __device__ void init(int t, int st, int dk) {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int c = t + G * i, row = c / NCH, ch = c % NCH;
            off[i] = ch * 4 < dk ? (row * st + ch * 4) * 4 : static_cast<int>(OUTSIDE);
        }
    }
    __device__ void load(const float* head, int st, int r0, int T, int dk) {
        const int64_t left = (static_cast<int64_t>(T - r0 - 1) * st + dk) * 4;  // r0 < T
        float* p = const_cast<float*>(head) + static_cast<int64_t>(r0) * st;
        const __amdgpu_buffer_rsrc_t rs =
            __builtin_amdgcn_make_buffer_rsrc(p, 0, left > 0x7fffffff ? 0x7fffffff : static_cast<int>(left), 0x00020000);
#pragma unroll
        for (int i = 0; i < CPT; ++i) r[i] = tile_load16(rs, off[i]);
    }
    __device__ void store(uint16_t* tile, int t) const {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(&r[i]);
            uint32_t h[2], m[2], l[2];
            split2(x[0] * UP<ALL>, x[1] * UP<ALL>, h[0], m[0], l[0]);
            split2(x[2] * UP<ALL>, x[3] * UP<ALL>, h[1], m[1], l[1]);
            uint16_t* p = at(tile, t, i);
            *reinterpret_cast<u32x2*>(p) = u32x2{h[0], h[1]};
            *reinterpret_cast<u32x2*>(p + PLANE) = u32x2{m[0], m[1]};
            *reinterpret_cast<u32x2*>(p + 2 * PLANE) = u32x2{l[0], l[1]};
        }
    }
    __device__ static uint16_t* at(uint16_t* tile, int t, int i) {
        const int c = t + G * i;
        return tile + lds_row<D>(c / NCH) * P + (c % NCH) * 4;
    }
};

// eight values as three operands
__device__ inline void split8(const float (&x)[8], bf16x8& h, bf16x8& m, bf16x8& l) {
    u32x4 p[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t a, b, c;
        split2(x[2 * i], x[2 * i + 1], a, b, c);
        p[0][i] = a, p[1][i] = b, p[2][i] = c;
    }
    h = *reinterpret_cast<bf16x8*>(&p[0]);
    m = *reinterpret_cast<bf16x8*>(&p[1]);
    l = *reinterpret_cast<bf16x8*>(&p[2]);
}

// Row `row` of a head, all of it on its way before any of it is split: chunk 2 kk + half holds columns 16 kk + 8 g + 4 half .. +3; zero past T and past dk.
// A chunk split, or multiplied into delta, where it is loaded waits there, a trip to memory for each of D / 8 chunks: T 241 x 10, 4 heads of 96 forward
// 18.4 -> 15.9 us; T 1037 x 2, 8 heads of 32 19.5 -> 18.7; dQ and dK/dV in one launch, T 836 x 2, 8 heads of 64 64.8 -> 58.7; long chains level.
template <int D>
struct Row {
    f32x4 x[D / 8];
    __device__ void load(const float* head, int64_t st, int row, int T, int dk, int g) {
#pragma unroll
        for (int j = 0; j < D / 8; ++j) {
            const int col = 16 * (j / 2) + 8 * g + 4 * (j % 2);
            f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
            if (row < T && col < dk) z = *reinterpret_cast<const f32x4*>(head + row * st + col);
            x[j] = z;
        }
    }
    // as three operands: chunk kk holds columns 16 kk + 8 g .. +7
    template <bool ALL = false>
    __device__ void split(bf16x8 (&out)[3][D / 16]) const {
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = x[2 * kk + e / 4][e % 4] * UP<ALL>;
            split8(v, out[0][kk], out[1][kk], out[2][kk]);
        }
    }
    // this lane's share of the product with another row
    __device__ float dot(const Row& o) const {
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < D / 8; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = fmaf(o.x[j][e], x[j][e], sum);
        return sum;
    }
};

// (rows of the tile) . b over the columns: all small products first, then the large ones on top of their sum
template <int D>
__device__ inline f32x16 dot3(const uint16_t* tile, const bf16x8 (&b)[3][D / 16], int c32, int g) {
    constexpr int P = D + 8, PLANE = 32 * P;
    const uint16_t* row = tile + lds_row<D>(c32) * P + g * 8;
    f32x16 t;
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = 0.0f;
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) {
        const bf16x8 h = lds_read8(row + kk * 16), m = lds_read8(row + PLANE + kk * 16), l = lds_read8(row + 2 * PLANE + kk * 16);
        t = mfma32(l, b[0][kk], t);
        t = mfma32(h, b[2][kk], t);
        t = mfma32(m, b[1][kk], t);
        t = mfma32(m, b[0][kk], t);
        t = mfma32(h, b[1][kk], t);
    }
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) t = mfma32(lds_read8(row + kk * 16), b[0][kk], t);
    return t;
}

// a C tile, its rows 0 .. 15 and 16 .. 31, as operands
struct Parts {
    bf16x8 h[2], m[2], l[2];
    __device__ inline explicit Parts(const f32x16& c) {
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const float x[8] = {c[8 * half], c[8 * half + 1], c[8 * half + 2], c[8 * half + 3],
                                c[8 * half + 4], c[8 * half + 5], c[8 * half + 6], c[8 * half + 7]};
            split8(x, h[half], m[half], l[half]);
        }
    }
    __device__ inline Parts() {}
};

// acc[n] += tile^T c for blocks db0 + n of the columns, c a C tile whose rows are the tile's rows. The tile's product is formed by
// itself, small products first, and added once: on the accumulator each of the twelve would be rounded at its size.
template <int D, int NB = D / 32>
__device__ inline void accumulate3(const uint16_t* tile, const Parts& c, f32x16* acc, int lane, int db0 = 0) {
    constexpr int PLANE = 32 * (D + 8);
    const auto &ch = c.h, &cm = c.m, &cl = c.l;
#pragma unroll
    for (int n = 0; n < NB; ++n) {
        const int db = min(db0 + n, D / 32 - 1);
        f32x16 t;
#pragma unroll
        for (int r = 0; r < 16; ++r) t[r] = 0.0f;
        bf16x8 h[2];
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            h[half] = tr_operand<D>(tile, 16 * half, db, lane);
            const bf16x8 m = tr_operand<D>(tile + PLANE, 16 * half, db, lane), l = tr_operand<D>(tile + 2 * PLANE, 16 * half, db, lane);
            t = mfma32(l, ch[half], t);
            t = mfma32(h[half], cl[half], t);
            t = mfma32(m, cm[half], t);
            t = mfma32(m, ch[half], t);
            t = mfma32(h[half], cm[half], t);
        }
#pragma unroll
        for (int half = 0; half < 2; ++half) t = mfma32(h[half], ch[half], t);
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[n][r] += t[r];
        if (D == 128) __builtin_amdgcn_sched_barrier(0);
    }
}

// m scale + log(l 2^-off): the logarithm of a mantissa and whole powers of two, added in 64 bits (logf of all of l and two sums
// in 32 bits, each rounded at the size of the result, had 4.2e-8 to 5.8e-8 of it as their error)
__device__ inline float log_sum(float m, float scale, float off, float l) {
    const double e = static_cast<double>(__builtin_amdgcn_frexp_expf(l)) - static_cast<double>(off);
    return static_cast<float>(static_cast<double>(m) * static_cast<double>(scale) + e * 0.69314718055994531 +
                              static_cast<double>(logf(__builtin_amdgcn_frexp_mantf(l))));
}

// ---- rows that are formed again ----
// An infinity leaves no rest (it is inf, NaN, NaN), a value past the largest bf16 rounds to one, and products with weights of up to 2^6
// or a long row's sum can leave fp32 where the mean does not. All of these end in results that are not finite, and such rows are
// formed once more from the tensors themselves, one key or query after the other as the scalar kernels do, over the visible ones only
// and with sums in 64 bits. A wavefront does this for the rows it is about to store, whose accumulators then hold them; its lanes are
// the rows of the other side, 64 at a time, and then the columns. What the test costs where it finds nothing, over 24 shapes: forward
// 1.000, dQ 1.005, dK/dV 1.013 of the time without it. Rows that are NaN end at the first 64 scores with one (T 4096 x 4, 16 heads, 64
// columns, forward 0.8 ms: 1.1 where all is NaN, 7.5 with one key that is), rows beside an infinity are walked to the end (45 to 56 ms).
//
// The last parts of values below 2^-109 are below the range of bf16. Beside others they do not count, and where everything is that
// small the results are: rows of a wavefront whose results are all below 2^-96, and not all zero, are formed again as well (not where ALL
// of fp32's range is split without loss).

// The kernel's arguments (AttnArgs is the first of them), read from memory where this is called: as the ones that the kernel has read
// they would be held in scalar registers through its loop, which spilled 50 of them in dK/dV.
__device__ inline AttnArgs arguments_again() {
    uint64_t at = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(at));
    return *(const AttnArgs*)(const __attribute__((address_space(4))) void*)at;
}
// The lane once more, without a register that holds it through the loop
__device__ inline int lane_again() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }
// Bit r: row r (a lane of either half each) is one of those. ok: the lane's row exists and is stored; NB blocks, of which this
// wavefront has every `step`-th from `first` on; sc: the factor they are stored with, or a power of two or so from it.
template <int NB, bool ALL = false>
__device__ inline uint32_t rows_to_redo(const f32x16* acc, float sc, bool ok, int first = 0, int step = 1) {
    float z[4] = {0.0f, 0.0f, 0.0f, 0.0f}, top[4] = {0.0f, 0.0f, 0.0f, 0.0f};  // z stays 0 under finite values
#pragma unroll
    for (int n = 0; n < NB; ++n)
        if (step == 1 || n % step == first)
#pragma unroll
            for (int r = 0; r < 16; ++r) z[r & 3] = fmaf(acc[n][r], 0.0f, z[r & 3]), top[r & 3] = fmaxf(top[r & 3], fabsf(acc[n][r]));
    const float t = fmaxf(fmaxf(top[0], top[1]), fmaxf(top[2], top[3]));
    uint64_t lanes = __ballot(ok && !((z[0] + z[1]) + (z[2] + z[3]) == 0.0f));
    if (!ALL && __ballot(ok && t * sc >= 0x1p-96f) == 0) lanes |= __ballot(ok && t > 0.0f);
    return static_cast<uint32_t>(lanes | lanes >> 32);
}
__device__ inline float dot_exact(const float* x, const float* y, int dk) {
    double sum = 0.0;
#pragma unroll 4
    for (int c = 0; c < dk; c += 4) {
        const f32x4 u = *reinterpret_cast<const f32x4*>(x + c), v = *reinterpret_cast<const f32x4*>(y + c);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum += static_cast<double>(u[e]) * static_cast<double>(v[e]);
    }
    return static_cast<float>(sum);
}
// sum[0], sum[1] += weight(i) rows[i][lane], rows[i][lane + 64] over i in [i0, i1), 64 weights at a time, one to a lane, and eight rows in
// flight; weight(i, w) is false for an i that has none. False, with sums of NaN, at the first weights of which one is NaN.
template <class Weight>
__device__ inline bool add_weighted_rows(int i0, int i1, const float* rows, int64_t st, int dk, int lane, double (&sum)[2], Weight weight) {
    const int c0 = min(lane, dk - 1), c1 = min(lane + 64, dk - 1);  // columns past the last one read it again
#pragma unroll 1
    for (int base = i0; base < i1; base += 64) {
        float w = 0.0f;
        const bool has = base + lane < i1 && weight(base + lane, w);
        if (__any(has && w != w)) {
            sum[0] = sum[1] = __builtin_nan("");
            return false;
        }
        const uint64_t mask = __ballot(has);
#pragma unroll 1
        for (int k = 0; k < 64; k += 8) {
            if ((mask >> k & 0xff) == 0) continue;
            float x0[8], x1[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float* row = rows + min(base + k + e, i1 - 1) * st;
                x0[e] = row[c0], x1[e] = row[c1];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if ((mask >> (k + e) & 1) == 0) continue;
                const double x = static_cast<double>(__uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), k + e)));
                sum[0] += x * static_cast<double>(x0[e]);
                sum[1] += x * static_cast<double>(x1[e]);
            }
        }
    }
    return true;
}
// Where a wavefront's row crosses LDS: the end of the kernel's, past the RED elements in which groups may still be joining their sums
template <int D, int WAVES, int RED, int N>
__device__ inline float* row_room(uint16_t (&lds)[N], int w) {
    static_assert(N >= RED + 2 * WAVES * D, "room for a row a wavefront");
    return reinterpret_cast<float*>(lds + N - 2 * WAVES * D) + w * D;
}
// A row of results, column by lane, into accumulators whose row it is
template <int D, int NB>
__device__ inline void put_row(float* buf, const double (&x)[2], int row, f32x16* acc, int lane, int db0 = 0) {
    const int g = lane >> 5, c32 = lane & 31;
    if (lane < D) buf[lane] = static_cast<float>(x[0]);
    if (lane + 64 < D) buf[lane + 64] = static_cast<float>(x[1]);
    tile_barrier<1>();
    if (c32 == row) {
#pragma unroll
        for (int n = 0; n < NB; ++n) {
            if (db0 + n >= D / 32) continue;
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[n][r] = buf[tr_col0<D>(db0 + n, r >> 2, g) + (r & 3)];
        }
    }
    tile_barrier<1>();
}
// O and LSE of query qi
__device__ inline void exact_o(const AttnArgs& a, int b, int h, int hk, int qi, int lane, double (&o)[2], float& lse) {
    const float* q = static_cast<const float*>(a.q) + b * a.q_sb + h * a.q_sh + qi * a.q_st;
    const float* k = static_cast<const float*>(a.k) + b * a.k_sb + hk * a.k_sh;
    const float* v = static_cast<const float*>(a.v) + b * a.v_sb + hk * a.v_sh;
    const int end = a.causal ? qi + 1 : a.T;
    const auto visible = [&](int kj) { return pk_visible(qi, kj, a.T, a.causal, a.window, a.sinks); };
    float m = -1e30f;
    bool nan = false;
#pragma unroll 1
    for (int base = 0; base < end && !nan; base += 64) {
        float s = -INFINITY;
        if (base + lane < end && visible(base + lane)) s = dot_exact(q, k + (base + lane) * a.k_st, a.dk_dim);
        nan = __any(s != s);
        m = fmaxf(m, s);
    }
    if (nan) {
        o[0] = o[1] = lse = __builtin_nanf("");
        return;
    }
#pragma unroll
    for (int i = 32; i >= 1; i >>= 1) m = fmaxf(m, __shfl_xor(m, i));
    double l = 0.0;
    o[0] = o[1] = 0.0;
    add_weighted_rows(0, end, v, a.v_st, a.dk_dim, lane, o, [&](int kj, float& w) {
        if (!visible(kj)) return false;
        w = __builtin_amdgcn_exp2f((dot_exact(q, k + kj * a.k_st, a.dk_dim) - m) * (a.scale * LOG2E));
        l += static_cast<double>(w);
        return true;
    });
#pragma unroll
    for (int i = 32; i >= 1; i >>= 1) l += __shfl_xor(l, i);
    o[0] /= l, o[1] /= l;
    lse = log_sum(m, a.scale, 0.0f, static_cast<float>(l));
}
// dQ of query qi without its factor `scale`
__device__ inline void exact_dq(const AttnArgs& a, int b, int h, int hk, int qi, float delta, int lane, double (&dq)[2]) {
    const float* q = static_cast<const float*>(a.q) + b * a.q_sb + h * a.q_sh + qi * a.q_st;
    const float* d_o = static_cast<const float*>(a.d_o) + b * a.do_sb + h * a.do_sh + qi * a.do_st;
    const float* k = static_cast<const float*>(a.k) + b * a.k_sb + hk * a.k_sh;
    const float* v = static_cast<const float*>(a.v) + b * a.v_sb + hk * a.v_sh;
    const int64_t lrow = (static_cast<int64_t>(b) * a.Hq + h) * a.T + qi;
    const float nlse = -a.lse[lrow] * LOG2E;
    dq[0] = dq[1] = 0.0;
    add_weighted_rows(0, a.causal ? qi + 1 : a.T, k, a.k_st, a.dk_dim, lane, dq, [&](int kj, float& w) {
        if (!pk_visible(qi, kj, a.T, a.causal, a.window, a.sinks)) return false;
        const float p = __builtin_amdgcn_exp2f(fmaf(dot_exact(q, k + kj * a.k_st, a.dk_dim), a.scale * LOG2E, nlse));
        w = p * (dot_exact(d_o, v + kj * a.v_st, a.dk_dim) - delta);
        return true;
    });
}
// dV (key_grad false) or dK without its factor `scale` of key kj, over queries [q0, q1) of heads [h0, h0 + nh)
__device__ inline void exact_dkdv(const AttnArgs& a, bool key_grad, int b, int hk, int h0, int nh, int q0, int q1, int kj, int lane, double (&out)[2]) {
    const float* k = static_cast<const float*>(a.k) + b * a.k_sb + hk * a.k_sh + kj * a.k_st;
    const float* v = static_cast<const float*>(a.v) + b * a.v_sb + hk * a.v_sh + kj * a.v_st;
    out[0] = out[1] = 0.0;
    bool more = true;
    for (int h = h0; h < h0 + nh && more; ++h) {
        const float* q = static_cast<const float*>(a.q) + b * a.q_sb + h * a.q_sh;
        const float* d_o = static_cast<const float*>(a.d_o) + b * a.do_sb + h * a.do_sh;
        const int64_t lrow = (static_cast<int64_t>(b) * a.Hq + h) * a.T;
        more = add_weighted_rows(q0, q1, key_grad ? q : d_o, key_grad ? a.q_st : a.do_st, a.dk_dim, lane, out, [&](int qi, float& w) {
            if (!pk_visible(qi, kj, a.T, a.causal, a.window, a.sinks)) return false;
            w = __builtin_amdgcn_exp2f(fmaf(dot_exact(q + qi * a.q_st, k, a.dk_dim), a.scale * LOG2E, -a.lse[lrow + qi] * LOG2E));
            if (key_grad) w *= dot_exact(d_o + qi * a.do_st, v, a.dk_dim) - a.delta[lrow + qi];
            return true;
        });
    }
}

// Tile buffers: two and one barrier a tile where a workgroup is one group, one and two barriers where two groups share the LDS.
template <int D, int QW, int KW>
constexpr int BUFS = KW == 1 && (D < 128 || QW > 4) ? 2 : 1;

// ---- forward: QW groups of 32 queries x KW groups of 32-key tiles ----
template <int D, int QW, int KW>
__global__ __launch_bounds__(64 * QW * KW, 2) void x3_fwd(AttnArgs a) {
    if (KW > 1) all_arguments(a);
    constexpr int BM = 32 * QW, DB = D / 32, G = 64 * QW, NBUF = BUFS<D, QW, KW>;
    constexpr int PLANE = Mover3<D, G>::PLANE, TILE = 6 * PLANE;
    constexpr int RED = KW > 1 ? QW * KW * (DB * 1024 + 128) * 2 : 0;  // in uint16
    __shared__ __attribute__((aligned(16))) uint16_t lds[NBUF * KW * TILE > RED ? NBUF * KW * TILE : RED];

    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = w / QW, qg = w % QW, gt = static_cast<int>(threadIdx.x) - kg * G;
    const int g = lane >> 5, c32 = lane & 31, dk = a.dk_dim;
    int b, h, hk, qblk;
    if (!map_query_block(a, (a.T + BM - 1) / BM, b, h, hk, qblk)) return;
    const int q0 = qblk * BM, qlo = q0 + qg * 32, qhi = qlo + 31, qi = qlo + c32;
    // plain addresses, as in split_fwd (us, with head_of | so: 128 columns, T 3473, 8 heads 241 | 231; T 492 x 33, 2 heads 62.4 | 59.4; 64, T 300 x 16, 8
    // heads 21.7 | 19.9; T 1024 x 4 40.8 | 40.2)
    const float *const kh = static_cast<const float*>(a.k) + (b * a.k_sb + hk * a.k_sh), *const vh = static_cast<const float*>(a.v) + (b * a.v_sb + hk * a.v_sh),
                *const qh = static_cast<const float*>(a.q) + (b * a.q_sb + h * a.q_sh);
    const int k_st = static_cast<int>(a.k_st), v_st = static_cast<int>(a.v_st);
    const float cexp = a.scale * LOG2E;

    Mover3<D, G> mk, mv;
    mk.init(gt, k_st, dk);
    mv.init(gt, v_st, dk);
    const KeyTiles kt(a, q0, BM, 32);
    const int iters = (kt.n + KW - 1) / KW;
    auto fetch = [&](int i) {  // this group's i-th tile (past its last: nothing)
        const int at = i * KW + kg;
        if (at < kt.n) {
            mk.load(kh, k_st, kt.tile(at) * 32, a.T, dk);
            mv.load(vh, v_st, kt.tile(at) * 32, a.T, dk);
        }
    };
    auto commit = [&](int i) {
        uint16_t* t = lds + (i % NBUF * KW + kg) * TILE;
        if (i * KW + kg < kt.n) mk.store(t, gt), mv.store(t + 3 * PLANE, gt);
    };
    fetch(0);
    bf16x8 qreg[3][D / 16];
    {
        Row<D> q;
        q.load(qh, a.q_st, qi, a.T, dk, g);
        q.split(qreg);
    }
    f32x16 acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;
    double lsum = 0.0;  // a sequence of tiles is a long chain of additions
    float m = -1e30f, mc = mul_rounded(m, cexp);  // the reference's running-max seed, src/ops.cpp:881; and m cexp as P is formed against it
    const QueryVis vis(qi, a.T, a.causal, a.window, a.sinks);
    commit(0);
    __syncthreads();

    for (int i = 0; i < iters; ++i) {
        if (i + 1 < iters) fetch(i + 1);  // in flight during the math
        const int at = i * KW + kg;
        const uint16_t* Ks = lds + (i % NBUF * KW + kg) * TILE;
        const int k0 = at < kt.n ? kt.tile(at) * 32 : a.T;
        // wavefront-uniform: is anything of this 32 x 32 block visible?
        if (k0 < a.T && qlo < a.T && !(a.causal && k0 > qhi) && !(a.window > 0 && k0 + 31 + a.window <= qlo && k0 >= a.sinks)) {
            f32x16 s = dot3<D>(Ks, qreg, c32, g);
            const MaskKind kind = mask_kind(k0, k0 + 31, qlo, qhi, a.T, a.causal, a.window, a.sinks);
            if (kind != MaskKind::NONE) mask_block(s, kind, vis, k0 + g * 4, -INFINITY);
            float mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
            mx = xhalf_max(mx);
            if (__any((mx - m) * cexp > LAZY_T)) {  // wavefront-uniform, rare after the first tiles
                const float mn = fmaxf(m, mx), mcn = mul_rounded(mn, cexp), alpha = __builtin_amdgcn_exp2f(mc - mcn);
                lsum *= static_cast<double>(alpha);
                m = mn, mc = mcn;
#pragma unroll
                for (int db = 0; db < DB; ++db)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
            }
            float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], cexp, -mc));
                ps[r & 3] += s[r];
            }
            lsum += static_cast<double>((ps[0] + ps[1]) + (ps[2] + ps[3]));  // per-lane partial; the two halves meet below
            accumulate3<D>(Ks + 3 * PLANE, Parts(s), acc, lane);
        }
        if (NBUF == 1) __syncthreads();
        if (i + 1 < iters) commit(i + 1);  // two buffers: last read one iteration ago, before the previous barrier
        __syncthreads();
    }

    const int le = lane_again(), ge = le >> 5, ce = le & 31, qe = qlo + ce;
    float l = xhalf_sum(static_cast<float>(lsum));
    float off = fmaf(m, cexp, -mc);  // what the rounding of mc left out
    if (KW > 1) {
        // the groups' running maxima and sums meet, then their accumulators scaled to the common maximum
        float* red = reinterpret_cast<float*>(lds) + qg * KW * (DB * 1024 + 128);
        float* ml = red + KW * DB * 1024;
        ml[kg * 128 + le] = m;
        ml[kg * 128 + 64 + le] = l;
        __syncthreads();
        float mt = m, lt = 0.0f;
#pragma unroll
        for (int k = 0; k < KW; ++k) mt = fmaxf(mt, ml[k * 128 + le]);
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const float mk = ml[k * 128 + le];
            lt += ml[k * 128 + 64 + le] * __builtin_amdgcn_exp2f(fmaf(mk - mt, cexp, -fmaf(mk, cexp, -mul_rounded(mk, cexp))));
        }
        const float alpha = __builtin_amdgcn_exp2f(fmaf(m - mt, cexp, -off));
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
        join_groups<DB, KW>(acc, red, kg, le);
        m = mt, l = lt, off = 0.0f;
    }
    float inv = 1.0f / l, lse = log_sum(m, a.scale, off, l);
    for (uint32_t again = rows_to_redo<DB>(acc, inv, qe < a.T, kg, KW); __builtin_expect(again != 0, 0); again &= again - 1) {
        const int row = __builtin_ctz(again);
        double x[2];
        float row_lse;
        exact_o(arguments_again(), b, h, hk, qlo + row, le, x, row_lse);
        put_row<D, DB>(row_room<D, QW * KW, RED>(lds, w), x, row, acc, le);
        if (ce == row) inv = 1.0f, lse = row_lse;
    }
    if (a.in_place) __syncthreads();  // every row has been read
    if (qe < a.T) {
        const int64_t ro = b * a.o_sb + h * a.o_sh + qe * a.o_st;
#pragma unroll
        for (int db = 0; db < DB; ++db)
            if (KW == 1 || db % KW == kg) store_block32<D>(a.o, ro, db, ge, acc[db], inv, dk);
        if (ge == 0 && kg == 0) a.lse[(static_cast<int64_t>(b) * a.Hq + h) * a.T + qe] = lse;
    }
}

// ---- dQ (and delta, when asked for with it): the same blocks ----
template <int D, int QW, int KW>
constexpr int dq_lds() {  // in uint16
    constexpr int TILES = BUFS<D, QW, KW> * KW * 6 * Mover3<D, 64 * QW>::PLANE, RED = KW > 1 ? QW * KW * (D / 32) * 2048 : 0;
    return TILES > RED ? TILES : RED;
}
template <int D, int QW, int KW, bool ALL, bool TURN, int N>
__device__ inline void dq_block(const AttnArgs& a, int fuse_delta, int b, int h, int hk, int qblk, uint16_t (&lds)[N]) {
    constexpr int BM = 32 * QW, DB = D / 32, G = 64 * QW, NBUF = BUFS<D, QW, KW>;
    constexpr int PLANE = Mover3<D, G>::PLANE, TILE = 6 * PLANE;
    constexpr int RED = KW > 1 ? QW * KW * DB * 2048 : 0;  // in uint16

    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = w / QW, qg = w % QW, gt = static_cast<int>(threadIdx.x) - kg * G;
    const int g = lane >> 5, c32 = lane & 31, dk = a.dk_dim;
    const int q0 = qblk * BM, qlo = q0 + qg * 32, qhi = qlo + 31, qi = qlo + c32;
    const float *const kh = head_of<float>(a.k, a.k_sb, b, a.k_sh, hk), *const vh = head_of<float>(a.v, a.v_sb, b, a.v_sh, hk),
                *const qh = head_of<float>(a.q, a.q_sb, b, a.q_sh, h);
    const int k_st = static_cast<int>(a.k_st), v_st = static_cast<int>(a.v_st);
    const float cexp = a.scale * LOG2E * (DOWN<ALL> * DOWN<ALL>);

    Mover3<D, G, ALL> mk, mv;
    mk.init(gt, k_st, dk);
    mv.init(gt, v_st, dk);
    const KeyTiles kt(a, q0, BM, 32);
    const int iters = (kt.n + KW - 1) / KW;
    auto fetch = [&](int i) {
        const int at = i * KW + kg;
        if (at < kt.n) {
            mk.load(kh, k_st, kt.tile(at) * 32, a.T, dk);
            mv.load(vh, v_st, kt.tile(at) * 32, a.T, dk);
        }
    };
    auto commit = [&](int i) {
        uint16_t* t = lds + (i % NBUF * KW + kg) * TILE;
        if (i * KW + kg < kt.n) mk.store(t, gt), mv.store(t + 3 * PLANE, gt);
    };
    fetch(0);
    bf16x8 qreg[3][D / 16], greg[3][D / 16];
    const int64_t lrow = (static_cast<int64_t>(b) * a.Hq + h) * a.T + min(qi, a.T - 1);
    float dl = 0.0f;
    const float lse = a.lse[lrow];
    {
        Row<D> q, d_o;
        q.load(qh, a.q_st, qi, a.T, dk, g);
        d_o.load(head_of<float>(a.d_o, a.do_sb, b, a.do_sh, h), a.do_st, qi, a.T, dk, g);
        if (fuse_delta) {
            Row<D> o;
            o.load(head_of<float>(a.o, a.o_sb, b, a.o_sh, h), a.o_st, qi, a.T, dk, g);
            dl = xhalf_sum(d_o.dot(o));
            if (qi < a.T && g == 0 && kg == 0) a.delta[lrow] = dl;
        } else {
            dl = a.delta[lrow];
        }
        q.template split<ALL>(qreg);
        d_o.template split<ALL>(greg);
    }
    const float nlse = -lse * LOG2E, dl_up = dl * UP<ALL>;
    const QueryVis vis(qi, a.T, a.causal, a.window, a.sinks);
    f32x16 acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;
    commit(0);
    __syncthreads();

    for (int i = 0; i < iters; ++i) {
        if (i + 1 < iters) fetch(i + 1);
        const int at = i * KW + kg;
        const uint16_t* Ks = lds + (i % NBUF * KW + kg) * TILE;
        const int k0 = at < kt.n ? kt.tile(at) * 32 : a.T;
        if (k0 < a.T && qlo < a.T && !(a.causal && k0 > qhi) && !(a.window > 0 && k0 + 31 + a.window <= qlo && k0 >= a.sinks)) {
            f32x16 s = dot3<D>(Ks, qreg, c32, g);
            const f32x16 dp = dot3<D>(Ks + 3 * PLANE, greg, c32, g);
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], cexp, nlse)) * fmaf(dp[r], DOWN<ALL>, -dl_up);
            const MaskKind kind = mask_kind(k0, k0 + 31, qlo, qhi, a.T, a.causal, a.window, a.sinks);
            if (kind != MaskKind::NONE) mask_block(s, kind, vis, k0 + g * 4, 0.0f);
            accumulate3<D>(Ks, Parts(s), acc, lane);
        }
        if (NBUF == 1) __syncthreads();
        if (i + 1 < iters) commit(i + 1);
        __syncthreads();
    }
    const int le = lane_again(), ge = le >> 5, qe = qlo + (le & 31);
    join_groups<DB, KW>(acc, reinterpret_cast<float*>(lds) + qg * KW * DB * 1024, kg, le);
    float sc = a.scale * (DOWN<ALL> * DOWN<ALL>);
    for (uint32_t again = rows_to_redo<DB, ALL>(acc, 1.0f, qe < a.T, kg, KW); __builtin_expect(again != 0, 0); again &= again - 1) {
        const int row = __builtin_ctz(again);
        double x[2];
        // (of ALL, delta is as it is only in memory)
        exact_dq(arguments_again(), b, h, hk, qlo + row, ALL ? a.delta[(static_cast<int64_t>(b) * a.Hq + h) * a.T + qlo + row] : __shfl(dl, row), le, x);
        put_row<D, DB>(row_room<D, QW * KW, RED>(lds, w), x, row, acc, le);
        if (ALL && (le & 31) == row) sc = a.scale;
    }
    if (a.in_place) __syncthreads();  // every row has been read
    if (qe < a.T) {
        const int64_t ro = b * a.dq_sb + h * a.dq_sh + qe * a.dq_st;
#pragma unroll
        for (int db = 0; db < DB; ++db)
            if (KW == 1 || db % KW == kg) store_block32<D>(a.dq, ro, db, ge, acc[db], sc, dk, turn_row<TURN>(a, h, qe));
    }
}
template <int D, int QW, int KW>
__global__ __launch_bounds__(64 * QW * KW, D <= 64 ? 2 : 1) void x3_dq(AttnArgs a, int fuse_delta) {
    all_arguments(a);
    __shared__ __attribute__((aligned(16))) uint16_t lds[dq_lds<D, QW, KW>()];
    int b, h, hk, qblk;
    if (map_query_block(a, (a.T + 32 * QW - 1) / (32 * QW), b, h, hk, qblk)) dq_block<D, QW, KW, false, false>(a, fuse_delta, b, h, hk, qblk, lds);
}

// The two products of a step that need no other go to two sets of wavefronts, as in the other dK/dV kernels: with both
// sides' resident rows and both accumulators one wavefront needs 320 registers at 128 columns before it has begun. A C
// tile crosses LDS in fp32, lane by lane as it lies in registers.
__device__ inline void put_tile(float* buf, const f32x16& t, int lane) {
#pragma unroll
    for (int qd = 0; qd < 4; ++qd)
        *reinterpret_cast<f32x4*>(buf + qd * 256 + lane * 4) = f32x4{t[qd * 4], t[qd * 4 + 1], t[qd * 4 + 2], t[qd * 4 + 3]};
}
__device__ inline f32x16 get_tile(const float* buf, int lane) {
    f32x16 t;
#pragma unroll
    for (int qd = 0; qd < 4; ++qd) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(buf + qd * 256 + lane * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) t[qd * 4 + e] = v[e];
    }
    return t;
}

// ---- dK, dV: QW groups of 32 keys, the query tiles of every query head of the group in turn ----
// A step is two phases. First: role 0 S = Q K^T and P, role 1 dP = dO V^T. Then, P handed over: role 0 dV^T += dO^T P, role 1 dS =
// P (dP - delta) and dK^T += Q^T dS. Each moves half of the next tile into LDS, role 1 ahead of its first product and role 0
// behind its second, so that one splits while the other multiplies: in a SIMD a matrix instruction leaves room for four others, and
// the loop has six of them for each (T 4096 x 2, 16 heads, head_dim 96, us: 1005 -> 968; head_dim 64, window 256, 4 KV heads, T
// 4096 x 4: 337 -> 323). At 128 columns there is one wavefront to a SIMD and both do it at the end of the first phase (1777; 1872).
template <int D, int QW>
constexpr int DKDV_TILE = 6 * Mover3<D, 64 * QW>::PLANE + 128;  // in uint16; LSE and delta of a tile's rows behind it
template <int D, int QW, bool ALL, bool TURN, int N>
__device__ inline void dkdv_block(const AttnArgs& a, int blk, int rr, int kvu, uint16_t (&lds)[N], float* pbuf) {
    constexpr int BNK = 32 * QW, DB = D / 32, G = 64 * QW;
    constexpr bool APART = D < 128;
    constexpr int PLANE = Mover3<D, G>::PLANE, TILE = DKDV_TILE<D, QW>;

    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int role = w / QW, qg = w % QW, gt = static_cast<int>(threadIdx.x) & (G - 1);
    const int g = lane >> 5, c32 = lane & 31, dk = a.dk_dim, rep = quotient(a.Hq, a.Hkv);
    const int nkb = (a.T + BNK - 1) / BNK;
    const int hs = a.head_split;  // > 1: this workgroup takes heads [h0, h0 + nh) of the group, see gqa_head_split
    // the sink keys' queries past their block's band go to workgroups of their own, blocks nkb .. nkb + nch - 1
    const SinkTail tl = a.tail ? sink_tail(a.T, a.window, a.sinks) : SinkTail{0, 0};
    const int chunk = blk - nkb;  // >= 0: a piece of the tail, for all query heads of the group
    if (chunk >= 0 && rr > 0) return;
    const int b = quotient(kvu, a.Hkv), hk = kvu - b * a.Hkv, h0 = chunk >= 0 ? 0 : quotient(rr * rep, hs), nh = chunk >= 0 ? rep : quotient((rr + 1) * rep, hs) - h0;
    const int k0 = chunk >= 0 ? 0 : blk * BNK, kw0 = k0 + qg * 32, kj = kw0 + c32;
    const float cexp = a.scale * LOG2E * (DOWN<ALL> * DOWN<ALL>);

    // query tiles that can see keys [k0, k0 + BNK) (paperkiln src/ops.cpp:960-965 inverted)
    const int khi = min(k0 + BNK, a.T) - 1;
    const int qt_lo = chunk >= 0 ? (tl.q0 + chunk * TAIL_CHUNK) / 32 : a.causal ? k0 / 32 : 0;
    const int q_end = chunk >= 0 ? min(a.T, tl.q0 + (chunk + 1) * TAIL_CHUNK) - 1
                      : tl.nch > 0 && k0 == 0 ? tl.q0 - 1
                      : a.window > 0 && k0 >= a.sinks ? min(a.T - 1, khi + a.window - 1) : a.T - 1;
    const int qt_hi = q_end / 32;
    const int nqt = qt_hi - qt_lo + 1, steps = nqt * nh;

    // role 0 moves Q and the rows' LSE, role 1 dO and their delta
    const int64_t s_sh = role == 0 ? a.q_sh : a.do_sh;
    const int s_st = static_cast<int>(role == 0 ? a.q_st : a.do_st);
    const float* const src = head_of<float>(role == 0 ? a.q : a.d_o, role == 0 ? a.q_sb : a.do_sb, b, s_sh, hk * rep + h0);  // the first query head's
    const float* const src_rows = role == 0 ? a.lse : a.delta;
    const float row_sc = role == 0 ? -LOG2E : UP<ALL>;
    Mover3<D, G, ALL> mv;
    mv.init(gt, s_st, dk);
    float row_r = 0.0f;
    int f_h = 0, f_t = 0;  // the (head, tile) of the next fetch
    auto fetch = [&]() {
        const int r0 = (qt_lo + f_t) * 32;
        mv.load(src + f_h * s_sh, s_st, r0, a.T, dk);
        if (gt < 32) row_r = src_rows[(static_cast<int64_t>(b) * a.Hq + hk * rep + h0 + f_h) * a.T + min(r0 + gt, a.T - 1)];  // rows past the end are masked
        if (++f_t == nqt) f_t = 0, ++f_h;
    };
    auto commit = [&](int i) {
        uint16_t* t = lds + (i & 1) * TILE;
        mv.store(t + role * 3 * PLANE, gt);
        if (gt < 32) reinterpret_cast<float*>(t + 6 * PLANE)[role * 32 + gt] = row_r * row_sc;
    };
    fetch();
    bf16x8 res[3][D / 16];  // K rows for role 0, V rows for role 1
    {
        Row<D> kv;
        kv.load(head_of<float>(role == 0 ? a.k : a.v, role == 0 ? a.k_sb : a.v_sb, b, role == 0 ? a.k_sh : a.v_sh, hk), role == 0 ? a.k_st : a.v_st, kj, a.T, dk, g);
        kv.template split<ALL>(res);
    }
    f32x16 acc[DB];  // dV^T, dK^T
#pragma unroll
    for (int n = 0; n < DB; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[n][r] = 0.0f;
    const KeyVis kvis(kj, a.T, a.causal, a.window, a.sinks);
    commit(0);
    if (steps > 1) fetch();
    __syncthreads();

    float* const pb = pbuf + qg * 1024;
    // one loop for each role: with the role tested inside, every step moves the accumulators at the join
    const auto loop = [&](auto role_c) {
        constexpr int ROLE = decltype(role_c)::value;
        int c_t = 0;
        for (int i = 0; i < steps; ++i) {
            const uint16_t* Qs = lds + (i & 1) * TILE;
            const uint16_t* Gs = Qs + 3 * PLANE;
            const float* rows = reinterpret_cast<const float*>(Qs + 6 * PLANE);
            const int qlo = (qt_lo + c_t) * 32, qhi = qlo + 31;
            if (++c_t == nqt) c_t = 0;
            // wavefront-uniform, the same for both roles: is anything of this 32 x 32 block visible?
            const bool live = qlo < a.T && kw0 < a.T && !(a.causal && kw0 > qhi) && !(a.window > 0 && kw0 + 31 + a.window <= qlo && kw0 >= a.sinks);
            // the other buffer was last read one step ago, before the previous barrier
            const auto stage = [&]() {
                if (i + 1 < steps) {
                    commit(i + 1);
                    if (i + 2 < steps) fetch();
                }
            };
            if (ROLE == 1 && APART) stage();
            f32x16 t;
            Parts parts;
            if (live) t = dot3<D>(ROLE == 0 ? Qs : Gs, res, c32, g);
            if (ROLE == 0 && live) {
                // lane = key kj; element r = query qlo + (r/4)*8 + 4g + r%4
#pragma unroll
                for (int qd = 0; qd < 4; ++qd) {
                    const f32x4 nl = *reinterpret_cast<const f32x4*>(rows + qd * 8 + g * 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) t[qd * 4 + e] = __builtin_amdgcn_exp2f(fmaf(t[qd * 4 + e], cexp, nl[e]));
                }
                const bool full = qhi < a.T && kw0 + 31 < a.T && (!a.causal || kw0 + 31 <= qlo) &&
                                  (a.window == 0 || kw0 + a.window > qhi || kw0 + 31 < a.sinks);
                if (!full) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) t[r] = kvis(qlo + (r >> 2) * 8 + g * 4 + (r & 3)) ? t[r] : 0.0f;
                }
                put_tile(pb, t, lane);
#pragma unroll
                for (int r = 0; r < 16; ++r) t[r] *= UP<ALL>;
                if (APART) parts = Parts(t);
            }
            if (!APART) stage();
            __syncthreads();
            if (ROLE == 1 && live) {
                const f32x16 p = get_tile(pb, lane);
#pragma unroll
                for (int qd = 0; qd < 4; ++qd) {
                    const f32x4 dl = *reinterpret_cast<const f32x4*>(rows + 32 + qd * 8 + g * 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) t[qd * 4 + e] = p[qd * 4 + e] * fmaf(t[qd * 4 + e], DOWN<ALL>, -dl[e]);
                }
            }
            if (live && (ROLE == 1 || !APART)) parts = Parts(t);
            if (live) accumulate3<D>(ROLE == 0 ? Gs : Qs, parts, acc, lane);
            if (ROLE == 0 && APART) stage();
            __syncthreads();
        }
    };
    if (role == 0)
        loop(std::integral_constant<int, 0>{});
    else
        loop(std::integral_constant<int, 1>{});
    // partial rows: the sink keys' of a split tail (and, unless the group's heads are split too, of the block's own band) go to
    // tail[unit][piece][dK | dV][32][dk], the others of a split group to part[unit][split][dK | dV][T][dk]
    const bool to_tail = tl.nch > 0 && k0 == 0 && kj < a.sinks && (chunk >= 0 || hs == 1), stored = kj < a.T && (chunk < 0 || to_tail);
    float sc = (role == 0 ? 1.0f : a.scale) * (DOWN<ALL> * DOWN<ALL>);
    for (uint32_t again = rows_to_redo<DB, ALL>(acc, 1.0f, stored); __builtin_expect(again != 0, 0); again &= again - 1) {
        const int row = __builtin_ctz(again);
        double x[2];
        exact_dkdv(arguments_again(), role == 1, b, hk, hk * rep + h0, nh, qt_lo * 32, q_end + 1, kw0 + row, lane, x);
        put_row<D, DB>(row_room<D, 2 * QW, 0>(lds, w), x, row, acc, lane);
        if (ALL && c32 == row) sc = role == 0 ? 1.0f : a.scale;
    }
    if (a.in_place) __syncthreads();  // every row has been read
    if (stored) {
        const bool parts = hs > 1 && !to_tail;
        const int64_t pk = to_tail ? ((static_cast<int64_t>(kvu) * (tl.nch + 1) + (chunk >= 0 ? chunk : tl.nch)) * 64 + kj) * dk
                                   : (static_cast<int64_t>(kvu) * hs + rr) * 2 * a.T * dk + static_cast<int64_t>(kj) * dk;
        const int64_t pv = pk + static_cast<int64_t>(to_tail ? 32 : a.T) * dk;
        const bool scratch = parts || to_tail;
        void* const room = to_tail ? a.tail : a.part;
        const int64_t row = scratch ? (role == 0 ? pv : pk) : role == 0 ? b * a.dv_sb + hk * a.dv_sh + kj * a.dv_st
                                                                       : b * a.dk_sb + hk * a.dk_sh + kj * a.dk_st;
        void* const dst = scratch ? room : role == 0 ? a.dv : a.dk;
#pragma unroll
        for (int db = 0; db < DB; ++db) store_block32<D>(dst, row, db, g, acc[db], sc, dk, role == 0 ? TurnRow() : turn_row<TURN>(a, hk, kj));
    }
}
template <int D, int QW>
__global__ __launch_bounds__(128 * QW, 2) void x3_dkdv(AttnArgs a) {
    all_arguments(a);
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * DKDV_TILE<D, QW>];
    __shared__ __attribute__((aligned(16))) float pbuf[QW * 1024];
    const int nblk = (a.T + 32 * QW - 1) / (32 * QW) + (a.tail ? sink_tail(a.T, a.window, a.sinks).nch : 0);
    int blk, rr, kvu;
    // block 0 of every unit first: without a band it is seen by every query, with one it owns the sink keys
    if (a.causal && nblk > 1 ? xcd_map_block_major(nblk, a.head_split, a.Hkv * a.B, blk, rr, kvu)
                             : xcd_map(nblk, a.head_split, a.Hkv * a.B, blk, rr, kvu))
        dkdv_block<D, QW, false, false>(a, blk, rr, kvu, lds, pbuf);
}

// ---- dK, dV and dQ in one launch, delta read (f32x3_takes_bwd) ----
template <int D, bool ALL, bool TURN>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void x3_bwd(AttnArgs a) {
    all_arguments(a);
    constexpr int Q = dq_lds<D, 2, 2>(), K = 2 * DKDV_TILE<D, 2>, N = Q > K + 4096 ? Q : K + 4096;
    __shared__ __attribute__((aligned(16))) uint16_t lds[N];
    const JoinedBlocks jb(a, 64);
    int rank, r, kvu;
    if (!jb.map(a, rank, r, kvu)) return;
    if (r < a.head_split) return dkdv_block<D, 2, ALL, TURN>(a, rank, r, kvu, lds, reinterpret_cast<float*>(lds + K));
    const int b = quotient(kvu, a.Hkv), hk = kvu - b * a.Hkv;
    dq_block<D, 2, 2, ALL, TURN>(a, 0, b, hk * (jb.each - a.head_split) + r - a.head_split, hk, jb.ranks - 1 - rank, lds);
}

// ---- dQ above 64 columns: the same two phases ----
// First: role 0 S = K Q^T and P, role 1 dP - delta; both tiles are handed over, and each role forms dS for itself and takes half the
// columns of dQ^T += K^T dS. The next tile is moved as in x3_dkdv (T 4403, 8 heads, head_dim 128, us: 456 -> 436).
template <int D>
__global__ __launch_bounds__(512, 2) void x3_dq_wide(AttnArgs a, int fuse_delta) {
    all_arguments(a);
    constexpr int QW = 4, BM = 32 * QW, DB = D / 32, G = 64 * QW, HB = (DB + 1) / 2;
    constexpr int PLANE = Mover3<D, G>::PLANE, TILE = 6 * PLANE;
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * TILE];
    __shared__ __attribute__((aligned(16))) float cbuf[2][QW * 1024];

    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int role = w / QW, qg = w % QW, gt = static_cast<int>(threadIdx.x) & (G - 1);
    const int g = lane >> 5, c32 = lane & 31, dk = a.dk_dim;
    int b, h, hk, qblk;
    if (!map_query_block(a, (a.T + BM - 1) / BM, b, h, hk, qblk)) return;
    const int q0 = qblk * BM, qlo = q0 + qg * 32, qhi = qlo + 31, qi = qlo + c32;
    const float cexp = a.scale * LOG2E;

    // role 0 moves K, role 1 V
    const float* const src = head_of<float>(role == 0 ? a.k : a.v, role == 0 ? a.k_sb : a.v_sb, b, role == 0 ? a.k_sh : a.v_sh, hk);
    const int s_st = static_cast<int>(role == 0 ? a.k_st : a.v_st);
    Mover3<D, G> mv;
    mv.init(gt, s_st, dk);
    const KeyTiles kt(a, q0, BM, 32);
    auto fetch = [&](int i) { mv.load(src, s_st, kt.tile(i) * 32, a.T, dk); };
    auto commit = [&](int i) { mv.store(lds + (i & 1) * TILE + role * 3 * PLANE, gt); };
    fetch(0);
    bf16x8 res[3][D / 16];  // Q rows for role 0, dO rows for role 1
    const int64_t lrow = (static_cast<int64_t>(b) * a.Hq + h) * a.T + min(qi, a.T - 1);
    // -LSE log2(e) for role 0, delta for role 1
    float row_r = role == 0 ? a.lse[lrow] : fuse_delta ? 0.0f : a.delta[lrow];
    {
        Row<D> r;
        r.load(head_of<float>(role == 0 ? a.q : a.d_o, role == 0 ? a.q_sb : a.do_sb, b, role == 0 ? a.q_sh : a.do_sh, h), role == 0 ? a.q_st : a.do_st, qi, a.T, dk, g);
        if (role == 1 && fuse_delta) {
            Row<D> o;
            o.load(head_of<float>(a.o, a.o_sb, b, a.o_sh, h), a.o_st, qi, a.T, dk, g);
            row_r = xhalf_sum(r.dot(o));
            if (qi < a.T && g == 0) a.delta[lrow] = row_r;
        }
        if (role == 0) row_r = -row_r * LOG2E;
        r.split(res);
    }
    const QueryVis vis(qi, a.T, a.causal, a.window, a.sinks);
    f32x16 acc[HB];
#pragma unroll
    for (int db = 0; db < HB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;
    commit(0);
    if (kt.n > 1) fetch(1);
    __syncthreads();

    const auto loop = [&](auto role_c) {
        constexpr int ROLE = decltype(role_c)::value;
        for (int i = 0; i < kt.n; ++i) {
            const uint16_t* Ks = lds + (i & 1) * TILE;
            const int k0 = kt.tile(i) * 32;
            const bool live = k0 < a.T && qlo < a.T && !(a.causal && k0 > qhi) && !(a.window > 0 && k0 + 31 + a.window <= qlo && k0 >= a.sinks);
            const auto stage = [&]() {
                if (i + 1 < kt.n) {
                    commit(i + 1);
                    if (i + 2 < kt.n) fetch(i + 2);
                }
            };
            if (ROLE == 1) stage();
            f32x16 t;
            if (live) {
                t = dot3<D>(ROLE == 0 ? Ks : Ks + 3 * PLANE, res, c32, g);
#pragma unroll
                for (int r = 0; r < 16; ++r) t[r] = ROLE == 0 ? __builtin_amdgcn_exp2f(fmaf(t[r], cexp, row_r)) : t[r] - row_r;
                const MaskKind kind = mask_kind(k0, k0 + 31, qlo, qhi, a.T, a.causal, a.window, a.sinks);
                if (kind != MaskKind::NONE) mask_block(t, kind, vis, k0 + g * 4, 0.0f);
                put_tile(cbuf[ROLE] + qg * 1024, t, lane);
            }
            __syncthreads();
            if (live) {
                const f32x16 o = get_tile(cbuf[1 - ROLE] + qg * 1024, lane);
#pragma unroll
                for (int r = 0; r < 16; ++r) t[r] *= o[r];
                accumulate3<D, HB>(Ks, Parts(t), acc, lane, ROLE * HB);
            }
            if (ROLE == 0) stage();
            __syncthreads();
        }
    };
    if (role == 0)
        loop(std::integral_constant<int, 0>{});
    else
        loop(std::integral_constant<int, 1>{});
    const int le = lane_again(), ge = le >> 5, qe = qlo + (le & 31);
    // (role 1's last block is a copy of the one before where their number is odd; the rows' delta has been in memory since the first barrier)
    for (uint32_t again = rows_to_redo<HB>(acc, 1.0f, qe < a.T); __builtin_expect(again != 0, 0); again &= again - 1) {
        const int row = __builtin_ctz(again);
        double x[2];
        exact_dq(arguments_again(), b, h, hk, qlo + row, a.delta[(static_cast<int64_t>(b) * a.Hq + h) * a.T + qlo + row], le, x);
        put_row<D, HB>(row_room<D, 2 * QW, 0>(lds, w), x, row, acc, le, role * HB);
    }
    if (a.in_place) __syncthreads();  // every row has been read
    if (qe < a.T) {
        const int64_t ro = b * a.dq_sb + h * a.dq_sh + qe * a.dq_st;
#pragma unroll
        for (int db = 0; db < HB; ++db)
            if (role * HB + db < DB) store_block32<D>(a.dq, ro, role * HB + db, ge, acc[db], a.scale, dk);
    }
}

// Which form a launch takes, from its number of 32-row blocks and the length of a block's chain; NONE leaves it to the kernels
// on the fp32 instruction, which split a block's tiles four or eight ways (attn_f32_split.hip) and are ahead while that is what
// fills the chip. PAIR: 64 rows, two groups of two wavefronts that take every other tile; WIDE: 128 rows (256 at 128 columns).
// Over 840 random shapes of 100 to 6000 tokens and 100 or more blocks the launches that come here are 1.2 (32 columns) to 1.7
// (96) times as fast as on the fp32 instruction in the geometric mean. Measured (us, fp32 | PAIR | WIDE; causal unless said):
//   forward, 64 columns    T 1024 x 4, 8 heads 57 | 42 | 60;   T 4096 x 4, 16 heads 1155 | 814 | 716;  T 2048, 8 heads 48 | 74 | 115
//   dQ                     80 | 56 | 75;                       1595 | 1077 | 953;                      68 | 89 | 136
//   dK/dV (64 | 128 keys)  101 | 70 | 79;                      2282 | 1450 | 1390;                     81 | 124 | 146
//   128 columns            T 4096 x 4, 16 heads: forward 2135 | 2257 | 1374, dQ 3262 | 2140, dK/dV 4240 | 3450 | 3470
//                          T 2420, 8 heads 146 | 164 | 281;  T 4403, 8 heads 426 | 356 | 526;  no mask, T 1634, 8 heads 151 | 119 | 209
enum class Form { NONE, PAIR, WIDE };

int64_t blocks_of(const AttnArgs& a, int64_t units) { return static_cast<int64_t>((a.T + 31) / 32) * units; }
// all blocks about as long as the longest: half the launch is not over before it
bool level(const AttnArgs& a) { return !a.causal || 2 * chain_tokens(a) <= a.T; }

Form fwd_form(const AttnArgs& a) {
    const int64_t blocks = blocks_of(a, static_cast<int64_t>(a.Hq) * a.B);
    if (a.T <= (a.dk_dim > 96 ? 128 : 32)) return Form::NONE;  // one tile to a block, or hardly more
    if (a.dk_dim <= 32) return blocks < (level(a) ? 800 : 900) ? Form::NONE : blocks < 3000 ? Form::PAIR : Form::WIDE;
    if (a.dk_dim <= 64) return blocks < (level(a) ? 500 : 700) ? Form::NONE : blocks < 2500 ? Form::PAIR : Form::WIDE;
    if (a.dk_dim <= 96) return blocks < (level(a) ? 250 : 640) ? Form::NONE : blocks < (level(a) ? 1100 : 2100) ? Form::PAIR : Form::WIDE;
    if (blocks < (level(a) ? 260 : 700)) return Form::NONE;
    return blocks < (level(a) ? 1050 : 1500) ? Form::PAIR : Form::WIDE;
}
Form dq_form(const AttnArgs& a) {
    const int64_t blocks = blocks_of(a, static_cast<int64_t>(a.Hq) * a.B);
    if (a.T <= 32) return Form::NONE;
    if (a.dk_dim <= 32) return blocks < (level(a) ? 400 : 750) ? Form::NONE : Form::PAIR;
    if (a.dk_dim <= 64) return blocks < (level(a) ? 300 : 660) ? Form::NONE : blocks < 2500 ? Form::PAIR : Form::WIDE;
    return blocks < (level(a) ? 260 : chain_tokens(a) < 600 ? 600 : 730) ? Form::NONE : Form::WIDE;
}
// The query heads of a group are dealt out where the launch would be on the fp32 instruction, which is what its workspace is sized
// for (f32_deals_heads): with 64 keys to a workgroup the others have enough of them. The blocks are those of all splits.
int head_split(const AttnArgs& a) { return f32_deals_heads(a) ? a.head_split : 1; }
Form dkdv_form(const AttnArgs& a) {
    const int64_t blocks = blocks_of(a, static_cast<int64_t>(a.Hkv) * a.B * head_split(a));
    const int chain = chain_tokens(a);
    // a sink keys' block that walks every query of every head of its group (32 heads on 8, T 1625, window 122: 100 us | 136; T 843 x
    // 6, window 79: 139 | 206)
    if (a.window > 0 && a.sinks > 0 && blocks < (a.Hq > a.Hkv ? 2000 : 800)) return Form::NONE;
    if (a.dk_dim <= 32) return blocks < (level(a) ? (chain < 130 ? 2000 : chain < 400 ? 1000 : 840) : 1250) ? Form::NONE : Form::PAIR;
    if (a.dk_dim <= 64) return blocks < (!level(a) ? 700 : chain <= 200 ? 400 : 512) ? Form::NONE : Form::PAIR;
    if (a.dk_dim <= 96) return blocks < (level(a) ? 260 : 600) ? Form::NONE : blocks < (level(a) ? 600 : 900) ? Form::PAIR : Form::WIDE;
    return blocks < (level(a) ? 260 : 450) ? Form::NONE : Form::PAIR;
}
// Whether the queries past the band of the sink keys' block go to workgroups of their own: split_tail_pays, and the pieces, which
// walk all heads of a group, are shorter than the block's chain through its share of the heads.
bool tail_pays(const AttnArgs& a, int block_rows) {
    const SinkTail t = sink_tail(a.T, a.window, a.sinks);
    const int64_t rep = a.Hq / a.Hkv, share = (rep + a.head_split - 1) / a.head_split, left = a.T - t.q0;
    return split_tail_pays(a, a.head_split, block_rows) && share * left > rep * (left < TAIL_CHUNK ? left : TAIL_CHUNK);
}

template <int D, int QW, int KW>
int run_fwd(const AttnArgs& a, hipStream_t st) {
    const int nqb = (a.T + 32 * QW - 1) / (32 * QW);
    hipLaunchKernelGGL((x3_fwd<D, QW, KW>), dim3(xcd_grid(nqb, a.Hq / a.Hkv, a.Hkv * a.B)), dim3(64 * QW * KW), 0, st, a);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
template <int D, int QW, int KW>
int run_dq(const AttnArgs& a, bool fuse_delta, hipStream_t st) {
    const int nqb = (a.T + 32 * QW - 1) / (32 * QW);
    hipLaunchKernelGGL((x3_dq<D, QW, KW>), dim3(xcd_grid(nqb, a.Hq / a.Hkv, a.Hkv * a.B)), dim3(64 * QW * KW), 0, st, a, fuse_delta ? 1 : 0);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
template <int D>
int run_dq_wide(const AttnArgs& a, bool fuse_delta, hipStream_t st) {
    hipLaunchKernelGGL((x3_dq_wide<D>), dim3(xcd_grid((a.T + 127) / 128, a.Hq / a.Hkv, a.Hkv * a.B)), dim3(512), 0, st, a, fuse_delta ? 1 : 0);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
template <int D, int QW>
int run_dkdv(const AttnArgs& a_in, hipStream_t st) {
    AttnArgs a = a_in;
    a.head_split = head_split(a);
    if (!tail_pays(a, 32 * QW)) a.tail = nullptr;
    const int nkb = (a.T + 32 * QW - 1) / (32 * QW);
    hipLaunchKernelGGL((x3_dkdv<D, QW>), dim3(xcd_grid(nkb + tail_blocks(a), a.head_split, a.Hkv * a.B)), dim3(128 * QW), 0, st, a);
    PK_HIP(hipGetLastError());
    return a.head_split > 1 ? launch_gqa_reduce(a, st) : a.tail ? launch_sink_tail_reduce(a, st) : PK_OK;
}

template <int D, bool ALL>
void launch_x3_bwd(const AttnArgs& a, dim3 grid, hipStream_t st) {
    if (a.turn)
        hipLaunchKernelGGL((x3_bwd<D, ALL, true>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((x3_bwd<D, ALL, false>), grid, dim3(256), 0, st, a);
}
template <int D>
int run_bwd(const AttnArgs& a_in, hipStream_t st) {
    AttnArgs a = a_in;
    a.head_split = head_split(a);
    a.tail = nullptr;
    if (const int rc = launch_row_delta(a, false, st)) return rc;
    const dim3 grid(JoinedBlocks(a, 64).grid(a));
    if (f32x3_bwd_keeps_all(a_in))
        launch_x3_bwd<D, true>(a, grid, st);
    else
        launch_x3_bwd<D, false>(a, grid, st);
    PK_HIP(hipGetLastError());
    return a.head_split > 1 ? launch_gqa_reduce(a, st) : PK_OK;
}

}  // namespace

// what the fp32 split kernels ask of their tensors holds for these as well
bool f32x3_takes_fwd(const AttnArgs& a) { return f32_split_serves(a) && fwd_form(a) != Form::NONE; }
bool f32x3_takes_dq(const AttnArgs& a) { return f32_split_serves(a) && dq_form(a) != Form::NONE; }
bool f32x3_takes_dkdv(const AttnArgs& a) { return f32_split_serves(a) && dkdv_form(a) != Form::NONE; }

int launch_f32x3_fwd(const AttnArgs& a, hipStream_t st) {
    const bool wide = fwd_form(a) == Form::WIDE;
    if (a.dk_dim <= 32) return wide ? run_fwd<32, 4, 1>(a, st) : run_fwd<32, 2, 2>(a, st);
    if (a.dk_dim <= 64) return wide ? run_fwd<64, 4, 1>(a, st) : run_fwd<64, 2, 2>(a, st);
    if (a.dk_dim <= 96) return wide ? run_fwd<96, 4, 1>(a, st) : run_fwd<96, 2, 2>(a, st);
    if (!wide) return run_fwd<128, 2, 2>(a, st);
    // 256 rows are mostly cut off by the ends of short sequences and bands (T 230 x 40, 8 heads 90 us, with 128 rows 71)
    return chain_tokens(a) <= 320 ? run_fwd<128, 4, 1>(a, st) : run_fwd<128, 8, 1>(a, st);
}
int launch_f32x3_dq(const AttnArgs& a, bool fuse_delta, hipStream_t st) {
    const bool wide = dq_form(a) == Form::WIDE;
    if (a.dk_dim <= 32) return run_dq<32, 2, 2>(a, fuse_delta, st);
    if (a.dk_dim <= 64) return wide ? run_dq<64, 4, 1>(a, fuse_delta, st) : run_dq<64, 2, 2>(a, fuse_delta, st);
    return a.dk_dim <= 96 ? run_dq_wide<96>(a, fuse_delta, st) : run_dq_wide<128>(a, fuse_delta, st);
}
// dQ and dK/dV in one launch behind one of delta: while either alone is about one round of the chip, its longest chains of tiles are as
// long as the launch and half of the chip waits for them; together one's chains run beside the other's. Over some rounds it is the same
// work with a pass over O and dO more. In 64-row blocks of queries, one after the other (or on the fp32 instruction) | joined, us, causal
// unless said:
//   64 columns   T 1024 x 4, 8 heads (512) 122 | 110;   T 313 x 4, 16 heads (320) 73 | 36;   T 836 x 2, 8 heads (224) 81 | 61;
//                T 1841, 8 heads (232) 136 | 120;   T 360 x 3, 8 heads (144) 38 | 31;   no mask, T 777 x 4, 12 heads (624) 210 | 177
//     below      T 963, 4 heads (64) 50 | 66;   T 894 x 4, 2 heads (112) 45 | 60;   T 3305, 4 heads on 2 (208) 197 | 202
//     above      T 5833, 8 heads (736) 688 | 710;   T 1024 x 8, 16 heads (2048) 351 | 362;   T 4096 x 4, 16 heads (4096) 2417 | 2562
//   32 columns   T 1037 x 2, 8 heads (272) 62 | 51;   T 181 x 13, 16 heads (624) 42 | 29;   no mask, T 1639, 8 heads (208) 109 | 85
//   128 columns, one workgroup to a CU   T 270 x 3, 16 heads (240) 122 | 58;   T 1796, 2 heads (58) 244 | 200;   T 2132, 8 heads (272) 393 | 291;
//                no mask, T 710, 8 heads (96) 129 | 91;   above: T 440 x 19, 4 heads (532) 146 | 158;   T 87 x 51, 4 on one (408) 57 | 66;
//                no mask, T 1010 x 14, 2 heads (448) 353 | 388;   T 44 x 99, 2 heads (198) 30 | 33
//   96 columns   T 241 x 10, 4 heads (160) 52 | 34;   T 936, 16 heads of 80 (240) 130 | 96;   below, above: T 2413, 4 heads of 80 (152) 184 | 210;   T 2309 x 2,
//                8 heads (592) 421 | 499;   from 2600 tokens on, where the launch of both on the fp32 instruction ends, from 88 blocks on (0.86 of the time over
//                81 shapes): T 3300 x 2, 1 head of 80 (104) 323 | 277;   T 6000, 1 head (94) 575 | 494;   no mask, above: T 44 x 99, 2 heads (198) 24 | 27;
//                T 312 x 15, 4 on 2 (300) 81 | 94
//   no mask, 512 workgroups there at once at 64 columns: up to 256 blocks of either kind are one round instead of two, up to 384 two that are full, from 540
//     on one round less than apart (T 4549 x 3, 2 heads (432) 643 | 732);   with groups the blocks of keys are the longer ones: T 3183, 8 on 2 (400) 452 | 533;
//     T 2003, 16 on 4 (512) 344 | 382;   32 columns, T 3353, 8 on 4 (424) 308 | 365
//   bands, every head its own: 48, T 165 x 6, 8 heads, window 86 (144) 35 | 19;   T 4383, 8 heads, 26 (552) 51 | 41;   T 975 x 13, 2 heads of 64, 408,
//     1 sink (416) 107 | 74;   not: T 1238, 16 heads of 32, 204, 4 sinks, whose block is walked whole (320) 46 | 64;   T 2377, 8 on 2 of 64 (304) 89 | 118
//     whose sink keys' block is walked for up to 600 queries more while there are blocks enough beside it: 64, T 419 x 6, 8 heads, 40, 1 sink (336) 54 | 40;
//     T 426 x 14, 4 heads, 36, 4 (392) 78 | 40;  48, T 1140 x 11, 2 heads, 556 (396) 126 | 85;  96, T 707 x 10, 2 heads, 321, 1 (240) 107 | 76;  not: 64,
//     T 962, 8 heads, 331, 16 (128) 58 | 66;  T 934, 12 heads of 48, 396, 1 (180) 64.7 | 65.3;  80, T 654, 8 heads, 180, 16 (88) 49 | 65;  128, T 490 x
//     3, 2 heads, 99, 16 (48) 42 | 67;  32, T 137 x 3, 16 heads, 27, 16 (144) 11.6 | 14.9;  T 1554, 8 heads, 1017, 4 (200) 57 | 75
//     long bands: 32, T 4127, 2 heads, 966 (130) 37 | 50;  T 1204, 8 heads, 574 (152) 29 | 34;  above, 64, T 4520, 8 heads, 1279 (568) 226 | 241;  96,
//     T 3220, 8 heads, 305 (408) 99 | 131;  T 4790, 4 heads, 74 (300) 59 | 67
//     below      T 1460, 8 heads (184) 56 | 65;   above   T 3072, 16 heads on 4 (768) 243 | 249;   no mask, T 3830, 8 on 2 (480) 371 | 423
//
// Where one of the two by itself would be on the fp32 instruction, values keep all the bits that they have there (UP). Scores from 2^80 on are
// out of range then: at the smallest scale that is 2^40 in the exponent, whose last place is 2^17.
bool f32x3_bwd_keeps_all(const AttnArgs& a) { return dq_form(a) == Form::NONE || dkdv_form(a) == Form::NONE || f32_split_takes_bwd(a); }
bool f32x3_takes_bwd(const AttnArgs& a) {
    if (!f32_split_serves(a) || a.T <= 32 || (a.scale < 0x1p-40f && f32x3_bwd_keeps_all(a))) return false;
    const int64_t q = static_cast<int64_t>((a.T + 63) / 64) * a.Hq * a.B;
    const bool groups = a.Hq > a.Hkv;
    if (a.window > 0) {
        const int chain = chain_tokens(a), tail = a.sinks > 0 ? a.T - a.window : 0;
        return !groups && tail <= (q >= (a.dk_dim <= 32 ? 260 : 200) ? 600 : 300) &&
               q >= (a.dk_dim <= 32 ? (chain > 400 || tail > 100 ? 200 : 130) : a.dk_dim <= 64 ? 100 : a.dk_dim <= 96 ? 88 : 50) &&
               q <= (a.dk_dim <= 64 ? (chain > 1000 ? 500 : chain > 400 ? 700 : 800) : a.T > 2500 || a.window < 32 ? 290 : 420);
    }
    if (a.dk_dim > 96) return q >= 40 && q <= (a.causal ? (a.T <= 130 ? 300 : 420) : a.T <= 64 ? 130 : a.T <= 130 ? 200 : 260);
    if (a.dk_dim > 64) return q >= (a.causal && a.T > 300 && a.T <= 2600 ? 170 : 88) && q <= (a.causal ? 330 : a.T <= 100 ? 120 : 290);
    if (a.dk_dim <= 32)
        return !a.causal ? q >= 180 && q <= (groups && a.T >= 800 ? 390 : 440) : q >= (a.T <= 130 ? 116 : a.T <= 600 ? 190 : 260) && q <= 640;
    if (!a.causal) return q >= 124 && q <= 960 && (a.T < 1000 || (groups ? q <= 300 : q <= 384 || q >= 540));
    return q >= (a.T <= 600 ? 140 : a.T <= 2000 ? 180 : 260) && q <= (a.T <= 1500 ? 1000 : 700);
}
int launch_f32x3_bwd(const AttnArgs& a, hipStream_t st) { return a.dk_dim <= 32 ? run_bwd<32>(a, st) : a.dk_dim <= 64 ? run_bwd<64>(a, st) : a.dk_dim <= 96 ? run_bwd<96>(a, st) : run_bwd<128>(a, st); }
int launch_f32x3_dkdv(const AttnArgs& a, hipStream_t st) {
    if (a.dk_dim <= 32) return run_dkdv<32, 2>(a, st);
    if (a.dk_dim <= 64) return run_dkdv<64, 2>(a, st);
    if (a.dk_dim <= 96) return dkdv_form(a) == Form::WIDE ? run_dkdv<96, 4>(a, st) : run_dkdv<96, 2>(a, st);
    return run_dkdv<128, 2>(a, st);
}

}  // namespace pk
