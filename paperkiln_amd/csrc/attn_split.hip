// bf16 attention (forward, dQ, dK/dV) in workgroups whose wavefronts share the CONTRACTION: KW groups of wavefronts take
// every KW-th tile of the keys (of the queries for dK/dV) of one block of rows, and their partial results meet in LDS at
// the end. Mathematics and operand layouts are those of attn_fwd_mfma.hip / attn_bwd_mfma.hip.
//
// What bounds it: the other bf16 kernels give a workgroup 128 or 256 rows and let it walk every visible tile alone. With
// few (batch, head) units or short sequences that is a handful of workgroups on 256 CUs, each a serial chain of tiles of
// about half a microsecond. Here a block is 32 rows and four wavefronts split its tiles: four times the workgroups, a
// quarter of the chain, and a sequence of 128 tokens is one tile per wavefront -- one round trip to memory.
//
// Which of these kernels a launch takes, or whether it takes one of the others, depends on its number of blocks (fwd_form,
// dq_form, dkdv_form): the same call gives the same bits every time, but a unit in a batch need not give those it gives alone.
//
// The same kernels, with wavefronts that own different rows and share the tiles (QW = 4, KW = 1), are the path of most dQ and dK/dV
// launches at head_dim 64 (dkdv_form_64) and of every head size that is a multiple of 8 up to 128 but not 64 or 128 (D is the size rounded up to 32; chunks past the real
// size read as zero and are not stored). Rows that are not aligned run in fp32 arithmetic there (attn_generic.hip), and these
// are no less exact (EXACT; head_dim 64 and 128 round P and dS to one bf16 operand): P and dS enter their products as several
// operands, the rounded value and the remainders.
#include <algorithm>
#include <type_traits>

#include "attn_split.h"

namespace pk {
namespace {

constexpr float LOG2E = 1.4426950408889634f;
// How many operands P and dS are (EXACT). Gradients can be fp32: three, all 24 bits; with two their error against float64 was
// 2.5e-6 of their norm at every size, three leave 2 to 9e-7, the scalar kernels 2e-7 to 1.5e-6 (eleven shapes of 97 to 4096
// tokens, head_dim 24 to 120). O is bf16 always: with two its error is the scalar kernels' to four digits, with three too.
// The third costs (us, B=2 T=4096 H=16, dQ and dK/dV): head_dim 32 110 -> 140, 148 -> 195; 96 219 -> 254, 326 -> 409.
constexpr int FWD_PARTS = 2, BWD_PARTS = 3;
// The maximum that P is formed against moves only when a row outgrows it by this many powers of two: some row of 32 finds a
// new maximum in most tiles, and rescaling costs three instructions per accumulator element. P then reaches 2^6, which its
// operands and the fp32 sums hold as they hold 1.
constexpr float LAZY_T = 6.0f;

// Where a row of a tile that serves row reads and transposing reads sits in LDS: at 64 columns in the order that keeps both free
// of bank conflicts (lds_row, mfma_common.h).
template <int D>
__device__ constexpr int tile_row(int r) {
    return lds_row<D == 64 ? 64 : 128>(r);
}

// A tile of ROWS rows of a [T, dk] bf16 matrix, moved by G threads: thread t of the group carries the 16-byte chunks
// t, t + G, ... Rows past T and chunks past dk read as zero.
template <int D, int G, int ROWS>
struct Mover {
    static constexpr int NCH = D / 8, CPT = ROWS * NCH / G;
    static_assert(CPT >= 1 && ROWS * NCH % G == 0, "every thread moves the same number of chunks");
    int off[CPT];  // byte offsets inside a tile
    u32x4 r[CPT];
    __device__ void init(int t, int st, int dk) {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int c = t + G * i, row = c / NCH, ch = c % NCH;
            off[i] = ch * 8 < dk ? (row * st + ch * 8) * 2 : static_cast<int>(OUTSIDE);
        }
    }
    __device__ void load(const uint16_t* head, int st, int r0, int T, int dk) {
        const __amdgpu_buffer_rsrc_t rs = tile_rsrc(head, 0, st, r0, T, dk);
#pragma unroll
        for (int i = 0; i < CPT; ++i) r[i] = tile_load16(rs, off[i]);
    }
    // ORDERED: rows in the order of tile_row
    template <bool ORDERED>
    __device__ void store(uint16_t* lds, int pitch, int t) const {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int c = t + G * i, row = c / NCH;
            *reinterpret_cast<u32x4*>(lds + (ORDERED ? tile_row<D>(row) : row) * pitch + (c % NCH) * 8) = r[i];
        }
    }
};

// Row r0 + c32 of a head as an operand held in registers: chunk kk covers d = 16kk + 8g .. +7; zero past T and past dk. BRANCH: under a
// condition instead of through a buffer, which keeps the loads where they are written. In the long loops of P and dS in several parts the scheduler
// needs that (forward, us, buffer | branch: 96 columns, T 1500 x 4, 8 heads 44.0 | 41.6, T 2500, 4 heads 24.8 | 23.5; 48, T 4000 x 2, window 500 27.2 | 26.1; backward
// 79.7 | 77.1, but 96 columns 111.5 | 113.8; 80, no mask, T 2000 x 4 286 | 291); in the backward at 64 columns the buffer is ahead (T 4096 x 2, 8 heads 154 | 156), and
// in the forward at 128 (T 200, 4 heads 6.8 | 7.2).
template <int D, bool BRANCH>
__device__ inline void load_row(const uint16_t* head, int st, int r0, int T, int dk, int c32, int g, bf16x8* out) {
    if constexpr (BRANCH) {
#pragma unroll
        for (int kk = 0; kk < D / 16; ++kk) {
            u32x4 z = {0, 0, 0, 0};
            const int col = kk * 16 + g * 8;
            if (r0 + c32 < T && col < dk) z = *reinterpret_cast<const u32x4*>(head + static_cast<int64_t>(r0 + c32) * st + col);
            out[kk] = *reinterpret_cast<bf16x8*>(&z);
        }
        return;
    }
    const __amdgpu_buffer_rsrc_t rs = tile_rsrc(head, 0, st, r0, T, dk);
    const int row = (c32 * st + g * 8) * 2;
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) {
        const u32x4 v = tile_load16(rs, kk * 16 + g * 8 < dk ? row + 32 * kk : static_cast<int>(OUTSIDE));
        out[kk] = *reinterpret_cast<const bf16x8*>(&v);
    }
}

// Elements 8H .. 8H+7 of a C tile as N bf16 k-chunks: the rounded values, then what the rounding before left over, rounded.
// 8 significant bits each and signs of their own: three hold the 24 bits of the fp32 values.
template <int H, int N>
__device__ inline void split_operand(const f32x16& c, bf16x8 (&part)[N]) {
    u32x4 p[N];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float x0 = c[8 * H + 2 * i], x1 = c[8 * H + 2 * i + 1];
#pragma unroll
        for (int n = 0; n < N; ++n) {
            p[n][i] = pack_bf16(x0, x1);
            x0 -= __uint_as_float(p[n][i] << 16), x1 -= __uint_as_float(p[n][i] & 0xffff0000u);
        }
    }
#pragma unroll
    for (int n = 0; n < N; ++n) part[n] = *reinterpret_cast<bf16x8*>(&p[n]);
}

// P of a raw score and the row's LSE (nl: -LSE of the row when EXACT, else -LSE log2 e). EXACT: the difference is formed in one
// rounding, of the difference; in units of log2 the scale, the LSE and the product would each be rounded at the size of the LSE.
template <bool EXACT>
__device__ inline float weight_of(float s, float scale, float cexp, float nl) {
    return __builtin_amdgcn_exp2f(EXACT ? fmaf(s, scale, nl) * LOG2E : fmaf(s, cexp, nl));
}

// sum + the products of eight elements, in order
__device__ inline float add_products(bf16x8 x, bf16x8 y, float sum) {
    const u32x4 xv = *reinterpret_cast<const u32x4*>(&x);
    const u32x4 yv = *reinterpret_cast<const u32x4*>(&y);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        sum = fmaf(__uint_as_float(xv[i] << 16), __uint_as_float(yv[i] << 16), sum);
        sum = fmaf(__uint_as_float(xv[i] & 0xFFFF0000u), __uint_as_float(yv[i] & 0xFFFF0000u), sum);
    }
    return sum;
}

// Whether dP starts from -delta instead of zero, a subtraction an element less: dQ 1.6 %, dK/dV 2.5 % over 17 shapes. The sum is then
// rounded at delta's size four times instead of once, which dS, one bf16 operand there, does not show: errors of dQ and dK against
// float64 are 1.63e-3 to 1.79e-3 of their norms and the same to four digits either way over 28 inputs, V with a mean of 30 standard
// deviations among them. Not where P and dS keep all their bits (EXACT), nor at 128 columns, where it spilled 30 registers more; dQ not where
// four wavefronts share the tiles (T 1661, 16 heads 21.5 us | 24.5), nor dQ or dK/dV in the joined launch for sizes whose launch of it alone is
// another kernel, which subtracts delta at the end: where V is the same in every row dS is zero and dQ and dK are the rounding of dP alone, two to
// four times as much from -delta (dK, T 150 x 4, 16 heads 1.9e-3 | 5.3e-4, alone 4.4e-4; T 64 x 31, 4 heads 3.1e-3 | 8.5e-4, alone 1.5e-3). Joined launch, from
// -delta | from zero, us: dQ, T 470 x 8, 8 heads 20.1 | 20.4, T 1024 x 8 50.1 | 50.9, T 1661, 16 heads 45.5 | 46.4; dK/dV, T 470 x 8 19.1 | 19.5, T 923
// x 7, 4 heads 29.4 | 30.1, T 150 x 4 9.5 | 9.6; 1.007 over 60 shapes, one by 4 % (subtracted behind dV's product 1.014, one by 7).
template <int D, bool EXACT>
constexpr bool FROM_DELTA = !EXACT && D == 64;

// acc[db] += M^T c for the 32 rows of an LDS tile that start at row0, M the tile (columns 32 db ..), c a C tile whose rows
// are the tile's rows, as PARTS operands
template <int D, int PARTS, bool ORDERED>
__device__ inline void accumulate_tr(const uint16_t* tile, int pitch, int row0, const f32x16& c, f32x16* acc, int lane) {
    constexpr int DB = D / 32;
    const auto half = [&](auto hc) {
        constexpr int H = decltype(hc)::value;
        bf16x8 part[PARTS];
        if constexpr (PARTS == 1)
            part[0] = c_to_operand<H>(c);
        else
            split_operand<H>(c, part);
        // a product that waits for the one before it takes half as long again: the rounded operand into every block, then
        // the remainders
        bf16x8 m[DB];
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            m[db] = ORDERED && D == 64 ? lds_read_tr_operand_perm<64>(tile, pitch, row0 + 16 * H, db, lane)
                                       : lds_read_tr_operand(tile, pitch, row0 + 16 * H, db * 32, lane);
            acc[db] = mfma32(m[db], part[0], acc[db]);
        }
#pragma unroll
        for (int n = 1; n < PARTS; ++n)
#pragma unroll
            for (int db = 0; db < DB; ++db) acc[db] = mfma32(m[db], part[n], acc[db]);
    };
    half(std::integral_constant<int, 0>{});
    half(std::integral_constant<int, 1>{});
}

// The launch bounds of all three kernels ask for two wavefronts to a SIMD where the registers allow it. Left to itself the
// compiler kept the accumulators of head sizes above 64 in accumulation registers beside 200 others, one wavefront to a SIMD,
// whose products, exponentials and LDS reads then took turns; within 256 registers they need no copies either. Forward, B=2
// T=4096 H=16 (with the alternating products and the lazy maximum below): head_dim 96 261 -> 179 us, 48 166 -> 137, 32 104 ->
// 93; backward 594 -> 542, 416 -> 360, 313 -> 259 (with two operands each for P and dS; with three 653, 450, 334).

// ---- forward: QW groups of 32 queries x KW groups of key tiles of 32 NB keys ----
template <int D, int QW, int KW, int NB, bool EXACT>
__global__ __launch_bounds__(64 * QW * KW, 2) void split_fwd(AttnArgs a) {
    if (KW > 1 || !EXACT) all_arguments(a);
    constexpr int BM = 32 * QW, BN = 32 * NB, KK = D / 16, DB = D / 32, G = 64 * QW;
    constexpr int KS = D + 8;                              // row reads conflict-free
    constexpr int VS = (D / 32) % 2 ? D : D + 32;          // 4-row transposing reads conflict-free
    constexpr int TILE = BN * (KS + VS), NBUF = QW > 1 ? 2 : 1;
    constexpr int RED = KW > 1 ? QW * KW * (DB * 1024 + 128) * 2 : 0;  // in uint16
    __shared__ __attribute__((aligned(16))) uint16_t lds[NBUF * KW * TILE > RED ? NBUF * KW * TILE : RED];

    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = w / QW, qg = w % QW, gt = static_cast<int>(threadIdx.x) - kg * G;
    const int g = lane >> 5, c32 = lane & 31, dk = a.dk_dim;
    const int nqb = (a.T + BM - 1) / BM;
    int b, h, hk, qblk;
    if (!map_query_block(a, nqb, b, h, hk, qblk)) return;
    const int q0 = qblk * BM, qlo = q0 + qg * 32, qhi = qlo + 31, qi = qlo + c32;
    // plain addresses: formed with head_of, and Q's row through a buffer, the loops of long chains and of bands were behind (us: 96 columns, T 5637, 2
    // heads 48 | 53; T 4000, 3 heads 35 | 40; 64, T 980 x 10, 16 heads, window 41, 16 sinks 23.6 | 25.4; T 4096 x 4, 16 heads, window 256 45.3 | 48.1)
    const uint16_t *const kh = static_cast<const uint16_t*>(a.k) + (b * a.k_sb + hk * a.k_sh), *const vh = static_cast<const uint16_t*>(a.v) + (b * a.v_sb + hk * a.v_sh),
                   *const qh = static_cast<const uint16_t*>(a.q) + (b * a.q_sb + h * a.q_sh);
    const int k_st = static_cast<int>(a.k_st), v_st = static_cast<int>(a.v_st);
    const float cexp = a.scale * LOG2E;

    Mover<D, G, BN> mk, mv;
    mk.init(gt, k_st, dk);
    mv.init(gt, v_st, dk);
    const KeyTiles kt(a, q0, BM, BN);
    const int iters = (kt.n + KW - 1) / KW;
    auto fetch = [&](int i) {  // this group's i-th tile (past its last: nothing)
        const int at = i * KW + kg;
        if (at < kt.n) {
            const int r0 = kt.tile(at) * BN;
            mk.load(kh, k_st, r0, a.T, dk);
            mv.load(vh, v_st, r0, a.T, dk);
        }
    };
    auto commit = [&](int buf) {
        uint16_t* t = lds + (buf % NBUF * KW + kg) * TILE;
        mk.template store<false>(t, KS, gt);
        mv.template store<false>(t + BN * KS, VS, gt);
    };
    fetch(0);
    bf16x8 qreg[KK];
    load_row<D, (QW > 1) || (EXACT && D <= 96)>(qh, static_cast<int>(a.q_st), qlo, a.T, dk, c32, g, qreg);
    f32x16 acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;
    float m = -1e30f, l = 0.0f;  // the reference's running-max seed, src/ops.cpp:881
    const QueryVis vis(qi, a.T, a.causal, a.window, a.sinks);
    const KeyRange range(a, qlo);
    commit(0);
    tile_barrier<QW>();

    for (int i = 0; i < iters; ++i) {
        if (i + 1 < iters) fetch(i + 1);  // in flight during the math
        const int at = i * KW + kg;
        const uint16_t* Ks = lds + (i % NBUF * KW + kg) * TILE;
        const uint16_t* Vs = Ks + BN * KS;
        const int n0 = at < kt.n ? kt.tile(at) * BN : a.T;
        f32x16 s[NB];
        bool live[NB], any = false;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {  // wavefront-uniform: is anything of this 32 x 32 block visible?
            live[nb] = range.live(n0 + nb * 32);
            any = any || live[nb];
        }
        if (any) {
            float mx = -INFINITY;
            bool all = true;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                all = all && live[nb];
#pragma unroll
                for (int r = 0; r < 16; ++r) s[nb][r] = 0.0f;
            }
            if (NB > 1 && all) {  // alternating: independent products follow one another
#pragma unroll
                for (int kk = 0; kk < KK; ++kk)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
                        s[nb] = mfma32(lds_read8(Ks + (nb * 32 + c32) * KS + kk * 16 + g * 8), qreg[kk], s[nb]);
            } else {
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) {
                    if (!live[nb]) continue;
#pragma unroll
                    for (int kk = 0; kk < KK; ++kk)
                        s[nb] = mfma32(lds_read8(Ks + (nb * 32 + c32) * KS + kk * 16 + g * 8), qreg[kk], s[nb]);
                }
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                if (!live[nb]) continue;
                const int k0 = n0 + nb * 32;
                if (!range.full(k0))
                    mask_block(s[nb], mask_kind(k0, k0 + 31, qlo, qhi, a.T, a.causal, a.window, a.sinks), vis, k0 + g * 4, -INFINITY);
#pragma unroll
                for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[nb][r]);
            }
            mx = xhalf_max(mx);
            if (__any((mx - m) * cexp > LAZY_T)) {  // wavefront-uniform, rare after the first tiles
                const float mn = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f((m - mn) * cexp);
                l *= alpha;
                m = mn;
#pragma unroll
                for (int db = 0; db < DB; ++db)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
            }
            const float mc = m * cexp;
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) {
                if (!live[nb]) continue;
                float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    s[nb][r] = __builtin_amdgcn_exp2f(fmaf(s[nb][r], cexp, -mc));
                    ps[r & 3] += s[nb][r];
                }
                l += (ps[0] + ps[1]) + (ps[2] + ps[3]);  // per-lane partial; the two halves meet below
                accumulate_tr<D, EXACT ? FWD_PARTS : 1, false>(Vs, VS, nb * 32, s[nb], acc, lane);
            }
        }
        if (i + 1 < iters) commit(i + 1);  // two buffers: last read one iteration ago, before the previous barrier
        tile_barrier<QW>();
    }

    l = xhalf_sum(l);
    const int64_t ro = b * a.o_sb + h * a.o_sh + qi * a.o_st;
    if constexpr (KW > 1) {
        if (QW == 1) __syncthreads();  // every group has read its last tile
        // the groups' running maxima and sums meet with their accumulators, each scaled to the common maximum
        float* red = reinterpret_cast<float*>(lds) + qg * KW * (DB * 1024 + 128);
        float* ml = red + KW * DB * 1024;
        ml[kg * 128 + lane] = m;
        ml[kg * 128 + 64 + lane] = l;
        float mt = m, lt = 0.0f, weight[KW];
        join_shares<DB, KW, 2>(acc, red, kg, lane, [&]() {
#pragma unroll
            for (int k = 0; k < KW; ++k) mt = fmaxf(mt, ml[k * 128 + lane]);
#pragma unroll
            for (int k = 0; k < KW; ++k) {
                weight[k] = __builtin_amdgcn_exp2f((ml[k * 128 + lane] - mt) * cexp);
                lt += ml[k * 128 + 64 + lane] * weight[k];
            }
            return weight;
        }, [&](int db, int qd, const f32x4 (&v)[2]) {
            if (qi < a.T) store_half(false, a.o, ro, db, qd, g, v, 1.0f / lt, dk);
        });
        m = mt, l = lt;
    }
    bool stored = KW > 1;
    if constexpr (KW == 1 && WHOLE_ROWS<D, EXACT>)
        if (dk == D) {
            using Rows = RowStrip<D>;
            static_assert(QW * Rows::ELEMS <= NBUF * KW * TILE, "the wavefronts' strips");
            uint16_t* const strip = lds + qg * Rows::ELEMS;
#pragma unroll
            for (int db = 0; db < DB; ++db) store_block(false, strip, c32 * Rows::S, db, g, acc[db], 1.0f / l, D);
            Rows::out(strip, static_cast<uint16_t*>(a.o) + b * a.o_sb + h * a.o_sh + qlo * a.o_st, a.o_st, 0, a.T - qlo, lane);
            stored = true;
        }
    if (qi < a.T) {
        const float inv = 1.0f / l;
        if (!stored)
#pragma unroll
            for (int db = 0; db < DB; ++db) store_block(false, a.o, ro, db, g, acc[db], inv, dk);
        if (g == 0 && kg == 0) a.lse[(static_cast<int64_t>(b) * a.Hq + h) * a.T + qi] = m * a.scale + logf(l);
    }
}

// ---- dQ (and delta, when asked for with it): the same blocks ----
template <int D, int QW, int KW, int NB>
constexpr int dq_lds() {  // in uint16
    constexpr int TILES = (QW > 1 ? 2 : 1) * KW * 2 * 32 * NB * (D + 8), RED = KW > 1 ? QW * KW * (D / 32) * 2048 : 0;
    return TILES > RED ? TILES : RED;
}
template <int D, int QW, int KW, int NB, bool EXACT, bool MINUS_DELTA = FROM_DELTA<D, EXACT> && (QW > 1 || KW == 8), bool TURN = false>
__device__ inline void dq_block(const AttnArgs& a, int fuse_delta, int b, int h, int hk, int qblk, uint16_t* lds) {
    constexpr int BM = 32 * QW, BN = 32 * NB, KK = D / 16, DB = D / 32, G = 64 * QW, S = D + 8;
    constexpr int TILE = 2 * BN * S, NBUF = QW > 1 ? 2 : 1;

    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = w / QW, qg = w % QW, gt = static_cast<int>(threadIdx.x) - kg * G;
    const int g = lane >> 5, c32 = lane & 31, dk = a.dk_dim;
    const int q0 = qblk * BM, qlo = q0 + qg * 32, qhi = qlo + 31, qi = qlo + c32;
    const uint16_t *const kh = head_of<uint16_t>(a.k, a.k_sb, b, a.k_sh, hk), *const vh = head_of<uint16_t>(a.v, a.v_sb, b, a.v_sh, hk),
                   *const qh = head_of<uint16_t>(a.q, a.q_sb, b, a.q_sh, h);
    const int k_st = static_cast<int>(a.k_st), v_st = static_cast<int>(a.v_st);
    const float cexp = a.scale * LOG2E;

    Mover<D, G, BN> mk, mv;
    mk.init(gt, k_st, dk);
    mv.init(gt, v_st, dk);
    const KeyTiles kt(a, q0, BM, BN);
    const int iters = (kt.n + KW - 1) / KW;
    auto fetch = [&](int i) {
        const int at = i * KW + kg;
        if (at < kt.n) {
            const int r0 = kt.tile(at) * BN;
            mk.load(kh, k_st, r0, a.T, dk);
            mv.load(vh, v_st, r0, a.T, dk);
        }
    };
    auto commit = [&](int buf) {
        uint16_t* t = lds + (buf % NBUF * KW + kg) * TILE;
        mk.template store<true>(t, S, gt);
        mv.template store<true>(t + BN * S, S, gt);
    };
    fetch(0);
    bf16x8 qreg[KK], greg[KK];
    load_row<D, EXACT && (QW > 1) && D <= 64>(qh, static_cast<int>(a.q_st), qlo, a.T, dk, c32, g, qreg);
    load_row<D, EXACT && (QW > 1) && D <= 64>(head_of<uint16_t>(a.d_o, a.do_sb, b, a.do_sh, h), static_cast<int>(a.do_st), qlo, a.T, dk, c32, g, greg);
    // everything is asked for before anything is waited for
    const int64_t lrow = (static_cast<int64_t>(b) * a.Hq + h) * a.T + min(qi, a.T - 1);
    const float lse = a.lse[lrow];
    float dl = 0.0f;
    if (fuse_delta) {
        bf16x8 oreg[KK];
        load_row<D, EXACT && (QW > 1) && D <= 64>(head_of<uint16_t>(a.o, a.o_sb, b, a.o_sh, h), static_cast<int>(a.o_st), qlo, a.T, dk, c32, g, oreg);
        float part = 0.0f;
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) part = add_products(oreg[kk], greg[kk], part);
        dl = xhalf_sum(part);
        if (qi < a.T && g == 0 && kg == 0) a.delta[lrow] = dl;
    } else {
        dl = a.delta[lrow];
    }
    const float nlse = EXACT ? -lse : -lse * LOG2E;
    const QueryVis vis(qi, a.T, a.causal, a.window, a.sinks);
    const KeyRange range(a, qlo);
    f32x16 acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;
    commit(0);
    tile_barrier<QW>();

    for (int i = 0; i < iters; ++i) {
        if (i + 1 < iters) fetch(i + 1);
        const int at = i * KW + kg;
        const uint16_t* Ks = lds + (i % NBUF * KW + kg) * TILE;
        const uint16_t* Vs = Ks + BN * S;
        const int n0 = at < kt.n ? kt.tile(at) * BN : a.T;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int k0 = n0 + nb * 32;
            if (!range.live(k0)) continue;
            f32x16 s, dp;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0.0f, dp[r] = MINUS_DELTA ? -dl : 0.0f;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                s = mfma32(lds_read8(Ks + (nb * 32 + tile_row<D>(c32)) * S + kk * 16 + g * 8), qreg[kk], s);
                dp = mfma32(lds_read8(Vs + (nb * 32 + tile_row<D>(c32)) * S + kk * 16 + g * 8), greg[kk], dp);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) dp[r] = weight_of<EXACT>(s[r], a.scale, cexp, nlse) * (MINUS_DELTA ? dp[r] : dp[r] - dl);
            if (!range.full(k0)) mask_block(dp, mask_kind(k0, k0 + 31, qlo, qhi, a.T, a.causal, a.window, a.sinks), vis, k0 + g * 4, 0.0f);
            accumulate_tr<D, EXACT ? BWD_PARTS : 1, true>(Ks, S, nb * 32, dp, acc, lane);
        }
        if (i + 1 < iters) commit(i + 1);
        tile_barrier<QW>();
    }
    if (KW > 1 && QW == 1) __syncthreads();  // every group has read its last tile
    const int64_t ro = b * a.dq_sb + h * a.dq_sh + qi * a.dq_st;
    if constexpr (KW > 1)
        join_shares<DB, KW, 2>(acc, reinterpret_cast<float*>(lds) + qg * KW * DB * 1024, kg, lane, no_weights, [&](int db, int qd, const f32x4 (&v)[2]) {
            if (qi < a.T) store_half(a.grad_f32 != 0, a.dq, ro, db, qd, g, v, a.scale, dk, turn_row<TURN>(a, h, qi));
        });
    else {
        if constexpr (WHOLE_ROWS<D, EXACT>)
            if (dk == D && !a.grad_f32) {
                using Rows = RowStrip<D>;
                static_assert(QW * Rows::ELEMS <= NBUF * KW * TILE, "the wavefronts' strips");
                uint16_t* const strip = lds + qg * Rows::ELEMS;
#pragma unroll
                for (int db = 0; db < DB; ++db)
                    store_block(false, strip, c32 * Rows::S, db, g, acc[db], a.scale, D, turn_row<TURN>(a, h, min(qi, a.T - 1)));
                return Rows::out(strip, static_cast<uint16_t*>(a.dq) + b * a.dq_sb + h * a.dq_sh + qlo * a.dq_st, a.dq_st, 0, a.T - qlo, lane);
            }
        if (qi < a.T)
#pragma unroll
            for (int db = 0; db < DB; ++db) store_block(a.grad_f32 != 0, a.dq, ro, db, g, acc[db], a.scale, dk, turn_row<TURN>(a, h, qi));
    }
}
template <int D, int QW, int KW, int NB, bool EXACT>
__global__ __launch_bounds__(64 * QW * KW, 2) void split_dq(AttnArgs a, int fuse_delta) {
    all_arguments(a);
    __shared__ __attribute__((aligned(16))) uint16_t lds[dq_lds<D, QW, KW, NB>()];
    int b, h, hk, qblk;
    if (map_query_block(a, (a.T + 32 * QW - 1) / (32 * QW), b, h, hk, qblk)) dq_block<D, QW, KW, NB, EXACT>(a, fuse_delta, b, h, hk, qblk, lds);
}

// The block of `rows` keys of a workgroup, or its piece of a dealt sink tail (past the blocks); rr: its share of the group's heads
__device__ inline bool map_key_block(const AttnArgs& a, int rows, int& blk, int& rr, int& kvu, int id = static_cast<int>(blockIdx.x)) {
    const int nblk = (a.T + rows - 1) / rows + (a.tail ? sink_tail(a.T, a.window, a.sinks).nch : 0);
    // block 0 of every unit first: without a band it is seen by every query, with one it owns the sink keys
    return a.causal && nblk > 1 ? xcd_map_block_major(nblk, a.head_split, a.Hkv * a.B, blk, rr, kvu, id)
                                : xcd_map(nblk, a.head_split, a.Hkv * a.B, blk, rr, kvu, id);
}

// ---- dK, dV: QW groups of 32 keys x KW groups of query tiles of 32 NB ----
// A wavefront owns 32 keys (K and V resident as B operands, lane = key) and both accumulators, so P goes from its
// exponentials into dV and into dS without leaving the registers. The steps are the query tiles that can see the block,
// for every query head of the KV head's group in turn.
//
// OWN_DELTA: the rows' delta is formed here, from O and the tile of dO; otherwise it is read. Of one wavefront to a group and tiles of 32 in the
// order of dq_block and to the same bits; else a thread's chunks of both, then the lanes that hold a row.
//
// dV and dK are joined together up to 64 columns; above, the LDS for both would keep a second workgroup off the CU.
template <int D>
constexpr bool JOIN_BOTH = D <= 64;
template <int D, int QW, int KW, int NB>
constexpr int dkdv_lds() {  // in uint16; LSE and delta of a tile's rows behind it
    constexpr int TILES = (QW > 1 ? 2 : 1) * KW * (2 * 32 * NB * (D + 8) + 128 * NB), RED = KW > 1 ? QW * KW * (D / 32) * (JOIN_BOTH<D> ? 4096 : 2048) : 0;
    return TILES > RED ? TILES : RED;
}
template <int D, int QW, int KW, int NB, bool EXACT, bool OWN_DELTA, bool MINUS_DELTA = FROM_DELTA<D, EXACT>, bool TURN = false>
__device__ inline void dkdv_block(const AttnArgs& a, int blk, int rr, int kvu, uint16_t* lds) {
    // a lane holds the row of O whose row of dO its wavefront has just written; or the chunks of O beside its chunks of dO
    static_assert(!OWN_DELTA || (QW == 1 && NB == 1) || (QW > 1 && (D == 32 || D == 64)), "a row's chunks are in 4 or 8 neighbouring lanes");
    constexpr bool BY_ROW = OWN_DELTA && QW == 1, BY_CHUNK = OWN_DELTA && QW > 1;
    // where dP does not start from -delta: it is subtracted behind dV's product, or, where the kernel's other form starts from it, at once
    constexpr bool LATE = !FROM_DELTA<D, EXACT>;
    constexpr int BNK = 32 * QW, BMQ = 32 * NB, KK = D / 16, DB = D / 32, G = 64 * QW, S = D + 8;
    constexpr int ROWC = 2 * BMQ * 2;                    // LSE and delta of a tile's rows, in uint16
    constexpr int TILE = 2 * BMQ * S + ROWC, NBUF = QW > 1 ? 2 : 1;

    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = w / QW, qg = w % QW, gt = static_cast<int>(threadIdx.x) - kg * G;
    const int g = lane >> 5, c32 = lane & 31, dk = a.dk_dim, rep = quotient(a.Hq, a.Hkv);
    const int nkb = (a.T + BNK - 1) / BNK;
    // hs > 1: the query heads of the group are dealt to hs workgroups (gqa_head_split); this one takes heads
    // [h0, h0 + nh) of the group and leaves fp32 partial sums for launch_gqa_reduce
    const int hs = a.head_split;
    // the sink keys' queries past their block's band go to workgroups of their own, blocks nkb .. nkb + nch - 1
    const SinkTail tl = a.tail ? sink_tail(a.T, a.window, a.sinks) : SinkTail{0, 0};
    const int chunk = blk - nkb;  // >= 0: a piece of the tail, for all query heads of the group
    if (chunk >= 0 && rr > 0) return;
    const int b = quotient(kvu, a.Hkv), hk = kvu - b * a.Hkv, h0 = chunk >= 0 ? 0 : quotient(rr * rep, hs), nh = chunk >= 0 ? rep : quotient((rr + 1) * rep, hs) - h0;
    const int k0 = chunk >= 0 ? 0 : blk * BNK, kw0 = k0 + qg * 32, kj = kw0 + c32;
    const float cexp = a.scale * LOG2E;

    // query tiles that can see keys [k0, k0 + BNK) (paperkiln src/ops.cpp:960-965 inverted)
    const int khi = min(k0 + BNK, a.T) - 1;
    const int qt_lo = chunk >= 0 ? (tl.q0 + chunk * TAIL_CHUNK) / BMQ : a.causal ? k0 / BMQ : 0;
    const int q_end = chunk >= 0 ? min(a.T, tl.q0 + (chunk + 1) * TAIL_CHUNK) - 1
                      : tl.nch > 0 && k0 == 0 ? tl.q0 - 1
                      : a.window > 0 && k0 >= a.sinks ? min(a.T - 1, khi + a.window - 1) : a.T - 1;
    const int qt_hi = q_end / BMQ;
    const int nqt = qt_hi - qt_lo + 1, steps = nqt * nh, iters = (steps + KW - 1) / KW;

    const int q_st = static_cast<int>(a.q_st), g_st = static_cast<int>(a.do_st), o_st = static_cast<int>(a.o_st);
    // the first query head's; the others follow at q_sh, ...
    const uint16_t *const q0h = head_of<uint16_t>(a.q, a.q_sb, b, a.q_sh, hk * rep + h0), *const g0h = head_of<uint16_t>(a.d_o, a.do_sb, b, a.do_sh, hk * rep + h0),
                   *const o0h = OWN_DELTA ? head_of<uint16_t>(a.o, a.o_sb, b, a.o_sh, hk * rep + h0) : nullptr, *const kh = head_of<uint16_t>(a.k, a.k_sb, b, a.k_sh, hk),
                   *const vh = head_of<uint16_t>(a.v, a.v_sb, b, a.v_sh, hk);
    Mover<D, G, BMQ> mq, mg;
    mq.init(gt, q_st, dk);
    mg.init(gt, g_st, dk);
    float row_r = 0.0f;
    bf16x8 oreg[BY_ROW ? KK : 1];
    typename std::conditional<BY_CHUNK, Mover<D, G, BMQ>, int>::type mo;
    if constexpr (BY_CHUNK) mo.init(gt, o_st, dk);
    // steps advance by KW; the (head, tile) of the next fetch is counted up
    int f_h = 0, f_t = kg;
    while (f_t >= nqt) f_t -= nqt, ++f_h;
    int c_t = f_t;
    auto fetch = [&](int i) {
        if (i * KW + kg < steps) {
            const int r0 = (qt_lo + f_t) * BMQ;
            mq.load(q0h + f_h * a.q_sh, q_st, r0, a.T, dk);
            mg.load(g0h + f_h * a.do_sh, g_st, r0, a.T, dk);
            if (gt < 2 * BMQ) {  // LSE in the first BMQ threads, delta in the next; rows past the end are masked
                const int t = min(r0 + gt % BMQ, a.T - 1);
                const int64_t lrow = (static_cast<int64_t>(b) * a.Hq + hk * rep + h0 + f_h) * a.T + t;
                if (gt < BMQ)
                    row_r = a.lse[lrow];
                else if (!OWN_DELTA)
                    row_r = a.delta[lrow];
            }
            if constexpr (BY_CHUNK) mo.load(o0h + f_h * a.o_sh, o_st, r0, a.T, dk);
            if constexpr (BY_ROW) load_row<D, EXACT && (QW > 1) && D <= 64>(o0h + f_h * a.o_sh, o_st, r0, a.T, dk, c32, g, oreg);
            f_t += KW;
            while (f_t >= nqt) f_t -= nqt, ++f_h;
        }
    };
    auto commit = [&](int buf) {
        uint16_t* t = lds + (buf % NBUF * KW + kg) * TILE;
        mq.template store<true>(t, S, gt);
        mg.template store<true>(t + BMQ * S, S, gt);
        float out = gt >= BMQ ? (MINUS_DELTA ? -row_r : row_r) : EXACT ? -row_r : -row_r * LOG2E;
        if constexpr (BY_CHUNK) {
#pragma unroll
            for (int i = 0; i < Mover<D, G, BMQ>::CPT; ++i) {
                float part = add_products(*reinterpret_cast<const bf16x8*>(&mo.r[i]), *reinterpret_cast<const bf16x8*>(&mg.r[i]), 0.0f);
                part += lane_moved<0xB1>(part);  // lane ^ 1
                part += lane_moved<0x4E>(part);  // lane ^ 2
                if (D == 64) part += lane_moved<0x141>(part);  // the other four of eight
                if (gt % (D / 8) == 0) reinterpret_cast<float*>(t + 2 * BMQ * S)[BMQ + (gt + G * i) / (D / 8)] = MINUS_DELTA ? -part : part;
            }
            if (gt >= BMQ) return;
        }
        if constexpr (BY_ROW) {
            tile_barrier<1>();
            float part = 0.0f;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) part = add_products(oreg[kk], lds_read8(t + BMQ * S + tile_row<D>(c32) * S + kk * 16 + g * 8), part);
            part = xhalf_sum(part);
            if (g == 1) out = MINUS_DELTA ? -part : part;
        }
        if (gt < 2 * BMQ) reinterpret_cast<float*>(t + 2 * BMQ * S)[gt] = out;
    };
    fetch(0);
    bf16x8 kreg[KK], vreg[KK];
    load_row<D, EXACT && (QW > 1) && D <= 64>(kh, static_cast<int>(a.k_st), kw0, a.T, dk, c32, g, kreg);
    load_row<D, EXACT && (QW > 1) && D <= 64>(vh, static_cast<int>(a.v_st), kw0, a.T, dk, c32, g, vreg);
    f32x16 acc[2 * DB];  // dV^T, dK^T
#pragma unroll
    for (int n = 0; n < 2 * DB; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[n][r] = 0.0f;
    const KeyVis kvis(kj, a.T, a.causal, a.window, a.sinks);
    const QueryRange range(a, kw0);
    commit(0);
    tile_barrier<QW>();

    for (int i = 0; i < iters; ++i) {
        if (i + 1 < iters) fetch(i + 1);
        const uint16_t* Qs = lds + (i % NBUF * KW + kg) * TILE;
        const uint16_t* Gs = Qs + BMQ * S;
        const float* rows = reinterpret_cast<const float*>(Qs + 2 * BMQ * S);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int qlo = (qt_lo + c_t) * BMQ + nb * 32;
            if ((KW > 1 && i * KW + kg >= steps) || !range.live(qlo)) continue;
            f32x16 s, dp;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                f32x4 dl = {0.0f, 0.0f, 0.0f, 0.0f};
                if (MINUS_DELTA) dl = *reinterpret_cast<const f32x4*>(rows + BMQ + nb * 32 + qd * 8 + g * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) dp[qd * 4 + e] = dl[e];
            }
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) s = mfma32(lds_read8(Qs + (nb * 32 + tile_row<D>(c32)) * S + kk * 16 + g * 8), kreg[kk], s);
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) dp = mfma32(lds_read8(Gs + (nb * 32 + tile_row<D>(c32)) * S + kk * 16 + g * 8), vreg[kk], dp);
            if (!MINUS_DELTA && !LATE) {
                f32x4 dl[4];  // all asked for before any is used: one by one 1.015 over the 60 shapes
#pragma unroll
                for (int qd = 0; qd < 4; ++qd) dl[qd] = *reinterpret_cast<const f32x4*>(rows + BMQ + nb * 32 + qd * 8 + g * 4);
#pragma unroll
                for (int qd = 0; qd < 4; ++qd)
#pragma unroll
                    for (int e = 0; e < 4; ++e) dp[qd * 4 + e] -= dl[qd][e];
            }
            // lane = key kj; element r = query qlo + (r/4)*8 + 4g + r%4
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                const f32x4 nl = *reinterpret_cast<const f32x4*>(rows + nb * 32 + qd * 8 + g * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[qd * 4 + e] = weight_of<EXACT>(s[qd * 4 + e], a.scale, cexp, nl[e]);
            }
            if (!range.full(qlo)) {
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = kvis(qlo + (r >> 2) * 8 + g * 4 + (r & 3)) ? s[r] : 0.0f;
            }
            accumulate_tr<D, EXACT ? BWD_PARTS : 1, true>(Gs, S, nb * 32, s, acc, lane);
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                f32x4 dl = {0.0f, 0.0f, 0.0f, 0.0f};
                if (LATE) dl = *reinterpret_cast<const f32x4*>(rows + BMQ + nb * 32 + qd * 8 + g * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) dp[qd * 4 + e] = s[qd * 4 + e] * (LATE ? dp[qd * 4 + e] - dl[e] : dp[qd * 4 + e]);
            }
            accumulate_tr<D, EXACT ? BWD_PARTS : 1, true>(Qs, S, nb * 32, dp, acc + DB, lane);
        }
        c_t += KW;
        while (c_t >= nqt) c_t -= nqt;
        if (i + 1 < iters) commit(i + 1);
        tile_barrier<QW>();
    }
    if (KW > 1 && QW == 1) __syncthreads();  // every group has read its last tile
    // partial rows: the sink keys' of a split tail (and, unless the group's heads are split too, of the block's own band) go to
    // tail[unit][piece][dK | dV][32][dk], the others of a split group to part[unit][split][dK | dV][T][dk]
    const bool to_tail = tl.nch > 0 && k0 == 0 && kj < a.sinks && (chunk >= 0 || hs == 1);
    const bool parts = hs > 1 && !to_tail;
    const int64_t pk = to_tail ? ((static_cast<int64_t>(kvu) * (tl.nch + 1) + (chunk >= 0 ? chunk : tl.nch)) * 64 + kj) * dk
                               : (static_cast<int64_t>(kvu) * hs + rr) * 2 * a.T * dk + static_cast<int64_t>(kj) * dk;
    const int64_t pv = pk + static_cast<int64_t>(to_tail ? 32 : a.T) * dk;
    const bool scratch = parts || to_tail, mine = kj < a.T && (chunk < 0 || to_tail);
    void* const room = to_tail ? a.tail : a.part;
    const int64_t rv = scratch ? pv : b * a.dv_sb + hk * a.dv_sh + kj * a.dv_st;
    const int64_t rk = scratch ? pk : b * a.dk_sb + hk * a.dk_sh + kj * a.dk_st;
    void* const dst_v = scratch ? room : a.dv;
    void* const dst_k = scratch ? room : a.dk;
    const bool f32 = scratch || a.grad_f32;
    if constexpr (KW > 1) {
        constexpr int N = JOIN_BOTH<D> ? 2 * DB : DB;
#pragma unroll
        for (int n0 = 0; n0 < 2 * DB; n0 += N) {
            if (n0 > 0) __syncthreads();
            join_shares<N, KW, 2>(acc + n0, reinterpret_cast<float*>(lds) + qg * KW * N * 1024, kg, lane, no_weights, [&](int n, int qd, const f32x4 (&v)[2]) {
                const bool is_v = n0 + n < DB;
                if (mine) store_half(f32, is_v ? dst_v : dst_k, is_v ? rv : rk, is_v ? n : n0 + n - DB, qd, g, v, is_v ? 1.0f : a.scale, dk, is_v ? TurnRow() : turn_row<TURN>(a, hk, kj));
            });
        }
    } else {
        if constexpr (WHOLE_ROWS<D, EXACT>)
            if (dk == D && !a.grad_f32 && hs == 1 && tl.nch == 0) {
                using Rows = RowStrip<D>;
                static_assert(QW * Rows::ELEMS <= NBUF * KW * TILE, "the wavefronts' strips");
                uint16_t* const strip = lds + qg * Rows::ELEMS;
                const int k1 = kj - c32;
#pragma unroll
                for (int db = 0; db < DB; ++db) store_block(false, strip, c32 * Rows::S, db, g, acc[db], 1.0f, D);
                Rows::out(strip, static_cast<uint16_t*>(a.dv) + b * a.dv_sb + hk * a.dv_sh + k1 * a.dv_st, a.dv_st, 0, a.T - k1, lane);
#pragma unroll
                for (int db = 0; db < DB; ++db)
                    store_block(false, strip, c32 * Rows::S, db, g, acc[DB + db], a.scale, D, turn_row<TURN>(a, hk, min(kj, a.T - 1)));
                return Rows::out(strip, static_cast<uint16_t*>(a.dk) + b * a.dk_sb + hk * a.dk_sh + k1 * a.dk_st, a.dk_st, 0, a.T - k1, lane);
            }
        if constexpr (WHOLE_ROWS<D, EXACT> && !TURN)
            if (dk == D && tl.nch == 0) {  // fp32: a share's partial sums, or the gradients
                using Lines = LineStrip<>;
                static_assert(QW * Lines::FLOATS * 2 <= NBUF * KW * TILE, "the wavefronts' strips");
                float* const strip = reinterpret_cast<float*>(lds) + qg * Lines::FLOATS;
                const int k1 = kj - c32;
#pragma unroll
                for (int n = 0; n < 2 * DB; ++n) {
                    const bool is_v = n < DB;
                    const float sc = is_v ? 1.0f : a.scale;
#pragma unroll
                    for (int qd = 0; qd < 4; ++qd)
                        Lines::put(strip, c32, 8 * qd + 4 * g, f32x4{acc[n][qd * 4] * sc, acc[n][qd * 4 + 1] * sc, acc[n][qd * 4 + 2] * sc, acc[n][qd * 4 + 3] * sc});
                    float* const to = parts  ? a.part + ((static_cast<int64_t>(kvu) * hs + rr) * 2 + (is_v ? 1 : 0)) * a.T * D
                                      : is_v ? static_cast<float*>(a.dv) + b * a.dv_sb + hk * a.dv_sh
                                             : static_cast<float*>(a.dk) + b * a.dk_sb + hk * a.dk_sh;
                    const int64_t st = parts ? D : is_v ? a.dv_st : a.dk_st;
                    Lines::out(strip, to + k1 * st + (is_v ? n : n - DB) * 32, st, a.T - k1, lane);
                }
                return;
            }
        if (!mine) return;
#pragma unroll
        for (int n = 0; n < 2 * DB; ++n) {
            if (n < DB)
                store_block(f32, dst_v, rv, n, g, acc[n], 1.0f, dk);
            else
                store_block(f32, dst_k, rk, n - DB, g, acc[n], a.scale, dk, turn_row<TURN>(a, hk, kj));
        }
    }
}
template <int D, int QW, int KW, int NB, bool EXACT, int OCC>
__global__ __launch_bounds__(64 * QW * KW, OCC) void split_dkdv(AttnArgs a) {
    all_arguments(a);
    __shared__ __attribute__((aligned(16))) uint16_t lds[dkdv_lds<D, QW, KW, NB>()];
    int blk, rr, kvu;
    if (map_key_block(a, 32 * QW, blk, rr, kvu)) dkdv_block<D, QW, KW, NB, EXACT, false>(a, blk, rr, kvu, lds);
}

// ---- dK, dV and dQ in one launch, as in attn_f32_split.hip ----
// Blocks 0 .. dkdv_ids - 1 are the dK/dV launch's, which forms its own delta, and the others the dQ launch's.
template <int D, bool EXACT, bool TURN>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void split_bwd(AttnArgs a, int dkdv_ids) {
    all_arguments(a);
    constexpr int Q = dq_lds<D, 1, 4, 1>(), K = dkdv_lds<D, 1, 4, 1>();
    __shared__ __attribute__((aligned(16))) uint16_t lds[Q > K ? Q : K];
    const int id = static_cast<int>(blockIdx.x);
    int blk, rr, kvu, b, h, hk, qblk;
    if (id < dkdv_ids) {
        if (map_key_block(a, 32, blk, rr, kvu, id)) dkdv_block<D, 1, 4, 1, EXACT, true, FROM_DELTA<D, EXACT>, TURN>(a, blk, rr, kvu, lds);
    } else if (map_query_block(a, (a.T + 31) / 32, b, h, hk, qblk, id - dkdv_ids)) {
        dq_block<D, 1, 4, 1, EXACT, false, TURN>(a, 1, b, h, hk, qblk, lds);
    }
}

// ---- the same of wavefronts that own their rows (split_takes_joined) ----
// dK/dV forms delta from the chunks of O beside those of dO while it moves a tile (up to 64 columns, whose chunks are in 4 or 8 neighbouring
// lanes; above, it is read): a launch of delta before this one cost 4 us more, of 13 to 60.
template <int D, bool EXACT, bool DQ_MINUS, bool DKDV_MINUS, bool TURN>
__global__ __launch_bounds__(256, 2) void split_joined(AttnArgs a) {
    all_arguments(a);
    constexpr bool OWN_DELTA = D <= 64;
    constexpr int Q = dq_lds<D, 4, 1, 2>(), K = dkdv_lds<D, 4, 1, 2>();
    __shared__ __attribute__((aligned(16))) uint16_t lds[Q > K ? Q : K];
    const JoinedBlocks jb(a, 128);
    int rank, r, kvu;
    if (!jb.map(a, rank, r, kvu)) return;
    if (r < a.head_split) return dkdv_block<D, 4, 1, 2, EXACT, OWN_DELTA, DKDV_MINUS, TURN>(a, rank, r, kvu, lds);
    const int b = quotient(kvu, a.Hkv), hk = kvu - b * a.Hkv;
    dq_block<D, 4, 1, 2, EXACT, DQ_MINUS, TURN>(a, OWN_DELTA, b, hk * (jb.each - a.head_split) + r - a.head_split, hk, jb.ranks - 1 - rank, lds);
}

// How a launch shares its work out: four wavefronts with 32 rows each (WIDE; in tiles of 32, SHORT) or two (HALF), or one block of
// 32 rows whose tiles are split between four or eight wavefronts.
enum class Form { NONE, WIDE, SHORT, HALF, FOUR, EIGHT };

// head_dim 64, launches that fill the chip: rows owned by wavefronts, against the kernels of the other files. A wavefront that holds
// K and V of its 32 keys needs no P from another, no ring and one barrier a tile, and at 64 columns two of its workgroups fit
// a CU where one of the others does (bf16, forward + backward kernels of head_dim 64, us, other | WIDE | HALF):
//   dK/dV    causal T 512 x 16, 8 heads 25.4 | 21.5 | 22.9;  T 1024 x 8, 8 heads 34 | 31 | 32;  T 2048 x 4, 14 heads on 2 110 | 89 | 89;
//            T 4096 x 4, 16 heads 327 | 281 | 302;  T 4016, 16 heads 83 | 98 | 100;  T 2378 x 3, 4 heads 34 | 56 | 56
//            no mask T 777 x 6, 12 heads 49 | 36 | 38;  T 1749, 16 heads 67 | 53 | 66;  T 195 x 57, 2 heads 11.2 | 11.8 | 13.5
//            window 69, 16 sinks, T 1889, 16 heads 30 | 24 | 24;  window 256, 4 sinks, T 4096 x 4, 16 heads 127 | 120 | 124
//   dQ       causal T 2048 x 4, 14 heads 64 | 59 | 63;  T 4096 x 4, 16 heads 223 | 212 | 243;  T 3190 x 2, 8 heads 75 | 65 | 66
//            no mask T 777 x 6, 12 heads 29.8 | 28.1 | 29.7;  window 43, T 1976, few heads (bands of 300 to 1700 blocks) 1.1 times with HALF
//   forward  window 256, T 4096 x 4, 16 heads 59 | 58 | 65, SHORT 45;  window 128, T 700 x 8, 16 heads 20.5 | 20.1 | 18.1, SHORT 15.8;
//            without a band the forward of attn_fwd_mfma.hip is ahead
// Long causal chains of few units stay with 64 keys a wavefront (mfma_dkdv3).
bool narrow_band(const AttnArgs& a) { return a.window > 0 && a.window <= 512 && chain_tokens(a) < a.T; }
Form fwd_form_64(const AttnArgs& a) {
    const int64_t blocks = static_cast<int64_t>((a.T + 31) / 32) * a.Hq * a.B;
    if (!narrow_band(a) || 2 * a.window > a.T) return Form::NONE;
    return blocks >= 1700 ? Form::SHORT : blocks >= 300 ? Form::HALF : Form::NONE;
}
Form dq_form_64(const AttnArgs& a) {
    const int64_t units = static_cast<int64_t>(a.Hq) * a.B, n = (a.T + 127) / 128;
    if (chain_tokens(a) < a.T) {
        const int64_t blocks = static_cast<int64_t>((a.T + 31) / 32) * units;
        return narrow_band(a) && a.T >= 256 && blocks >= 300 && blocks < 1700 ? Form::HALF : Form::NONE;
    }
    // (without a mask 64 queries a wavefront, mfma_dq3, are ahead from 4096 tokens on: T 5856 x 2, 16 heads 394 | 422)
    if (!a.causal) return a.T >= 100 && a.T < 4096 && units * n >= (a.T < 1000 ? 200 : 330) ? Form::WIDE : Form::NONE;
    return a.T >= 256 && units * (n + 1) >= 400 ? Form::WIDE : Form::NONE;
}
// splits: how many workgroups share the heads of a group
Form dkdv_form_64(const AttnArgs& a, int splits) {
    const int64_t units = static_cast<int64_t>(a.Hkv) * a.B * splits, n = (a.T + 127) / 128;
    if (a.T <= 64 || (splits > 1 && a.T < 400)) return Form::NONE;
    if (chain_tokens(a) < a.T) {
        if (a.sinks > 0) return a.window <= 256 && units * n >= 300 ? Form::HALF : Form::NONE;
        return 3 * a.window <= 2 * a.T && units * n >= 230 ? Form::HALF : Form::NONE;
    }
    if (!a.causal) return a.T > 250 ? (units * n >= 160 ? Form::WIDE : Form::NONE) : units * n >= 440 ? Form::HALF : Form::NONE;
    if (units * (n + 1) < (a.T >= 2000 ? 560 : 500)) return Form::NONE;  // the longest chains against all there is to do
    return a.T >= 400 ? Form::WIDE : Form::HALF;
}

// Which form, from the number of 32-row blocks of the launch (`blocks`) and the length of a block's chain. A block split between
// eight wavefronts has the shortest chain but fills half a CU or more, so it wins while the blocks come to about one
// per CU; between four, up to two or three per CU; beyond that the chip is full either way and rows that share a
// tile's trip to LDS win. Measured (us, bf16, causal; eight | four | the kernels of head_dim 64 / 128 without a split):
//   forward, head_dim 64      T 512, 8 heads 7.5 | 8.4 | 11.0;  32 heads 12.1 | 9.0 | 11.3;  64 heads 22 | 14.6 | 11.8
//                             T 4096, 1 head 21 | 35 | 58;  4 heads 29 | 35 | 58;  8 heads 51 | 51 | 59
//                             T 1024, 32 heads 26 | 21 | 19;  T 2048, 16 heads 34 | 31 | 32;  T 128, 1 head 5.6 | 5.3 | 5.9
//   dQ, head_dim 64           T 512, 32 heads 15 | 11 | 17;  T 1024, 32 heads 32 | 25 | 27;  T 4096, 8 heads 60 | 59 | 89
//   dK/dV, head_dim 64        T 512, 32 heads 16 | 16 | 22;  T 1024, 32 heads 34 | 38 | 33;  T 4096, 4 heads 35 | 50 | 79
//   forward, head_dim 128     T 512, 8 heads 11 | 12 | 16;  32 heads 18 | 18 | 16;  T 1024, 16 heads 22 | 23 | 26
//   dQ, head_dim 128          T 512, 8 heads 16 | 14 | 22;  T 2048, 8 heads 41 | 40 | 68;  16 heads 84 | 79 | 72
//   dK/dV, head_dim 128       T 512, 32 heads - | 24 | 34;  T 2048, 8 heads - | 48 | 66;  16 heads - | 94 | 69
// Where the kernels without a split exist, they win on short chains as soon as the blocks exceed the CUs, on even chains
// from there on, and always where a chain is a single tile of theirs (us, split | unsplit, forward, dQ, dK/dV):
//   head_dim 64, T 64, 16 units 5.3 6.6 6.7 | 4.3 5.4 5.7;     T 180, 32 units 6.5 8.5 8.8 | 6.7 9.3 9.5, 64 units 8.0 10.1 15.9 | 6.8 9.4 9.7
//   T 600, window 128, 16 units 10.5 13.7 15.0 | 9.2 11.2 10.9;  T 929, no mask, 16 units 16.8 20.1 25.0 | 17.5 25.9 28.6
//   head_dim 128, T 600, window 60, 16 units 12.2 17.8 18.2 | 11.0 13.6 10.5;  T 1100, no mask, 16 units 41 60 72 | 29 43 54
// From 4096 tokens on head_dim 128 stays with the unsplit kernels whatever the number of units. That is not for speed (causal,
// forward, dQ, dK/dV, us, unsplit | split: 4096 x 1 head 86 118 94 | 32 67 67, 4 heads 88 120 96 | 42 98 80; 8192 x 1 167 223 179
// | 54 206 126; window 256, 2 heads 17 20 26 | 10 14 31). A unit alone, a unit in a batch and the prefix of a longer sequence are
// then the same bits (O, LSE and dQ), which the tests of long sequences compare.
// Everywhere else the sums' order, and so the last bits, depend on how many blocks a launch has.
bool unsplit_is_ahead(const AttnArgs& a, int64_t blocks) {
    if (a.dk_dim != 64 && a.dk_dim != 128) return false;  // they take these head sizes only
    if (a.dk_dim == 128 && a.T >= 4096) return true;
    const int chain = chain_tokens(a);
    if (blocks <= 256) return false;
    if ((chain < 512 || a.dk_dim == 128) && blocks > 540) return true;
    return chain < 256 || (even_chains(a) && !(a.dk_dim == 64 && chain >= 768 && blocks <= 600));
}
// Head sizes other than 64 and 128, FOUR | WIDE. Many short chains of equal length are ahead unsplit from two blocks a CU on
// (head_dim 80, T 64 x 87, 8 heads, no mask: forward 10.8 | 7.0 us, dQ 27 | 18, dK/dV 47 | 21; T 2089 x 4, window 20: dQ 38 | 29,
// dK/dV 71 | 33), long causal ones stay split for longer, the more so the fewer columns (forward: head_dim 32, T 3201 x 3, 4 heads 30 | 67, T 5179 x
// 2, 8 heads 91 | 105; head_dim 96, T 1886 x 3, 8 heads 45 | 53, T 4618, 16 heads 148 | 128).
bool wide_chains(const AttnArgs& a, int64_t blocks) { return a.dk_dim > 32 && even_chains(a) && chain_tokens(a) <= 160 && blocks > 550; }
Form fwd_form(const AttnArgs& a) {
    if (a.dk_dim == 64)
        if (const Form f = fwd_form_64(a); f != Form::NONE) return f;
    const int64_t blocks = static_cast<int64_t>((a.T + 31) / 32) * a.Hq * a.B;
    const bool plain = a.dk_dim == 64 || a.dk_dim == 128;
    if (unsplit_is_ahead(a, blocks) || (plain && a.T <= 64)) return Form::NONE;
    // (six tiles on eight wavefronts, T 170, 38 heads of 128: four 8.8 us, eight 9.8, unsplit 9.0)
    if (blocks <= 256) return chain_tokens(a) <= (plain ? 192 : 160) ? Form::FOUR : Form::EIGHT;
    if (!plain) {
        const int chain = chain_tokens(a);
        const int64_t longest = a.dk_dim <= 32 ? (chain >= (a.causal ? 400 : 2000) ? 2600 : 1100) : (a.causal && chain >= 900 ? 1450 : 1100);
        return blocks <= longest && !wide_chains(a, blocks) ? Form::FOUR : Form::WIDE;
    }
    // past 512 blocks eight wavefronts a block, two workgroups to a CU, are a second round (no mask, T 1700, 10 heads of 64:
    // eight 34 us, four 24, unsplit 28; causal, T 850, 19 heads of 128: 25, 17, 24)
    if (blocks <= 600)
        return chain_tokens(a) >= (a.dk_dim == 64 ? 1536 : 768) ? (blocks <= 512 ? Form::EIGHT : Form::FOUR)
               : a.dk_dim == 64 && a.causal                    ? Form::FOUR
                                                               : Form::NONE;
    return blocks <= 1100 && chain_tokens(a) >= 3000 ? Form::EIGHT : Form::NONE;
}
Form dq_form(const AttnArgs& a) {
    if (a.dk_dim == 64)
        if (const Form f = dq_form_64(a); f != Form::NONE) return f;
    const int64_t blocks = static_cast<int64_t>((a.T + 31) / 32) * a.Hq * a.B;
    const bool plain = a.dk_dim == 64 || a.dk_dim == 128;
    // (causal, T 80, 77 heads of 128: four wavefronts 10.8 us, unsplit 10.1; T 100 11.0 and 11.6)
    if (unsplit_is_ahead(a, blocks) || (plain && a.T <= (a.dk_dim == 128 && a.causal ? 96 : 64))) return Form::NONE;
    // above 96 columns eight wavefronts of this kernel do not fit the registers
    const Form best = a.dk_dim > 96 || chain_tokens(a) <= 160 ? Form::FOUR : Form::EIGHT;
    if (blocks <= 256) return best;
    if (!plain) {  // FOUR | WIDE: T 5395, 8 heads, head_dim 32: 75 us | 126; T 1169 x 2, 16 heads, 80: 41 | 46
        const bool far = a.causal && chain_tokens(a) >= (a.dk_dim <= 32 ? 1200 : 900);
        return blocks <= (!far || a.dk_dim > 96 ? 1100 : a.dk_dim <= 32 ? 2600 : 1250) && !wide_chains(a, blocks) ? Form::FOUR : Form::WIDE;
    }
    if (blocks <= 600) return chain_tokens(a) >= 1536 ? best : a.dk_dim == 64 || chain_tokens(a) >= 768 ? Form::FOUR : Form::NONE;
    return blocks <= 1100 && a.dk_dim == 64 && chain_tokens(a) >= 1000 ? Form::FOUR : Form::NONE;
}
// Every head its own, head_dim 64 and 128: where the unsplit kernels are ahead of a block split between four wavefronts. At 128
// one such workgroup fills a CU, so that short chains are behind even in one round (causal, four | unsplit, us: T 80, 77 heads
// 11.3 | 10.0, T 170, 38 heads 13.6 | 12.5, T 250, 29 heads 14.6 | 15.4), and the blocks of a second round have to be few against
// the chain (T 300, 38 heads 22 | 18; T 400, 21 heads 19 | 20.5, 34 heads 25 | 21; T 600, 17 heads 26 | 29, 26 heads 30 | 28; T
// 1000, 16 heads 39 | 40; T 4000, 5 heads 106 | 92). At 64 two do: T 300, 50 heads 11.4 | 13.3, 60 heads 14.6 | 13.2.
bool short_chains(const AttnArgs& a, int64_t blocks) {
    const int chain = chain_tokens(a);
    if (a.dk_dim == 64) return blocks > 512 && chain < 400;
    if (blocks <= 256) return a.T <= (a.window > 0 ? 250 : 180);
    return blocks > std::min(512, 256 + std::max(chain - 350, 0) * 2 / 5);
}
Form dkdv_small_form(const AttnArgs& a) {
    const int64_t blocks = static_cast<int64_t>((a.T + 31) / 32) * a.Hkv * a.B * a.head_split;
    const bool plain = a.dk_dim == 64 || a.dk_dim == 128;
    if (unsplit_is_ahead(a, blocks) || (plain && a.head_split == 1 && (a.T <= 72 || (a.Hq == a.Hkv && short_chains(a, blocks)))))
        return Form::NONE;
    // a band over two tiles and groups of two: the sum over the dealt heads takes longer than they do (T 40, window 13, four
    // heads on two: head_dim 64 10.0 us | 8.6, 128 13.2 | 9.8; groups of four 10.4 | 11.7, 13.7 | 14.2)
    if (plain && a.window > 0 && a.T <= 64 && a.Hq <= 2 * a.Hkv) return Form::NONE;
    const Form best = a.dk_dim > 64 || chain_tokens(a) <= 160 ? Form::FOUR : Form::EIGHT;  // registers, as above
    if (!plain) {  // split | WIDE: T 2933 x 2, 4 heads, head_dim 96: 96 us | 135; T 1714 x 2, 8 heads, 32: 40 | 57
        const bool far = a.causal && chain_tokens(a) >= 1500 && a.dk_dim <= 96;
        const bool wide = a.dk_dim > 64 && wide_chains(a, blocks);  // at 48, T 239 x 9, 8 KV heads, window 47, WIDE is behind: 22 | 16
        return blocks <= (!far ? 700 : a.dk_dim <= 32 ? 1600 : 800) && !wide ? best : Form::WIDE;
    }
    // at 64 eight wavefronts are ahead in one round only, or nearly so where the causal chains are long (us, eight | four | unsplit:
    // T 350, 25 heads 16 | 10.4 | 13.9; T 600, 29 heads 25 | 15.5 | 19; T 2200, 13 heads 37 | 34 | 57, 14 heads 55 | 37 | 46;
    // T 3000, 4 heads 31 | 37 | 63)
    const Form later = a.dk_dim == 64 && blocks > 256 && !(blocks <= 450 && chain_tokens(a) >= 2000 && !even_chains(a)) ? Form::FOUR : best;
    if (blocks <= 600) return later;
    return blocks <= 1100 && a.dk_dim == 64 && chain_tokens(a) >= 2000 ? later : Form::NONE;
}

// The query heads of a group are dealt out where the kernels below this file's lines, or mfma_dkdv3, would be: the workspace is
// sized for that.
int splits_of(const AttnArgs& a) { return bf16_deals_heads(a) ? a.head_split : 1; }
Form dkdv_form(const AttnArgs& a) {
    if (a.dk_dim == 64)
        if (const Form f = dkdv_form_64(a, splits_of(a)); f != Form::NONE) return f;
    return dkdv_small_form(a);
}

template <int D, int QW, int KW, int NB, bool EXACT>
void run_fwd(const AttnArgs& a, hipStream_t st) {
    const int nqb = (a.T + 32 * QW - 1) / (32 * QW);
    hipLaunchKernelGGL((split_fwd<D, QW, KW, NB, EXACT>), dim3(xcd_grid(nqb, a.Hq / a.Hkv, a.Hkv * a.B)), dim3(64 * QW * KW), 0, st, a);
}
template <int D, int QW, int KW, int NB, bool EXACT>
void run_dq(const AttnArgs& a, bool fuse_delta, hipStream_t st) {
    const int nqb = (a.T + 32 * QW - 1) / (32 * QW);
    hipLaunchKernelGGL((split_dq<D, QW, KW, NB, EXACT>), dim3(xcd_grid(nqb, a.Hq / a.Hkv, a.Hkv * a.B)), dim3(64 * QW * KW), 0, st, a,
                       fuse_delta ? 1 : 0);
}
template <int D, int QW, int KW, int NB, bool EXACT>
void run_dkdv(const AttnArgs& a, hipStream_t st) {
    const int nkb = (a.T + 32 * QW - 1) / (32 * QW);
    const dim3 grid(xcd_grid(nkb + tail_blocks(a), a.head_split, a.Hkv * a.B));
    // Two wavefronts to a SIMD cost head sizes up to 96 a few spilled registers: not while there is a workgroup for each CU at
    // most (us, head_dim 80, one | two: T 4263, 6 heads, 204 workgroups 193 | 237; 16 heads on 4, T 1466 x 9, 432: 302 | 272,
    // T 743 x 19, 456: 211 | 185). A few hundred workgroups with one head each are behind with two (4 heads, T 1466 x 9: 78 | 94).
    if (D == 96 && QW > 1 && static_cast<int64_t>(nkb) * a.head_split * a.Hkv * a.B > 256)
        hipLaunchKernelGGL((split_dkdv<D, QW, KW, NB, EXACT, 2>), grid, dim3(64 * QW * KW), 0, st, a);
    else
        hipLaunchKernelGGL((split_dkdv<D, QW, KW, NB, EXACT, D <= 64 ? 2 : 1>), grid, dim3(64 * QW * KW), 0, st, a);
}

template <int D, bool EXACT>
int fwd_of(const AttnArgs& a, Form f, hipStream_t st) {
    if (f == Form::EIGHT) run_fwd<D, 1, 8, 1, EXACT>(a, st);
    if (f == Form::FOUR) run_fwd<D, 1, 4, 1, EXACT>(a, st);
    if constexpr (EXACT)
        if (f == Form::WIDE) run_fwd<D, 4, 1, 2, EXACT>(a, st);
    if constexpr (!EXACT && D == 64) {
        if (f == Form::SHORT) run_fwd<D, 4, 1, 1, EXACT>(a, st);
        if (f == Form::HALF) run_fwd<D, 2, 1, 2, EXACT>(a, st);
    }
    PK_HIP(hipGetLastError());
    return PK_OK;
}
template <int D, bool EXACT>
int dq_of(const AttnArgs& a, Form f, bool fuse_delta, hipStream_t st) {
    if constexpr (D <= 96)
        if (f == Form::EIGHT) run_dq<D, 1, 8, 1, EXACT>(a, fuse_delta, st);
    if (f == Form::FOUR) run_dq<D, 1, 4, 1, EXACT>(a, fuse_delta, st);
    if constexpr (EXACT || D == 64)
        if (f == Form::WIDE) run_dq<D, 4, 1, 2, EXACT>(a, fuse_delta, st);
    if constexpr (!EXACT && D == 64)
        if (f == Form::HALF) run_dq<D, 2, 1, 2, EXACT>(a, fuse_delta, st);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
template <int D, bool EXACT>
int dkdv_of(const AttnArgs& a, Form f, hipStream_t st) {
    if constexpr (D <= 64)
        if (f == Form::EIGHT) run_dkdv<D, 1, 8, 1, EXACT>(a, st);
    if (f == Form::FOUR) run_dkdv<D, 1, 4, 1, EXACT>(a, st);
    if constexpr (EXACT || D == 64)
        if (f == Form::WIDE) run_dkdv<D, 4, 1, 2, EXACT>(a, st);
    if constexpr (!EXACT && D == 64)
        if (f == Form::HALF) run_dkdv<D, 2, 1, 2, EXACT>(a, st);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
template <int D, bool EXACT>
int bwd_of(const OneLaunch& l, hipStream_t st) {
    const dim3 grid(l.dkdv_ids + l.dq_ids);
    if (l.a.turn)
        hipLaunchKernelGGL((split_bwd<D, EXACT, true>), grid, dim3(256), 0, st, l.a, l.dkdv_ids);
    else
        hipLaunchKernelGGL((split_bwd<D, EXACT, false>), grid, dim3(256), 0, st, l.a, l.dkdv_ids);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
// f<D, EXACT>() for the instantiation that serves head_dim dk
#define PK_SPLIT_DISPATCH(call)                        \
    do {                                               \
        const int dk = a.dk_dim;                       \
        if (dk == 64) return call(64, false);          \
        if (dk == 128) return call(128, false);        \
        if (dk <= 32) return call(32, true);           \
        if (dk <= 64) return call(64, true);           \
        if (dk <= 96) return call(96, true);           \
        return call(128, true);                        \
    } while (0)

}  // namespace

bool split_serves(const AttnArgs& a) { return a.dk_dim % 8 == 0 && a.dk_dim <= 128 && bf16_rows_aligned(a); }
bool split_takes_fwd(const AttnArgs& a) { return fwd_form(a) != Form::NONE; }
bool split_takes_dq(const AttnArgs& a) { return dq_form(a) != Form::NONE; }
bool split_takes_dkdv(const AttnArgs& a) { return dkdv_form(a) != Form::NONE; }
bool split_deals_heads(const AttnArgs& a) { return a.head_split > 1 && dkdv_small_form(a) != Form::NONE; }
int launch_split_fwd(const AttnArgs& a, hipStream_t st) {
#define PK_CALL(D, E) fwd_of<D, E>(a, fwd_form(a), st)
    PK_SPLIT_DISPATCH(PK_CALL);
#undef PK_CALL
}
int launch_split_dq(const AttnArgs& a, bool fuse_delta, hipStream_t st) {
#define PK_CALL(D, E) dq_of<D, E>(a, dq_form(a), fuse_delta, st)
    PK_SPLIT_DISPATCH(PK_CALL);
#undef PK_CALL
}
int launch_split_dkdv(const AttnArgs& a_in, hipStream_t st) {
    AttnArgs a = a_in;
    const Form f = dkdv_form(a);
    a.head_split = splits_of(a);
    if (!split_tail_pays(a, a.head_split, f == Form::WIDE ? 128 : f == Form::HALF ? 64 : 32)) a.tail = nullptr;
    const auto run = [&]() -> int {
#define PK_CALL(D, E) dkdv_of<D, E>(a, f, st)
        PK_SPLIT_DISPATCH(PK_CALL);
#undef PK_CALL
    };
    if (const int rc = run()) return rc;
    return a.head_split > 1 ? launch_gqa_reduce(a, st) : a.tail ? launch_sink_tail_reduce(a, st) : PK_OK;
}

// dQ and dK/dV in one launch: while their workgroups find room on the chip together, two to a CU up to 64 columns and one above.
// Measured, the launches of a backward one after the other | this one (us): head_dim 64 T 64, 16 heads 11.1 | 7.0, T 300 x 2, 8 heads 23 | 17;
// 128 T 128 x 2, 8 heads 16 | 12, T 25 x 8, 1 head 11.0 | 12.3, T 64 x 25, 4 heads, window 18 16 | 22; 96 no mask, T 2000, 4 heads 74 | 87; 24 T 4000,
// 1 head 53 | 58. Over 460 random shapes of up to 1000 blocks it is 1.15 to 1.6 times as fast as they are below these lines.
bool split_takes_bwd(const AttnArgs& a) {
    const OneLaunch l(a);
    const int ids = l.dkdv_ids + l.dq_ids;
    // bands of more than a thousand keys, T 3201, window 1268, 4 heads on 1: 57 | 71
    if (chain_tokens(a) > (chain_tokens(a) < a.T ? 1024 : 2600)) return false;
    if (a.dk_dim <= 32) return ids <= (even_chains(a) ? 400 : 960);
    if (a.dk_dim <= 64) return ids <= (a.T <= 64 ? 400 : even_chains(a) ? 640 : 800);  // (one tile: T 31 x 84, 4 heads of 64 10.9 | 13.3)
    if (a.dk_dim <= 96) return ids <= (even_chains(a) ? 380 : 400);
    return ids <= 256 && (a.dk_dim < 128 || a.T > 32);
}
// Blocks of 128 keys and of 128 queries in one launch. Where either launch by itself is a round of the chip or less, its longest chains
// last as long as it does; together one's run beside the other's, and rows that share a tile's trip to LDS do half of the work there that blocks
// of 32 do. `u` blocks of queries, `n` to a head. Measured, one after the other (or in blocks of 32) | joined, us:
//   64 columns     T 470 x 8, 8 heads (u 256) 31 | 21;  T 923 x 7, 4 heads (224) 48 | 33;  T 1104 x 2, 16 heads on 8 (288) 67 | 46;  T 150 x 4, 16
//                  heads (128) 15.4 | 11.0;  T 1024 x 8, 8 heads (512) 57 | 52;  T 4945, 8 heads (312) 190 | 138;  no mask, T 423 x 14, 2 heads (112) 30 | 19
//     below        T 1066, 16 heads on 4 (144) 38 | 39;  T 1982, 8 on 4 (128) 51 | 61;  T 3520, 8 heads (224) 82 | 94;  no mask, T 3347, 4 on 1 (108) 90 | 114
//     above        T 1182 x 8, 8 heads (640) 69 | 75;  T 2048 x 4, 14 heads on 2 (896) 149 | 153;  no mask, T 777 x 6, 12 heads (504) 65 | 69
//   32, 48         T 148 x 58, 2 heads of 48 (232) 21 | 13;  T 486 x 3, 16 heads on 4 (192) 34 | 26;  T 1746, 32 on 8 of 48 (448) 127 | 111
//     below, above T 961, 16 heads (128) 29 | 35;  T 1715, 14 on 2 of 48 (196) 72 | 79;  T 1951, 32 on 16 (512) 106 | 110
//   80, 96 (delta in a launch of its own)  T 49 x 131, 2 heads (262) 37 | 21;  T 393 x 7, 14 on 2 (392) 70 | 56;  T 2515, 14 on 2 (280) 217 | 173
//     below, above T 1110, 16 heads (144) 63 | 69;  T 2573, 8 on 4 (168) 125 | 157;  T 129 x 15, 16 on 8 (480) 40 | 44
//   bands, every head its own  64: T 651 x 2, 8 heads, window 235 (96) 26 | 17;  T 4247, 8 heads, 336 (272) 36 | 32;  T 159 x 7, 16 on 8 23 | 18
//     not          T 1128, 16 heads, 178, 1 sink, whose block is walked whole (144) 33 | 42;  T 1777, 16 on 8 44 | 116;  T 211 x 8, 4 heads (64) 11 | 14;
//                  32 columns under long bands: T 3810, 8 heads, 1771 (240) 76 | 90;  T 2632, 16 heads, 1403 (336) 79 | 84
//   past 512 workgroups, which are there at once, both kinds share a second round: 64, T 4950, 8 heads, window 25 (312) 18.4 | 21.2;  no mask, T 4433,
//     8 on 4 (280) 256 | 290;  96, no mask, T 222 x 53, 4 heads (424) 49 | 56;  T 37 x 49, 8 heads (392) 19 | 22;  and with groups, whose blocks of keys
//     walk all heads: T 3156, 16 on 4 (400) 423 | 525;  T 1424, 16 on 4 (192) 128 | 135
bool split_takes_joined(const AttnArgs& a) {
    if (a.dk_dim > 96 || a.T <= 32) return false;
    const int64_t n = (a.T + 127) / 128, u = n * a.Hq * a.B;
    if (a.window > 0)
        return a.Hq == a.Hkv && (a.sinks == 0 || a.T <= 600) &&
               (a.dk_dim == 64 ? u >= (chain_tokens(a) <= 1024 ? 84 : 150) && u <= (a.T > 2500 && a.window < 128 ? 256 : 450)
                               : chain_tokens(a) <= 1024 && u >= 190 && u <= 390);
    if (a.dk_dim == 64)
        return a.causal ? u >= (n == 1 ? 60 : n <= 4 ? 104 : n <= 12 ? 150 : n <= 17 ? 200 : 290) && u <= (n <= 2 ? 440 : 560)
                        : u >= (n == 1 ? 60 : n <= 8 ? 110 : n <= 32 ? 150 : 170) && u <= (n <= 32 ? 300 : 256);
    if (a.dk_dim < 64)
        return a.causal ? n <= 16 && u >= (n == 1 ? 60 : n <= 2 ? 112 : n <= 7 ? 190 : 300) && u <= 450
                        : n <= 12 && u >= (n == 1 ? 60 : n <= 6 ? 84 : 200) && u <= 300;
    if (!a.causal && n > 8 && a.Hq > a.Hkv) return false;
    return u >= (n == 1 ? 80 : n <= 5 ? 150 : n <= 12 ? 200 : 232) && u <= (a.causal ? 420 : a.T <= 64 ? 380 : 400);
}
template <int D, bool EXACT, bool DQ_MINUS = false, bool DKDV_MINUS = false>
int joined_of(const AttnArgs& a, hipStream_t st) {
    const dim3 grid(JoinedBlocks(a, 128).grid(a));
    if (a.turn)
        hipLaunchKernelGGL((split_joined<D, EXACT, DQ_MINUS, DKDV_MINUS, true>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((split_joined<D, EXACT, DQ_MINUS, DKDV_MINUS, false>), grid, dim3(256), 0, st, a);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
int launch_split_joined(const AttnArgs& a_in, hipStream_t st) {
    AttnArgs a = a_in;
    a.head_split = splits_of(a);
    a.tail = nullptr;
    if (a.dk_dim > 64)
        if (const int rc = launch_row_delta(a, true, st)) return rc;
    const auto run = [&]() -> int {
        if (a.dk_dim == 64) {
            const Form alone = dq_form(a);
            const bool dkdv = split_takes_dkdv(a_in) || mfma_dkdv3_takes(a_in);
            if (alone == Form::NONE || alone == Form::FOUR) return dkdv ? joined_of<64, false, false, true>(a, st) : joined_of<64, false>(a, st);
            return dkdv ? joined_of<64, false, true, true>(a, st) : joined_of<64, false, true>(a, st);
        }
        if (a.dk_dim <= 32) return joined_of<32, true>(a, st);
        if (a.dk_dim <= 64) return joined_of<64, true>(a, st);
        return joined_of<96, true>(a, st);
    };
    if (const int rc = run()) return rc;
    return a.head_split > 1 ? launch_gqa_reduce(a, st) : PK_OK;
}
int launch_split_bwd(const AttnArgs& a, hipStream_t st) {
    const OneLaunch l(a);
    const auto run = [&]() -> int {
#define PK_CALL(D, E) bwd_of<D, E>(l, st)
        PK_SPLIT_DISPATCH(PK_CALL);
#undef PK_CALL
    };
    if (const int rc = run()) return rc;
    return l.finish(st);
}

}  // namespace pk
