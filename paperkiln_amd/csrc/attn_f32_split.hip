// fp32 attention (forward, dQ, dK/dV) in workgroups whose wavefronts share the CONTRACTION, the fp32 counterpart of
// attn_split.hip: one block of 32 rows per workgroup, KW wavefronts that take every KW-th 32-row tile of the other side,
// each from LDS of its own, results joined at the end. Operand layouts of v_mfma_f32_32x32x2_f32 as in
// attn_f32_mfma.hip; products and sums are fp32 throughout.
//
// What bounds it: a 32 x 32 block is D matrix instructions of 64 clocks per product, so four wavefronts of a CU are bound
// by the matrix pipe as soon as each has something to do. The kernels of attn_f32_mfma.hip give a workgroup 128 rows and
// let each wavefront walk every tile: 256 workgroups of very different length at B=4 H=8 T=1024, where the longest is
// half the launch. Here there are four times as many, a quarter or an eighth as long.
//
// They are also the path of every head size that is a multiple of 4 up to 128 but not 32, 64 or 128 (columns padded to
// D = 32, 64, 96 or 128, zero past the real size and not stored).
#include "attn_split.h"

namespace pk {
namespace {

constexpr float LOG2E = 1.4426950408889634f;

__device__ inline f32x16 mfma2(float a, float b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
__device__ inline int crow(int r, int g) { return (r >> 2) * 8 + 4 * g + (r & 3); }

// rows r0 .. T - 1 of a head; r0 < T. Whatever lies past them reads as zero.
__device__ inline __amdgpu_buffer_rsrc_t rows_from(const float* head, int st, int r0, int T, int dk) {
    const int64_t left = (static_cast<int64_t>(T - r0 - 1) * st + dk) * 4;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(head) + static_cast<int64_t>(r0) * st, 0,
                                             left > 0x7fffffff ? 0x7fffffff : static_cast<int>(left), 0x00020000);
}

// A 32-row tile of a [T, dk] fp32 matrix, moved by one wavefront through a buffer resource (rows past T and chunks past
// dk read as zero) into LDS rows of pitch D + 4: 16-byte row reads of 16 rows then touch all 64 banks once.
template <int D>
struct Mover32 {
    static constexpr int NCH = D / 4, CPT = 32 * NCH / 64, P = D + 4;
    int off[CPT];
    u32x4 r[CPT];
    __device__ void init(int lane, int st, int dk) {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int c = lane + 64 * i, row = c / NCH, ch = c % NCH;
            off[i] = ch * 4 < dk ? (row * st + ch * 4) * 4 : static_cast<int>(OUTSIDE);
        }
    }
    __device__ void load(const float* head, int st, int r0, int T, int dk) {
        const __amdgpu_buffer_rsrc_t rs = rows_from(head, st, r0, T, dk);
#pragma unroll
        for (int i = 0; i < CPT; ++i) r[i] = tile_load16(rs, off[i]);
    }
    __device__ void store(float* lds, int lane) const {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int c = lane + 64 * i;
            *reinterpret_cast<u32x4*>(lds + (c / NCH) * P + (c % NCH) * 4) = r[i];
        }
    }
};

// Row r0 + c32 of a head as an operand: chunk j holds columns 8j + 4g .. +3; zero past T and past dk.
template <int D>
__device__ inline void load_row32(const float* head, int st, int r0, int T, int dk, int c32, int g, f32x4* out) {
    const __amdgpu_buffer_rsrc_t rs = rows_from(head, st, r0, T, dk);
    const int row = c32 * st * 4 + 16 * g;
#pragma unroll
    for (int j = 0; j < D / 8; ++j) {
        const u32x4 v = tile_load16(rs, 8 * j + 4 * g < dk ? row + 32 * j : static_cast<int>(OUTSIDE));
        out[j] = *reinterpret_cast<const f32x4*>(&v);
    }
}

// The same of a tensor with any row stride (O's is not asked about). The branch around each load keeps it where it is written: free to move, the
// scheduler holds the row through the products before its use (backward, 128 columns, T 300, 4 heads: 46.5 us | 52.6; 32, T 2900, 4 heads 86 | 96).
template <int D>
__device__ inline void load_row_of_o(const float* head, int64_t st, int row, int T, int dk, int g, f32x4* out) {
#pragma unroll
    for (int j = 0; j < D / 8; ++j) {
        const int col = 8 * j + 4 * g;
        f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
        if (row < T && col < dk) z = *reinterpret_cast<const f32x4*>(head + row * st + col);
        out[j] = z;
    }
}

// The order inside both products is pinned -- the fragments of the next group of matrix instructions, then this group --
// so that no fragment is waited for and no more than two groups of them hold registers (left to itself the scheduler
// reads a whole tile ahead and spills at D = 128).
//
// (rows of the tile) . b, contracted over the columns; b from registers, or from an LDS tile of the same layout
template <int D, typename B>
__device__ inline f32x16 rows_dot(const float* tile, B b, int c32, int g) {
    constexpr int NJ = D / 8, P = D + 4;
    const float* row = tile + c32 * P + 4 * g;
    f32x16 t;
#pragma unroll
    for (int r = 0; r < 16; ++r) t[r] = 0.0f;
    f32x4 a = *reinterpret_cast<const f32x4*>(row), bb = b(0);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        f32x4 na = a, nb = bb;
        if (j + 1 < NJ) {
            na = *reinterpret_cast<const f32x4*>(row + 8 * (j + 1));
            nb = b(j + 1);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) t = mfma2(a[i], bb[i], t);
        a = na, bb = nb;
    }
    return t;
}
// acc[db] += tile^T c: register r of the C tile is the operand of the tile's row crow(r, g)
template <int D>
__device__ inline void accumulate_tr32(const float* tile, const f32x16& c, f32x16* acc, int c32, int g) {
    constexpr int DB = D / 32, P = D + 4;
    float m[DB], n[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) m[db] = tile[crow(0, g) * P + c32 + 32 * db];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        if (r + 1 < 16) {
#pragma unroll
            for (int db = 0; db < DB; ++db) n[db] = tile[crow(r + 1, g) * P + c32 + 32 * db];
        }
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[db] = mfma2(m[db], c[r], acc[db]);
#pragma unroll
        for (int db = 0; db < DB; ++db) m[db] = n[db];
    }
#pragma unroll
    for (int r = 0; r + 1 < 16; ++r) {
        __builtin_amdgcn_sched_group_barrier(0x100, DB, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, DB, 0);
    }
}

// a quad of a lane's output row
__device__ inline void store_quad(void* base, int64_t row_off, int db, int qd, int g, const f32x4& v, float sc, int dk, const TurnRow& turn = {}) {
    const int col = 32 * db + 8 * qd + 4 * g;
    const f32x4 o = {v[0] * sc, v[1] * sc, v[2] * sc, v[3] * sc};
    if (col < dk) *reinterpret_cast<f32x4*>(static_cast<float*>(base) + row_off + col) = turn.quad(o, col, dk);
}

// Both tensors of a wavefront's next tile on their way together, or one behind the other's product. Where chains are a tile or two, as in
// most launches of these kernels, the second trip to memory is a fifth of the launch. Above 64 columns the registers do not hold both; dQ and
// dK/dV take it at 32 columns in one launch (by themselves they run four and three wavefronts to a SIMD; at 64 T 512, 8 heads is 28.0 us | 29.5).
//
// With it, the addresses formed once (head_of) and all wavefronts in the join, T 128 x 2, 4 heads of 32: forward 5.6 -> 4.9 us, backward 9.7 -> 8.5; T 2900,
// 4 heads 37.7 -> 37.2, 99.9 -> 86.1; 128 columns, T 300, 4 heads 21.2 -> 20.6, 55.2 -> 46.5; 96, no mask, T 700, 4 heads 29.5 -> 28.1, 56.1 -> 56.5.
template <int D>
constexpr bool BOTH_AHEAD = D <= 64;

// ---- forward ----
// The launch bounds ask for the wavefronts that the LDS leaves room for: four to a SIMD at head_dim 32, two at 64 (backward,
// head_dim 24, T 402 x 22, 16 heads: 204 -> 173 us; head_dim 64, T 731 x 4, 28 heads on 4, window 309: 296 -> 242).
template <int D, int KW>
__global__ __launch_bounds__(64 * KW, D <= 32 ? 4 : D <= 64 ? 2 : 1) void f32_split_fwd(AttnArgs a) {
    all_arguments(a);
    constexpr int DB = D / 32, P = D + 4, TILE = 2 * 32 * P, RED = KW * (DB * 1024 + 128);
    __shared__ __attribute__((aligned(16))) float lds[KW * TILE > RED ? KW * TILE : RED];
    const int lane = threadIdx.x & 63, kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, c32 = lane & 31, dk = a.dk_dim;
    int b, h, hk, qblk;
    if (!map_query_block(a, (a.T + 31) / 32, b, h, hk, qblk)) return;
    const int q0 = qblk * 32, qhi = q0 + 31, qi = q0 + c32;
    const float *const kh = head_of<float>(a.k, a.k_sb, b, a.k_sh, hk), *const vh = head_of<float>(a.v, a.v_sb, b, a.v_sh, hk), *const qh = head_of<float>(a.q, a.q_sb, b, a.q_sh, h);
    const int k_st = static_cast<int>(a.k_st), v_st = static_cast<int>(a.v_st);
    const float cexp = a.scale * LOG2E;
    float* const Ks = lds + kg * TILE;
    float* const Vs = Ks + 32 * P;

    Mover32<D> mk, mv;
    mk.init(lane, k_st, dk);
    mv.init(lane, v_st, dk);
    const KeyTiles kt(a, q0, 32, 32);
    if (kg < kt.n) mk.load(kh, k_st, kt.tile(kg) * 32, a.T, dk);
    f32x4 qreg[D / 8];
    load_row32<D>(qh, static_cast<int>(a.q_st), q0, a.T, dk, c32, g, qreg);
    if (BOTH_AHEAD<D> && kg < kt.n) mv.load(vh, v_st, kt.tile(kg) * 32, a.T, dk);
    f32x16 acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;
    float m = -1e30f, l = 0.0f;  // the reference's running-max seed, src/ops.cpp:881
    const QueryVis vis(qi, a.T, a.causal, a.window, a.sinks);

    for (int at = kg; at < kt.n; at += KW) {
        const int k0 = kt.tile(at) * 32;
        mk.store(Ks, lane);
        tile_barrier<1>();
        if (!BOTH_AHEAD<D>) mv.load(vh, v_st, k0, a.T, dk);
        f32x16 s = rows_dot<D>(Ks, [&](int j) { return qreg[j]; }, c32, g);
        mv.store(Vs, lane);
        tile_barrier<1>();
        if (at + KW < kt.n) {
            mk.load(kh, k_st, kt.tile(at + KW) * 32, a.T, dk);
            if (BOTH_AHEAD<D>) mv.load(vh, v_st, kt.tile(at + KW) * 32, a.T, dk);
        }
        if (!((a.causal && k0 > qhi) || (a.window > 0 && k0 + 31 + a.window <= q0 && k0 >= a.sinks))) {
            const MaskKind kind = mask_kind(k0, k0 + 31, q0, qhi, a.T, a.causal, a.window, a.sinks);
            if (kind != MaskKind::NONE) mask_block(s, kind, vis, k0 + g * 4, -INFINITY);
            float mx = -INFINITY;
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[r]);
            mx = xhalf_max(mx);
            if (__any(mx > m)) {  // wavefront-uniform
                const float mn = fmaxf(m, mx), alpha = __builtin_amdgcn_exp2f((m - mn) * cexp);
                l *= alpha;
                m = mn;
#pragma unroll
                for (int db = 0; db < DB; ++db)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[db][r] *= alpha;
            }
            const float mc = m * cexp;
            float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], cexp, -mc));
                ps[r & 3] += s[r];
            }
            l += (ps[0] + ps[1]) + (ps[2] + ps[3]);  // per-lane partial; the two halves meet below
            accumulate_tr32<D>(Vs, s, acc, c32, g);
        }
        tile_barrier<1>();
    }

    l = xhalf_sum(l);
    __syncthreads();  // every wavefront has read its last tile
    float* ml = lds + KW * DB * 1024;
    ml[kg * 128 + lane] = m;
    ml[kg * 128 + 64 + lane] = l;
    const int64_t ro = b * a.o_sb + h * a.o_sh + qi * a.o_st;
    float mt = m, lt = 0.0f, weight[KW];
    join_shares<DB, KW, 1>(acc, lds, kg, lane, [&]() {
#pragma unroll
        for (int k = 0; k < KW; ++k) mt = fmaxf(mt, ml[k * 128 + lane]);
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            weight[k] = __builtin_amdgcn_exp2f((ml[k * 128 + lane] - mt) * cexp);
            lt += ml[k * 128 + 64 + lane] * weight[k];
        }
        return weight;
    }, [&](int db, int qd, const f32x4 (&v)[1]) {
        if (qi < a.T) store_quad(a.o, ro, db, qd, g, v[0], 1.0f / lt, dk);
    });
    if (qi < a.T && g == 0 && kg == 0) a.lse[(static_cast<int64_t>(b) * a.Hq + h) * a.T + qi] = mt * a.scale + logf(lt);
}

// ---- dQ (and delta, when asked for with it) ----
template <int D, int KW>
constexpr int dq_lds() {  // floats
    constexpr int TILE = 2 * 32 * (D + 4), RED = KW * (D / 32) * 1024;
    return KW * TILE > RED ? KW * TILE : RED;
}
template <int D, int KW, bool BOTH, bool TURN = false>
__device__ inline void dq_block(const AttnArgs& a, int fuse_delta, int id, float* lds) {
    constexpr int DB = D / 32, P = D + 4, TILE = 2 * 32 * P;
    const int lane = threadIdx.x & 63, kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, c32 = lane & 31, dk = a.dk_dim;
    int b, h, hk, qblk;
    if (!map_query_block(a, (a.T + 31) / 32, b, h, hk, qblk, id)) return;
    const int q0 = qblk * 32, qhi = q0 + 31, qi = q0 + c32;
    const float *const kh = head_of<float>(a.k, a.k_sb, b, a.k_sh, hk), *const vh = head_of<float>(a.v, a.v_sb, b, a.v_sh, hk), *const qh = head_of<float>(a.q, a.q_sb, b, a.q_sh, h);
    const float *const gh = head_of<float>(a.d_o, a.do_sb, b, a.do_sh, h), *const oh = head_of<float>(a.o, a.o_sb, b, a.o_sh, h);
    const int k_st = static_cast<int>(a.k_st), v_st = static_cast<int>(a.v_st);
    const float cexp = a.scale * LOG2E;
    float* const Ks = lds + kg * TILE;
    float* const Vs = Ks + 32 * P;

    Mover32<D> mk, mv;
    mk.init(lane, k_st, dk);
    mv.init(lane, v_st, dk);
    const KeyTiles kt(a, q0, 32, 32);
    if (kg < kt.n) mk.load(kh, k_st, kt.tile(kg) * 32, a.T, dk);
    f32x4 qreg[D / 8], greg[D / 8];
    load_row32<D>(qh, static_cast<int>(a.q_st), q0, a.T, dk, c32, g, qreg);
    if (BOTH && kg < kt.n) mv.load(vh, v_st, kt.tile(kg) * 32, a.T, dk);
    load_row32<D>(gh, static_cast<int>(a.do_st), q0, a.T, dk, c32, g, greg);
    // everything is asked for before anything is waited for
    const int64_t lrow = (static_cast<int64_t>(b) * a.Hq + h) * a.T + min(qi, a.T - 1);
    const float lse = a.lse[lrow];
    float dl = 0.0f;
    if (fuse_delta) {
        f32x4 oreg[D / 8];
        load_row_of_o<D>(oh, a.o_st, qi, a.T, dk, g, oreg);
        float part = 0.0f;
#pragma unroll
        for (int j = 0; j < D / 8; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i) part = fmaf(oreg[j][i], greg[j][i], part);
        dl = xhalf_sum(part);
        if (qi < a.T && g == 0 && kg == 0) a.delta[lrow] = dl;
    } else {
        dl = a.delta[lrow];
    }
    const float nlse = -lse * LOG2E;
    const QueryVis vis(qi, a.T, a.causal, a.window, a.sinks);
    f32x16 acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;

    for (int at = kg; at < kt.n; at += KW) {
        const int k0 = kt.tile(at) * 32;
        mk.store(Ks, lane);
        tile_barrier<1>();
        if (!BOTH) mv.load(vh, v_st, k0, a.T, dk);
        f32x16 s = rows_dot<D>(Ks, [&](int j) { return qreg[j]; }, c32, g);
        mv.store(Vs, lane);
        tile_barrier<1>();
        if (at + KW < kt.n) {
            mk.load(kh, k_st, kt.tile(at + KW) * 32, a.T, dk);
            if (BOTH) mv.load(vh, v_st, kt.tile(at + KW) * 32, a.T, dk);
        }
        if (!((a.causal && k0 > qhi) || (a.window > 0 && k0 + 31 + a.window <= q0 && k0 >= a.sinks))) {
            const f32x16 dp = rows_dot<D>(Vs, [&](int j) { return greg[j]; }, c32, g);
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = __builtin_amdgcn_exp2f(fmaf(s[r], cexp, nlse)) * (dp[r] - dl);
            const MaskKind kind = mask_kind(k0, k0 + 31, q0, qhi, a.T, a.causal, a.window, a.sinks);
            if (kind != MaskKind::NONE) mask_block(s, kind, vis, k0 + g * 4, 0.0f);
            accumulate_tr32<D>(Ks, s, acc, c32, g);
        }
        tile_barrier<1>();
    }
    __syncthreads();  // every wavefront has read its last tile
    const int64_t ro = b * a.dq_sb + h * a.dq_sh + qi * a.dq_st;
    join_shares<DB, KW, 1>(acc, lds, kg, lane, no_weights, [&](int db, int qd, const f32x4 (&v)[1]) {
        if (qi < a.T) store_quad(a.dq, ro, db, qd, g, v[0], a.scale, dk, turn_row<TURN>(a, h, qi));
    });
}
template <int D, int KW>
__global__ __launch_bounds__(64 * KW, D <= 32 ? 4 : D <= 64 ? 2 : 1) void f32_split_dq(AttnArgs a, int fuse_delta) {
    all_arguments(a);
    __shared__ __attribute__((aligned(16))) float lds[dq_lds<D, KW>()];
    dq_block<D, KW, false>(a, fuse_delta, static_cast<int>(blockIdx.x), lds);
}

// ---- dK, dV: a block of 32 keys, the query tiles (of every query head of the group in turn) split ----
// OWN_DELTA: the rows' delta is formed here, from O and the tile of dO, in the order of dq_block and to the same bits; otherwise
// it is read.
//
// K and V of the block stay in LDS, one copy for all wavefronts, where registers are short and the LDS has the room (at D = 128
// for K only).
template <int D>
constexpr bool V_IN_LDS = D == 64 || D == 96;
template <int D>
constexpr bool K_IN_LDS = V_IN_LDS<D> || D == 128;
template <int D, int KW>
constexpr int dkdv_lds() {  // floats
    constexpr int TILE = 2 * 32 * (D + 4) + 64, RED = 2 * KW * (D / 32) * 1024;
    return (K_IN_LDS<D> + V_IN_LDS<D>) * 32 * (D + 4) + (KW * TILE > RED ? KW * TILE : RED);
}
template <int D, int KW, bool OWN_DELTA, bool TURN = false>
__device__ inline void dkdv_block(const AttnArgs& a, int id, float* lds) {
    constexpr int DB = D / 32, P = D + 4, TILE = 2 * 32 * P + 64;
    constexpr bool BOTH = D == 32 && OWN_DELTA;
    constexpr bool V_LDS = V_IN_LDS<D>, K_LDS = K_IN_LDS<D>;
    constexpr int KVB = (K_LDS + V_LDS) * 32 * P;
    const int lane = threadIdx.x & 63, kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, c32 = lane & 31, dk = a.dk_dim, rep = quotient(a.Hq, a.Hkv);
    const int nkb = (a.T + 31) / 32;
    const int hs = a.head_split;  // > 1: this workgroup takes heads [h0, h0 + nh) of the group, see gqa_head_split
    // the sink keys' queries past their block's band go to workgroups of their own, blocks nkb .. nkb + nch - 1
    const SinkTail tl = a.tail ? sink_tail(a.T, a.window, a.sinks) : SinkTail{0, 0};
    const int nblk = nkb + tl.nch;
    int blk, rr, kvu;
    // block 0 of every unit first: without a band it is seen by every query, with one it owns the sink keys
    if (a.causal && nblk > 1 ? !xcd_map_block_major(nblk, hs, a.Hkv * a.B, blk, rr, kvu, id) : !xcd_map(nblk, hs, a.Hkv * a.B, blk, rr, kvu, id))
        return;
    const int chunk = blk - nkb;  // >= 0: a piece of the tail, for all query heads of the group
    if (chunk >= 0 && rr > 0) return;
    const int b = quotient(kvu, a.Hkv), hk = kvu - b * a.Hkv, h0 = chunk >= 0 ? 0 : quotient(rr * rep, hs), nh = chunk >= 0 ? rep : quotient((rr + 1) * rep, hs) - h0;
    const int k0 = chunk >= 0 ? 0 : blk * 32, kj = k0 + c32;
    const float cexp = a.scale * LOG2E;
    float* const Qs = lds + KVB + kg * TILE;
    float* const Gs = Qs + 32 * P;
    float* const rows = Gs + 32 * P;  // -LSE log2(e) and delta of the tile's rows

    // query tiles that can see keys [k0, k0 + 32) (paperkiln src/ops.cpp:960-965 inverted)
    const int khi = min(k0 + 32, a.T) - 1;
    const int qt_lo = chunk >= 0 ? (tl.q0 + chunk * TAIL_CHUNK) / 32 : a.causal ? k0 / 32 : 0;
    const int q_end = chunk >= 0 ? min(a.T, tl.q0 + (chunk + 1) * TAIL_CHUNK) - 1
                      : tl.nch > 0 && k0 == 0 ? tl.q0 - 1
                      : a.window > 0 && k0 >= a.sinks ? min(a.T - 1, khi + a.window - 1) : a.T - 1;
    const int qt_hi = q_end / 32;
    const int nqt = qt_hi - qt_lo + 1, steps = nqt * nh;

    const int q_st = static_cast<int>(a.q_st), g_st = static_cast<int>(a.do_st);
    const float *const kh = head_of<float>(a.k, a.k_sb, b, a.k_sh, hk), *const vh = head_of<float>(a.v, a.v_sb, b, a.v_sh, hk);
    // of the first query head in hand; the others follow at q_sh, ...
    const float *const q0h = head_of<float>(a.q, a.q_sb, b, a.q_sh, hk * rep + h0), *const g0h = head_of<float>(a.d_o, a.do_sb, b, a.do_sh, hk * rep + h0),
                *const o0h = OWN_DELTA ? head_of<float>(a.o, a.o_sb, b, a.o_sh, hk * rep + h0) : nullptr;
    Mover32<D> mq, mg;
    mq.init(lane, q_st, dk);
    mg.init(lane, g_st, dk);
    float row_r = 0.0f;
    int f_h = 0, f_t = kg;  // head and tile of the next fetch
    while (f_t >= nqt) f_t -= nqt, ++f_h;
    int c_h = 0, c_r0 = 0;  // query head (from h0 on) and first row of the step in hand
    f32x4 oreg[OWN_DELTA ? D / 8 : 1];
    auto fetch_g = [&]() {
        mg.load(g0h + c_h * a.do_sh, g_st, c_r0, a.T, dk);
        if constexpr (OWN_DELTA) load_row_of_o<D>(o0h + c_h * a.o_sh, a.o_st, c_r0 + c32, a.T, dk, g, oreg);
    };
    auto fetch_q = [&]() {
        const int r0 = (qt_lo + f_t) * 32;
        mq.load(q0h + f_h * a.q_sh, q_st, r0, a.T, dk);
        const int64_t lrow = (static_cast<int64_t>(b) * a.Hq + hk * rep + h0 + f_h) * a.T + min(r0 + c32, a.T - 1);  // rows past the end are masked
        if (g == 0)
            row_r = a.lse[lrow];
        else if (!OWN_DELTA)
            row_r = a.delta[lrow];
        c_h = f_h, c_r0 = r0;
        f_t += KW;
        while (f_t >= nqt) f_t -= nqt, ++f_h;
    };
    if (kg < steps) fetch_q();
    f32x4 kreg[D / 8], vreg[D / 8];
    if (K_LDS) {
        for (int c = static_cast<int>(threadIdx.x); c < (K_LDS + V_LDS) * 32 * (D / 4); c += 64 * KW) {
            const int which = c / (32 * (D / 4)), row = c / (D / 4) % 32, col = c % (D / 4) * 4;
            const float* src = which == 0 ? kh + (k0 + row) * a.k_st : vh + (k0 + row) * a.v_st;
            f32x4 z = {0.0f, 0.0f, 0.0f, 0.0f};
            if (k0 + row < a.T && col < dk) z = *reinterpret_cast<const f32x4*>(src + col);
            *reinterpret_cast<f32x4*>(lds + (which * 32 + row) * P + col) = z;
        }
        __syncthreads();
    }
    if (!K_LDS) load_row32<D>(kh, static_cast<int>(a.k_st), k0, a.T, dk, c32, g, kreg);
    if (!V_LDS) load_row32<D>(vh, static_cast<int>(a.v_st), k0, a.T, dk, c32, g, vreg);
    if (BOTH && kg < steps) fetch_g();
    // (rows of a tile) . (K or V rows of the block)
    auto dot = [&](const float* tile, bool in_lds, const f32x4* reg, const float* shared) {
        if (in_lds)
            return rows_dot<D>(tile, [&](int j) { return *reinterpret_cast<const f32x4*>(shared + c32 * P + 8 * j + 4 * g); }, c32, g);
        return rows_dot<D>(tile, [&](int j) { return reg[j]; }, c32, g);
    };
    f32x16 acc[2 * DB];  // dV^T, dK^T
#pragma unroll
    for (int n = 0; n < 2 * DB; ++n)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[n][r] = 0.0f;
    const KeyVis kvis(kj, a.T, a.causal, a.window, a.sinks);

    for (int step = kg; step < steps; step += KW) {
        const int qlo = c_r0, qhi = qlo + 31;
        mq.store(Qs, lane);
        if (!OWN_DELTA || g == 0) rows[lane] = g == 0 ? -row_r * LOG2E : row_r;
        tile_barrier<1>();
        if (!BOTH) fetch_g();
        f32x16 s = dot(Qs, K_LDS, kreg, lds);
        mg.store(Gs, lane);
        tile_barrier<1>();
        if constexpr (OWN_DELTA) {
            float part = 0.0f;
#pragma unroll
            for (int j = 0; j < D / 8; ++j) {
                const f32x4 gv = *reinterpret_cast<const f32x4*>(Gs + c32 * P + 8 * j + 4 * g);
#pragma unroll
                for (int i = 0; i < 4; ++i) part = fmaf(oreg[j][i], gv[i], part);
            }
            part = xhalf_sum(part);
            if (g == 1) rows[lane] = part;
            tile_barrier<1>();
        }
        if (step + KW < steps) {
            fetch_q();
            if (BOTH) fetch_g();
        }
        if (!((a.causal && k0 > qhi) || (a.window > 0 && k0 + 31 + a.window <= qlo && k0 >= a.sinks))) {
            // lane = key kj; element r = query qlo + crow(r, g)
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                const f32x4 nl = *reinterpret_cast<const f32x4*>(rows + qd * 8 + g * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[qd * 4 + e] = __builtin_amdgcn_exp2f(fmaf(s[qd * 4 + e], cexp, nl[e]));
            }
            const bool full = qhi < a.T && k0 + 31 < a.T && (!a.causal || k0 + 31 <= qlo) &&
                              (a.window == 0 || k0 + a.window > qhi || k0 + 31 < a.sinks);
            if (!full) {
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = kvis(qlo + crow(r, g)) ? s[r] : 0.0f;
            }
            accumulate_tr32<D>(Gs, s, acc, c32, g);
            f32x16 dp = dot(Gs, V_LDS, vreg, lds + 32 * P);
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                const f32x4 dl = *reinterpret_cast<const f32x4*>(rows + 32 + qd * 8 + g * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) dp[qd * 4 + e] = s[qd * 4 + e] * (dp[qd * 4 + e] - dl[e]);
            }
            accumulate_tr32<D>(Qs, dp, acc + DB, c32, g);
        }
        tile_barrier<1>();
    }
    __syncthreads();  // every wavefront has read its last tile
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
    join_shares<2 * DB, KW, 1>(acc, lds + KVB, kg, lane, no_weights, [&](int n, int qd, const f32x4 (&v)[1]) {
        if (mine) store_quad(n < DB ? dst_v : dst_k, n < DB ? rv : rk, n < DB ? n : n - DB, qd, g, v[0], n < DB ? 1.0f : a.scale, dk, n < DB ? TurnRow() : turn_row<TURN>(a, hk, kj));
    });
}
template <int D, int KW>
__global__ __launch_bounds__(64 * KW, D <= 32 && KW == 4 ? 3 : D <= 64 ? 2 : 1) void f32_split_dkdv(AttnArgs a) {
    all_arguments(a);
    __shared__ __attribute__((aligned(16))) float lds[dkdv_lds<D, KW>()];
    dkdv_block<D, KW, false>(a, static_cast<int>(blockIdx.x), lds);
}

// ---- dK, dV and dQ in one launch ----
// Two launches of a handful of workgroups each, the second waiting for the first one's delta, are two round trips to memory with
// most CUs idle. Here blocks 0 .. dkdv_ids - 1 are the dK/dV launch's, which forms its own delta, and the others the dQ launch's.
template <int D, bool TURN>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void f32_split_bwd(AttnArgs a, int dkdv_ids) {
    all_arguments(a);
    constexpr int Q = dq_lds<D, 4>(), K = dkdv_lds<D, 4>();
    __shared__ __attribute__((aligned(16))) float lds[Q > K ? Q : K];
    const int id = static_cast<int>(blockIdx.x);
    if (id < dkdv_ids)
        dkdv_block<D, 4, true, TURN>(a, id, lds);
    else
        dq_block<D, 4, D == 32, TURN>(a, 1, id - dkdv_ids, lds);
}

// A block's tiles split between four or eight wavefronts, or not this kernel.
enum class Form { NONE, FOUR, EIGHT };

// Which form, from the number of 32-row blocks of the launch and the length of a block's chain; the kernels of attn_f32_mfma.hip
// (128 rows a workgroup) where they are ahead: head_dim 128 once there are about four blocks per CU -- a split block's
// tiles then cross the L2 four times as often as theirs and hide it behind twice the matrix work only -- and many short
// sequences. Measured (us, causal; eight | four | 128 rows):
//   forward, head_dim 64    T 512, 8 heads 15 | 16 | 46;  T 2048, 8 heads 51 | 60 | 168;  B=4 T=1024 H=8 58 | 54 | 88
//                           B=2 T=4096 H=16 653 | 609 | 656;  B=32 T=128 H=8 28 | 19 | 18
//   dQ, head_dim 64         T 2048, 8 heads 68 | 84 | 222;  B=4 T=1024 H=8 89 | 79 | 117;  B=2 T=4096 H=16 912 | 833 | 919
//   dK/dV, head_dim 64      T 512, 8 heads 23 | 25 | 97;  B=4 T=1024 H=8 96 | 105 | 169;  B=8 T=1024 H=16 384 | 423 | 338
//                           B=2 T=4096 H=16 1130 | 1299 | 1177
//   head_dim 32             B=4 T=1024 H=8: forward 30 | 31 | 46, dQ 43 | 43 | 64, dK/dV 59 | 53 | 100
//   head_dim 128            T 512, 8 heads: forward - | 27 | 73, dQ - | 38 | 105, dK/dV - | 55 | 174
//                           B=4 T=1024 H=8: - | 115 | 146, - | 162 | 204, - | 276 | 306
//                           B=16 T=512 H=8: - | 152 | 140, - | 220 | 218, - | 381 | 190
bool has_own_kernel(const AttnArgs& a) { return a.dk_dim == 32 || a.dk_dim == 64 || a.dk_dim == 128; }
// and where all chains are equally long (no mask, or a window; forward, dQ, dK/dV):
//   head_dim 128, T 600, window 120, 24 heads 33 48 75 | 42 61 77, 38 heads 50 72 113 | 43 63 79;  T 600, no mask, 16 heads
//   62 86 135 | 92 124 162, 38 heads 95 131 250 | 95 128 167;  T 2400, window 100, 8 heads 49 71 107 | 43 63 79
//   head_dim 64, T 1200, window 64, 16 heads 16 28 32 | 22 29 35, 24 heads 19 30 44 | 22 30 36, 38 heads 29 44 68 | 37 57 68
bool query_kernel_is_ahead(const AttnArgs& a, int64_t blocks, bool dq) {
    if (!has_own_kernel(a)) return false;
    const int chain = chain_tokens(a);
    if (dq && a.T <= 32) return true;  // one tile, nothing to split: T 30, 16 heads of 128 12.9 us against 17.5, of 64 8.6 and 10.2
    if (a.T <= 160 && blocks > (a.T <= (dq && a.dk_dim == 128 ? 96 : 64) ? 256 : dq ? 512 : 600)) return true;
    if (a.dk_dim == 128) return blocks > (a.T <= 96 ? 300 : even_chains(a) || chain < 400 ? 512 : 1200);
    if (a.T <= 200 && even_chains(a) && blocks > 512) return true;
    return !dq && blocks > 1500 && (a.T <= 200 || (even_chains(a) && chain > 128));
}
Form query_form(const AttnArgs& a, bool dq) {  // forward, dQ
    const int64_t blocks = static_cast<int64_t>((a.T + 31) / 32) * a.Hq * a.B;
    if (query_kernel_is_ahead(a, blocks, dq)) return Form::NONE;
    const int chain = chain_tokens(a);
    const int64_t short_chain = dq ? 0 : 200;
    return a.dk_dim <= 64 && ((blocks <= 600 && chain >= 1000) || (blocks <= short_chain && chain >= 256)) ? Form::EIGHT : Form::FOUR;
}
Form fwd_form(const AttnArgs& a) { return query_form(a, false); }
Form dq_form(const AttnArgs& a) { return query_form(a, true); }
// The 128-key kernel walks the whole group of query heads in one workgroup: it is behind while those leave CUs idle,
// however many blocks a split of keys and heads comes to (a group of four, head_dim 128, T 600, window 120: 8 KV heads
// 252 us against 100, 24 KV heads 256 against 268; T 2400, window 100, 8 KV heads 258 against 356). Causal, every head its own
// (us, this kernel | the 128-key one): head_dim 128, T 1100, 24 heads 255 | 287, 32 heads 328 | 287; head_dim 64, T 400, 64
// heads 54 | 65, 96 heads 77 | 66.
bool key_kernel_is_ahead(const AttnArgs& a, int64_t blocks) {
    if (!has_own_kernel(a)) return false;
    const int chain = chain_tokens(a);
    const int64_t groups = static_cast<int64_t>((a.T + 127) / 128) * a.Hkv * a.B;  // workgroups of the 128-key kernel
    // One tile, nothing to split but the heads of a group: T 26, 8 heads of 128 x 7 14 us against 21, of 64 9.2 and 11.6; groups
    // of two, 48 of 128 22 and 25; groups of four, 64 of 128 37 and 26, 68 37 and 42.
    if (a.T <= 32 && (a.Hq <= 2 * a.Hkv || (a.Hq <= 4 * a.Hkv && a.dk_dim >= 64 && groups > 64))) return true;
    if (a.dk_dim == 128 && groups >= (a.T <= 64 ? 80 : 100) && chain < 400) return true;
    if (a.T <= 160) return a.Hq == a.Hkv ? blocks > (a.T <= (a.dk_dim > 32 ? 96 : 64) ? 256 : 600) : groups >= 128;
    if (a.dk_dim == 128) return a.Hq == a.Hkv ? blocks > (even_chains(a) ? 512 : a.T < 800 ? 800 : 900) : groups >= 112;
    if (a.dk_dim == 64 && chain <= 160 && even_chains(a) && groups > 192 && groups <= 256) return true;  // one to a CU
    // groups of heads in causal pairs of 128-key blocks that come to most of a round (T 200, 218 units of two heads 159 | 101, 167,
    // 252 of four 240 | 151; 401, 128 of two 212 | 136; 500, 88 of four 340 | 292)
    if (a.dk_dim == 64 && a.Hq > a.Hkv && a.causal && a.window == 0 && a.T <= 512 && (a.T + 127) / 128 % 2 == 0 && groups > 340 && groups <= 512)
        return true;
    return a.Hq == a.Hkv && ((a.dk_dim == 64 && blocks > 1400 && a.T < 3000) || (a.T <= 450 && blocks > 1000));
}
Form dkdv_form(const AttnArgs& a) {
    const int64_t blocks = static_cast<int64_t>((a.T + 31) / 32) * a.Hkv * a.B * a.head_split;
    if (key_kernel_is_ahead(a, blocks)) return Form::NONE;
    if (a.dk_dim > 64) return Form::FOUR;
    return a.dk_dim > 32 || (blocks <= 320 && chain_tokens(a) >= 512) ? Form::EIGHT : Form::FOUR;
}

template <int D, int KW>
void run_fwd(const AttnArgs& a, hipStream_t st) {
    hipLaunchKernelGGL((f32_split_fwd<D, KW>), dim3(xcd_grid((a.T + 31) / 32, a.Hq / a.Hkv, a.Hkv * a.B)), dim3(64 * KW), 0, st, a);
}
template <int D, int KW>
void run_dq(const AttnArgs& a, bool fuse_delta, hipStream_t st) {
    hipLaunchKernelGGL((f32_split_dq<D, KW>), dim3(xcd_grid((a.T + 31) / 32, a.Hq / a.Hkv, a.Hkv * a.B)), dim3(64 * KW), 0, st, a,
                       fuse_delta ? 1 : 0);
}
template <int D, int KW>
void run_dkdv(const AttnArgs& a, hipStream_t st) {
    hipLaunchKernelGGL((f32_split_dkdv<D, KW>), dim3(xcd_grid((a.T + 31) / 32 + tail_blocks(a), a.head_split, a.Hkv * a.B)), dim3(64 * KW), 0, st, a);
}

template <int D>
void run_bwd(const OneLaunch& l, hipStream_t st) {
    const dim3 grid(l.dkdv_ids + l.dq_ids);
    if (l.a.turn)
        hipLaunchKernelGGL((f32_split_bwd<D, true>), grid, dim3(256), 0, st, l.a, l.dkdv_ids);
    else
        hipLaunchKernelGGL((f32_split_bwd<D, false>), grid, dim3(256), 0, st, l.a, l.dkdv_ids);
}

}  // namespace

// a lane's byte offset inside a 32-row tile is kept in 31 bits
bool f32_split_serves(const AttnArgs& a) {
    auto ok = [](int64_t st) { return st > 0 && st < (int64_t{1} << 22); };
    return a.dk_dim % 4 == 0 && a.dk_dim <= 128 && ok(a.q_st) && ok(a.k_st) && ok(a.v_st) && (!a.d_o || ok(a.do_st));
}
bool f32_split_takes_fwd(const AttnArgs& a) { return f32_split_serves(a) && fwd_form(a) != Form::NONE; }
bool f32_split_takes_dq(const AttnArgs& a) { return f32_split_serves(a) && dq_form(a) != Form::NONE; }
bool f32_split_takes_dkdv(const AttnArgs& a) { return f32_split_serves(a) && dkdv_form(a) != Form::NONE; }

int launch_f32_split_fwd(const AttnArgs& a, hipStream_t st) {
    const bool eight = fwd_form(a) == Form::EIGHT;
    if (a.dk_dim <= 32)
        eight ? run_fwd<32, 8>(a, st) : run_fwd<32, 4>(a, st);
    else if (a.dk_dim <= 64)
        eight ? run_fwd<64, 8>(a, st) : run_fwd<64, 4>(a, st);
    else if (a.dk_dim <= 96)
        run_fwd<96, 4>(a, st);
    else
        run_fwd<128, 4>(a, st);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
int launch_f32_split_dq(const AttnArgs& a, bool fuse_delta, hipStream_t st) {
    const bool eight = dq_form(a) == Form::EIGHT;
    if (a.dk_dim <= 32)
        eight ? run_dq<32, 8>(a, fuse_delta, st) : run_dq<32, 4>(a, fuse_delta, st);
    else if (a.dk_dim <= 64)
        eight ? run_dq<64, 8>(a, fuse_delta, st) : run_dq<64, 4>(a, fuse_delta, st);
    else if (a.dk_dim <= 96)
        run_dq<96, 4>(a, fuse_delta, st);
    else
        run_dq<128, 4>(a, fuse_delta, st);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
int launch_f32_split_dkdv(const AttnArgs& a_in, hipStream_t st) {
    AttnArgs a = a_in;
    if (!split_tail_pays(a, a.head_split, 32)) a.tail = nullptr;
    const bool eight = dkdv_form(a) == Form::EIGHT;
    if (a.dk_dim <= 32)
        eight ? run_dkdv<32, 8>(a, st) : run_dkdv<32, 4>(a, st);
    else if (a.dk_dim <= 64)
        run_dkdv<64, 8>(a, st);
    else if (a.dk_dim <= 96)
        run_dkdv<96, 4>(a, st);
    else
        run_dkdv<128, 4>(a, st);
    PK_HIP(hipGetLastError());
    return a.head_split > 1 ? launch_gqa_reduce(a, st) : a.tail ? launch_sink_tail_reduce(a, st) : PK_OK;
}

// dQ and dK/dV in one launch: while their workgroups find room on the chip together, one to a CU above 32 columns, or nearly do
// where causal chains are of very different length. Measured, the launches of a backward one after the other | this one (us):
//   head_dim 32   T 194, 16 heads 19.0 | 13.9;  T 623 x 2, 8 heads 36 | 28;  T 640, 32 heads on 8 50 | 50
//            64   T 511, 8 heads 41 | 29;  T 872 x 8, 1 head 68 | 46;  T 41 x 7, 8 heads, no mask 21 | 12.6;  T 2931, 4 heads 174 | 181
//            128  T 370, 16 heads 74 | 68;  no mask: T 56 x 46, 2 heads 41 | 47, T 1179 x 3, 2 heads 233 | 314
// Over 300 random shapes of up to 1000 blocks it is 1.2 to 1.7 times as fast as they are below these lines.
bool f32_split_takes_bwd(const AttnArgs& a) {
    if (!f32_split_serves(a)) return false;
    const OneLaunch l(a);
    const int ids = l.dkdv_ids + l.dq_ids;
    if (a.dk_dim <= 32) return ids <= (even_chains(a) ? 800 : 960);
    if (ids <= 256) return true;
    if (a.dk_dim > 96 || a.T <= 32 || chain_tokens(a) > 2600) return false;  // (one tile: T 24 x 104, 2 heads of 64 16.3 | 21.1)
    return ids <= (even_chains(a) ? 300 : 700);
}
int launch_f32_split_bwd(const AttnArgs& a, hipStream_t st) {
    const OneLaunch l(a);
    if (a.dk_dim <= 32)
        run_bwd<32>(l, st);
    else if (a.dk_dim <= 64)
        run_bwd<64>(l, st);
    else if (a.dk_dim <= 96)
        run_bwd<96>(l, st);
    else
        run_bwd<128>(l, st);
    PK_HIP(hipGetLastError());
    return l.finish(st);
}

}  // namespace pk
