// dQ of a block of 32 NW queries in bf16 (see attn_bwd_mfma.hip for the mathematics): what the launches of dQ alone and those
// that take blocks of keys as well (attn_bwd_dkdv2.hip) share.
#pragma once
#include "mfma_common.h"
#include "pk_internal.h"

namespace pk {
namespace {

constexpr float LOG2E = 1.4426950408889634f;

// ---- shared tile movers ---------------------------------------------------
template <int D, int ROWS, int NW = 4>
struct Tile {
    static constexpr int S = D + 8;             // row pitch (elements)
    static constexpr int NCH = D / 8;           // 16-byte chunks per row
    static constexpr int CPT = ROWS * NCH / (64 * NW);
    // this thread's byte offsets inside a tile whose rows are st_t elements apart
    __device__ static void offsets(int64_t st_t, int* boff) {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int c = threadIdx.x + 64 * NW * i;
            boff[i] = static_cast<int>((c / NCH) * st_t + (c % NCH) * 8) * 2;
        }
    }
    // rows r0 .. r0+ROWS-1 of the matrix at base + off; rows past T read as zero
    __device__ static void load(const void* base, int64_t off, int64_t st_t, int r0, int T, const int* boff, u32x4* r) {
        const __amdgpu_buffer_rsrc_t rs = tile_rsrc(base, off, st_t, r0, T, D);
#pragma unroll
        for (int i = 0; i < CPT; ++i) r[i] = tile_load16(rs, boff[i]);
    }
    __device__ static void store(uint16_t* lds, const u32x4* r) {
#pragma unroll
        for (int i = 0; i < CPT; ++i) {
            const int c = threadIdx.x + 64 * NW * i;
            const int row = c / NCH, ch = c % NCH;
            *reinterpret_cast<u32x4*>(lds + lds_row<D>(row) * S + ch * 8) = r[i];
        }
    }
};

// Row `row` of a head as an MFMA operand held in registers:
// element chunk kk covers d = 16kk + 8g .. +7.
template <int D>
__device__ inline void load_row_operand(const void* base, int64_t off, int64_t st_t, int row, int T,
                                        int g, bf16x8* out) {
#pragma unroll
    for (int kk = 0; kk < D / 16; ++kk) {
        u32x4 z = {0, 0, 0, 0};
        if (row < T)
            z = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(base) + off + row * st_t +
                                                kk * 16 + g * 8);
        out[kk] = *reinterpret_cast<bf16x8*>(&z);
    }
}

template <bool F32>
__device__ inline void store4(void* base, int64_t idx, float x0, float x1, float x2, float x3) {
    if (F32) {
        f32x4 v = {x0, x1, x2, x3};
        *reinterpret_cast<f32x4*>(static_cast<float*>(base) + idx) = v;
    } else {
        u32x2 v = {pack_bf16(x0, x1), pack_bf16(x2, x3)};
        *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(base) + idx) = v;
    }
}

// FUSE_DELTA: the workgroup also forms delta for its own rows (it holds their dO
// already; O costs one more row read), uses it and writes it for a dK/dV kernel
// that reads it after this one. Saves the separate pass over O and dO.
template <int D, int NW>
constexpr int DQ_LDS = 2 * 64 * Tile<D, 64, NW>::S;  // in uint16
template <int D, bool GF32, bool FUSE_DELTA, int NW>
__device__ inline void dq_block(const AttnArgs& a, int b, int h, int hk, int qblk, uint16_t* lds) {
    constexpr int BM = 32 * NW, BN = 64;
    constexpr int KK = D / 16, DB = D / 32;
    using KT = Tile<D, BN, NW>;
    uint16_t* const Ks = lds;
    uint16_t* const Vs = lds + BN * KT::S;

    const int lane = threadIdx.x & 63;
    // the wavefront index as a scalar: every test on it becomes a scalar branch
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 5, c32 = lane & 31;
    const int q0 = qblk * BM;
    const int qlo = q0 + w * 32, qhi = qlo + 31, qi = qlo + c32;
    const int64_t kb = b * a.k_sb + hk * a.k_sh, vb = b * a.v_sb + hk * a.v_sh;
    const float cexp = a.scale * LOG2E;

    bf16x8 qreg[KK], greg[KK];
    load_row_operand<D>(a.q, b * a.q_sb + h * a.q_sh, a.q_st, qi, a.T, g, qreg);
    load_row_operand<D>(a.d_o, b * a.do_sb + h * a.do_sh, a.do_st, qi, a.T, g, greg);
    float nlse = 0.0f, dl = 0.0f;
    const int64_t lrow = (static_cast<int64_t>(b) * a.Hq + h) * a.T + qi;
    if (qi < a.T) nlse = -a.lse[lrow] * LOG2E;
    if (FUSE_DELTA) {
        bf16x8 oreg[KK];  // zero rows past the end, as dO
        load_row_operand<D>(a.o, b * a.o_sb + h * a.o_sh, a.o_st, qi, a.T, g, oreg);
        float part = 0.0f;  // this lane's half of the row: d = 16kk + 8g .. +7
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const u32x4 ov = *reinterpret_cast<const u32x4*>(&oreg[kk]);
            const u32x4 gv = *reinterpret_cast<const u32x4*>(&greg[kk]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                part = fmaf(__uint_as_float(ov[i] << 16), __uint_as_float(gv[i] << 16), part);
                part = fmaf(__uint_as_float(ov[i] & 0xFFFF0000u), __uint_as_float(gv[i] & 0xFFFF0000u), part);
            }
        }
        dl = xhalf_sum(part);
        if (qi < a.T && g == 0) a.delta[lrow] = dl;
    } else if (qi < a.T) {
        dl = a.delta[lrow];
    }
    const QueryVis qvis(qi, a.T, a.causal, a.window, a.sinks);
    f32x16 dq_acc[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) dq_acc[db][r] = 0.0f;

    const int qmax = min(q0 + BM, a.T) - 1;
    const int hi = (a.causal ? qmax : a.T - 1) / BN;
    const int lo = a.window > 0 ? max(0, q0 + 1 - a.window) / BN : 0;
    const int ns = a.window > 0 ? min((a.sinks + BN - 1) / BN, lo) : 0;
    int t = ns > 0 ? 0 : lo;

    u32x4 kr[KT::CPT], vr[KT::CPT];
    int koff[KT::CPT], voff[KT::CPT];
    KT::offsets(a.k_st, koff);
    KT::offsets(a.v_st, voff);
    KT::load(a.k, kb, a.k_st, t * BN, a.T, koff, kr);
    KT::load(a.v, vb, a.v_st, t * BN, a.T, voff, vr);
    KT::store(Ks, kr);
    KT::store(Vs, vr);
    __syncthreads();

    while (t <= hi) {
        const int n0 = t * BN;
        const int tn = (t + 1 == ns) ? lo : t + 1;
        if (tn <= hi) {
            KT::load(a.k, kb, a.k_st, tn * BN, a.T, koff, kr);
            KT::load(a.v, vb, a.v_st, tn * BN, a.T, voff, vr);
        }
        const bool skip = qlo >= a.T || (a.causal && n0 > qhi) ||
                          (a.window > 0 && n0 + BN - 1 + a.window <= qlo && n0 >= a.sinks);
        if (!skip) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
                // a 32-key half no query of this wavefront can see (past the diagonal, or before the band and without
                // a sink key) costs nothing; which of the mask's tests the half can fail decides its masking loop
                const int k0 = n0 + nb * 32, k1 = k0 + 31;
                if ((a.causal && k0 > qhi) || (a.window > 0 && k1 + a.window <= qlo && k0 >= a.sinks)) continue;
                const MaskKind kind = mask_kind(k0, k1, qlo, qhi, a.T, a.causal, a.window, a.sinks);
                f32x16 s, dp;
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = dp[r] = 0.0f;
                // matrix phases issue ahead of co-resident waves' exponent phases
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) {
                    const bf16x8 kf = lds_read8(Ks + (nb * 32 + lds_row<D>(c32)) * KT::S + kk * 16 + g * 8);
                    s = mfma32(kf, qreg[kk], s);
                    const bf16x8 vf = lds_read8(Vs + (nb * 32 + lds_row<D>(c32)) * KT::S + kk * 16 + g * 8);
                    dp = mfma32(vf, greg[kk], dp);
                }
                __builtin_amdgcn_s_setprio(0);
                // lane = query qi; element r = key n0 + nb*32 + (r/4)*8 + 4g + r%4
#pragma unroll
                for (int r = 0; r < 16; ++r) dp[r] = __builtin_amdgcn_exp2f(fmaf(s[r], cexp, nlse)) * (dp[r] - dl);
                // off the common path: interior blocks carry no mask arithmetic at all
                if (kind != MaskKind::NONE) mask_block(dp, kind, qvis, k0 + g * 4, 0.0f);
                const bf16x8 d0 = c_to_operand<0>(dp), d1 = c_to_operand<1>(dp);
                __builtin_amdgcn_s_setprio(1);
                // dQ^T += K^T dS^T, DB independent chains per k-chunk
#pragma unroll
                for (int db = 0; db < DB; ++db)
                    dq_acc[db] = mfma32(lds_read_tr_operand_perm<D>(Ks, KT::S, nb * 32, db, lane), d0, dq_acc[db]);
#pragma unroll
                for (int db = 0; db < DB; ++db)
                    dq_acc[db] = mfma32(lds_read_tr_operand_perm<D>(Ks, KT::S, nb * 32 + 16, db, lane), d1, dq_acc[db]);
                __builtin_amdgcn_s_setprio(0);
            }
        }
        __syncthreads();
        if (tn <= hi) {
            KT::store(Ks, kr);
            KT::store(Vs, vr);
        }
        __syncthreads();
        t = tn;
    }

    if constexpr (!GF32 && NW <= 4) {  // (no tile is read any more; eight wavefronts' rows would not fit)
        using Rows = RowStrip<D>;
        static_assert(NW * Rows::ELEMS <= DQ_LDS<D, NW>, "the wavefronts' strips");
        uint16_t* const strip = lds + w * Rows::ELEMS;
        const int q1 = qi - c32;
#pragma unroll
        for (int db = 0; db < DB; ++db) store_acc_bf16<D>(Rows::row(strip, c32), db, g, dq_acc[db], a.scale);
        Rows::out(strip, static_cast<uint16_t*>(a.dq) + b * a.dq_sb + h * a.dq_sh + q1 * a.dq_st, a.dq_st, 0, a.T - q1, lane);
    } else if (qi < a.T) {
        const int64_t ob = b * a.dq_sb + h * a.dq_sh + qi * a.dq_st;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
            if (!GF32) {
                store_acc_bf16<D>(static_cast<uint16_t*>(a.dq) + ob, db, g, dq_acc[db], a.scale);
                continue;
            }
#pragma unroll
            for (int qd = 0; qd < 4; ++qd)
                store4<GF32>(a.dq, ob + TrMap<D>::col0(db, qd, g), dq_acc[db][qd * 4] * a.scale,
                             dq_acc[db][qd * 4 + 1] * a.scale, dq_acc[db][qd * 4 + 2] * a.scale,
                             dq_acc[db][qd * 4 + 3] * a.scale);
        }
    }
}

}  // namespace
}  // namespace pk
