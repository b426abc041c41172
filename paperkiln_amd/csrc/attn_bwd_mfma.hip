// bf16 flash-attention recompute backward for gfx950. Replaces the backward
// closure of ops::fused_attention / ops::swa_attention (paperkiln
// src/ops.cpp:902-933, 997-1026), which reads the saved [T,T] matrix A: here P
// is rebuilt from Q, K and the forward's logsumexp, so the tape node keeps
// only O and LSE.
//
//   delta_i = sum_d O_id dO_id            (= the reference's `dot`, :920-921)
//   P_ij    = exp(scale*s_ij - LSE_i)     (0 where masked)
//   dV = P^T dO          dP = dO V^T      dS = P .* (dP - delta)
//   dQ = scale * dS K    dK = scale * dS^T Q
//
// No atomics, deterministic. The full backward is two launches, mfma_dq (which
// also forms delta) then mfma_dkdv2; asked for by parts it is three:
//   mfma_delta    one pass over O and dO (only when delta is wanted without dQ).
//   mfma_dkdv2    (attn_bwd_dkdv2.hip) a workgroup owns 128 keys of one KV
//                 head and loops over the query heads of its GQA group and
//                 over the query tiles that can see it.
//   mfma_dq       a workgroup owns 128 queries of one head (32 per
//                 wavefront, Q and dO in registers), loops over the visible
//                 key tiles: S^T = K Q^T, dP^T = V dO^T (lane = query, so LSE
//                 and delta are per-lane scalars), dQ^T += K^T dS^T.
#include <cstdlib>

#include "attn_bwd_dq.h"
#include "mfma_common.h"
#include "pk_internal.h"

namespace pk {
namespace {

// ---- delta --------------------------------------------------------------
template <int D>
__global__ __launch_bounds__(256) void mfma_delta(AttnArgs a) {
    constexpr int LPR = D / 8;        // lanes per row, 16 bytes each
    constexpr int RPB = 256 / LPR;    // rows per block
    const int sub = threadIdx.x % LPR;
    const int64_t row = static_cast<int64_t>(blockIdx.x) * RPB + threadIdx.x / LPR;
    const int64_t rows = static_cast<int64_t>(a.B) * a.Hq * a.T;
    float s = 0.0f;
    if (row < rows) {
        const int t = row % a.T;
        const int h = (row / a.T) % a.Hq;
        const int b = row / (static_cast<int64_t>(a.T) * a.Hq);
        const u32x4 ov = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.o) + b * a.o_sb +
                                                         h * a.o_sh + t * a.o_st + sub * 8);
        const u32x4 gv = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.d_o) +
                                                         b * a.do_sb + h * a.do_sh + t * a.do_st + sub * 8);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            s = fmaf(__uint_as_float(ov[i] << 16), __uint_as_float(gv[i] << 16), s);
            s = fmaf(__uint_as_float(ov[i] & 0xFFFF0000u), __uint_as_float(gv[i] & 0xFFFF0000u), s);
        }
    }
#pragma unroll
    for (int o = LPR / 2; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if (row < rows && sub == 0) a.delta[row] = s;
}

template <int D, bool GF32, bool FUSE_DELTA, int NW>
__global__ __launch_bounds__(64 * NW, 2) void mfma_dq(AttnArgs a) {
    __shared__ __attribute__((aligned(16))) uint16_t lds[DQ_LDS<D, NW>];
    const int nqb = (a.T + 32 * NW - 1) / (32 * NW), rep = quotient(a.Hq, a.Hkv);
    int blk, rr, kvu;
    if (!map_causal_blocks(a, nqb, rep, blk, rr, kvu)) return;
    const int b = quotient(kvu, a.Hkv), hk = kvu - b * a.Hkv, npass = (a.paired && blk != nqb - 1 - blk) ? 2 : 1;
    for (int pass = 0; pass < npass; ++pass) {
        dq_block<D, GF32, FUSE_DELTA, NW>(a, b, hk * rep + rr, hk, pass == 0 ? nqb - 1 - blk : blk, lds);
        __syncthreads();  // the next pass refills the tile buffers
    }
}

template <int D, bool GF32>
int launch_dq(const AttnArgs& a_in, bool fuse_delta, hipStream_t st) {
    AttnArgs a = a_in;
    // dQ with 8 wavefronts (256 queries) per K/V tile where the paired causal grid still gives every CU two
    // workgroups in turn, as in the forward kernel; 4 wavefronts otherwise.
    const int nb256 = (a.T + 255) / 256;
    const bool wide = D == 128 && a.causal && a.window == 0 && static_cast<int64_t>((nb256 + 1) / 2) * a.Hq * a.B >= 512;
    const int nbq = wide ? nb256 : (a.T + 127) / 128;
    // as in the forward kernel (16 heads x 1024 x 16, head_dim 64: 76 us singly, 80 paired)
    a.paired = (D == 128 || nbq <= 2) && pair_causal_blocks(nbq, static_cast<int64_t>(a.Hq) * a.B, a.causal, a.window, wide ? 256 : 512);
    const dim3 grid = causal_blocks_grid(a, nbq, a.Hq / a.Hkv);
    if (wide && fuse_delta) hipLaunchKernelGGL((mfma_dq<D, GF32, true, 8>), grid, dim3(512), 0, st, a);
    if (wide && !fuse_delta) hipLaunchKernelGGL((mfma_dq<D, GF32, false, 8>), grid, dim3(512), 0, st, a);
    if (!wide && fuse_delta) hipLaunchKernelGGL((mfma_dq<D, GF32, true, 4>), grid, dim3(256), 0, st, a);
    if (!wide && !fuse_delta) hipLaunchKernelGGL((mfma_dq<D, GF32, false, 4>), grid, dim3(256), 0, st, a);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
// Any head size, LPR lanes a row and 16 bytes a lane at a time
template <bool BF16, int LPR>
__global__ __launch_bounds__(256) void row_delta(AttnArgs a) {
    constexpr int W = BF16 ? 8 : 4;
    const int sub = threadIdx.x % LPR;
    const int blocks = (a.T + 256 / LPR - 1) / (256 / LPR), hb = blockIdx.x / blocks;
    const int row = (blockIdx.x % blocks) * (256 / LPR) + static_cast<int>(threadIdx.x) / LPR;
    const int h = hb % a.Hq, b = hb / a.Hq;
    float s = 0.0f;
    if (row < a.T) {
        const int64_t oo = b * a.o_sb + h * a.o_sh + row * a.o_st, go = b * a.do_sb + h * a.do_sh + row * a.do_st;
        for (int c = sub * W; c < a.dk_dim; c += LPR * W) {
            const u32x4 ov = *reinterpret_cast<const u32x4*>(static_cast<const char*>(a.o) + (oo + c) * (BF16 ? 2 : 4));
            const u32x4 gv = *reinterpret_cast<const u32x4*>(static_cast<const char*>(a.d_o) + (go + c) * (BF16 ? 2 : 4));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (BF16) {
                    s = fmaf(__uint_as_float(ov[i] << 16), __uint_as_float(gv[i] << 16), s);
                    s = fmaf(__uint_as_float(ov[i] & 0xFFFF0000u), __uint_as_float(gv[i] & 0xFFFF0000u), s);
                } else {
                    s = fmaf(__uint_as_float(ov[i]), __uint_as_float(gv[i]), s);
                }
            }
        }
    }
#pragma unroll
    for (int o = LPR / 2; o >= 1; o >>= 1) s += __shfl_xor(s, o, 64);
    if (row < a.T && sub == 0) a.delta[static_cast<int64_t>(hb) * a.T + row] = s;
}
template <int D>
int launch_delta(const AttnArgs& a, hipStream_t st) {
    constexpr int RPB = 256 / (D / 8);
    const int64_t rows = static_cast<int64_t>(a.B) * a.Hq * a.T;
    hipLaunchKernelGGL((mfma_delta<D>), dim3((rows + RPB - 1) / RPB), dim3(256), 0, st, a);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
// Which dQ kernel: wavefronts that split the keys for small launches and for head sizes other than 64 and 128, 64
// queries per wavefront (one wavefront per SIMD) for long sequences, 32 otherwise.
int run_dq(const AttnArgs& a, bool fuse_delta, hipStream_t st) {
    if (split_takes_dq(a)) return launch_split_dq(a, fuse_delta, st);
    if (mfma_dq3_takes(a)) return launch_mfma_dq3(a, fuse_delta, st);
    if (a.dk_dim == 128) return a.grad_f32 ? launch_dq<128, true>(a, fuse_delta, st) : launch_dq<128, false>(a, fuse_delta, st);
    return a.grad_f32 ? launch_dq<64, true>(a, fuse_delta, st) : launch_dq<64, false>(a, fuse_delta, st);
}

}  // namespace

bool bf16_deals_heads(const AttnArgs& a) { return a.head_split > 1 && (split_deals_heads(a) || mfma_dkdv3_takes(a)); }

int launch_row_delta(const AttnArgs& a, bool bf16, hipStream_t st) {
    const int lanes = bf16 || a.dk_dim > 32 ? 16 : 8;
    const dim3 grid((a.T + 256 / lanes - 1) / (256 / lanes) * a.Hq * a.B);
    if (bf16)  // asked for above 64 columns
        hipLaunchKernelGGL((row_delta<true, 16>), grid, dim3(256), 0, st, a);
    else if (lanes == 16)
        hipLaunchKernelGGL((row_delta<false, 16>), grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL((row_delta<false, 8>), grid, dim3(256), 0, st, a);
    PK_HIP(hipGetLastError());
    return PK_OK;
}
Bwd bwd_of_bf16(const AttnArgs& a) {
    if (joined_takes_bwd(a)) return Bwd::JOINED;
    return split_takes_joined(a) ? Bwd::SPLIT_JOINED : split_takes_bwd(a) ? Bwd::SPLIT : Bwd::APART;
}
int launch_mfma_bwd(const AttnArgs& a, int stages, hipStream_t st) {
    // delta and dQ asked for together: dQ forms delta itself and runs first, dK/dV reads what it wrote
    const bool fused = (stages & PK_BWD_DELTA) && (stages & PK_BWD_DQ);
    const Bwd form = stages == PK_BWD_ALL && !a.in_place ? bwd_of_bf16(a) : Bwd::APART;
    if (form != Bwd::APART) return form == Bwd::JOINED ? launch_joined_bwd(a, st) : form == Bwd::SPLIT ? launch_split_bwd(a, st) : launch_split_joined(a, st);
    int rc = PK_OK;
    if (fused)
        rc = run_dq(a, true, st);
    else if (stages & PK_BWD_DELTA)
        rc = a.dk_dim == 128 ? launch_delta<128>(a, st) : a.dk_dim == 64 ? launch_delta<64>(a, st)
                                                                        : launch_generic_bwd(a, true, PK_BWD_DELTA, st);
    if (rc) return rc;
    if (stages & PK_BWD_DKDV) {
        // split queries as above; without a band: 64 keys per wavefront, one wavefront per SIMD; with one: 32 keys, two
        // per SIMD
        rc = split_takes_dkdv(a) ? launch_split_dkdv(a, st) : mfma_dkdv3_takes(a) ? launch_mfma_dkdv3(a, st) : launch_mfma_dkdv2(a, st);
        if (rc) return rc;
    }
    return !fused && (stages & PK_BWD_DQ) ? run_dq(a, false, st) : PK_OK;
}

}  // namespace pk
