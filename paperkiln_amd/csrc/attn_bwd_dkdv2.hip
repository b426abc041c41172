// dK / dV of the recompute backward, second generation (see attn_bwd_mfma.hip
// for the mathematics and the operand layouts).
//
// Measured: the one-wavefront-per-SIMD kernel that keeps K, V, dK^T and dV^T
// of 32 keys in one wavefront's registers leaves the matrix pipe idle while
// that wavefront does its exp2 / LDS work, and cannot be run two per SIMD
// (it needs > 256 registers). Here the work of one 32-key block is split
// between TWO wavefronts that share a SIMD:
//
//   role 0 (wavefronts 0-3):  S = Q K^T -> P = exp2(S*c - LSE) -> dV^T += dO^T P
//   role 1 (wavefronts 4-7):  dP = dO V^T -> dS = P .* (dP - delta) -> dK^T += Q^T dS
//
// Each holds one operand (K or V) and one accumulator (dV^T or dK^T): ~180
// registers, two wavefronts per SIMD, 16 MFMAs each per 32 x 32 block, no
// recomputation. P goes from role 0 to role 1 through LDS as packed fp16 pairs in
// the accumulator's own element order (lane-private 32 bytes, conflict-free). Role 1
// runs ONE STEP BEHIND role 0, so the hand-over needs no extra barrier: the
// step barrier that publishes the next Q / dO tile also publishes P.
//
// Step = 64 queries of one query head. Q / dO tiles sit in a three-deep LDS
// ring (role 0 reads step s, role 1 step s-1, step s+1 is being stored).
#include <cstdlib>
#include <type_traits>

#include "attn_bwd_dq.h"
#include "mfma_common.h"
#include "pk_internal.h"

namespace pk {
namespace {

// Two geometries. 128 keys per workgroup (8 wavefronts, 64-query steps, one workgroup per CU) is the general one.
// With a narrow band a key block meets only a handful of query steps, and the fixed costs of a workgroup -- resident
// rows, first tiles, pipeline fill, epilogue -- weigh as much as its steps; there a workgroup takes 64 keys with 4
// wavefronts and 32-query steps, so that TWO workgroups fit a CU (registers: still two wavefronts per SIMD; LDS: 61 KB
// each) and one's fixed costs run beside the other's steps. Finer tiles also waste less on the band's edges.
typedef __fp16 h16x2 __attribute__((ext_vector_type(2)));

template <bool F32>
__device__ inline void store4g(void* base, int64_t idx, float x0, float x1, float x2, float x3) {
    if (F32) {
        f32x4 v = {x0, x1, x2, x3};
        *reinterpret_cast<f32x4*>(static_cast<float*>(base) + idx) = v;
    } else {
        u32x2 v = {pack_bf16(x0, x1), pack_bf16(x2, x3)};
        *reinterpret_cast<u32x2*>(static_cast<uint16_t*>(base) + idx) = v;
    }
}

template <int D, int BMQ>
using Ring = uint16_t[2][3][BMQ * (D + 8)];  // [Q | dO][ring slot]
template <int BNK, int BMQ>
using Weights = uint16_t[2][BMQ / 32][BNK / 32][2 * 64 * 8];  // [step parity][query block][key block][half][lane][8]
template <int BMQ>
using Rows = float[3][BMQ];

// A workgroup's blocks of BNK keys, by its number in the launch; JOINED: the block jblk of unit jkvu.
// TAIL: the launch carries the extra workgroups of a split sink tail (a separate instantiation, so
// that the plain causal kernel keeps its register budget)
// JOINED: delta is formed here, from the chunks of O beside those of dO, while a tile is moved, and the heads of a group may be dealt to
// a.head_split workgroups of which this is the rr-th (gqa_head_split); otherwise delta is read and all heads are walked.
template <int D, bool GF32, bool TAIL, int BNK, int BMQ, bool JOINED>
__device__ inline void dkdv2_blocks(const AttnArgs& a, Ring<D, BMQ>& tiles, Weights<BNK, BMQ>& Pbuf, Rows<BMQ>& nlse_s, Rows<BMQ>& dl_s,
                                    int jblk = 0, int jkvu = 0, int share = 0) {
    constexpr int KK = D / 16, DB = D / 32;
    constexpr int NTHR = 4 * BNK, NKB = BNK / 32, NQB = BMQ / 32;  // threads; 32-key blocks; 32-query blocks per step
    constexpr int S = D + 8;            // tile row pitch (elements): 16-byte row reads conflict-free
    constexpr int NCH = D / 8;          // 16-byte chunks per row
    constexpr int CPT = BMQ * NCH / NTHR;  // chunks per thread per tensor per step
    static_assert(CPT >= 1 && BMQ * NCH % NTHR == 0, "every thread stages the same number of chunks");
    static_assert(!JOINED || NCH == 8 || NCH == 16, "a row's chunks are in 8 or 16 neighbouring lanes");
    uint16_t (*const Qs)[BMQ * S] = tiles[0];
    uint16_t (*const dOs)[BMQ * S] = tiles[1];

    const int lane = threadIdx.x & 63;
    // the wavefront index as a scalar: every test on it becomes a scalar branch
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int role = w / NKB, kbw = w % NKB;
    const int g = lane >> 5, c32 = lane & 31;
    // Lane parts of the two LDS operand addresses (elements): a 16-byte row read at
    // (row c32, column 8g) and a transposing read as lds_read_tr_operand_perm lays it out.
    const int row_lane = lds_row<D>(c32) * S + g * 8;
    const int tr_lane = lds_row<D>(4 * g + ((lane & 15) >> 2)) * S + TrMap<D>::src_col(0, (lane >> 4) & 1, lane & 3);
    const int nkb = (a.T + BNK - 1) / BNK, rep = quotient(a.Hq, a.Hkv), hs = JOINED ? a.head_split : 1;
    // Full-causal: key block i is seen by T - 128i queries.
    int blk = jblk, rr = share, kvu = jkvu;
    // Band mask with a few sink keys: the queries past block 0's band are cut into chunks that get
    // workgroups of their own (ids nkb .. nkb + nch - 1 of the unit), see sink_tail.
    const SinkTail tl = TAIL ? sink_tail(a.T, a.window, a.sinks) : SinkTail{0, 0};
    if (JOINED) {
    } else if (TAIL) {
        if (!xcd_map(nkb + tl.nch, 1, a.Hkv * a.B, blk, rr, kvu)) return;
    } else if (a.window > 0 && a.sinks > 0 && nkb > 1) {
        if (!xcd_map_block0_first(nkb, a.Hkv * a.B, blk, kvu)) return;
    } else if (!map_causal_blocks(a, nkb, 1, blk, rr, kvu)) {
        return;
    }
    const int chunk = (TAIL && blk >= nkb) ? blk - nkb : -1;  // >= 0: this workgroup takes a chunk of the sink tail
    if (TAIL && chunk >= 0) blk = 0;
    const int b = quotient(kvu, a.Hkv), hk = kvu - b * a.Hkv, h0 = JOINED ? quotient(rr * rep, hs) : 0, nh = JOINED ? quotient((rr + 1) * rep, hs) - h0 : rep;
    const float cexp = a.scale * LOG2E;
    const int npass = (!JOINED && a.paired && blk != nkb - 1 - blk) ? 2 : 1;

    for (int pass = 0; pass < npass; ++pass) {
        const int kblk = pass == 0 ? blk : nkb - 1 - blk;  // heavy block first
        const int k0 = kblk * BNK;
        const int kw0 = k0 + kbw * 32;  // this wavefront's 32 keys
        const int kj = kw0 + c32;

        // The wavefront's resident operand: K for role 0, V for role 1 (B operand,
        // lane = key, chunk kk covers d = 16kk + 8g .. +7). Keys past the end
        // re-read the last row; their P is masked to zero and nothing is stored.
        bf16x8 kv[KK];
        {
            const void* src = role == 0 ? a.k : a.v;
            const int64_t off = role == 0 ? b * a.k_sb + hk * a.k_sh : b * a.v_sb + hk * a.v_sh;
            const int64_t st = role == 0 ? a.k_st : a.v_st;
            const int t = min(kj, a.T - 1);
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                const u32x4 z = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(src) + off + t * st +
                                                                kk * 16 + g * 8);
                kv[kk] = *reinterpret_cast<const bf16x8*>(&z);
            }
        }
        // Query tiles that can see keys [k0, k0+127] (paperkiln src/ops.cpp:960-965 inverted).
        const int khi = min(k0 + BNK, a.T) - 1;
        int qt_lo = a.causal ? k0 / BMQ : 0;
        int qt_hi = (a.window > 0 && (k0 >= a.sinks || TAIL)) ? min(a.T - 1, khi + a.window - 1) / BMQ
                                                              : (a.T - 1) / BMQ;
        if (TAIL && chunk >= 0) {
            qt_lo = (tl.q0 + chunk * TAIL_CHUNK) / BMQ;
            qt_hi = min(a.T - 1, tl.q0 + (chunk + 1) * TAIL_CHUNK - 1) / BMQ;
        } else if (TAIL && kblk == 0) {
            qt_hi = tl.q0 / BMQ - 1;  // the band part of block 0 ends where the chunks begin, whatever the block size
        }
        const int nqt = qt_hi - qt_lo + 1;
        const int steps = nqt * nh;

        u32x4 qr[CPT], gr[CPT], orow[JOINED ? CPT : 1];
        float lse_r = 0.0f, dl_r = 0.0f;
        // Steps are fetched in order, so the (head, query tile) of the next fetch is counted up, not divided out of
        // the step number, and a thread's position inside a tile (row tid / NCH + RPI i, chunk tid % NCH) is formed once.
        // (Tile positions as scalar bases plus per-thread 32-bit offsets, as the 64-key kernel keeps them, take a
        // third of the vector instructions out of the staging and measured no faster here, slower at head_dim 64.)
        int f_h = hk * rep + h0, f_qt = 0;
        const int frow = static_cast<int>(threadIdx.x) / NCH, fch = static_cast<int>(threadIdx.x) % NCH;
        constexpr int RPI = NTHR / NCH;  // tile rows between a thread's consecutive chunks
        auto fetch = [&]() {  // global -> registers, rows past the end clamped
            const int q0 = (qt_lo + f_qt) * BMQ;
            const uint16_t* qb = static_cast<const uint16_t*>(a.q) + b * a.q_sb + f_h * a.q_sh + fch * 8;
            const uint16_t* gb = static_cast<const uint16_t*>(a.d_o) + b * a.do_sb + f_h * a.do_sh + fch * 8;
#pragma unroll
            for (int i = 0; i < CPT; ++i) {
                const int t = min(q0 + frow + RPI * i, a.T - 1);
                qr[i] = *reinterpret_cast<const u32x4*>(qb + t * a.q_st);
                gr[i] = *reinterpret_cast<const u32x4*>(gb + t * a.do_st);
                if (JOINED)
                    orow[i] = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(a.o) + b * a.o_sb + f_h * a.o_sh + fch * 8 + t * a.o_st);
            }
            if (threadIdx.x < BMQ) {
                const int t = min(q0 + static_cast<int>(threadIdx.x), a.T - 1);
                const int64_t lrow = (static_cast<int64_t>(b) * a.Hq + f_h) * a.T + t;
                lse_r = a.lse[lrow];  // scaled when it is stored: arithmetic on it here would wait for every load just issued
                if (!JOINED) dl_r = a.delta[lrow];
            }
            const bool wrap = f_qt + 1 == nqt;
            f_qt = wrap ? 0 : f_qt + 1;
            f_h += wrap;
        };
        auto commit = [&](int slot) {  // registers -> LDS ring slot
            // The store addresses are rebuilt from the thread index at every call (the
            // empty statement hides its value): a handful of shifts, where addresses
            // kept live across the step were the ones the allocator sent to scratch.
            int tid = threadIdx.x;
            asm volatile("" : "+v"(tid));
#pragma unroll
            for (int i = 0; i < CPT; ++i) {
                const int c = tid + NTHR * i;
                const int row = c / NCH, ch = c % NCH;
                *reinterpret_cast<u32x4*>(Qs[slot] + lds_row<D>(row) * S + ch * 8) = qr[i];
                *reinterpret_cast<u32x4*>(dOs[slot] + lds_row<D>(row) * S + ch * 8) = gr[i];
                if (JOINED) {
                    float part = 0.0f;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        part = fmaf(__uint_as_float(orow[i][e] << 16), __uint_as_float(gr[i][e] << 16), part);
                        part = fmaf(__uint_as_float(orow[i][e] & 0xFFFF0000u), __uint_as_float(gr[i][e] & 0xFFFF0000u), part);
                    }
                    part += lane_moved<0xB1>(part);   // lane ^ 1
                    part += lane_moved<0x4E>(part);   // lane ^ 2
                    part += lane_moved<0x141>(part);  // the other four of eight
                    if (NCH == 16) part += lane_moved<0x140>(part);  // the other eight of sixteen
                    if (ch == 0) dl_s[slot][row] = part;
                }
            }
            if (tid < BMQ) {
                nlse_s[slot][tid] = -lse_r * LOG2E;
                if (!JOINED) dl_s[slot][tid] = dl_r;
            }
        };
        // wavefront-uniform: is anything of (query block qb of the step at query tile `qt`) x (this key block) visible?
        auto block_live = [&](int qt, int qb, int& qlo) {
            qlo = (qt_lo + qt) * BMQ + qb * 32;
            const int qhi = qlo + 31;
            if (qlo >= a.T || kw0 >= a.T) return false;
            if (a.causal && kw0 > qhi) return false;
            if (a.window > 0 && kw0 + 31 + a.window <= qlo && kw0 >= a.sinks) return false;
            return true;
        };

        if (steps > 0) {
            fetch();
            commit(0);
            if (steps > 1) fetch();
        }
        // Every load issued so far -- the resident K / V rows above all -- has landed before the step loop is
        // entered. Without this the wait-count bookkeeping carries "kv may still be in flight" around the loop
        // and puts a vmcnt wait in front of each MFMA that reads kv, which in every later step waits for the
        // NEXT tile's prefetch instead (a full memory latency per step).
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
        __syncthreads();

        // transposed operand (k-chunk = rows row0 + {4g..4g+3} u {8+4g..}) of column block db, from a
        // pointer that already carries the lane part
        auto tr_operand = [&](const uint16_t* p, int row0, int db) {
            p += row0 * S + TrMap<D>::src_col(db, 0, 0);
            const s16x4 lo = lds_read_tr4(p), hi = lds_read_tr4(p + TR_HI_ROWS<D> * S);
            typedef short s16x8 __attribute__((ext_vector_type(8)));
            const s16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            return *reinterpret_cast<const bf16x8*>(&v);
        };
        // The step loop and the stores are instantiated once per role and entered through one branch on the role: with
        // the role tested inside the loop the two sides of the branch each get their own copy of the accumulators,
        // which are moved back at the join in every step (64 register moves a step, found in the compiled loop).
        auto run_role = [&](auto role_tag) {
        constexpr int rl = decltype(role_tag)::value;
        f32x16 acc[DB];  // dV^T (role 0) or dK^T (role 1)
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[db][r] = 0.0f;
        // iteration s: role 0 works on step s, role 1 on step s-1; the query tile of either is counted, not divided out
        int c_qt = 0, slot = 0;  // query tile and ring slot of the step this role works on
        for (int s = 0; s <= steps; ++s) {
            if (s + 1 < steps) {
                commit((s + 1) % 3);  // slot last read (by role 1) before the previous barrier
                if (s + 2 < steps) fetch();
            }
            if (rl == 0) {
                if (s < steps) {
                    // One register each for the row-read and the transposing-read address of
                        // this step; every fragment is then an immediate offset away. Left to
                        // itself the compiler keeps a dozen pre-offset copies and spills.
                    int xrow = slot * (BMQ * S) + row_lane;                     // Q rows
                    int ytr = (3 + slot) * (BMQ * S) + tr_lane;                 // dO transposed
                    asm volatile("" : "+v"(xrow), "+v"(ytr));
                    const uint16_t* flat = &tiles[0][0][0];
#pragma unroll
                    for (int qb = 0; qb < NQB; ++qb) {
                        int qlo;
                        if (!block_live(c_qt, qb, qlo)) continue;
                        // One accumulator chain: the other role's wavefront on this SIMD issues
                        // into the gaps a dependent MFMA pair leaves, and the registers of a
                        // second chain would push the kernel into scratch.
                        f32x16 sc;
#pragma unroll
                        for (int r = 0; r < 16; ++r) sc[r] = 0.0f;
#pragma unroll
                        for (int kk = 0; kk < KK; ++kk)
                            sc = mfma32(lds_read8(flat + xrow + qb * 32 * S + kk * 16), kv[kk], sc);
                        const int qhi = qlo + 31;
                        const bool full = qhi < a.T && kw0 + 31 < a.T && (!a.causal || kw0 + 31 <= qlo) &&
                                          (a.window == 0 || kw0 + a.window > qhi || kw0 + 31 < a.sinks);
                        // lane = key kj; element r = query qlo + (r/4)*8 + 4g + r%4
#pragma unroll
                        for (int qd = 0; qd < 4; ++qd) {
                            const f32x4 nl = *reinterpret_cast<const f32x4*>(&nlse_s[slot][qb * 32 + qd * 8 + g * 4]);
#pragma unroll
                            for (int e = 0; e < 4; ++e)
                                sc[qd * 4 + e] = __builtin_amdgcn_exp2f(fmaf(sc[qd * 4 + e], cexp, nl[e]));
                        }
                        if (!full) {  // off the common path: interior tiles carry no mask arithmetic at all
                            const KeyVis kvis(kj, a.T, a.causal, a.window, a.sinks);
#pragma unroll
                            for (int r = 0; r < 16; ++r)
                                sc[r] = kvis(qlo + (r >> 2) * 8 + g * 4 + (r & 3)) ? sc[r] : 0.0f;
                        }
                        const bf16x8 p0 = c_to_operand<0>(sc), p1 = c_to_operand<1>(sc);
                        // hand-over copy in fp16: P is in [0, 1], where fp16 carries 11 significant
                        // bits against bf16's 8, so dS is built from a P as good as the old fp32 one
                        // the two 16-byte halves of a lane sit 1 KB apart: consecutive lanes then
                        // write consecutive 16-byte chunks and no two lanes share a bank
                        uint16_t* pb = Pbuf[s & 1][qb][kbw] + lane * 8;
                        h16x2 ph[8];
#pragma unroll
                        for (int i = 0; i < 8; ++i) {
                            const f32x2 pr = {sc[2 * i], sc[2 * i + 1]};
                            ph[i] = __builtin_convertvector(pr, h16x2);  // round to nearest even
                        }
                        *reinterpret_cast<u32x4*>(pb) = *reinterpret_cast<u32x4*>(&ph[0]);
                        *reinterpret_cast<u32x4*>(pb + 512) = *reinterpret_cast<u32x4*>(&ph[4]);
                        // dV^T += dO^T P
#pragma unroll
                        for (int db = 0; db < DB; ++db)
                            acc[db] = mfma32(tr_operand(flat + ytr, qb * 32, db), p0, acc[db]);
#pragma unroll
                        for (int db = 0; db < DB; ++db)
                            acc[db] = mfma32(tr_operand(flat + ytr, qb * 32 + 16, db), p1, acc[db]);
                    }
                    c_qt = c_qt + 1 == nqt ? 0 : c_qt + 1;
                    slot = slot == 2 ? 0 : slot + 1;
                }
            } else {
                if (s >= 1) {
                    const int sp = s - 1;
                    int xrow = (3 + slot) * (BMQ * S) + row_lane;               // dO rows
                    int ytr = slot * (BMQ * S) + tr_lane;                       // Q transposed
                    asm volatile("" : "+v"(xrow), "+v"(ytr));
                    const uint16_t* flat = &tiles[0][0][0];
#pragma unroll
                    for (int qb = 0; qb < NQB; ++qb) {
                        int qlo;
                        if (!block_live(c_qt, qb, qlo)) continue;
                        f32x16 dp;
#pragma unroll
                        for (int r = 0; r < 16; ++r) dp[r] = 0.0f;
#pragma unroll
                        for (int kk = 0; kk < KK; ++kk)
                            dp = mfma32(lds_read8(flat + xrow + qb * 32 * S + kk * 16), kv[kk], dp);
                        const uint16_t* pb = Pbuf[sp & 1][qb][kbw] + lane * 8;
                        u32x4 praw[2];
                        praw[0] = *reinterpret_cast<const u32x4*>(pb);
                        praw[1] = *reinterpret_cast<const u32x4*>(pb + 512);
                        const h16x2* ph = reinterpret_cast<const h16x2*>(praw);
                        // dS = P .* (dP - delta); P arrives as fp16 pairs of elements (2i, 2i+1)
#pragma unroll
                        for (int qd = 0; qd < 4; ++qd) {
                            const f32x4 dl = *reinterpret_cast<const f32x4*>(&dl_s[slot][qb * 32 + qd * 8 + g * 4]);
                            dp[qd * 4 + 0] = static_cast<float>(ph[2 * qd][0]) * (dp[qd * 4 + 0] - dl[0]);
                            dp[qd * 4 + 1] = static_cast<float>(ph[2 * qd][1]) * (dp[qd * 4 + 1] - dl[1]);
                            dp[qd * 4 + 2] = static_cast<float>(ph[2 * qd + 1][0]) * (dp[qd * 4 + 2] - dl[2]);
                            dp[qd * 4 + 3] = static_cast<float>(ph[2 * qd + 1][1]) * (dp[qd * 4 + 3] - dl[3]);
                        }
                        const bf16x8 d0 = c_to_operand<0>(dp), d1 = c_to_operand<1>(dp);
                        // dK^T += Q^T dS
#pragma unroll
                        for (int db = 0; db < DB; ++db)
                            acc[db] = mfma32(tr_operand(flat + ytr, qb * 32, db), d0, acc[db]);
#pragma unroll
                        for (int db = 0; db < DB; ++db)
                            acc[db] = mfma32(tr_operand(flat + ytr, qb * 32 + 16, db), d1, acc[db]);
                    }
                    c_qt = c_qt + 1 == nqt ? 0 : c_qt + 1;
                    slot = slot == 2 ? 0 : slot + 1;
                }
            }
            __syncthreads();
        }

        // Pieces of a split sink tail: the sink keys' rows go to the workspace as fp32 partial sums
        // (a chunk writes nothing else; the band part of block 0 writes its other rows as usual).
        const bool piece = TAIL && kblk == 0;
        if (piece && kbw == 0 && kj < a.sinks) {
            float* rows = sink_tail_rows(a.tail, kvu, tl.nch, chunk >= 0 ? chunk : tl.nch, rl == 0 ? 1 : 0, D) + kj * D;
            const float sc = rl == 0 ? 1.0f : a.scale;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int qd = 0; qd < 4; ++qd)
                    store4g<true>(rows, TrMap<D>::col0(db, qd, g), acc[db][qd * 4] * sc, acc[db][qd * 4 + 1] * sc,
                                  acc[db][qd * 4 + 2] * sc, acc[db][qd * 4 + 3] * sc);
        }
        if (JOINED && hs > 1) {  // partial sums of this share of the heads, for launch_gqa_reduce
            static_assert(!JOINED || NTHR / 64 * LineStrip<64>::FLOATS * 2 <= 6 * BMQ * S, "the wavefronts' strips");
            float* const strip = reinterpret_cast<float*>(Qs[0]) + static_cast<int>(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * LineStrip<64>::FLOATS;
            const int k1 = kj - c32;
            const int64_t row = ((static_cast<int64_t>(kvu) * hs + rr) * 2 + (rl == 0 ? 1 : 0)) * a.T + k1;
            store_rows_f32<D>(strip, a.part + row * D, D, a.T - k1, acc, rl == 0 ? 1.0f : a.scale, lane);
        } else if (!GF32 && chunk < 0) {  // (no tile is read any more)
            using Rows = RowStrip<D>;
            static_assert(NTHR / 64 * Rows::ELEMS <= 6 * BMQ * S, "the wavefronts' strips");
            uint16_t* const strip = Qs[0] + static_cast<int>(__builtin_amdgcn_readfirstlane(threadIdx.x >> 6)) * Rows::ELEMS;
            const int k1 = kj - c32, from = piece ? a.sinks - k1 : 0;
            const int64_t st = rl == 0 ? a.dv_st : a.dk_st;
            const float sc = rl == 0 ? 1.0f : a.scale;
#pragma unroll
            for (int db = 0; db < DB; ++db) store_acc_bf16<D>(Rows::row(strip, c32), db, g, acc[db], sc);
            Rows::out(strip, static_cast<uint16_t*>(rl == 0 ? a.dv : a.dk) + (rl == 0 ? b * a.dv_sb + hk * a.dv_sh : b * a.dk_sb + hk * a.dk_sh) + k1 * st, st, from,
                      a.T - k1, lane);
        } else if (kj < a.T && chunk < 0 && !(piece && kj < a.sinks)) {
            void* dst = rl == 0 ? a.dv : a.dk;
            const int64_t ob = rl == 0 ? b * a.dv_sb + hk * a.dv_sh + kj * a.dv_st
                                         : b * a.dk_sb + hk * a.dk_sh + kj * a.dk_st;
            const float sc = rl == 0 ? 1.0f : a.scale;
#pragma unroll
            for (int db = 0; db < DB; ++db) {
#pragma unroll
                for (int qd = 0; qd < 4; ++qd)
                    store4g<GF32>(dst, ob + TrMap<D>::col0(db, qd, g), acc[db][qd * 4] * sc, acc[db][qd * 4 + 1] * sc,
                                  acc[db][qd * 4 + 2] * sc, acc[db][qd * 4 + 3] * sc);
            }
        }
        };  // run_role
        if (role == 0)
            run_role(std::integral_constant<int, 0>{});
        else
            run_role(std::integral_constant<int, 1>{});
        __syncthreads();  // the next pass refills the ring
    }
}
template <int D, bool GF32, bool TAIL, int BNK, int BMQ>
__global__ __launch_bounds__(4 * BNK, 2) void mfma_dkdv2(AttnArgs a) {
    __shared__ __attribute__((aligned(16))) Ring<D, BMQ> tiles;
    __shared__ __attribute__((aligned(16))) Weights<BNK, BMQ> Pbuf;
    __shared__ __attribute__((aligned(16))) Rows<BMQ> nlse_s;  // -LSE * log2(e)
    __shared__ __attribute__((aligned(16))) Rows<BMQ> dl_s;
    dkdv2_blocks<D, GF32, TAIL, BNK, BMQ, false>(a, tiles, Pbuf, nlse_s, dl_s);
}

// ---- dQ and dK/dV at head_dim 128 in one launch: blocks of 64 keys and of 128 queries (joined_takes_bwd) ----
// By rank: two blocks of keys for each share of the group's heads and one of queries for each head. Under a band every unit's block of sink keys comes first, then
// a unit's blocks along its band; else the longest of every unit.
template <bool GF32>
__global__ __launch_bounds__(256, 2) void joined_bwd(AttnArgs a) {
    __shared__ union {
        struct {
            __attribute__((aligned(16))) Ring<128, 32> tiles;
            __attribute__((aligned(16))) Weights<64, 32> p;
            __attribute__((aligned(16))) Rows<32> nlse, delta;
        } k;
        __attribute__((aligned(16))) uint16_t q[DQ_LDS<128, 4>];
    } lds;
    const int nkb = (a.T + 63) / 64, ranks = (a.T + 127) / 128, rep = quotient(a.Hq, a.Hkv), keys = 2 * a.head_split, each = keys + rep;
    int rank, r, kvu, at;
    if (a.window > 0) {
        if (!xcd_map_block0_first(ranks * each, a.Hkv * a.B, at, kvu)) return;
        rank = at / each, r = at % each;
    } else if (a.causal && ranks > 1 ? !xcd_map_block_major(ranks, each, a.Hkv * a.B, rank, r, kvu)
                                     : !xcd_map(ranks, each, a.Hkv * a.B, rank, r, kvu)) {
        return;
    }
    const int b = quotient(kvu, a.Hkv), hk = kvu - b * a.Hkv;
    if (r >= keys)
        dq_block<128, GF32, true, 4>(a, b, hk * rep + r - keys, hk, a.window > 0 ? rank : ranks - 1 - rank, lds.q);
    else if (2 * rank + r % 2 < nkb)
        dkdv2_blocks<128, GF32, false, 64, 32, true>(a, lds.k.tiles, lds.k.p, lds.k.nlse, lds.k.delta, 2 * rank + r % 2, kvu, r / 2);
}

// dK / dV rows [0, sinks) of every (batch, KV head) = the band part plus the chunks, in that order. One element a thread: a
// unit's rows as a loop of one workgroup were a chain of up to 32 x (nch + 1) dependent loads behind each other.
template <bool GF32>
__global__ __launch_bounds__(256) void sink_tail_reduce(AttnArgs a, int nch) {
    const int kvu = blockIdx.x, hk = kvu % a.Hkv, b = kvu / a.Hkv, D = a.dk_dim;
    const int idx = blockIdx.y * 256 + threadIdx.x;
    if (idx < 2 * a.sinks * D) {
        const int which = idx / (a.sinks * D), j = (idx / D) % a.sinks, d = idx % D;
        float sum = sink_tail_rows(a.tail, kvu, nch, nch, which, D)[j * D + d];
#pragma unroll 4
        for (int c = 0; c < nch; ++c) sum += sink_tail_rows(a.tail, kvu, nch, c, which, D)[j * D + d];
        void* dst = which == 0 ? a.dk : a.dv;
        const int64_t at = which == 0 ? b * a.dk_sb + hk * a.dk_sh + j * a.dk_st + d
                                      : b * a.dv_sb + hk * a.dv_sh + j * a.dv_st + d;
        if (GF32) {
            static_cast<float*>(dst)[at] = sum;
        } else {
            const uint32_t two = pack_bf16(sum, 0.0f);
            static_cast<uint16_t*>(dst)[at] = static_cast<uint16_t>(two & 0xffffu);
        }
    }
}

// The sink tail that a launch of this kernel deals out, if any (nch = 0: none). A tail step keeps two of the eight wavefronts
// busy but takes as long as a full one (measured).
SinkTail dealt_tail(const AttnArgs& a) {
    const SinkTail tl = a.tail ? sink_tail(a.T, a.window, a.sinks) : SinkTail{0, 0};
    return sink_tail_pays(tl, a.T, a.window, a.Hkv * a.B, 64, 3, 1.0f) ? tl : SinkTail{0, 0};
}

template <int D, bool GF32, int BNK, int BMQ>
int launch_geo(const AttnArgs& a_in, hipStream_t st) {
    AttnArgs a = a_in;
    const int nkb = (a.T + BNK - 1) / BNK;
    a.paired = pair_causal_blocks(nkb, static_cast<int64_t>(a.Hkv) * a.B, a.causal, a.window, 256);
    const SinkTail tl = dealt_tail(a);
    if (tl.nch == 0) a.tail = nullptr;
    if (tl.nch > 0) {
        hipLaunchKernelGGL((mfma_dkdv2<D, GF32, true, BNK, BMQ>), dim3(xcd_grid(nkb + tl.nch, 1, a.Hkv * a.B)), dim3(4 * BNK), 0,
                           st, a);
        PK_HIP(hipGetLastError());
        return launch_sink_tail_reduce(a, st);
    }
    const int ids = a.window > 0 && a.sinks > 0 && nkb > 1 ? xcd_grid_block0_first(nkb, a.Hkv * a.B)
                                                           : xcd_grid(a.paired ? (nkb + 1) / 2 : nkb, 1, a.Hkv * a.B);
    hipLaunchKernelGGL((mfma_dkdv2<D, GF32, false, BNK, BMQ>), dim3(ids), dim3(4 * BNK), 0, st, a);
    PK_HIP(hipGetLastError());
    return PK_OK;
}

// Short sequences and bands of a few key blocks: the small geometry, two workgroups per CU or (head_dim 64) four, which
// hides the two memory round trips at the start of each and wastes less of the last tile. Measured, small | large
// (us): B=4 H=16 T=4096, head_dim 128, window 128 190 | 229, 512 264 | 276, 1024 404 | 387; 16 heads, no band, T 48 x 170
// at head_dim 64 29 | 57, at 128 59 | 82; T 128 x 64 28 | 36 and 52 | 67; T 400 x 20 41 | 49 and 76 | 81; T 900 x 3,
// head_dim 64 32 | 26.
// The large one is ahead in spite of that where its workgroups, one to a CU, come to one round of the chip, or nearly whole to
// two, and the small one's do not save a part of them in the last tile: head_dim 64, causal, T 200 x 128 heads 15 | 11, 256 x
// 128 16 | 12, 512 x 128 29 | 25, 96 x 256 13 | 10, 400 x 64 17 | 15, 320 x 96 15 | 13; no mask, 400 x 128 36 | 30, 512 x 128
// 40 | 33, 320 x 160 28 | 23, 160 x 256 (a part saved) 20 | 25; one head more in eight and it is behind (512 x 160, causal
// 33 | 34, 256 x 160 14 | 16). At head_dim 128 only where one round is whole (causal, 256 x 128 22 | 19, 96 x 256 17 | 15) or all
// chains are as long (no mask, 400 x 48 25 | 22, 480 x 64 29 | 27).
// At head_dim 64 a wide band has to come with many of its workgroups (3571 tokens, window 315, 8 heads 20 | 16; 2000 x 4,
// window 300, 16 heads 56 | 64; 2000 x 2, 16 heads, window 512 48 | 39), sink keys with a narrow one, whose tail then hides the
// sinks' (16 heads of 500 tokens, window 100, 4 sinks: x 16 40 | 52, x 6 24 | 23; 2000 x 4, window 300, 16 sinks 74 | 71) or is
// dealt out (64 heads of 2000, window 128, 4 sinks, left whole 76 | 60; window 32, dealt out 53 | 64).
template <int D>
bool small_geometry_is_ahead(const AttnArgs& a) {
    const int64_t units = static_cast<int64_t>(a.Hkv) * a.B;
    const int64_t small = (a.T + 63) / 64 * units, large = (a.T + 127) / 128 * units;  // workgroups of either
    if (a.window == 0) {
        if (a.T > 512 || (a.T > 256 && small < 256)) return false;
        const bool saves = small * 5 < large * 8;
        if (D == 128) return large > 256 || (a.causal || a.T <= 300 ? saves || large < 240 : false);
        if (large <= 256) return a.T <= 32;
        if (large > 512) return true;
        return a.causal ? !((a.T > 256 && large <= 300) || (a.T > 128 && large > 480 && small == 2 * large)) : saves || large < 450;
    }
    if (a.window > 512) return false;
    if (D == 128) return true;
    if (a.T <= 128 && a.Hq > a.Hkv) return false;  // a group's heads in turn, a step or two of 64 queries each: T 60, 14 on 2 17 | 20
    if (a.sinks > 0) return a.window <= 128 && small >= 1024 && (units > 96 || dealt_tail(a).nch > 0);
    return a.window <= 64 || (a.window <= 128 ? large < 160 || large > 256 : small >= 1100);
}

template <int D, bool GF32>
int launch(const AttnArgs& a, hipStream_t st) {
    if (small_geometry_is_ahead<D>(a)) return launch_geo<D, GF32, 64, 32>(a, st);
    return launch_geo<D, GF32, 128, 64>(a, st);
}

}  // namespace

int launch_sink_tail_reduce(const AttnArgs& a, hipStream_t st) {
    const int nch = sink_tail(a.T, a.window, a.sinks).nch;
    const dim3 grid(a.Hkv * a.B, (2 * a.sinks * a.dk_dim + 255) / 256);
    if (a.grad_f32)
        hipLaunchKernelGGL(sink_tail_reduce<true>, grid, dim3(256), 0, st, a, nch);
    else
        hipLaunchKernelGGL(sink_tail_reduce<false>, grid, dim3(256), 0, st, a, nch);
    PK_HIP(hipGetLastError());
    return PK_OK;
}

// Where either launch by itself is a round of the chip or less, its longest chains last as long as it does, and together one's run beside the
// other's; dK/dV forms delta while it moves its tiles, 20 vector instructions a 16-byte chunk. From 4096 tokens on without a band the launches
// stay apart, which keeps dQ's bits whatever the number of units. In 64-row blocks of queries (q), one after the other | joined, us:
//   causal     T 222 x 5, 16 heads (320) 27 | 20;  T 79 x 18, 4 heads (144) 18 | 11;  T 571 x 2, 8 heads (144) 41 | 32;  T 1792, 16 heads (448) 111 | 101;
//              T 307 x 4, 16 on 8 (320) 48 | 35;  T 739, 28 on 4 (336) 67 | 54;  T 2531, 7 on one (280) 152 | 134
//     not      T 609 x 6, 1 head (60) 25 | 34;  T 1423, 8 heads (184) 64 | 74;  T 3991, 4 on 2 (252) 175 | 191;  T 2422 x 3, 8 heads (912) 164 | 200
//   no mask    T 54 x 10, 8 heads (80) 14.5 | 8.5;  T 1061 x 4, 2 heads (136) 88 | 59;  T 2309, 8 heads (296) 172 | 140;  T 611, 28 on 4 (280) 70 | 52
//     not      T 1229, 4 heads (80) 54 | 67;  T 352 x 16, 4 heads (384) 40 | 42;  T 1461 x 3, 7 on one (483) 136 | 175;  T 2006, 4 heads (128), where
//              blocks of 32 rows are a round 70 | 100;  T 62 x 11, 32 on 16 (352) 20 | 24;  T 49 x 69, 4 on 2 (276) 18 | 22
//   band       T 559 x 4, 8 heads, 71 (288) 30 | 20;  T 140 x 11, 8 heads, 27, 1 sink (264) 24 | 16;  T 1317, 16 on 8, 123 (336) 36 | 28
//     not      with sinks in long sequences, whose block is walked whole (T 1409, 16 heads, 325 (368) 59 | 87; T 394, 28 on 4, 74 (196) 126 | 145);
//              T 59 x 29, 16 heads (464) 24 | 29;  T 2839, 14 on 2, 154 (630) 57 | 89;  few blocks: T 1702, 2 heads, 73 (54) 11.6 | 16.0;  T 1758, 4 on 2,
//              386 (112) 40 | 45;  groups of more than two whose heads are not dealt out, whose blocks of keys walk them all: T 3396, 7 on one, 477 (378)
//              92 | 162;  T 372 x 2, 16 on 4, 219 (192) 41 | 54;  T 168 x 4, 16 on 4, 17 (192) 22 | 23;  a tail of sinks beside few blocks: T 697, 8
//              heads, 181, 4 (88) 26 | 37;  and in long sequences a second round of 512 workgroups: T 3220, 8 heads, 305 (408) 46.7 | 48.4
bool joined_takes_bwd(const AttnArgs& a) {
    if (a.dk_dim != 128) return false;
    const bool groups = a.Hq > a.Hkv;
    const int64_t q = static_cast<int64_t>((a.T + 63) / 64) * a.Hq * a.B;
    if (a.window > 0)
        return a.window <= 512 && (a.Hq <= 2 * a.Hkv || bf16_deals_heads(a)) &&
               (a.sinks == 0 || (groups ? a.T <= 160 : a.T <= 700 && (a.T - a.window <= 300 || q >= 200))) &&
               q >= (groups ? (a.window > 200 ? 120 : 76) : a.T <= 130 ? 52 : 70) && q <= (a.T <= 64 || a.T > 1000 ? 320 : 600);
    if (a.T >= 4096) return false;
    if (a.T <= 130) return q >= 56 && q <= (a.T > 64 || !groups ? 500 : a.Hq == 2 * a.Hkv ? 270 : 340);
    if (!a.causal) return q >= 130 && q <= 330;
    return a.T <= 800 ? q >= 140 && q <= 600 : q >= (a.T <= 2600 ? 260 : 320) && q <= 500;
}
int launch_joined_bwd(const AttnArgs& a_in, hipStream_t st) {
    AttnArgs a = a_in;
    if (!bf16_deals_heads(a)) a.head_split = 1;
    const int ranks = (a.T + 127) / 128, each = 2 * a.head_split + a.Hq / a.Hkv;
    const dim3 grid(a.window > 0 ? xcd_grid_block0_first(ranks * each, a.Hkv * a.B) : xcd_grid(ranks, each, a.Hkv * a.B));
    if (a.grad_f32)
        hipLaunchKernelGGL(joined_bwd<true>, grid, dim3(256), 0, st, a);
    else
        hipLaunchKernelGGL(joined_bwd<false>, grid, dim3(256), 0, st, a);
    PK_HIP(hipGetLastError());
    return a.head_split > 1 ? launch_gqa_reduce(a, st) : PK_OK;
}
int launch_mfma_dkdv2(const AttnArgs& a, hipStream_t st) {
    if (a.dk_dim == 128) return a.grad_f32 ? launch<128, true>(a, st) : launch<128, false>(a, st);
    return a.grad_f32 ? launch<64, true>(a, st) : launch<64, false>(a, st);
}

}  // namespace pk
