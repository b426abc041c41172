// What the attention kernels whose wavefronts split the contraction share (attn_split.hip: bf16, attn_f32_split.hip:
// fp32). Accumulator blocks are 32 x 32 C tiles with lane = row of the output and the columns in natural order.
#pragma once
#include "mfma_common.h"
#include "pk_internal.h"

namespace pk {
namespace {

// The KW groups' accumulators of N blocks added up: group kg ends up with the sums of blocks kg, kg + KW, ... (in group
// order, so repeatable). `red` is LDS for KW N KB per row group, free to overwrite when this is called.
template <int N, int KW>
__device__ inline void join_groups(f32x16* acc, float* red, int kg, int lane) {
    if (KW == 1) return;
#pragma unroll
    for (int n = 0; n < N; ++n) {
        if (n % KW == kg) continue;
        f32x4* p = reinterpret_cast<f32x4*>(red) + ((kg * N + n) * 4) * 64 + lane;
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
            const f32x4 v = {acc[n][qd * 4], acc[n][qd * 4 + 1], acc[n][qd * 4 + 2], acc[n][qd * 4 + 3]};
            p[qd * 64] = v;
        }
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < N; ++n) {
        if (n % KW != kg) continue;
        f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.0f;
#pragma unroll
        for (int k = 0; k < KW; ++k) {
            const f32x4* p = reinterpret_cast<const f32x4*>(red) + ((k * N + n) * 4) * 64 + lane;
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                f32x4 v;
                if (k == n % KW)
                    v = {acc[n][qd * 4], acc[n][qd * 4 + 1], acc[n][qd * 4 + 2], acc[n][qd * 4 + 3]};
                else
                    v = p[qd * 64];
#pragma unroll
                for (int e = 0; e < 4; ++e) s[qd * 4 + e] += v[e];
            }
        }
        acc[n] = s;
    }
}

// The same where all wavefronts add and store: every block is four quads of eight columns (four to a lane), the shares of Q quads are dealt out
// to the KW wavefronts in turn (block by block, three of four watch one at 32 columns). `red`: 1024 N KW floats of LDS, free to overwrite. out takes
// (block, first quad, sums); weights(), asked for behind the barrier: what wavefront k's part is multiplied by, or nullptr.
template <int N, int KW, int Q, typename W, typename F>
__device__ inline void join_shares(const f32x16* acc, float* red, int kg, int lane, W weights, F out) {
    constexpr int QUADS = 4 * N, ITEMS = QUADS / Q;
    f32x4* const all = reinterpret_cast<f32x4*>(red) + lane;
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
            const f32x4 v = {acc[n][qd * 4], acc[n][qd * 4 + 1], acc[n][qd * 4 + 2], acc[n][qd * 4 + 3]};
            all[(kg * QUADS + n * 4 + qd) * 64] = v;
        }
    __syncthreads();
    const float* const weight = weights();
#pragma unroll
    for (int i = 0; i < (ITEMS + KW - 1) / KW; ++i) {
        const int item = i * KW + kg;
        if (ITEMS % KW != 0 && item >= ITEMS) break;
        f32x4 s[Q];
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            s[q] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int k = 0; k < KW; ++k) {
                const f32x4 v = all[(k * QUADS + item * Q + q) * 64];
#pragma unroll
                for (int e = 0; e < 4; ++e) s[q][e] = weight ? fmaf(v[e], weight[k], s[q][e]) : s[q][e] + v[e];
            }
        }
        out(item * Q / 4, item * Q % 4, s);
    }
}
__device__ inline const float* no_weights() { return nullptr; }

// A head's first element. The value is formed here and kept: left to itself the compiler reads the arguments again, a round trip through the
// scalar cache each, wherever the next tensor is addressed -- seven times before the first product.
// With it, LSE asked for with the rest and all wavefronts in the join, bf16 launches of short chains, us: T 128, 4 heads of 64 forward 5.4 -> 4.8,
// backward 8.0 -> 7.7; T 200, 4 heads of 128 8.5 -> 7.0, 15.6 -> 14.9; T 90 x 2, 4 heads of 32 backward 7.8 -> 6.5; T 1000 x 2, 8 heads of 80
// 48.6 -> 46.2; 96 columns, T 400, 4 heads 8.7 -> 7.8, 19.4 -> 16.6. Long chains level, backward at 64 columns 1 to 2 % ahead; not in
// the forwards of bf16 and of three parts (split_fwd, x3_fwd).
template <typename T>
__device__ inline const T* head_of(const void* base, int64_t sb, int b, int64_t sh, int h) {
    const T* p = static_cast<const T*>(base) + (b * sb + h * sh);
    asm volatile("" : "+s"(p));
    return p;
}

// A gradient's row on its way out: turned back by its position's cosines and sines where the arguments say so (AttnArgs::turn). A launch of
// its own that did this reads and writes dQ and dK again: 3 to 5 us of a layer's backward pass, against 0.3 to 2.5 of the launch here (8 x 1024
// tokens, 8 heads of 64, bf16: 56.3 -> 58.9 and one of 5.1 less). The others keep kernels without it: the registers that its test takes are 0.5 to
// 0.8 % of those too.
struct TurnRow {
    const float* at = nullptr;
    bool on = false;
    TurnRow() = default;
    __device__ TurnRow(const AttnArgs& a, int head, int row) : at(a.turn + static_cast<int64_t>(row) * a.dk_dim), on(head < a.turn_heads) {}
    // columns col .. col + 3 (a multiple of 4)
    __device__ f32x4 quad(f32x4 v, int col, int dk) const {
        if (!on) return v;
        const f32x4 t = *reinterpret_cast<const f32x4*>(at + min(col, dk - 4));
        return f32x4{v[0] * t[0] + v[1] * t[1], v[1] * t[0] - v[0] * t[1], v[2] * t[2] + v[3] * t[3], v[3] * t[2] - v[2] * t[3]};
    }
};
template <bool TURN>
__device__ inline TurnRow turn_row(const AttnArgs& a, int head, int row) {
    if constexpr (TURN)
        return TurnRow(a, head, row);
    else
        return TurnRow();
}

// One 32 x 32 accumulator block (lane = row of the output, natural column order) scaled and written; columns past dk are
// not. Both lanes of a pair (c, c + 32) hold the same row and must be active.
__device__ inline void store_block(bool f32, void* base, int64_t row_off, int db, int g, const f32x16& acc, float sc, int dk, const TurnRow& turn = {}) {
    if (f32) {
        float* row = static_cast<float*>(base) + row_off;
#pragma unroll
        for (int qd = 0; qd < 4; ++qd) {
            const int col = 32 * db + 8 * qd + 4 * g;
            const f32x4 v = {acc[qd * 4] * sc, acc[qd * 4 + 1] * sc, acc[qd * 4 + 2] * sc, acc[qd * 4 + 3] * sc};
            if (col < dk) *reinterpret_cast<f32x4*>(row + col) = turn.quad(v, col, dk);
        }
    } else {
        uint16_t* row = static_cast<uint16_t*>(base) + row_off;
#pragma unroll
        for (int qp = 0; qp < 2; ++qp) {
            const int lo = qp * 8, hi = qp * 8 + 4, at = 32 * db + 16 * qp + 4 * g;
            const f32x4 x = turn.quad(f32x4{acc[lo] * sc, acc[lo + 1] * sc, acc[lo + 2] * sc, acc[lo + 3] * sc}, at, dk),
                        y = turn.quad(f32x4{acc[hi] * sc, acc[hi + 1] * sc, acc[hi + 2] * sc, acc[hi + 3] * sc}, at + 8, dk);
            const auto r0 = __builtin_amdgcn_permlane32_swap(pack_bf16(x[0], x[1]), pack_bf16(y[0], y[1]), false, false);
            const auto r1 = __builtin_amdgcn_permlane32_swap(pack_bf16(x[2], x[3]), pack_bf16(y[2], y[3]), false, false);
            const u32x4 v = {r0[0], r1[0], r0[1], r1[1]};
            const int col = 32 * db + 8 * (2 * qp + g);
            if (col < dk) *reinterpret_cast<u32x4*>(row + col) = v;
        }
    }
}
// Rows of D bf16 that can be whole lines (RowStrip); EXACT kernels serve the sizes between. Backward in one launch, T 512 x 16, 8 heads 32.8 -> 30.1 us, 1024 x 8
// 49.4 -> 47.6, no mask, T 777 x 6, 12 heads 62.6 -> 61.2; window 128, 4 sinks, T 700 x 8, 16 heads, forward 16.2 -> 15.0 and backward 45.6 -> 44.2. Blocks of 32
// rows whose tiles are split between wavefronts write what each has joined, as before: a pass through a strip is another barrier of a launch of 5 to 10 us.
template <int D, bool EXACT>
constexpr bool WHOLE_ROWS = D % 64 == 0 && !EXACT;

// Quads qd and qd + 1 (even, odd) of such a block
__device__ inline void store_half(bool f32, void* base, int64_t row_off, int db, int qd, int g, const f32x4 (&v)[2], float sc, int dk,
                                  const TurnRow& turn = {}) {
    if (f32) {
        float* row = static_cast<float*>(base) + row_off;
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const int col = 32 * db + 8 * (qd + q) + 4 * g;
            const f32x4 o = {v[q][0] * sc, v[q][1] * sc, v[q][2] * sc, v[q][3] * sc};
            if (col < dk) *reinterpret_cast<f32x4*>(row + col) = turn.quad(o, col, dk);
        }
    } else {
        const int at = 32 * db + 8 * qd + 4 * g;
        const f32x4 x = turn.quad(f32x4{v[0][0] * sc, v[0][1] * sc, v[0][2] * sc, v[0][3] * sc}, at, dk),
                    y = turn.quad(f32x4{v[1][0] * sc, v[1][1] * sc, v[1][2] * sc, v[1][3] * sc}, at + 8, dk);
        const auto r0 = __builtin_amdgcn_permlane32_swap(pack_bf16(x[0], x[1]), pack_bf16(y[0], y[1]), false, false);
        const auto r1 = __builtin_amdgcn_permlane32_swap(pack_bf16(x[2], x[3]), pack_bf16(y[2], y[3]), false, false);
        const u32x4 o = {r0[0], r1[0], r0[1], r1[1]};
        const int col = 32 * db + 8 * (qd + g);
        if (col < dk) *reinterpret_cast<u32x4*>(static_cast<uint16_t*>(base) + row_off + col) = o;
    }
}

// A group of several wavefronts has two tile buffers and one barrier per tile; a group of one wavefront has one buffer and
// none: a wavefront's LDS operations complete in order, so it overwrites its tile behind its own last read of it.
template <int QW>
__device__ inline void tile_barrier() {
    if (QW > 1)
        __syncthreads();
    else
        __builtin_amdgcn_wave_barrier();
}

// How many tokens of the other side a block of rows walks at most: what its chain of tiles is as long as.
inline int chain_tokens(const AttnArgs& a) { return a.window > 0 && a.window + 64 < a.T ? a.window + 64 : a.T; }
// Whether all blocks of a launch have about the same chain. Under a full causal mask they do not: the longest are twice the
// mean and decide when an unsplit launch ends.
inline bool even_chains(const AttnArgs& a) { return !a.causal || chain_tokens(a) < a.T; }
// Whether a dK/dV launch deals the queries past the band of the sink keys' block to workgroups of their own (sink_tail): the
// block's chain through all of them, against the rest of the launch, two workgroups to a CU with a band of queries and about
// three tiles of overhead each. (fp32, head_dim 64, T 2476, window 64, 4 sinks, 4 heads: 86 us with that chain.)
// (bf16, head_dim 32, T 4213, window 1224, 16 sinks, 8 heads, blocks of 128 rows: 355 us with that chain, 146 with the tail dealt out.)
// Where the heads of a group are dealt out a piece still walks all of them, the block its share: no use if that is no shorter (us, with
// pieces | without: bf16, head_dim 128, T 615, 7 heads on one, window 25 64 | 24; T 517 x 2, window 68 47 | 26; fp32, head_dim 64, T 636,
// 28 heads on 4, window 21 130 | 37; T 527 x 3, 7 on one 99 | 33).
inline bool split_tail_pays(const AttnArgs& a, int head_split, int block_rows) {
    const SinkTail t = sink_tail(a.T, a.window, a.sinks);
    const int64_t blocks = static_cast<int64_t>((a.T + block_rows - 1) / block_rows) * a.Hkv * a.B * head_split;
    const int64_t left = a.T - t.q0, rep = quotient(a.Hq, a.Hkv), share = (rep + head_split - 1) / head_split;
    return a.tail && t.nch > 0 && left > (blocks + 511) / 512 * (a.window + 128) &&
           (share == rep || share * left > rep * (left < TAIL_CHUNK ? left : TAIL_CHUNK));
}
inline int tail_blocks(const AttnArgs& a) { return a.tail ? sink_tail(a.T, a.window, a.sinks).nch : 0; }

// A backward whose dK/dV and dQ blocks of 32 rows go into one launch (no gradient where an input is, AttnArgs::in_place: each kind of block
// reads what the other's would overwrite): the arguments of its dK/dV part, and the two kinds' ids. Heads
// of a group are dealt out where the workspace holds their partial sums.
struct OneLaunch {
    AttnArgs a;
    int dkdv_ids, dq_ids;
    explicit OneLaunch(const AttnArgs& args) : a(args) {
        if (!a.part) a.head_split = 1;
        if (!split_tail_pays(a, a.head_split, 32)) a.tail = nullptr;
        const int nblk = (a.T + 31) / 32, units = a.Hkv * a.B;
        dkdv_ids = xcd_grid(nblk + tail_blocks(a), a.head_split, units);
        dq_ids = xcd_grid(nblk, a.Hq / a.Hkv, units);
    }
    // partial sums, as after a dK/dV launch
    int finish(hipStream_t st) const { return a.head_split > 1 ? launch_gqa_reduce(a, st) : a.tail ? launch_sink_tail_reduce(a, st) : PK_OK; }
};

// The same for blocks of more rows, which read delta: blocks of `rows` keys and blocks of as many queries by rank, the longest of either
// first. A rank of a (batch, KV head) unit is a block of keys for each share of the group's heads, then one of queries for each head.
struct JoinedBlocks {
    int ranks, each;
    __host__ __device__ JoinedBlocks(const AttnArgs& a, int rows) : ranks((a.T + rows - 1) / rows), each(a.head_split + quotient(a.Hq, a.Hkv)) {}
    __host__ int grid(const AttnArgs& a) const { return xcd_grid(ranks, each, a.Hkv * a.B); }
    // r: the share of the heads whose dK, dV (r < a.head_split), or the head (the others) whose dQ this workgroup forms
    __device__ bool map(const AttnArgs& a, int& rank, int& r, int& kvu) const {
        return a.causal && ranks > 1 ? xcd_map_block_major(ranks, each, a.Hkv * a.B, rank, r, kvu) : xcd_map(ranks, each, a.Hkv * a.B, rank, r, kvu);
    }
};

// The tiles of BN keys that queries [q0, q0 + BM) can see, as a list: sink tiles [0, ns), then [lo, hi].
struct KeyTiles {
    int ns, lo, n;
    __device__ KeyTiles(const AttnArgs& a, int q0, int BM, int BN) {
        const int qmax = min(q0 + BM, a.T) - 1;
        const int hi = (a.causal ? qmax : a.T - 1) / BN;
        lo = a.window > 0 ? max(0, q0 + 1 - a.window) / BN : 0;
        ns = a.window > 0 ? min((a.sinks + BN - 1) / BN, lo) : 0;
        n = ns + hi - lo + 1;
    }
    __device__ int tile(int i) const { return i < ns ? i : lo + i - ns; }
};

// What of a tile a wavefront's 32 rows see, as comparisons with four numbers formed once: written out for every tile the tests were
// half the instructions of a loop at 64 columns.
//
// Its 32 queries from qlo on against the 32 keys from k0 on: is any pair visible, are all?
struct KeyRange {
    int end, band, full_end, full_band, sinks;
    __device__ KeyRange(const AttnArgs& a, int qlo) {
        end = qlo >= a.T ? -1 : a.causal ? min(a.T - 1, qlo + 31) : a.T - 1;
        band = a.window > 0 ? qlo - 30 - a.window : 0;
        full_end = a.causal ? min(a.T - 32, qlo - 31) : a.T - 32;
        full_band = a.window > 0 ? qlo + 32 - a.window : 0;
        sinks = a.window > 0 ? a.sinks : 0;
    }
    __device__ bool live(int k0) const { return k0 <= end && (k0 >= band || k0 < sinks); }
    __device__ bool full(int k0) const { return k0 <= full_end && (k0 >= full_band || k0 + 31 < sinks); }
};
// Its 32 keys from k0 on against the 32 queries from qlo on.
struct QueryRange {
    int lo, end, full_lo, full_end;
    __device__ QueryRange(const AttnArgs& a, int k0) {
        const bool band = a.window > 0;
        lo = a.causal ? k0 - 31 : 0;
        end = k0 >= a.T ? -1 : band && k0 >= a.sinks ? min(a.T - 1, k0 + 30 + a.window) : a.T - 1;
        full_lo = a.causal ? k0 + 31 : 0;
        full_end = k0 + 31 >= a.T ? -1 : band && k0 + 31 >= a.sinks ? min(a.T - 32, k0 + a.window - 32) : a.T - 32;
    }
    __device__ bool live(int qlo) const { return qlo >= lo && qlo <= end; }
    __device__ bool full(int qlo) const { return qlo >= full_lo && qlo <= full_end; }
};

__device__ inline bool map_query_block(const AttnArgs& a, int nqb, int& b, int& h, int& hk, int& qblk, int id = static_cast<int>(blockIdx.x)) {
    const int rep = quotient(a.Hq, a.Hkv);
    int blk, rr, kvu;
    // causal blocks without a band: the heaviest blocks of every unit first
    if (a.causal && a.window == 0 ? !xcd_map_block_major(nqb, rep, a.Hkv * a.B, blk, rr, kvu, id)
                                  : !xcd_map(nqb, rep, a.Hkv * a.B, blk, rr, kvu, id))
        return false;
    b = quotient(kvu, a.Hkv), hk = kvu - b * a.Hkv, h = hk * rep + rr;
    qblk = nqb - 1 - blk;
    return true;
}

}  // namespace
}  // namespace pk
