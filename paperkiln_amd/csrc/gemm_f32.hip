// The fp32 matrix product on the matrix cores (v_mfma_f32_16x16x4_f32): C = op(A) op(B) (+ C or an addend), row-major, up
// to eight products in one launch.
//
// The fp32 matrix rate is a sixteenth of the bf16 one: a wavefront's 32 x 32 outputs need 8 bytes a cycle, which L1 and L2
// deliver without LDS. Fragments are therefore loaded from global memory straight into the layout the instruction reads,
// two chunks of the contraction ahead of the multiplications, and there is no barrier in the loop. What bounds a small
// product is latency, and that a projection of a few hundred tokens has 16 to 200 blocks of 32 x 32 for 1024 SIMDs: the
// wavefronts of a workgroup split the contraction and add their accumulators through LDS at the end, in a fixed order.
//
// Against the library, which serves the larger products (GPU time, 512 tokens of width 128): level for the fused
// q/k/v projection, 4.0 us and 6.0 for the down projection; but a launch here costs the host 3 us, not 10 to 25, sums
// an addend on the way out, and takes all the weight gradients of a block together. 2048 tokens of width 512 against
// 1536 columns: 45 us and 28.
#include "mfma_common.h"
#include "tensor.h"

#include <algorithm>

namespace pk {
namespace {

struct Job {
    const float* a;
    const float* b;
    float* c;
    const float* addend;
    float* gu;  // the gated forms' [M, 2 N] matrix [gate | up]
    int lda, ldb, ldc, M, N, K;
};
// What becomes of a tile. GATE: B is [gate | up], N columns each, and a tile is the same columns of both: C = silu(gate) up, and both
// of them to gu if it is given. GATE_GRAD: the product is C's gradient d for the gate and up in gu: C is [M, 2 N] and gets theirs.
// TURN: C is a [q | k | v] projection whose q and k turn by their positions (a lane's partner of a pair is its neighbour).
enum class End { PLAIN, GATE, GATE_GRAD, TURN };
// One product's numbers are found at one place, several products' only once the workgroup knows whose tile it has: a second
// round trip to the arguments, 0.4 to 0.8 us of the 3.5 to 8 that a small product takes.
template <int MAX>
struct Jobs {
    int count;
    int first[MAX + 1];  // job j's tiles are first[j] .. first[j + 1] - 1
    Job job[MAX];
};

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));  // a row may start at any element

// One chunk of KC steps of the contraction for NBLK blocks of 16 rows (of A) or columns (of B). The instruction takes four
// steps, one for each 16 lanes. Which four does not matter as long as A and B agree: lanes 16 g .. 16 g + 15 take steps
// 4 g .. 4 g + 3 of every 16, so that a row of an operand whose steps are adjacent is read 64 bytes at a time, 16 bytes a
// lane. (With the 32 x 32 instruction, whose two steps leave a lane's 16 bytes alone in their line, the loads kept the
// CU's address unit busy for twice as long as the multiplications took.)
// ROWS: element (k, i) is p[k ld + i], otherwise p[i ld + k]. off: the lane's byte offset of step 4 g of a chunk at step 0;
// k0: the chunk's first step. Everything that changes from load to load is in scalar registers.
template <bool ROWS, int NBLK, int KC>
__device__ inline void load_chunk(__amdgpu_buffer_rsrc_t p, int ld, const int (&off)[NBLK], int k0, float (&f)[NBLK][KC / 4]) {
#pragma unroll
    for (int s = 0; s < KC / 4; s += 4)
#pragma unroll
        for (int b = 0; b < NBLK; ++b) {
            if (ROWS) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    f[b][s + e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(p, off[b], (k0 + 4 * s + e) * ld * 4, 0));
            } else {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(p, off[b] + 16 * s, k0 * 4, 0);
#pragma unroll
                for (int e = 0; e < 4; ++e) f[b][s + e] = __uint_as_float(v[e]);
            }
        }
}
// The same where the contraction is shorter than a chunk: zeros past its end.
template <bool ROWS, int NBLK, int KC>
__device__ inline void load_short(const float* p, int64_t ld, const int (&idx)[NBLK], int k0, int K, float (&f)[NBLK][KC / 4]) {
#pragma unroll
    for (int b = 0; b < NBLK; ++b)
#pragma unroll
        for (int s = 0; s < KC / 4; ++s) {
            const int at = k0 + 4 * (s & ~3) + (s & 3), k = min(at, K - 1);
            const float v = ROWS ? p[k * ld + idx[b]] : p[idx[b] * ld + k];
            f[b][s] = at < K ? v : 0.0f;
        }
}

__host__ __device__ inline int64_t extent(int64_t rows, int64_t cols, int64_t ld) { return ((rows - 1) * ld + cols) * 4; }
__device__ inline int bytes_of(int rows, int cols, int64_t ld) { return static_cast<int>(extent(rows, cols, ld)); }

// A workgroup's tile is MB x NB blocks of 16 x 16; its KW wavefronts split the contraction chunk by chunk. SUMS 2: a wavefront has two
// sums, of every other step of a chunk, so that four wavefronts' chains of additions, with which a sum's error grows, are as short
// as eight wavefronts' (at the sizes named below no slower: 4.69 us | 4.68, 3.78 | 3.80, 5.72 | 5.75, 5.87 | 5.88 with one | two).
//
// NORM: A's rows count normalised (Norm in tensor.h). A wavefront adds up the squares of what it loads of them and multiplies it by the
// norm's weight; the rows' sums meet where the tiles' do, and every workgroup of a row of tiles writes its share of the normalised rows'
// columns, of a short contraction out of the registers they still lie in. A launch of its own was 2.8 us and the wait for it, of a chain of 44
// launches in a small model's step (512 x 384 x 128: 2.8 and 5.0 us | 5.6; gate and up, 512 x 688 x 128: 2.8 and 5.4 | 6.2, as 32 x 32: what
// every workgroup adds is a microsecond, and of 16 x 32 there are two rounds, 7.2). The step: 3.75 -> 3.67 ms for 16.
template <bool TA, bool TB, int MB, int NB, int KW, int SUMS, int MAX, End END, bool NORM>
__global__ __launch_bounds__(64 * KW, 2) void gemm_f32_k(const Jobs<MAX> jobs, const int tiles, const float beta, const Turn turn, const Norm norm) {
    static_assert(!NORM || (!TA && MAX == 1 && MB <= 2 && NB <= 2), "rows of one A, small tiles");
    constexpr int KC = MB * NB <= 4 ? 32 : 16, BUFS = MB * NB <= (NORM ? 2 : 4) ? 3 : 2, TM = 16 * MB;
    constexpr int HALF = END == End::GATE ? NB / 2 : NB, TN = 16 * HALF;  // blocks of columns of C
    constexpr int ITEMS = (MB * HALF + KW - 1) / KW;                      // blocks that a wavefront adds up and stores
    constexpr bool EARLY = END != End::GATE && ITEMS == 1;
    // every XCD takes a contiguous range of the tiles: neighbours share operand rows or columns in its L2
    const int t = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (t >= tiles) return;
    int j = 0;
    if constexpr (MAX > 1)
        while (t >= jobs.first[j + 1]) ++j;
    const int M = jobs.job[j].M, N = jobs.job[j].N, K = jobs.job[j].K;
    const int tn = (N + TN - 1) / TN, at_row = quotient(t - jobs.first[j], tn), m0 = at_row * TM, n0 = (t - jobs.first[j] - at_row * tn) * TN;
    const int lane = threadIdx.x & 63, kw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, grp = lane >> 4;
    const float* const a = jobs.job[j].a;
    const float* const b = jobs.job[j].b;
    const int64_t lda = jobs.job[j].lda, ldb = jobs.job[j].ldb;
    int row[MB], col[NB];  // rows and columns past the edge read the last one; they are not stored
#pragma unroll
    for (int i = 0; i < MB; ++i) row[i] = min(m0 + i * 16 + l16, M - 1);
#pragma unroll
    for (int i = 0; i < NB; ++i) col[i] = min(n0 + i % HALF * 16 + l16, N - 1) + (i >= HALF ? N : 0);

    f32x4 acc[SUMS][MB][NB];
#pragma unroll
    for (int i = 0; i < SUMS; ++i)
#pragma unroll
        for (int x = 0; x < MB; ++x)
#pragma unroll
            for (int y = 0; y < NB; ++y) acc[i][x][y] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    const auto ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a), 0, bytes_of(TA ? K : M, TA ? M : K, lda), 0x00020000);
    const auto rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(b), 0, bytes_of(TB ? N : K, TB ? K : END == End::GATE ? 2 * N : N, ldb), 0x00020000);
    int oa[MB], ob[NB];
#pragma unroll
    for (int i = 0; i < MB; ++i) oa[i] = static_cast<int>(TA ? 4 * grp * lda + row[i] : row[i] * lda + 4 * grp) * 4;
#pragma unroll
    for (int i = 0; i < NB; ++i) ob[i] = static_cast<int>(TB ? col[i] * ldb + 4 * grp : 4 * grp * ldb + col[i]) * 4;
    float fa[BUFS][MB][KC / 4], fb[BUFS][NB][KC / 4];
    float fw[NORM ? BUFS : 1][1][KC / 4], squares[MB];
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(NORM ? norm.w : a), 0, K * 4, 0x00020000);
    const int ow[1] = {16 * grp};
#pragma unroll
    for (int x = 0; x < MB; ++x) squares[x] = 0.0f;
    const int chunks = (K + KC - 1) / KC;
    auto load = [&](int chunk, int buf) {
        const int over = max((chunk + 1) * KC - K, 0), k0 = chunk * KC - over;
        if (over == 0) {
            load_chunk<TA, MB, KC>(ra, jobs.job[j].lda, oa, k0, fa[buf]);
            load_chunk<!TB, NB, KC>(rb, jobs.job[j].ldb, ob, k0, fb[buf]);
            if constexpr (NORM) load_chunk<false, 1, KC>(rw, 0, ow, k0, fw[buf]);
        } else if (K >= KC) {  // the last chunk, moved back to end where the contraction does: its first steps are done already
            load_chunk<TA, MB, KC>(ra, jobs.job[j].lda, oa, k0, fa[buf]);
            load_chunk<!TB, NB, KC>(rb, jobs.job[j].ldb, ob, k0, fb[buf]);
            if constexpr (NORM) load_chunk<false, 1, KC>(rw, 0, ow, k0, fw[buf]);
#pragma unroll
            for (int s = 0; s < KC / 4; ++s) {
                const bool done = 4 * grp + 4 * (s & ~3) + (s & 3) < over;
#pragma unroll
                for (int x = 0; x < MB; ++x) fa[buf][x][s] = done ? 0.0f : fa[buf][x][s];
#pragma unroll
                for (int y = 0; y < NB; ++y) fb[buf][y][s] = done ? 0.0f : fb[buf][y][s];
            }
        } else {
            load_short<TA, MB, KC>(a, lda, row, 4 * grp, K, fa[buf]);
            load_short<!TB, NB, KC>(b, ldb, col, 4 * grp, K, fb[buf]);
            if constexpr (NORM) load_chunk<false, 1, KC>(rw, 0, ow, 0, fw[buf]);  // zeros past the end
        }
    };
    auto multiply = [&](int buf) {
        if constexpr (NORM)
#pragma unroll
            for (int s = 0; s < KC / 4; ++s)
#pragma unroll
                for (int x = 0; x < MB; ++x) {
                    squares[x] = fmaf(fa[buf][x][s], fa[buf][x][s], squares[x]);
                    fa[buf][x][s] *= fw[buf][0][s];
                }
#pragma unroll
        for (int s = 0; s < KC / 4; ++s)
#pragma unroll
            for (int x = 0; x < MB; ++x)
#pragma unroll
                for (int y = 0; y < NB; ++y)
                    acc[s % SUMS][x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[buf][x][s], fb[buf][y][s], acc[s % SUMS][x][y], 0, 0, 0);
    };
    const int mine = kw < chunks ? (chunks - kw + KW - 1) / KW : 0;  // chunks kw, kw + KW, ... are this wavefront's
#pragma unroll
    for (int u = 0; u < BUFS; ++u)
        if (u < mine) load(kw + u * KW, u);
    // what the tile meets on its way out is asked for behind the first chunks, not when the contraction is over: a trip to memory of the 4 to 6 us
    // of a small product (with a residual, us: 512 x 128 x 128 and 344 4.5 -> 4.0, 1024 x 256 x 256 and 688 6.9 -> 6.0; gate and up, 512 x 344 x 128 6.3 ->
    // 5.2). Tiles of several blocks to a wavefront ask block by block, but for whole blocks (gate and up, 1024 x 688 x 256 17.3 -> 14.6; 392 tiles of weight
    // gradients 27.0 -> 25.3): held over the loop those blocks cost it registers (28.0).
    const float* const add = jobs.job[j].addend ? jobs.job[j].addend : beta != 0.0f ? jobs.job[j].c : nullptr;
    const int64_t ldc = jobs.job[j].ldc;
    constexpr bool MEETS = END == End::GATE_GRAD || END == End::TURN;  // two numbers an element
    f32x4 met[EARLY ? ITEMS : 1][MEETS ? 2 : 1];
    const int base = END == End::TURN ? m0 - quotient(m0, turn.seq_len) * turn.seq_len : 0;
    auto meet = [&](int x, int y, f32x4 (&v)[MEETS ? 2 : 1]) {
        const int n = min(n0 + y * 16 + l16, N - 1);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (END == End::TURN) {
                const int pair = max(turned_pair(turn, n), 0), at = turned_position<TM>(turn, base, x * 16 + 4 * grp + r);
                const float2 cs = *reinterpret_cast<const float2*>(turn.table + (static_cast<int64_t>(at) * (turn.head_dim / 2) + pair) * 2);
                v[0][r] = cs.x, v[1][r] = cs.y;
                continue;
            }
            const int64_t o = min(m0 + x * 16 + 4 * grp + r, M - 1) * ldc + n;
            if constexpr (END == End::GATE_GRAD)
                v[0][r] = jobs.job[j].gu[o], v[1][r] = jobs.job[j].gu[o + N];
            else
                v[0][r] = add[o];
        }
    };
    if constexpr (EARLY)
        if (MEETS || add)
#pragma unroll
            for (int q = 0; q < ITEMS; ++q) {
                const int g = min(q * KW + kw, MB * HALF - 1);
                meet(g / HALF, g % HALF, met[q]);
            }
    __builtin_amdgcn_sched_barrier(0);
    int i = 0;
    for (; i + BUFS <= mine; i += BUFS) {
#pragma unroll
        for (int u = 0; u < BUFS; ++u) {
            multiply(u);
            if (i + u + BUFS < mine) load(kw + (i + u + BUFS) * KW, u);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int u = 0; u < BUFS - 1; ++u)
        if (i + u < mine) multiply(u);

    float* const out = jobs.job[j].c;
    auto store = [&](int x, int y, f32x4 v, const f32x4 (&e)[MEETS ? 2 : 1]) {
        const int n = n0 + y * 16 + l16;
        if constexpr (END == End::TURN) {
            const bool turns = turned_pair(turn, n) >= 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float w = lane_moved<0xB1>(v[r]), t = l16 & 1 ? w * e[1][r] + v[r] * e[0][r] : v[r] * e[0][r] - w * e[1][r];
                v[r] = turns ? t : v[r];
            }
        }
        if (n >= N) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m0 + x * 16 + 4 * grp + r;
            if (m < M) {
                const int64_t o = m * ldc + n;
                if constexpr (END == End::GATE_GRAD)
                    gated_grad(e[0][r], e[1][r], v[r], out[o], out[o + N]);
                else
                    out[o] = END != End::TURN && add ? e[0][r] + v[r] : v[r];
            }
        }
    };
    auto store_gated = [&](int x, int y, f32x4 gate, f32x4 up) {
        float* const gu = jobs.job[j].gu;
        const int n = n0 + y * 16 + l16;
        if (n >= N) return;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m0 + x * 16 + 4 * grp + r;
            if (m < M) {
                out[m * ldc + n] = gated(gate[r], up[r]);
                if (gu) {
                    gu[m * ldc * 2 + n] = gate[r];
                    gu[m * ldc * 2 + N + n] = up[r];
                }
            }
        }
    };
    __shared__ f32x4 part[KW][MB * NB][64];
#pragma unroll
    for (int x = 0; x < MB; ++x)
#pragma unroll
        for (int y = 0; y < NB; ++y) part[kw][x * NB + y][lane] = SUMS > 1 ? acc[0][x][y] + acc[SUMS - 1][x][y] : acc[0][x][y];
    __shared__ float of_row[NORM ? KW : 1][NORM ? TM : 1];
    if constexpr (NORM)
#pragma unroll
        for (int x = 0; x < MB; ++x) {  // a row's other steps are 16, 32 and 48 lanes on
            float q = squares[x];
            q += __shfl_xor(q, 16);
            q += __shfl_xor(q, 32);
            if (grp == 0) of_row[kw][x * 16 + l16] = q;
        }
    __syncthreads();
    float inverse[MB];  // 1 / rms of row l16 of a block
    if constexpr (NORM) {
#pragma unroll
        for (int x = 0; x < MB; ++x) {
            float q = of_row[0][x * 16 + l16];
#pragma unroll
            for (int k = 1; k < KW; ++k) q += of_row[k][x * 16 + l16];
            inverse[x] = 1.0f / sqrtf(q / static_cast<float>(K) + norm.eps);
        }
        if (norm.y) {  // column tile c writes chunks c, c + tn, ...: of a short contraction out of the registers they still lie in
            const int at_col = t - jobs.first[j] - at_row * tn;
            float* const y = static_cast<float*>(norm.y);
#pragma unroll
            for (int x = 0; x < MB; ++x) {
                const int m = m0 + x * 16 + l16;
                if (at_col == 0 && kw == 0 && grp == 0 && m < M) norm.rinv[m] = inverse[x];
            }
            if (chunks <= BUFS * KW && K % KC == 0) {
#pragma unroll
                for (int u = 0; u < BUFS; ++u) {
                    const int c = kw + u * KW;
                    if (c >= chunks || c - quotient(c, tn) * tn != at_col) continue;
#pragma unroll
                    for (int x = 0; x < MB; ++x) {
                        const int m = m0 + x * 16 + l16;
#pragma unroll
                        for (int s = 0; s < KC / 4; s += 4) {
                            const f32x4 v = {fa[u][x][s], fa[u][x][s + 1], fa[u][x][s + 2], fa[u][x][s + 3]};
                            if (m < M) *reinterpret_cast<f32x4*>(y + static_cast<int64_t>(m) * K + c * KC + 4 * grp + 4 * s) = v * inverse[x];
                        }
                    }
                }
            } else {
                for (int c = at_col; c < chunks; c += tn)
#pragma unroll
                    for (int x = 0; x < MB; ++x) {
                        const int m = m0 + x * 16 + l16, k = c * KC + 4 * (kw * 4 + grp);
                        if (m < M && 4 * (kw * 4 + grp) < KC && k < K) {
                            const f32x4 v = *reinterpret_cast<const f32x4*>(a + m * lda + k), w = *reinterpret_cast<const f32x4*>(norm.w + k);
                            *reinterpret_cast<f32x4*>(y + static_cast<int64_t>(m) * K + k) = v * w * inverse[x];
                        }
                    }
            }
        }
    }
#pragma unroll
    for (int g0 = 0; g0 < MB * HALF; g0 += KW) {
        const int g = g0 + kw;
        if (g < MB * HALF) {
            const int at = g / HALF * NB + g % HALF;
            f32x4 s = part[0][at][lane];
#pragma unroll
            for (int k = 1; k < KW; ++k) s += part[k][at][lane];
            f32x4 by;
            if constexpr (NORM) {
#pragma unroll
                for (int r = 0; r < 4; ++r) by[r] = __shfl(g < HALF ? inverse[0] : inverse[MB - 1], 4 * grp + r);
                s *= by;
            }
            if constexpr (END == End::GATE) {
                f32x4 up = part[0][at + HALF][lane];
#pragma unroll
                for (int k = 1; k < KW; ++k) up += part[k][at + HALF][lane];
                if constexpr (NORM) up *= by;
                store_gated(g / HALF, g % HALF, s, up);
            } else {
                if constexpr (!EARLY)
                    if (MEETS || add) meet(g / HALF, g % HALF, met[0]);
                store(g / HALF, g % HALF, s, met[EARLY ? g0 / KW : 0]);
            }
        }
    }
}

template <bool TA, bool TB, int MB, int NB, int KW, End END, int SUMS = 1, int MAX>
void launch(Jobs<MAX>& jobs, float beta, hipStream_t st, const Turn& turn, const Norm* norm) {
    constexpr int TM = 16 * MB, TN = 16 * (END == End::GATE ? NB / 2 : NB);
    int tiles = 0;
    for (int j = 0; j < jobs.count; ++j) {
        jobs.first[j] = tiles;
        tiles += ((jobs.job[j].M + TM - 1) / TM) * ((jobs.job[j].N + TN - 1) / TN);
    }
    for (int j = jobs.count; j <= MAX; ++j) jobs.first[j] = tiles;
    const dim3 grid((tiles + 7) / 8 * 8), block(64 * KW);
    if constexpr (MAX == 1 && MB <= 2 && NB <= 2 && (END == End::GATE || END == End::TURN))
        if (norm) {
            hipLaunchKernelGGL((gemm_f32_k<TA, TB, MB, NB, KW, SUMS, MAX, END, true>), grid, block, 0, st, jobs, tiles, beta, turn, *norm);
            hip_check(hipGetLastError(), "gemm_f32");
            return;
        }
    hipLaunchKernelGGL((gemm_f32_k<TA, TB, MB, NB, KW, SUMS, MAX, END, false>), grid, block, 0, st, jobs, tiles, beta, turn, Norm{});
    hip_check(hipGetLastError(), "gemm_f32");
}

// Which tile, by the number of 32 x 32 ones. A small tile keeps more CUs busy, a large one reads its operands less often. Measured
// on projections, heads and weight gradients of 64 to 8192 tokens:
//   More than 640 (2.5 to a CU): 64 x 64 (2048 x 1000 x 128: 10.4 us against 15.7), except for weight gradients, whose long
//   contraction the small ones walk with more wavefronts (512 x 1536 x 8192: 117 us against 152). Theirs are 32 x 64, which cross
//   the L2 three times for every four of 32 x 32, where they come to rounds that are full enough: above 768 (us, 32 x 32 | 32 x 64: 2048 x
//   1536 x 1224 90 | 70, 896 x 896 x 1144 29 | 24, 1536 x 1152 x 1776 73 | 69; 512 x 1376 x 8192, 688 tiles, 134 | 150), and
//   where they make one a CU, with eight wavefronts (768 x 576 x 6232 65 | 58, 640 x 640 x 896 13.2 | 11.7, 700 x 700 x 3000 37 | 29).
//   Up to 64: 16 x 16, up to 128: 16 x 32, which makes a tile for each CU, in two sums a wavefront. A wavefront's loads and products for a chunk are a half or
//   less (us, 32 x 32 with eight | 16 x 32 | 16 x 16 wavefronts: 512 x 128 x 688, B transposed 7.9 | 6.2 | 5.0; 512 x 128 x 344 5.4 |
//   4.8 | 4.0; 512 x 256 x 688 7.8 | 6.0 | 6.6; 1024 x 128 x 688, B transposed 7.8 | 6.3 | 6.5).
//   In between 32 x 32; eight wavefronts split the contraction where it is long and there is a tile or less to a CU. Short
//   contractions of more tiles than that are over sooner as 16 x 32, for which the last round is half as long (1000 x 576 x
//   192: 7.7 us against 9.4, 256 x 1376 x 256: 5.8 against 6.8; with B transposed, whose rows those tiles read twice, they are not).
template <bool TA, bool TB, End END, int MAX>
void launch_by_size(Jobs<MAX>& jobs, float beta, hipStream_t st, const Turn& turn = {}, const Norm* norm = nullptr) {
    int64_t tiles = 0;
    int longest = 0;
    for (int j = 0; j < jobs.count; ++j) {
        tiles += static_cast<int64_t>((jobs.job[j].M + 31) / 32) * ((jobs.job[j].N * (END == End::GATE ? 2 : 1) + 31) / 32);
        longest = std::max(longest, jobs.job[j].K);
    }
    if (tiles > 640 && (!TA || longest < 256))
        launch<TA, TB, 4, 4, 4, END>(jobs, beta, st, turn, norm);
    else if (TA && longest >= 256 && tiles > 768)
        launch<TA, TB, 2, 4, 4, END>(jobs, beta, st, turn, norm);
    else if (TA && longest >= 256 && tiles > 320 && tiles <= 512)
        launch<TA, TB, 2, 4, 8, END>(jobs, beta, st, turn, norm);
    else if (tiles <= 64 && END != End::GATE)
        launch<TA, TB, 1, END == End::GATE ? 2 : 1, 4, END, 2>(jobs, beta, st, turn, norm);
    else if (tiles <= 128)
        launch<TA, TB, 1, 2, 4, END, 2>(jobs, beta, st, turn, norm);
    else if (!TA && !TB && !norm && tiles > 256 && longest <= 256)
        launch<TA, TB, 1, 2, 4, END>(jobs, beta, st, turn, norm);
    else if (tiles <= 256 && longest >= 256)
        launch<TA, TB, 2, 2, 8, END>(jobs, beta, st, turn, norm);
    else
        launch<TA, TB, 2, 2, 4, END>(jobs, beta, st, turn, norm);
}

template <int MAX>
bool multiply(const F32Product* ps, int count, bool tA, bool tB, float beta, hipStream_t st, End end = End::PLAIN, float* gu = nullptr,
              const Turn& turn = {}, const Norm* norm = nullptr) {
    Jobs<MAX> jobs{};
    jobs.count = count;
    for (int j = 0; j < count; ++j) {
        const F32Product& p = ps[j];
        const int64_t limit = int64_t{1} << 30;
        if (p.M <= 0 || p.N <= 0 || p.K <= 0 || p.M > limit || p.N > limit || p.K > limit || p.lda > limit || p.ldb > limit ||
            p.ldc > limit)
            return false;
        if (extent(tA ? p.K : p.M, tA ? p.M : p.K, p.lda) >= int64_t{1} << 31 || extent(tB ? p.N : p.K, tB ? p.K : end == End::GATE ? 2 * p.N : p.N, p.ldb) >= int64_t{1} << 31)
            return false;
        jobs.job[j].a = p.a;
        jobs.job[j].b = p.b;
        jobs.job[j].c = p.c;
        jobs.job[j].addend = p.addend;
        jobs.job[j].gu = gu;
        jobs.job[j].lda = static_cast<int>(p.lda);
        jobs.job[j].ldb = static_cast<int>(p.ldb);
        jobs.job[j].ldc = static_cast<int>(p.ldc);
        jobs.job[j].M = static_cast<int>(p.M);
        jobs.job[j].N = static_cast<int>(p.N);
        jobs.job[j].K = static_cast<int>(p.K);
    }
    if constexpr (MAX == 1) {
        if (end == End::GATE) launch_by_size<false, false, End::GATE>(jobs, beta, st, turn, norm);
        if (end == End::GATE_GRAD) launch_by_size<false, true, End::GATE_GRAD>(jobs, beta, st);
        if (end == End::TURN) launch_by_size<false, false, End::TURN>(jobs, beta, st, turn, norm);
        if (end != End::PLAIN) return true;
    }
    if (tA)
        launch_by_size<true, false, End::PLAIN>(jobs, beta, st);
    else if (tB)
        launch_by_size<false, true, End::PLAIN>(jobs, beta, st);
    else
        launch_by_size<false, false, End::PLAIN>(jobs, beta, st);
    return true;
}

// The normalised rows are written 16 bytes at a time. Not in the 64 x 64 tiles of more than 640 of 32 x 32, which have no registers for it.
bool norm_fits(const float* x, int64_t M, int64_t columns, int64_t K, const Norm* norm) {
    const auto at16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    return !norm || (((M + 31) / 32) * ((columns + 31) / 32) <= 640 && K % 4 == 0 && at16(x) && at16(norm->w) && at16(norm->y));
}

}  // namespace

bool gemm_f32(const F32Product* ps, int count, bool tA, bool tB, float beta, hipStream_t st) {
    if (count < 1 || count > 8 || (tA && tB) || (beta != 0.0f && beta != 1.0f)) return false;
    return count == 1 ? multiply<1>(ps, count, tA, tB, beta, st) : multiply<8>(ps, count, tA, tB, beta, st);
}
bool gemm_f32_gated(const float* x, const float* w, float* gu, float* h, int64_t M, int64_t N, int64_t K, hipStream_t st, const Norm* norm) {
    const F32Product p{x, K, w, 2 * N, h, N, nullptr, M, N, K};
    return norm_fits(x, M, 2 * N, K, norm) && multiply<1>(&p, 1, false, false, 0.0f, st, End::GATE, gu, {}, norm);
}
bool gemm_f32_gated_grad(const float* dy, const float* w, const float* gu, float* dgu, int64_t M, int64_t N, int64_t K, hipStream_t st) {
    const F32Product p{dy, K, w, K, dgu, 2 * N, nullptr, M, N, K};
    return multiply<1>(&p, 1, false, true, 0.0f, st, End::GATE_GRAD, const_cast<float*>(gu));
}
bool gemm_f32_turned(const float* x, const float* w, float* y, int64_t M, int64_t K, const Turn& turn, hipStream_t st, const Norm* norm) {
    const int64_t N = 3 * static_cast<int64_t>(turn.d);
    const F32Product p{x, K, w, N, y, N, nullptr, M, N, K};
    return turn.d % 2 == 0 && turn.head_dim % 2 == 0 && norm_fits(x, M, N, K, norm) && multiply<1>(&p, 1, false, false, 0.0f, st, End::TURN, nullptr, turn, norm);
}

}  // namespace pk
