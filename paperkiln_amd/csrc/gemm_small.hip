// The bf16 matrix product where it is small: C = op(A) op(B) (+ C or an addend), row-major, up to eight products in one
// launch, bf16 operands, fp32 accumulation.
//
// gemm_mfma.hip feeds 128 x 128 tiles through a ring in LDS. A projection of a few hundred tokens is a handful of those,
// over a contraction of a few slices, and takes 5 to 8 us of prologue, pipeline fill and strip-wise store, on a
// fraction of the CUs. Here a workgroup's four or eight wavefronts share a 32 x 32 tile and split its contraction,
// load their fragments from global memory straight into the layout the instruction reads -- everything a short
// contraction needs is in flight at once -- and meet once, in LDS, in a fixed order. What bounds it is that one round
// trip. Operands cross the L2 once per 32 rows, so it is behind as soon as the tiles are many (gemm_small_us).
#include "mfma_common.h"
#include "tensor.h"

#include <algorithm>

namespace pk {
namespace {

struct Job {
    const uint16_t* a;
    const uint16_t* b;
    void* c;
    const void* addend;
    uint16_t* gu;  // as in gemm_f32.hip
    int lda, ldb, ldc, M, N, K;
};
enum class End { PLAIN, GATE, GATE_GRAD, TURN };
// as in gemm_f32.hip: one product's numbers are found without a second round trip to the arguments (512 x 384 x 128 4.2 -> 3.3 us,
// 512 x 128 x 344 4.7 -> 3.6, 2048 x 128 x 128 4.0 -> 3.4)
template <int MAX>
struct Jobs {
    int count;
    int first[MAX + 1];  // job j's tiles are first[j] .. first[j + 1] - 1
    Job job[MAX];
};
constexpr int KC = 32;  // steps of the contraction per chunk: one v_mfma_f32_16x16x32_bf16

__host__ __device__ inline int64_t extent(int64_t rows, int64_t cols, int64_t ld) { return ((rows - 1) * ld + cols) * 2; }

// One chunk for two interleaved blocks of 16 rows (of A) or columns (of B): lane l holds of block b row or column
// 2 (l % 16) + b, steps 8 (l / 16) .. + 7. PAIRS: the steps are rows of the operand, and one dword of a row holds the lane's
// place in both blocks; otherwise the steps are adjacent, 16 bytes a lane, 64 a row. Interleaved rather than side by side, so
// that both kinds of operand fit each other and a lane's two columns of C are one dword of bf16.
template <bool PAIRS>
struct Chunk {
    u32x4 raw[2];  // PAIRS: dwords of steps 0-3, 4-7; otherwise the two blocks' fragments
    __device__ void load(__amdgpu_buffer_rsrc_t p, const int (&off)[2], int k0, int ld) {
        if (PAIRS) {
#pragma unroll
            for (int e = 0; e < 8; ++e) raw[e / 4][e % 4] = __builtin_amdgcn_raw_buffer_load_b32(p, off[0], (k0 + e) * ld * 2, 0);
        } else {
#pragma unroll
            for (int b = 0; b < 2; ++b) raw[b] = __builtin_amdgcn_raw_buffer_load_b128(p, off[b], k0 * 2, 0);
        }
    }
    __device__ void clear_first(int n, int grp) {  // zeros for the first n steps of the chunk (an even number if !PAIRS)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int step = 8 * grp + (PAIRS ? 4 * h + e : 2 * e);
                raw[h][e] = step < n ? 0u : raw[h][e];
            }
    }
    __device__ bf16x8 block(int b) const {
        u32x4 f = raw[b];
        if (PAIRS) {
#pragma unroll
            for (int e = 0; e < 4; ++e)  // steps 2e, 2e + 1 of the low (b = 0) or high halves
                f[e] = __builtin_amdgcn_perm(raw[e / 2][e % 2 * 2 + 1], raw[e / 2][e % 2 * 2], b == 0 ? 0x05040100u : 0x07060302u);
        }
        return *reinterpret_cast<const bf16x8*>(&f);
    }
};

// NORM: A's rows count normalised, as in gemm_f32.hip; the product of a row and the norm's weight is rounded where the normalised row would be.
// (512 x 384 x 128: 3.1 us of its own and 3.6 | 4.4; gate and up, 512 x 688 x 128: 3.1 and 4.1 | 5.1. A step of a bf16 model of 4 layers of
// width 256 with checkpointing, 512 tokens: 9.1 -> 8.5 ms for 12.)
template <bool TA, bool TB, bool CF32, int KW, int MAX, End END, bool NORM>
__global__ __launch_bounds__(64 * KW, 2) void gemm_small_k(const Jobs<MAX> jobs, const int tiles, const int accumulate, const Turn turn, const Norm norm) {
    static_assert(!NORM || (!TA && MAX == 1), "rows of one A");
    constexpr int BUFS = 4, NC = END == End::GATE ? 2 : 1;  // NC: columns of gate and of up, or of one matrix
    // every XCD takes a contiguous range of the tiles: neighbours share operand rows or columns in its L2
    const int t = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
    if (t >= tiles) return;
    int j = 0;
    if constexpr (MAX > 1)
        while (t >= jobs.first[j + 1]) ++j;
    const int M = jobs.job[j].M, N = jobs.job[j].N, K = jobs.job[j].K, lda = jobs.job[j].lda, ldb = jobs.job[j].ldb;
    const int tn = (N + 31) / 32, at_row = quotient(t - jobs.first[j], tn), m0 = at_row * 32, n0 = (t - jobs.first[j] - at_row * tn) * 32;
    const int lane = threadIdx.x & 63, kw = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, grp = lane >> 4;
    const auto ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(jobs.job[j].a), 0,
                                                      static_cast<int>(extent(TA ? K : M, TA ? M : K, lda)), 0x00020000);
    const auto rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(jobs.job[j].b), 0,
                                                      static_cast<int>(extent(TB ? N : K, TB ? K : N * NC, ldb)), 0x00020000);
    int oa[2], ob[2];  // rows and columns past the edge read the last ones; they are not stored
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        oa[b] = TA ? (8 * grp * lda + min(m0 + 2 * l16, M - 2)) * 2 : (min(m0 + 2 * l16 + b, M - 1) * lda + 8 * grp) * 2;
        ob[b] = TB ? (min(n0 + 2 * l16 + b, N - 1) * ldb + 8 * grp) * 2 : (8 * grp * ldb + min(n0 + 2 * l16, N - 2)) * 2;
    }
    f32x4 acc[NC][2][2];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) acc[c][x][y] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    int oc[NC][2];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int b = 0; b < 2; ++b) oc[c][b] = ob[b] + c * N * 2;

    Chunk<TA> fa[BUFS];
    Chunk<!TB> fb[BUFS][NC];
    f32x4 fw[NORM ? BUFS : 1][2];
    float squares[2] = {0.0f, 0.0f};
    const auto rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(norm.w), 0, K * 4, 0x00020000);
    const int chunks = (K + KC - 1) / KC;
    auto load = [&](int chunk, int buf) {
        // the last chunk of a contraction that is no multiple is moved back to end where that does: its first steps are done
        const int over = max((chunk + 1) * KC - K, 0), k0 = chunk * KC - over;
        fa[buf].load(ra, oa, k0, lda);
        if constexpr (NORM)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rw, 32 * grp + 16 * h, k0 * 4, 0);
                fw[buf][h] = *reinterpret_cast<const f32x4*>(&v);
            }
#pragma unroll
        for (int c = 0; c < NC; ++c) fb[buf][c].load(rb, oc[c], k0, ldb);
        if (over > 0) {
            fa[buf].clear_first(over, grp);
#pragma unroll
            for (int c = 0; c < NC; ++c) fb[buf][c].clear_first(over, grp);
        }
    };
    auto multiply = [&](int buf) {
        if constexpr (NORM)
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float lo = __uint_as_float(fa[buf].raw[b][e] << 16), hi = __uint_as_float(fa[buf].raw[b][e] & 0xffff0000u);
                    squares[b] = fmaf(hi, hi, fmaf(lo, lo, squares[b]));
                    fa[buf].raw[b][e] = pack_bf16(lo * fw[buf][e / 2][e % 2 * 2], hi * fw[buf][e / 2][e % 2 * 2 + 1]);
                }
        const bf16x8 a0 = fa[buf].block(0), a1 = fa[buf].block(1);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const bf16x8 b0 = fb[buf][c].block(0), b1 = fb[buf][c].block(1);
            acc[c][0][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b0, acc[c][0][0], 0, 0, 0);
            acc[c][0][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a0, b1, acc[c][0][1], 0, 0, 0);
            acc[c][1][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b0, acc[c][1][0], 0, 0, 0);
            acc[c][1][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1, b1, acc[c][1][1], 0, 0, 0);
        }
    };
    const int mine = kw < chunks ? (chunks - kw + KW - 1) / KW : 0;  // chunks kw, kw + KW, ... are this wavefront's
#pragma unroll
    for (int u = 0; u < BUFS; ++u)
        if (u < mine) load(kw + u * KW, u);
    // what the tile meets on its way out, asked for behind the first chunks as in gemm_f32.hip
    constexpr int RPW = 8 / KW;  // of the 2 x 4 rows a lane holds, each wavefront adds up this many
    const void* const add = jobs.job[j].addend ? jobs.job[j].addend : accumulate ? jobs.job[j].c : nullptr;
    const int64_t ldc = jobs.job[j].ldc;
    u32x2 met[RPW];
    const int pair = END == End::TURN ? turned_pair(turn, n0 + 2 * l16) : -1;
    if constexpr (END == End::TURN) {
        const int base = m0 - quotient(m0, turn.seq_len) * turn.seq_len;
#pragma unroll
        for (int q = 0; q < RPW; ++q) {
            const int row = kw * RPW + q, at = turned_position<32>(turn, base, 2 * (4 * grp + (row & 3)) + (row >> 2));
            if (pair >= 0) met[q] = *reinterpret_cast<const u32x2*>(turn.table + (static_cast<int64_t>(at) * (turn.head_dim / 2) + pair) * 2);
        }
    }
    if (END == End::GATE_GRAD || (END == End::PLAIN && add))
#pragma unroll
        for (int q = 0; q < RPW; ++q) {
            const int row = kw * RPW + q;
            const int64_t o = min(m0 + 2 * (4 * grp + (row & 3)) + (row >> 2), M - 1) * ldc + min(n0 + 2 * l16, N - 2);
            if (END == End::GATE_GRAD)
                met[q] = u32x2{*reinterpret_cast<const uint32_t*>(jobs.job[j].gu + o), *reinterpret_cast<const uint32_t*>(jobs.job[j].gu + o + N)};
            else if (CF32)
                met[q] = *reinterpret_cast<const u32x2*>(static_cast<const float*>(add) + o);
            else
                met[q] = u32x2{*reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(add) + o), 0};
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

    // lane (l16, grp), register r of block (x, y): row m0 + 2 (4 grp + r) + x, column n0 + 2 l16 + y
    __shared__ f32x4 part[KW][NC][2][2][64];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int y = 0; y < 2; ++y) part[kw][c][x][y][lane] = acc[c][x][y];
    __shared__ float of_row[NORM ? KW : 1][NORM ? 32 : 1];
    if constexpr (NORM)
#pragma unroll
        for (int b = 0; b < 2; ++b) {  // a row's other steps are 16, 32 and 48 lanes on
            float q = squares[b];
            q += __shfl_xor(q, 16);
            q += __shfl_xor(q, 32);
            if (grp == 0) of_row[kw][2 * l16 + b] = q;
        }
    __syncthreads();
    auto inverse = [&](int r) {  // 1 / rms of the tile's row r
        float q = of_row[0][NORM ? r : 0];
#pragma unroll
        for (int k = 1; k < KW; ++k) q += of_row[NORM ? k : 0][NORM ? r : 0];
        return 1.0f / sqrtf(q / static_cast<float>(K) + norm.eps);
    };
    if constexpr (NORM)
        if (norm.y) {
            const int at_col = t - jobs.first[j] - at_row * tn, share = (quotient(K + 3, 4) + tn - 1) / tn * 4, c0 = at_col * share, n = min(share, K - c0);
            const int r = static_cast<int>(threadIdx.x) % 32, m = m0 + r;
            if (m < M && (n > 0 || at_col == 0)) {
                const float by = inverse(r);
                if (at_col == 0 && static_cast<int>(threadIdx.x) < 32) norm.rinv[m] = by;
                uint16_t* const y = static_cast<uint16_t*>(norm.y) + static_cast<int64_t>(m) * K + c0;
                const uint16_t* const x = jobs.job[j].a + static_cast<int64_t>(m) * lda + c0;
                for (int c = static_cast<int>(threadIdx.x) / 32 * 4; c < n; c += 64 * KW / 32 * 4) {
                    u32x2 v = *reinterpret_cast<const u32x2*>(x + c);
                    const f32x4 w = *reinterpret_cast<const f32x4*>(norm.w + c0 + c);
#pragma unroll
                    for (int e = 0; e < 2; ++e)
                        v[e] = pack_bf16(__uint_as_float(v[e] << 16) * by * w[2 * e], __uint_as_float(v[e] & 0xffff0000u) * by * w[2 * e + 1]);
                    *reinterpret_cast<u32x2*>(y + c) = v;
                }
            }
        }
    const int n = n0 + 2 * l16;
    if (n >= N) return;
#pragma unroll
    for (int q = 0; q < RPW; ++q) {
        const int row = kw * RPW + q, x = row >> 2, r = row & 3;
        auto sum = [&](int c, int y) {
            float s = reinterpret_cast<const float*>(&part[0][c][x][y][lane])[r];
#pragma unroll
            for (int k = 1; k < KW; ++k) s += reinterpret_cast<const float*>(&part[k][c][x][y][lane])[r];
            return s;
        };
        float s0 = sum(0, 0), s1 = sum(0, 1);
        float by = 1.0f;
        if constexpr (NORM) by = inverse(2 * (4 * grp + r) + x), s0 *= by, s1 *= by;
        const int m = m0 + 2 * (4 * grp + r) + x;
        if (m >= M) continue;
        const int64_t o = m * ldc + n;
        // gate, up and their product's gradient count as they are stored, rounded
        const auto lo = [](uint32_t v) { return __uint_as_float(v << 16); };
        const auto hi = [](uint32_t v) { return __uint_as_float(v & 0xffff0000u); };
        if constexpr (END == End::GATE) {
            const uint32_t gate = pack_bf16(s0, s1), up = NORM ? pack_bf16(sum(1, 0) * by, sum(1, 1) * by) : pack_bf16(sum(1, 0), sum(1, 1));
            *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(jobs.job[j].c) + o) =
                pack_bf16(gated(lo(gate), lo(up)), gated(hi(gate), hi(up)));
            if (uint16_t* const gu = jobs.job[j].gu) {
                *reinterpret_cast<uint32_t*>(gu + m * ldc * 2 + n) = gate;
                *reinterpret_cast<uint32_t*>(gu + m * ldc * 2 + N + n) = up;
            }
            continue;
        }
        if constexpr (END == End::GATE_GRAD) {
            const uint32_t d = pack_bf16(s0, s1), gate = met[q][0], up = met[q][1];
            float dg[2], du[2];
            gated_grad(lo(gate), lo(up), lo(d), dg[0], du[0]);
            gated_grad(hi(gate), hi(up), hi(d), dg[1], du[1]);
            *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(jobs.job[j].c) + o) = pack_bf16(dg[0], dg[1]);
            *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(jobs.job[j].c) + o + N) = pack_bf16(du[0], du[1]);
            continue;
        }
        if constexpr (END == End::TURN) {
            if (pair >= 0) {
                const float c = __uint_as_float(met[q][0]), s = __uint_as_float(met[q][1]), t = s0 * c - s1 * s;
                s1 = s0 * s + s1 * c;
                s0 = t;
            }
        }
        if (CF32) {
            f32x2 v = {s0, s1};
            if (add) v[0] += __uint_as_float(met[q][0]), v[1] += __uint_as_float(met[q][1]);
            *reinterpret_cast<f32x2*>(static_cast<float*>(jobs.job[j].c) + o) = v;
        } else {
            if (add) {
                const uint32_t e = met[q][0];
                s0 += __uint_as_float(e << 16), s1 += __uint_as_float(e & 0xffff0000u);
            }
            *reinterpret_cast<uint32_t*>(static_cast<uint16_t*>(jobs.job[j].c) + o) = pack_bf16(s0, s1);
        }
    }
}

template <bool TA, bool TB, bool CF32, End END = End::PLAIN, int MAX>
void launch(Jobs<MAX>& jobs, bool accumulate, hipStream_t st, const Turn& turn = {}, const Norm* norm = nullptr) {
    int tiles = 0, longest = 0;
    for (int j = 0; j < jobs.count; ++j) {
        jobs.first[j] = tiles;
        tiles += ((jobs.job[j].M + 31) / 32) * ((jobs.job[j].N + 31) / 32);
        longest = std::max(longest, jobs.job[j].K);
    }
    for (int j = jobs.count; j <= MAX; ++j) jobs.first[j] = tiles;
    const dim3 grid((tiles + 7) / 8 * 8);
    // eight wavefronts where each still has a few chunks and two workgroups fit every CU
    const bool eight = longest >= 512 && tiles <= 1024;
    const auto start = [&](auto kw, auto normed, const Norm& n) {
        constexpr int KW = decltype(kw)::value;
        hipLaunchKernelGGL((gemm_small_k<TA, TB, CF32, KW, MAX, END, decltype(normed)::value>), grid, dim3(64 * KW), 0, st, jobs, tiles, accumulate ? 1 : 0,
                           turn, n);
    };
    const auto by_length = [&](auto normed, const Norm& n) {
        eight ? start(std::integral_constant<int, 8>{}, normed, n) : start(std::integral_constant<int, 4>{}, normed, n);
    };
    if constexpr (MAX == 1 && (END == End::GATE || END == End::TURN))
        norm ? by_length(std::true_type{}, *norm) : by_length(std::false_type{}, Norm{});
    else
        by_length(std::false_type{}, Norm{});
    hip_check(hipGetLastError(), "gemm_small");
}

}  // namespace

// Microseconds that this kernel takes, and the ring kernels (one product; several, grouped), as fitted to 250 sizes of 64 to 8192 tokens,
// widths 64 to 512 and vocabularies of 4000. Here a workgroup is a chain of its contraction's loads, and the launch all
// its tiles' operands through the L2s, in rounds of 256 tiles; there a tile is a chain of slices, cut up from 2048 on.
// (512 tokens: 128 x 384 projection 3.1 and 4.6, 344 x 128 3.5 and 6.2, its two gradients 3.8 and 7.5, 4.5 and 8.8;
// 4096 tokens, 512 x 1536: 30 and 12.)
double gemm_small_us(bool tA, bool tB, int64_t tiles, int64_t K) {
    const double chain = tA ? 0.0019 : tB ? 0.0035 : 0.0022, stream = tA ? 1.0e-5 : tB ? 1.3e-5 : 0.9e-5;
    return 2.8 + std::max(chain * K, static_cast<double>((tiles + 255) / 256 * 256) * (0.0011 + stream * K));
}
bool gemm_small_is_ahead(bool tA, bool tB, int64_t M, int64_t N, int64_t K) {
    const double ring = K >= 2048 ? (tA ? 13.5 : 15.5) : (tA ? 4.0 : 3.6) + 0.0072 * K;
    return gemm_small_us(tA, tB, ((M + 31) / 32) * ((N + 31) / 32), K) - 0.6 < ring;  // one product's arguments
}

namespace {
template <int MAX>
bool multiply(const SmallProduct* ps, int count, bool tA, bool tB, int c_dtype, float beta, hipStream_t st, End end = End::PLAIN,
              void* gu = nullptr, const Turn& turn = {}, const Norm* norm = nullptr) {
    Jobs<MAX> jobs{};
    jobs.count = count;
    for (int j = 0; j < count; ++j) {
        const SmallProduct& p = ps[j];
        const int64_t limit = int64_t{1} << 30;
        if (p.M < 2 || p.N < 2 || p.K < KC || p.M > limit || p.N > limit || p.K > limit) return false;
        if (extent(tA ? p.K : p.M, tA ? p.M : p.K, p.lda) >= limit || extent(tB ? p.N : p.K, tB ? p.K : end == End::GATE ? 2 * p.N : p.N, p.ldb) >= limit) return false;
        // pairs of columns, and of steps where those are adjacent, are read and written as one
        auto aligned = [](const void* q, int a) { return reinterpret_cast<uintptr_t>(q) % a == 0; };
        if (p.lda % 2 || p.ldb % 2 || p.ldc % 2 || p.N % 2 || (tA && p.M % 2) || (!(tA && !tB) && p.K % 2)) return false;
        if (!aligned(p.a, 4) || !aligned(p.b, 4) || !aligned(p.c, 8) || !aligned(p.addend, 8) || !aligned(gu, 4)) return false;
        jobs.job[j].a = static_cast<const uint16_t*>(p.a);
        jobs.job[j].b = static_cast<const uint16_t*>(p.b);
        jobs.job[j].c = p.c;
        jobs.job[j].addend = p.addend;
        jobs.job[j].gu = static_cast<uint16_t*>(gu);
        jobs.job[j].lda = static_cast<int>(p.lda);
        jobs.job[j].ldb = static_cast<int>(p.ldb);
        jobs.job[j].ldc = static_cast<int>(p.ldc);
        jobs.job[j].M = static_cast<int>(p.M);
        jobs.job[j].N = static_cast<int>(p.N);
        jobs.job[j].K = static_cast<int>(p.K);
    }
    const bool f32 = c_dtype == PK_F32, acc = beta != 0.0f;
    if constexpr (MAX == 1) {
        if (end == End::GATE) launch<false, false, false, End::GATE>(jobs, acc, st, turn, norm);
        if (end == End::GATE_GRAD) launch<false, true, false, End::GATE_GRAD>(jobs, acc, st);
        if (end == End::TURN) launch<false, false, false, End::TURN>(jobs, acc, st, turn, norm);
        if (end != End::PLAIN) return true;
    }
    if (tA)
        f32 ? launch<true, false, true>(jobs, acc, st) : launch<true, false, false>(jobs, acc, st);
    else if (tB)
        f32 ? launch<false, true, true>(jobs, acc, st) : launch<false, true, false>(jobs, acc, st);
    else
        f32 ? launch<false, false, true>(jobs, acc, st) : launch<false, false, false>(jobs, acc, st);
    return true;
}
// the normalised rows are written four columns at a time
bool norm_fits(const void* x, int64_t K, const Norm* norm) {
    const auto at = [](const void* p, int a) { return reinterpret_cast<uintptr_t>(p) % a == 0; };
    return !norm || (K % 4 == 0 && K <= 4096 && at(x, 8) && at(norm->w, 16) && at(norm->y, 8));
}
}  // namespace

bool gemm_small(const SmallProduct* ps, int count, bool tA, bool tB, int c_dtype, float beta, hipStream_t st) {
    if (count < 1 || count > 8 || (tA && tB) || (beta != 0.0f && beta != 1.0f)) return false;
    return count == 1 ? multiply<1>(ps, count, tA, tB, c_dtype, beta, st) : multiply<8>(ps, count, tA, tB, c_dtype, beta, st);
}
bool gemm_small_gated(const void* x, const void* w, void* gu, void* h, int64_t M, int64_t N, int64_t K, hipStream_t st, const Norm* norm) {
    const SmallProduct p{x, K, w, 2 * N, h, N, nullptr, M, N, K};
    return norm_fits(x, K, norm) && multiply<1>(&p, 1, false, false, PK_BF16, 0.0f, st, End::GATE, gu, {}, norm);
}
bool gemm_small_gated_grad(const void* dy, const void* w, const void* gu, void* dgu, int64_t M, int64_t N, int64_t K, hipStream_t st) {
    const SmallProduct p{dy, K, w, K, dgu, 2 * N, nullptr, M, N, K};
    return multiply<1>(&p, 1, false, true, PK_BF16, 0.0f, st, End::GATE_GRAD, const_cast<void*>(gu));
}
bool gemm_small_turned(const void* x, const void* w, void* y, int64_t M, int64_t K, const Turn& turn, hipStream_t st, const Norm* norm) {
    const int64_t N = 3 * static_cast<int64_t>(turn.d);
    const SmallProduct p{x, K, w, N, y, N, nullptr, M, N, K};
    return turn.d % 2 == 0 && turn.head_dim % 2 == 0 && norm_fits(x, K, norm) &&
           multiply<1>(&p, 1, false, false, PK_BF16, 0.0f, st, End::TURN, nullptr, turn, norm);
}

}  // namespace pk
