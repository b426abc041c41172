// bf16 GEMM on the gfx950 matrix cores for the Linear layers of the Llama block: the MI355X counterpart of the
// reference's tiled GEMM with transpose flags (paperkiln src/cuda_resident.cu:141-171, entry step_resident_gemm
// :226-263, reached through device::gemm, src/device.cpp:91-125).
//
//   C[M, N] (+)= op(A) op(B),   row-major, bf16 operands, fp32 accumulation, C in bf16 or fp32
//
// One workgroup of four wavefronts owns a 128 x 128 tile of C and walks the contraction in slices of 64; each
// wavefront owns 64 x 64 of it as 2 x 2 accumulators of v_mfma_f32_32x32x16_bf16. Operand tiles are staged in LDS,
// double-buffered, one barrier per slice, the next slice's global loads in flight while the current one is
// multiplied. An operand whose contraction index is contiguous in memory (A of "N", B of "T") is kept as
// [row][k] with a pitch of 72 elements and read with 16-byte row reads; one whose contraction index is the row
// index in memory (A of "T", B of "N") is kept as [k][column] with a pitch of 160 and read with
// ds_read_b64_tr_b16, so no operand is ever transposed in memory. Both pitches are conflict-free for their read.
// The product is formed as C^T (the B fragment in the MFMA's A slot), which leaves each lane with runs of four
// consecutive columns of one row of C; the tile then goes through LDS once so that the global stores are whole
// 16-byte chunks of consecutive columns.
//
// Long contractions with a small result (weight gradients over all tokens) are cut along the contraction axis
// into slices that separate workgroups multiply into fp32 partial tiles; the partial tiles are added in slice
// order by a second kernel -- no atomics, the same bits on every run.
#include <algorithm>
#include <memory>
#include <type_traits>

#include "mfma_common.h"
#include "tensor.h"

namespace pk {
namespace {

constexpr int BK = 64;
constexpr int PITCH_ROW = BK + 8;  // [rows][64 k]: 16-byte row reads conflict-free

// Tile geometry: WGM x WGN wavefronts, each owning FM x FN accumulators of 32 x 32.
//   Small: 2 x 2 wavefronts of 2 x 2 -> 128 x 128, 256 threads, two workgroups per CU. For outputs of a few
//          hundred tiles, where more and smaller workgroups fill the chip better.
//   Large: 2 x 4 wavefronts of 4 x 2 -> 256 x 256, 512 threads, one workgroup per CU: half the operand bytes per
//          MFMA, which is what the vector memory path (64 bytes per clock and CU) asks for on long runs.
//   KS > 1 (ring kernel only): KS sets of WGM x WGN wavefronts share the tile, set q multiplying the q-th part of every
//          64-deep slice; their accumulators are added through LDS at the end. Two wavefronts per SIMD from one
//          workgroup, for outputs of so few tiles that a CU gets no second workgroup.
template <int WGM_, int WGN_, int FM_, int FN_, int KS_ = 1>
struct Geo {
    static constexpr int WGM = WGM_, WGN = WGN_, FM = FM_, FN = FN_, KS = KS_;
    static constexpr int BM = WGM * FM * 32, BN = WGN * FN * 32, NTHR = WGM * WGN * KS * 64;
    // [64 k][columns] tiles: a pitch of 32 past a multiple of 128 keeps the transposing reads conflict-free
    static constexpr int PITCH_TR_A = BM + 32, PITCH_TR_B = BN + 32;
    static constexpr int A_EL = BM * PITCH_ROW > BK * PITCH_TR_A ? BM * PITCH_ROW : BK * PITCH_TR_A;
    static constexpr int B_EL = BN * PITCH_ROW > BK * PITCH_TR_B ? BN * PITCH_ROW : BK * PITCH_TR_B;
    static constexpr int CH_A = BM * BK / 8 / NTHR, CH_B = BN * BK / 8 / NTHR;  // 16-byte chunks per thread and slice
};
using GeoSmall = Geo<2, 2, 2, 2>;
using GeoLarge = Geo<2, 4, 4, 2>;
using GeoSmallK2 = Geo<2, 2, 2, 2, 2>;

struct GemmArgs {
    const uint16_t* a;
    const uint16_t* b;
    void* c;
    int M, N, K;
    int64_t lda, ldb, ldc;
    int beta;         // 0: C = product, 1: C = D + product
    const void* d;    // D of beta 1: C's type and row pitch; null = C itself (C += product)
    int k_per_split;  // contraction elements per blockIdx.z (a multiple of BK); K when not split
    int64_t part_stride;  // elements between the fp32 partial results of two slices (split only)
    int tiles_m, tiles_n;
    int splits;  // slices of the contraction (gemm_ring walks them itself; gemm_bf16 takes them from blockIdx.z)
};

// What the two passes of the tied head's cross-entropy do with a tile of logits instead of storing it (gemm_ring's
// EPI parameter). Pass 1: per row and per 64-column span of a wavefront, the span's maximum and its sum of
// exp(z - maximum), to stats[span][row], and the target column's logit to zt[row]. Pass 2: the same tile formed
// again, turned into dlogits = (exp(z - row_max) row_inv - [column == target]) gscale and stored as bf16. EPI 1 is the first
// pass, EPI 2 the second, EPI 4 the second over a vocabulary padded to a multiple of 8: its test of the columns keeps 95 scalar
// registers outside their file, which the whole of pass 2 would pay for (4096 rows x 32000 x 512: 165 -> 169 us).
struct HeadArgs {
    const int* target;     // [M]
    float2* stats;         // pass 1: [spans][M]
    float* zt;             // pass 1: [M]
    const float* row_max;  // pass 2: [M]
    const float* row_inv;  // pass 2: [M], 1 / sum_j exp(z_j - row_max)
    float gscale;          // pass 2
    int vocab;             // EPI 4: columns from here to N only pad the matrix; their dlogits are 0
    Turn turn;             // EPI 8
};
constexpr float LOG2E = 1.4426950408889634f;

// Several products of one launch (gemm_ring's EPI 3): C_p (+)= op(A_p) op(B_p), p < count, all with the contraction
// length, transposition flags and result type of the launch; the workgroups walk the tiles of all of them as one
// sequence (problem after problem, each row by row). For products that are each too small to fill the chip and would
// otherwise each cut their contraction into slices and add partial results afterwards.
constexpr int GROUP_MAX = 8;
struct GroupArgs {
    int count;
    int tile_end[GROUP_MAX];  // tiles of problems 0 .. p
    const uint16_t* a[GROUP_MAX];
    const uint16_t* b[GROUP_MAX];
    void* c[GROUP_MAX];
    int M[GROUP_MAX], N[GROUP_MAX], tiles_n[GROUP_MAX];
    int lda[GROUP_MAX], ldb[GROUP_MAX], ldc[GROUP_MAX];
};

// Transposing operand read in natural k order: lane (c32, g) receives rows row0 + 8g .. 8g + 7 of column
// col0 + c32 of a [k][column] tile.
__device__ inline bf16x8 read_tr_nat(const uint16_t* tile, int pitch, int row0, int col0, int lane) {
    const int g = lane >> 5, u = (lane >> 4) & 1, j = lane & 15;
    const uint16_t* p = tile + (row0 + 8 * g + (j >> 2)) * pitch + col0 + 16 * u + 4 * (j & 3);
    const s16x4 lo = lds_read_tr4(p), hi = lds_read_tr4(p + 4 * pitch);
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    const s16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return *reinterpret_cast<const bf16x8*>(&v);
}

// One operand tile of the slice starting at k0: global -> registers (NCH 16-byte chunks per thread).
// TR = false: memory is [row][k] (rows = the SPAN rows / columns of C this tile covers);
// TR = true:  memory is [k][column].
template <bool TR, int SPAN, int NTHR, int NCH>
__device__ inline void fetch_tile(const uint16_t* base, int64_t ld, int rc0, int rc_count, int k0, int k_end, u32x4 (&r)[NCH]) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int c = static_cast<int>(threadIdx.x) + NTHR * i;
        const u32x4 zero = {0u, 0u, 0u, 0u};
        if (!TR) {
            const int row = c >> 3, ch = c & 7;
            const bool ok = rc0 + row < rc_count && k0 + ch * 8 < k_end;
            r[i] = ok ? *reinterpret_cast<const u32x4*>(base + static_cast<int64_t>(rc0 + row) * ld + k0 + ch * 8) : zero;
        } else {
            constexpr int CPR = SPAN / 8;
            const int row = c / CPR, ch = c % CPR;
            const bool ok = k0 + row < k_end && rc0 + ch * 8 < rc_count;
            r[i] = ok ? *reinterpret_cast<const u32x4*>(base + static_cast<int64_t>(k0 + row) * ld + rc0 + ch * 8) : zero;
        }
    }
}
template <bool TR, int SPAN, int NTHR, int NCH>
__device__ inline void commit_tile(uint16_t* tile, const u32x4 (&r)[NCH]) {
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
        const int c = static_cast<int>(threadIdx.x) + NTHR * i;
        if (!TR) {
            *reinterpret_cast<u32x4*>(tile + (c >> 3) * PITCH_ROW + (c & 7) * 8) = r[i];
        } else {
            constexpr int CPR = SPAN / 8;
            *reinterpret_cast<u32x4*>(tile + (c / CPR) * (SPAN + 32) + (c % CPR) * 8) = r[i];
        }
    }
}

// Epilogue through LDS, one strip of 32 rows per wavefront row at a time: the strip as [WGM * 32][BN + pad]
// in the output's element type, then 16-byte chunks of consecutive columns to global memory (read-add-write
// when accumulating). `lds` is the kernel's whole LDS allocation, free to overwrite when this is called.
template <typename G, bool CF32>
__device__ inline void store_tile(const f32x16 (&acc)[G::FM][G::FN], void* lds, const GemmArgs& g, int m0, int n0, int wm, int wn,
                                  int c32, int gh, bool writer = true) {
    constexpr int BN = G::BN, NTHR = G::NTHR, FM = G::FM, FN = G::FN;
    typedef typename std::conditional<CF32, float, uint16_t>::type CT;
    constexpr int CP = BN + (CF32 ? 4 : 8);  // pitch in elements: rows stay 16-byte aligned
    constexpr int EPC = CF32 ? 4 : 8;        // elements per 16-byte chunk
    constexpr int CPR = BN / EPC;            // chunks per strip row
    CT* cs = reinterpret_cast<CT*>(lds);
    CT* cout = static_cast<CT*>(g.c) + (g.part_stride ? static_cast<int64_t>(blockIdx.z) * g.part_stride : 0);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                if (!writer) continue;  // wavefront-uniform: the wavefronts that hold the tile's sums
                const int row = wm * 32 + c32, col = (wn * FN + j) * 32 + qd * 8 + gh * 4;
                if (CF32) {
                    const f32x4 v = {acc[i][j][qd * 4], acc[i][j][qd * 4 + 1], acc[i][j][qd * 4 + 2], acc[i][j][qd * 4 + 3]};
                    *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(cs) + row * CP + col) = v;
                } else {
                    const u32x2 v = {pack_bf16(acc[i][j][qd * 4], acc[i][j][qd * 4 + 1]),
                                     pack_bf16(acc[i][j][qd * 4 + 2], acc[i][j][qd * 4 + 3])};
                    *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(cs) + row * CP + col) = v;
                }
            }
        __syncthreads();
        for (int c = threadIdx.x; c < G::WGM * 32 * CPR; c += NTHR) {
            const int srow = c / CPR, ch = c % CPR;
            // strip row srow belongs to wavefront row srow / 32, whose i-th block of 32 rows this is
            const int m = m0 + ((srow >> 5) * FM + i) * 32 + (srow & 31), n = n0 + ch * EPC;
            if (m >= g.M || n >= g.N) continue;
            u32x4 v = *reinterpret_cast<const u32x4*>(cs + srow * CP + ch * EPC);
            CT* dst = cout + static_cast<int64_t>(m) * g.ldc + n;
            if (g.beta) {
                const u32x4 old = *reinterpret_cast<const u32x4*>(dst);
                if (CF32) {
                    f32x4 s = *reinterpret_cast<const f32x4*>(&old) + *reinterpret_cast<const f32x4*>(&v);
                    v = *reinterpret_cast<const u32x4*>(&s);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float lo = __uint_as_float(old[e] << 16) + __uint_as_float(v[e] << 16);
                        const float hi = __uint_as_float(old[e] & 0xffff0000u) + __uint_as_float(v[e] & 0xffff0000u);
                        v[e] = pack_bf16(lo, hi);
                    }
                }
            }
            *reinterpret_cast<u32x4*>(dst) = v;
        }
        __syncthreads();
    }
}

template <typename G, bool TA, bool TB, bool CF32>
__global__ __launch_bounds__(G::NTHR, 2) void gemm_bf16(GemmArgs g) {
    constexpr int BM = G::BM, BN = G::BN, NTHR = G::NTHR, FM = G::FM, FN = G::FN;
    __shared__ __attribute__((aligned(16))) uint16_t lds[2 * (G::A_EL + G::B_EL)];  // [buffer][A | B]
    static_assert(G::WGM * 32 * (G::BN + 8) * (CF32 ? 4 : 2) <= sizeof(lds), "epilogue strip must fit the tile buffers");
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c32 = lane & 31, gh = lane >> 5, wm = w / G::WGN, wn = w % G::WGN;

    // XCD-aware tile order: workgroup ids go round-robin over the 8 XCDs, so XCD x takes the x-th eighth of the
    // tile list (columns fastest): the tiles that share rows of A meet in one L2.
    const int ntiles = g.tiles_m * g.tiles_n;
    const int per_xcd = (ntiles + 7) / 8;
    const int t = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
    if (t >= ntiles) return;
    const int m0 = (t / g.tiles_n) * BM, n0 = (t % g.tiles_n) * BN;
    const int k_begin = blockIdx.z * g.k_per_split, k_end = min(g.K, k_begin + g.k_per_split);

    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    u32x4 ra[G::CH_A], rb[G::CH_B];
    // A: !TA [M][K] row form; TA [K][M] transposed form.  B: TB [N][K] row form; !TB [K][N] transposed form.
    fetch_tile<TA, BM, NTHR, G::CH_A>(g.a, g.lda, m0, g.M, k_begin, k_end, ra);
    fetch_tile<!TB, BN, NTHR, G::CH_B>(g.b, g.ldb, n0, g.N, k_begin, k_end, rb);
    commit_tile<TA, BM, NTHR, G::CH_A>(lds, ra);
    commit_tile<!TB, BN, NTHR, G::CH_B>(lds + G::A_EL, rb);
    __syncthreads();

    int buf = 0;
    for (int k0 = k_begin; k0 < k_end; k0 += BK) {
        const bool more = k0 + BK < k_end;
        if (more) {
            fetch_tile<TA, BM, NTHR, G::CH_A>(g.a, g.lda, m0, g.M, k0 + BK, k_end, ra);
            fetch_tile<!TB, BN, NTHR, G::CH_B>(g.b, g.ldb, n0, g.N, k0 + BK, k_end, rb);
        }
        const uint16_t* As = lds + buf * (G::A_EL + G::B_EL);
        const uint16_t* Bs = As + G::A_EL;
#pragma unroll
        for (int kk = 0; kk < BK / 16; ++kk) {
            bf16x8 fa[FM], fb[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i)
                fa[i] = TA ? read_tr_nat(As, G::PITCH_TR_A, kk * 16, (wm * FM + i) * 32, lane)
                           : lds_read8(As + ((wm * FM + i) * 32 + c32) * PITCH_ROW + kk * 16 + gh * 8);
#pragma unroll
            for (int j = 0; j < FN; ++j)
                fb[j] = !TB ? read_tr_nat(Bs, G::PITCH_TR_B, kk * 16, (wn * FN + j) * 32, lane)
                            : lds_read8(Bs + ((wn * FN + j) * 32 + c32) * PITCH_ROW + kk * 16 + gh * 8);
            // C^T blocks: rows = columns of C (from B), lane = row of C (from A)
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) acc[i][j] = mfma32(fb[j], fa[i], acc[i][j]);
        }
        if (more) {
            uint16_t* nxt = lds + (buf ^ 1) * (G::A_EL + G::B_EL);
            commit_tile<TA, BM, NTHR, G::CH_A>(nxt, ra);
            commit_tile<!TB, BN, NTHR, G::CH_B>(nxt + G::A_EL, rb);
        }
        __syncthreads();
        buf ^= 1;
    }

    store_tile<G, CF32>(acc, lds, g, m0, n0, wm, wn, c32, gh);
}

// ---- the same tiles fed through a ring of LDS slots ---------------------------------------------------------------
// With one workgroup per CU (an output of 256 tiles or fewer, or tiles whose buffers fill the LDS) a slice's global
// loads have one slice of matrix work to hide behind, 512 clocks against a round trip of 1,500 - 2,000, and a loop
// that spends four scalar instructions per matrix instruction on addresses and branches is bound by instruction
// issue. Here the operand slices go from memory straight into LDS (buffer_load_dwordx4 ... lds: no staging
// registers, no LDS stores, a lane outside the buffer writes zeros), into a ring of NS slots; a slot is asked for anew
// as soon as its slice's last fragments are in registers; a tile's buffer descriptors are formed once and the position
// in the contraction is the instruction's scalar offset (which the hardware counts in its range check); the slice
// loop is unrolled over the ring, so every LDS address is a register formed once plus an immediate. The result leaves
// through a strip of LDS beside the ring, so the next tile's slices keep coming meanwhile.
//
// One load instruction fills 1 KB of LDS lane after lane, so a lane's place in LDS is fixed and what varies is which
// 16 bytes of memory it fetches. The tiles are therefore not padded but swizzled:
//   [row][64 k] operand (A of "N", B of "T"), rows of 128 bytes = 8 chunks: chunk c of row r lies at chunk
//     c ^ ((r & 7) ^ ((r >> 3) & 3)) of its row. The 16 rows a quarter-wavefront reads with one 16-byte row read
//     then cover all 64 banks once (and any 8 consecutive rows 32 banks once).
//   [64 k][columns] operand (A of "T", B of "N"), rows of 2 * SPAN bytes: the 64-byte segment s of row r lies at
//     segment s ^ (r & 3) within its group of four. The 4 rows x 64 bytes a half-wavefront reads with one
//     transposing read then cover all 64 banks once.
template <bool TR, int SPAN, int NW>
struct RingOp {
    static constexpr int CPR = TR ? SPAN / 8 : BK / 8;    // 16-byte chunks per LDS row
    static constexpr int ROWS = TR ? BK : SPAN;
    static constexpr int ROWB = CPR * 16;                 // bytes per LDS row
    static constexpr int NI = ROWS * CPR / 64;            // wavefront loads per slice
    static_assert(NI % NW == 0, "every wavefront issues the same number of loads");
    static constexpr int PER = NI / NW;                   // consecutive 1 KB pieces per wavefront
    static_assert(PER == 2 || PER == 4, "one m0 value and immediate offsets below 4096 per group");
    static constexpr int BYTES = NI * 1024;
    // the chunk of its LDS row that holds memory chunk c (and vice versa: the map is an involution)
    __device__ static int swz(int r, int c) { return TR ? c ^ ((r & 3) << 2) : c ^ ((r & 7) ^ ((r >> 3) & 3)); }
};
// Descriptor of an operand's tile: from BIAS bytes before the tile's first element of the contraction range to the
// operand's end (rows past the matrix, and rows past the contraction's end where the contraction index is the row,
// read as zeros); `step` bytes per slice.
struct TileDesc {
    u32x4 rsrc;
    int step;
};
template <bool TR>
__device__ inline TileDesc tile_desc(const uint16_t* base, int64_t ld, int rc0, int rc_count, int k_begin, int k_end) {
    const int64_t kspan = k_end - k_begin, rcs = rc_count - rc0;
    const char* p;
    int64_t left;
    TileDesc d;
    if (!TR) {  // [row][k]
        p = reinterpret_cast<const char*>(base + static_cast<int64_t>(rc0) * ld + k_begin);
        left = ((rcs - 1) * ld + kspan) * 2;
        d.step = BK * 2;
    } else {  // [k][column]
        // An odd number of columns (of A^T only) ends in the middle of a dword, which the range check drops whole: the last
        // row's last element would read as zero. That dword lies inside the row's pitch, a multiple of 8.
        p = reinterpret_cast<const char*>(base + static_cast<int64_t>(k_begin) * ld + rc0);
        left = ((kspan - 1) * ld + rcs + (rcs & 1)) * 2;
        d.step = static_cast<int>(BK * ld * 2);
    }
    const uint64_t a = reinterpret_cast<uint64_t>(p) - BIAS;
    d.rsrc[0] = static_cast<uint32_t>(a);
    d.rsrc[1] = static_cast<uint32_t>(a >> 32) & 0xffffu;
    d.rsrc[2] = static_cast<uint32_t>(left + BIAS);
    d.rsrc[3] = 0x00020000u;
    return d;
}
template <int N>
__device__ inline void wait_loads_then_barrier() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}
// GATED: the operand is [gate | up] of `half` columns each, and the tile holds, in 32-column blocks in turn, the same columns of both:
// a wavefront's two blocks of results are then a gate's and an up's, lane by lane. Column (of gate) a chunk begins at, from the
// tile's first on, and bytes from the tile's first to the chunk:
__device__ inline int gated_column(int c) { return (c >> 3) * 32 + (c & 3) * 8; }
__device__ inline uint32_t gated_bytes(int c, int half) { return (gated_column(c) + (c & 4 ? half : 0)) * 2u; }
// lane offsets of a wavefront's loads of one operand's slice, for a tile in the matrix's interior (every column there,
// every slice whole)
template <typename O, bool GATED = false>
__device__ inline void lane_offsets(uint32_t (&off)[O::PER], int w, int lane, int64_t ld, int half = 0) {
#pragma unroll
    for (int j = 0; j < O::PER; ++j) {
        const int u = (w * O::PER + j) * 64 + lane, r = u / O::CPR, c = O::swz(r, u % O::CPR);
        off[j] = static_cast<uint32_t>(r) * static_cast<uint32_t>(ld) * 2u + (GATED ? gated_bytes(c, half) : c * 16u) + BIAS - j * 1024u;
    }
}
// ... and with the chunks that must not be read sent outside the buffer: columns past the matrix's edge of a
// [k][column] operand (every slice of an edge tile), chunks past the contraction's end in the last, partial slice of
// a [row][k] operand (they are the next row's)
template <typename O, bool TR, bool GATED = false>
__device__ inline void lane_offsets_masked(uint32_t (&off)[O::PER], const uint32_t (&whole)[O::PER], int w, int lane, int rc0,
                                           int rc_count, int ktail) {
#pragma unroll
    for (int j = 0; j < O::PER; ++j) {
        const int u = (w * O::PER + j) * 64 + lane, r = u / O::CPR, c = O::swz(r, u % O::CPR);
        const bool ok = TR ? rc0 + (GATED ? gated_column(c) : c * 8) < rc_count : (ktail == 0 || c * 8 < ktail);
        off[j] = ok ? whole[j] : OUTSIDE;
    }
}
template <bool SPILLED = false>
__device__ inline void store16(u32x4 v, uint32_t off, u32x4 rsrc, uint32_t soff) {
    // invisible to the compiler's count of memory operations in flight, like the loads above; the data registers
    // may be overwritten by the next two instructions, which a 16-byte store does not allow: two idle states behind it. SPILLED: five in front of
    // it, for scalars that a vector instruction has just written (dma_piece).
    // sc1, agent scope: an XCD's L2 passes the line on at once instead of holding it until the kernel's end, when eight L2s of 4 MB would be written
    // back while nothing multiplies. Rows leave a strip as whole lines, so nothing is written twice. 8192 x 1536 x 512 17.6 -> 15.9 us, 8192 x 512 x 512
    // 8.0 -> 7.4, 8192 x 1376 x 512 17.0 -> 15.0, fp32 results 32000 x 512 x 4096 131.9 -> 129.1 and 512 x 2752 x 8192 34.8 -> 33.6, 4096 ^ 3 103.5 ->
    // 102.3. Not nt, which keeps the last-level cache from holding the lines as well: a little more of this, and 5 to 9 % of the kernels that read them next.
    if constexpr (SPILLED)
        asm volatile("s_nop 4\n\tbuffer_store_dwordx4 %0, %1, %2, %3 offen sc1\n\ts_nop 1" ::"v"(v), "v"(off), "s"(rsrc), "s"(soff) : "memory");
    else
        asm volatile("buffer_store_dwordx4 %0, %1, %2, %3 offen sc1\n\ts_nop 1" ::"v"(v), "v"(off), "s"(rsrc), "s"(soff) : "memory");
}
// The same where the compiler counts it, between loads whose waits are not to be waits for the stores as well. The compiler leaves the idle states
// out where the scalar offset is a register: without them the last dword of some lanes was the next value's (256 x 256 tiles).
__device__ inline void store16_counted(u32x4 v, uint32_t off, __amdgpu_buffer_rsrc_t rsrc, uint32_t soff) {
    constexpr int SC1 = 16;
    __builtin_amdgcn_raw_buffer_store_b128(v, rsrc, static_cast<int>(off), static_cast<int>(soff), SC1);
    asm volatile("s_nop 1" ::"v"(v) : "memory");
}
// What a workgroup stores per tile, for the count of memory operations in flight: FM strips of all WGM * 32 rows
// (bf16) or FM * WGM strips of 32 rows (fp32, whose wider rows would not fit a ring slot otherwise), each
// rows * chunks-per-row / threads stores per thread.
template <typename G, bool CF32>
struct TileStore {
    static constexpr int EPC = CF32 ? 4 : 8;  // elements per 16-byte chunk
    static constexpr int CPR = G::BN / EPC;   // chunks per strip row
    static constexpr int SR = CF32 ? 32 : G::WGM * 32;
    static constexpr int PHASES = CF32 ? G::FM * G::WGM : G::FM;
    static_assert(SR * CPR % G::NTHR == 0 && G::NTHR % CPR == 0, "whole stores per thread, one chunk column per thread");
    static constexpr int PER_PHASE = SR * CPR / G::NTHR;
    static constexpr int NST = PHASES * PER_PHASE;
    static constexpr int BYTES = SR * CPR * 16;
    // Place of column `col` of strip row `row`, in elements: rows are not padded (the strip lies beside the ring, and the two fill the
    // LDS to the byte), chunks are dealt over the banks by the row instead, two lanes of a half-wavefront to a bank as padding has it.
    __device__ static int at(int row, int col) { return row * G::BN + ((col / EPC) ^ (row & 31 & (CPR - 1))) * EPC + col % EPC; }
};
// LDS of a ring kernel: NS slots of one slice of both operands and, beside them, a strip of the result on its way out (or half of the
// second wavefront set's sums).
template <typename G, int NS>
struct RingLds {
    static constexpr int SLOT = (G::BM + G::BN) * BK * 2;
    static constexpr int SUMS = G::KS == 1 ? 0 : G::WGM * G::WGN * 64 * (G::FM / 2) * G::FN * 64;
    static constexpr int STRIP = TileStore<G, false>::BYTES > SUMS ? TileStore<G, false>::BYTES : SUMS;
    static_assert(TileStore<G, true>::BYTES <= STRIP, "both result types' strips");
    static constexpr int BYTES = NS * SLOT + STRIP;
    static_assert(NS >= 2 && BYTES <= 160 * 1024, "the ring and the strip must fit the LDS");
    static constexpr int PER_CU = BYTES <= 80 * 1024 ? 2 : 1;
};

// C = op(A) op(B), persistent: gridDim.x workgroups walk the virtual blocks v = blockIdx.x, + gridDim.x, ...
// (virtual block -> (contraction slice, tile) as gemm_bf16 maps (blockIdx.z, blockIdx.x), XCD by XCD), and the ring
// runs on across tile boundaries: the first slices of the next tile are on their way while the last ones of this tile
// are multiplied and its result is stored, so a tile's first round trip to memory is paid once per workgroup.
template <typename G, bool TA, bool TB, bool CF32, int NS, int EPI = 0>
__global__ __launch_bounds__(G::NTHR, (RingLds<G, NS>::PER_CU))
void gemm_ring(GemmArgs g, HeadArgs hd, GroupArgs gr) {
    static_assert(EPI == 0 || EPI == 3 || (G::KS == 1 && !CF32), "the head's epilogues: one wavefront set, bf16 result");
    constexpr bool GROUPED = EPI == 3;
    constexpr bool SPILLED = EPI == 1 || EPI == 2 || EPI == 4;  // 56 to 81 scalars of the head's passes lie in vector registers
    // A gated product's ends. 5, 6: B is [gate | up], N columns each; C = silu(gate) up, and (5) both of them to D, [M, 2 N]. 7: the
    // product is the gradient of C for the gate and up in D; C is [M, 2 N] and gets theirs.
    constexpr bool GATE = EPI == 5 || EPI == 6, GATE_GRAD = EPI == 7;
    // 8: C is a [q | k | v] projection whose q and k turn by their positions.
    constexpr bool TURN = EPI == 8;
    static_assert(!GATE || (!TB && G::FN == 2), "a wavefront holds a block of gate and one of up");
    constexpr int BM = G::BM, BN = G::BN, NTHR = G::NTHR, FM = G::FM, FN = G::FN, NW = NTHR / 64;
    using OA = RingOp<TA, BM, NW>;
    using OB = RingOp<!TB, BN, NW>;
    using ST = TileStore<G, CF32>;
    constexpr int SLOT = OA::BYTES + OB::BYTES, PERTOT = OA::PER + OB::PER;
    constexpr int BNC = GATE ? BN / 2 : BN;  // columns of C per tile
    constexpr int NST = EPI == 5 ? ST::NST / 2 * 3 : EPI == 6 ? ST::NST / 2 : EPI == 7 ? ST::NST * 2 : ST::NST;
    using RL = RingLds<G, NS>;
    static_assert(SLOT == RL::SLOT, "a slice of both operands");
    static_assert((NS - 2) * PERTOT + NST < 64, "memory operations in flight must fit the counter");
    __shared__ __attribute__((aligned(1024))) uint8_t lds[RL::BYTES];
    uint8_t* const strip = lds + NS * SLOT;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    constexpr int KS = G::KS, NWQ = G::WGM * G::WGN, KPW = BK / 16 / KS;  // k-chunks of a slice per wavefront
    static_assert(KS == 1 || KS == 2, "one or two wavefront sets");
    static_assert(KS == 1 || FM % 2 == 0, "half of the second set's sums at a time");
    const int ks = KS == 1 ? 0 : w / NWQ, wq = w - ks * NWQ;
    const int c32 = lane & 31, gh = lane >> 5, wm = wq / G::WGN, wn = wq % G::WGN;

    // Virtual blocks: u = slice z of the contraction, then tile t row by row; XCD x (workgroups with blockIdx % 8 == x)
    // takes the x-th eighth of that sequence, so the workgroups that run on an XCD at one time work on one slice of
    // the contraction -- they stream the same rows of both operands through the XCD's L2 (the weight-gradient products
    // of a d = 512 block fetch 40 MB instead of 89 and run 6 - 10 % faster than with every slice spread over all XCDs)
    // -- and on whole rows of tiles. (Walking tiles in blocks of 4 or 8 rows instead halves what the L2s fetch for
    // [4096, 32000] x 512, 543 -> ~270 MB, and changes its time by nothing -- the last-level cache serves those misses
    // at 7 TB/s -- while [8192, 2752] x 512, whose weight matrix fits an L2 whole, loses 20 %.)
    // The arguments' lines of memory looked at together, as in the attention kernels, where that is ahead: a block's weight gradients 42.5 -> 41.6 us (200
    // tiles of 8192 steps among them), 22.0 -> 20.9; one wavefront set, 8192 x 1536 x 512 20.15 -> 19.8; two sets and the head's passes without (24.8 | 25.3), and two sets
    // without the divisions of unsigned numbers (14.0 | 14.6).
    if constexpr (GROUPED)
        asm volatile("" ::"s"(gr.a[0]), "s"(gr.lda[0]), "s"(gr.M[0]), "s"(gr.count), "s"(gr.c[0]), "s"(gr.b[0]), "s"(gr.ldc[0]));
    else if constexpr (G::KS == 1 && EPI == 0)
        asm volatile("" ::"s"(g.a), "s"(g.ldc), "s"(g.splits));
    const int ntiles = GROUPED ? gr.tile_end[gr.count - 1] : g.tiles_m * g.tiles_n;
    const int total = ntiles * g.splits, per_xcd = (total + 7) / 8, V = per_xcd * 8;
    const int stride = static_cast<int>(gridDim.x);
    struct Block {
        int m0, n0, k_begin, k_end, z, p;  // p: which problem of a grouped launch
    };
    auto next_block = [&](int v, Block& bl) {  // first virtual block at or after v (in steps of the grid) that is a tile
        for (; v < V; v += stride) {
            const int u = (v & 7) * per_xcd + (v >> 3);
            if (u >= total) continue;
            const int z = KS == 1 || GROUPED ? quotient(u, ntiles) : u / ntiles;
            int t = u - z * ntiles, p = 0, tiles_n = g.tiles_n;
            if (GROUPED) {
                while (t >= gr.tile_end[p]) ++p;
                if (p > 0) t -= gr.tile_end[p - 1];
                tiles_n = gr.tiles_n[p];
            }
            const int tm = KS == 1 || GROUPED ? quotient(t, tiles_n) : t / tiles_n;
            bl.m0 = tm * BM;
            bl.n0 = (t - tm * tiles_n) * BNC;
            bl.z = z;
            bl.p = p;
            bl.k_begin = z * g.k_per_split;
            bl.k_end = min(g.K, bl.k_begin + g.k_per_split);
            return v;
        }
        return V;
    };
    // the operands and sizes of the problem a block belongs to
    struct Prob {
        const uint16_t* a;
        const uint16_t* b;
        void* c;
        int M, N;
        int64_t lda, ldb, ldc;
    };
    auto prob = [&](const Block& bl) -> Prob {
        if (GROUPED) return Prob{gr.a[bl.p], gr.b[bl.p], gr.c[bl.p], gr.M[bl.p], gr.N[bl.p], gr.lda[bl.p], gr.ldb[bl.p], gr.ldc[bl.p]};
        return Prob{g.a, g.b, g.c, g.M, g.N, g.lda, g.ldb, g.ldc};
    };

    // ---- fetch side: a stream of slices, tile after tile ----
    uint32_t offa[OA::PER], offb[OB::PER], offa_c[OA::PER], offb_c[OB::PER];
    if (!GROUPED) {  // a grouped launch forms them per tile: the row pitches are the problem's
        lane_offsets<OA>(offa, w, lane, g.lda);
        lane_offsets<OB, GATE>(offb, w, lane, g.ldb, g.N);
    }
    const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds));
    const uint32_t dst_a = lds0 + w * OA::PER * 1024u, dst_b = lds0 + OA::BYTES + w * OB::PER * 1024u;
    Block fb;
    int fv = next_block(static_cast<int>(blockIdx.x), fb);
    if (fv >= V) return;  // nothing for this workgroup (before any barrier)
    TileDesc da, db;
    int f_slice = 0, f_nslices = 0, f_ktail = 0;
    uint32_t soff_a = 0, soff_b = 0;
    auto open = [&]() {  // the fetch stream enters virtual block fv
        f_slice = 0;
        soff_a = soff_b = 0;
        if (fv >= V) {  // past the last block: descriptors stay, every offset goes outside
            f_nslices = 0;
            return;
        }
        f_nslices = (fb.k_end - fb.k_begin + BK - 1) / BK;
        f_ktail = (fb.k_end - fb.k_begin) % BK;
        const Prob fp = prob(fb);
        if (GROUPED) {
            lane_offsets<OA>(offa, w, lane, fp.lda);
            lane_offsets<OB>(offb, w, lane, fp.ldb);
        }
        da = tile_desc<TA>(fp.a, fp.lda, fb.m0, fp.M, fb.k_begin, fb.k_end);
        db = tile_desc<!TB>(fp.b, fp.ldb, fb.n0, GATE ? 2 * fp.N : fp.N, fb.k_begin, fb.k_end);
        // the masked lane offsets: used by every slice of a [k][column] operand, by the last slice of a [row][k] one
        if (TA ? fb.m0 + BM > fp.M : f_ktail != 0)
            lane_offsets_masked<OA, TA>(offa_c, offa, w, lane, fb.m0, fp.M, f_ktail);
        else {
#pragma unroll
            for (int j = 0; j < OA::PER; ++j) offa_c[j] = offa[j];
        }
        if (!TB ? fb.n0 + BNC > fp.N : f_ktail != 0)
            lane_offsets_masked<OB, !TB, GATE>(offb_c, offb, w, lane, fb.n0, fp.N, f_ktail);
        else {
#pragma unroll
            for (int j = 0; j < OB::PER; ++j) offb_c[j] = offb[j];
        }
    };
    // One call per slice of the stream, in order, also past the stream's end: a wavefront's count of loads in flight
    // stays the same, and the scalar offset is then outside every buffer, so nothing is fetched (the lanes write zeros
    // into a slot nobody reads).
    // A slice's loads are issued one by one between the matrix instructions of the slice in hand (all at once they
    // hold a wavefront for 500 clocks in which it issues nothing else, and every wavefront of the workgroup does so at
    // the same time): begin fixes where the slice goes and what it reads, piece<Q> issues its Q-th load, end moves
    // the stream on.
    uint32_t f_la = 0, f_lb = 0, f_sa = 0, f_sb = 0;
    bool f_ca = false, f_cb = false;  // this slice takes the masked lane offsets of A / of B
    auto fetch_begin = [&](int slot) {
        const bool none = f_nslices == 0, last = f_slice == f_nslices - 1;
        f_sa = none ? PAST_END : soff_a;
        f_sb = none ? PAST_END : soff_b;
        f_la = dst_a + static_cast<uint32_t>(slot) * SLOT;
        f_lb = dst_b + static_cast<uint32_t>(slot) * SLOT;
        f_ca = TA || last;
        f_cb = !TB || last;
    };
    auto fetch_piece = [&](auto qc) {
        constexpr int Q = decltype(qc)::value;
        if constexpr (Q < OA::PER) {
            dma_piece<Q, SPILLED ? 3 : 0>(f_la, f_ca ? offa_c[Q] : offa[Q], da.rsrc, f_sa);
        } else if constexpr (Q < PERTOT) {
            constexpr int J = Q - OA::PER;
            dma_piece<J, SPILLED ? 3 : 0>(f_lb, f_cb ? offb_c[J] : offb[J], db.rsrc, f_sb);
        }
    };
    auto fetch_end = [&]() {
        const bool none = f_nslices == 0;
        soff_a += da.step;
        soff_b += db.step;
        if (!none && ++f_slice == f_nslices) {
            fv = next_block(fv + stride, fb);
            open();
        }
    };
    auto fetch = [&](int slot) {  // the whole slice at once (before the first slice is multiplied)
        fetch_begin(slot);
        static_for<0, PERTOT>([&](auto pc) { fetch_piece(pc); });
        fetch_end();
    };

    // ---- lane parts of the fragment reads ----
    // [row][k]: row c32 of a 32-row block, chunk 2 kk + gh, one address per kk (the swizzle is an exclusive-or with a
    // lane value, so kk cannot be an immediate); [k][column]: rows 8 gh + j / 4 (+ 4), columns 16 u + 4 (j % 4) of
    // 32-column block b, one address per block the wavefront reads.
    const int tj = lane & 15, tu = (lane >> 4) & 1;
    uint32_t r_row[KPW], ra_tr[FM], rb_tr[FN];  // r_row: for this wavefront's own k-chunks ks KPW .. ks KPW + KPW - 1
#pragma unroll
    for (int kq = 0; kq < KPW; ++kq)
        r_row[kq] = static_cast<uint32_t>(c32 * 128 + (RingOp<false, 128, 4>::swz(c32, 2 * (ks * KPW + kq) + gh)) * 16);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int blk = wm * FM + i, r = 8 * gh + (tj >> 2);
        ra_tr[i] = static_cast<uint32_t>(r * OA::ROWB + (((blk & ~3) | ((blk & 3) ^ (r & 3))) * 32 + 16 * tu + 4 * (tj & 3)) * 2);
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int blk = wn * FN + j, r = 8 * gh + (tj >> 2);
        rb_tr[j] = static_cast<uint32_t>(r * OB::ROWB + (((blk & ~3) | ((blk & 3) ^ (r & 3))) * 32 + 16 * tu + 4 * (tj & 3)) * 2);
    }
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    auto read_tr = [](const uint8_t* p, int rowb) -> bf16x8 {
        const s16x4 lo = lds_read_tr4(reinterpret_cast<const uint16_t*>(p));
        const s16x4 hi = lds_read_tr4(reinterpret_cast<const uint16_t*>(p + 4 * rowb));
        const s16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        return *reinterpret_cast<const bf16x8*>(&v);
    };
    auto read_a = [&](const uint8_t* As, int i, int kq, int kk) -> bf16x8 {
        if (!TA) return lds_read8(reinterpret_cast<const uint16_t*>(As + r_row[kq] + (wm * FM + i) * 32 * 128));
        return read_tr(As + ra_tr[i] + kk * 16 * OA::ROWB, OA::ROWB);
    };
    auto read_b = [&](const uint8_t* Bs, int j, int kq, int kk) -> bf16x8 {
        if (TB) return lds_read8(reinterpret_cast<const uint16_t*>(Bs + r_row[kq] + (wn * FN + j) * 32 * 128));
        return read_tr(Bs + rb_tr[j] + kk * 16 * OB::ROWB, OB::ROWB);
    };

    // ---- epilogue: lane parts of the stores (tile-relative), formed once ----
    typedef typename std::conditional<CF32, float, uint16_t>::type CT;
    constexpr int ES = CF32 ? 4 : 2;
    const int st_ch = static_cast<int>(threadIdx.x) % ST::CPR;  // the chunk column this thread stores in every strip
    uint32_t coff[ST::PER_PHASE];
#pragma unroll
    for (int k = 0; k < ST::PER_PHASE; ++k) {
        const int srow = (static_cast<int>(threadIdx.x) + k * NTHR) / ST::CPR;
        // bf16 strips hold the i-th 32-row block of every wavefront row: strip row -> tile row (srow / 32) FM 32 + srow % 32
        const int trow = CF32 ? srow : (srow >> 5) * FM * 32 + (srow & 31);
        coff[k] = (static_cast<uint32_t>(trow) * static_cast<uint32_t>(g.ldc) + st_ch * ST::EPC) * ES;  // (not grouped)
    }

    f32x16 acc[FM][FN];
    auto zero_acc = [&]() {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    };
    // lane (c32, gh) holds, of row (wm FM + i) 32 + c32 of the tile, columns (wn FN + j) 32 + 8 qd + 4 gh + e
    auto drop_columns = [&](const Block& bl, int from) {  // columns from there on count for nothing
        const int col0 = bl.n0 + wn * FN * 32 + gh * 4;
        if (bl.n0 + BN <= from) return;  // wavefront-uniform
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (col0 + j * 32 + (r >> 2) * 8 + (r & 3) >= from) acc[i][j][r] = -INFINITY;
    };
    auto head_stats = [&](const Block& bl) {  // EPI 1
        const int span = (bl.n0 / BN) * G::WGN + wn;
        drop_columns(bl, g.N);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int row = bl.m0 + (wm * FM + i) * 32 + c32;
            // the target's place among this lane's 16 FN sums of the row, if it is there: 16 j + r
            const int tt = (row < g.M ? hd.target[row] : -1) - (bl.n0 + wn * FN * 32);
            const bool has = tt >= 0 && tt < FN * 32 && ((tt >> 2) & 1) == gh && row < g.M;
            const int at = has ? (tt >> 5) * 16 + ((tt >> 3) & 3) * 4 + (tt & 3) : -1;
            float mx = -INFINITY, zt = 0.0f;
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    mx = fmaxf(mx, acc[i][j][r]);
                    zt = at == j * 16 + r ? acc[i][j][r] : zt;
                }
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float ref = mx == -INFINITY ? 0.0f : mx * LOG2E;  // a span wholly past the last column sums to 0
            float sum = 0.0f;
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) sum += __builtin_amdgcn_exp2f(fmaf(acc[i][j][r], LOG2E, -ref));
            sum += __shfl_xor(sum, 32);
            if (row < g.M && gh == 0) hd.stats[static_cast<int64_t>(span) * g.M + row] = make_float2(mx, sum);
            if (has) hd.zt[row] = zt;
        }
    };
    auto head_dlogits = [&](const Block& bl) {  // EPI 2, 4: the sums become dlogits where they lie
        // The padding's logits are 0, not in the row's maximum: their exponentials would overflow where every real logit lies
        // far below 0, and dh multiply the infinities with the zero rows that pad B.
        if constexpr (EPI == 4) drop_columns(bl, hd.vocab);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int row = bl.m0 + (wm * FM + i) * 32 + c32;
            const bool in = row < g.M;
            const int tt = (in ? hd.target[row] : -1) - (bl.n0 + wn * FN * 32);
            const bool has = tt >= 0 && tt < FN * 32 && ((tt >> 2) & 1) == gh && in;
            // P gscale = exp2(z log2e - (max log2e - log2(gscale / sum))): the scaling rides in the exponent
            const float ref = in ? fmaf(hd.row_max[row], LOG2E, -__builtin_amdgcn_logf(hd.row_inv[row] * hd.gscale)) : 0.0f;
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = __builtin_amdgcn_exp2f(fmaf(acc[i][j][r], LOG2E, -ref));
            if (__builtin_amdgcn_ballot_w64(has) != 0) {  // few wavefronts hold a target column of one of their rows
                const int at = has ? (tt >> 5) * 16 + ((tt >> 3) & 3) * 4 + (tt & 3) : -1;
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] -= at == j * 16 + r ? hd.gscale : 0.0f;
            }
        }
    };
    // The ends of gated products, strip by strip as below. Gate, up and the gradient count as they are stored, rounded.
    const auto lo = [](uint32_t v) { return __uint_as_float(v << 16); };
    const auto hi = [](uint32_t v) { return __uint_as_float(v & 0xffff0000u); };
    auto write_strip = [&](uint16_t* cs, int i) {
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int qd = 0; qd < 4; ++qd) {
                const u32x2 v = {pack_bf16(acc[i][j][qd * 4], acc[i][j][qd * 4 + 1]), pack_bf16(acc[i][j][qd * 4 + 2], acc[i][j][qd * 4 + 3])};
                *reinterpret_cast<u32x2*>(cs + ST::at(wm * 32 + c32, (wn * FN + j) * 32 + qd * 8 + gh * 4)) = v;
            }
    };
    // descriptor of a [M, ld] matrix from the tile's first element on, `cols` columns from there to the last row's end
    auto tile_rsrc = [&](const void* base, const Block& bl, int64_t ld, int64_t cols) -> u32x4 {
        const uint64_t a = reinterpret_cast<uint64_t>(static_cast<const uint16_t*>(base) + bl.m0 * ld + bl.n0);
        const int64_t left = ((g.M - bl.m0 - 1) * ld + cols) * 2;
        return u32x4{static_cast<uint32_t>(a), static_cast<uint32_t>(a >> 32) & 0xffffu, left > 0x7ffffff0 ? 0x7ffffff0u : static_cast<uint32_t>(left),
                     0x00020000u};
    };
    auto store_gated = [&](const Block& bl) {
        constexpr int GPR = ST::CPR / 2;  // chunks of gate in a strip row; each with its chunk of up four further on
        static_assert(NTHR % GPR == 0 && ST::SR * GPR % NTHR == 0, "one chunk column per thread, whole rounds of rows");
        const int q = static_cast<int>(threadIdx.x) % GPR, cg = (q >> 2) * 8 + (q & 3), col = gated_column(cg);
        const u32x4 to_c = tile_rsrc(g.c, bl, g.N, g.N - bl.n0), to_d = tile_rsrc(g.d, bl, 2 * g.N, 2 * g.N - bl.n0);
        const uint32_t mask = bl.n0 + col < g.N ? 0u : OUTSIDE;
        uint16_t* const cs = reinterpret_cast<uint16_t*>(strip);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            write_strip(cs, i);
            __syncthreads();
            const uint32_t soff = static_cast<uint32_t>(i * 32) * g.N * 2u;
#pragma unroll
            for (int k = 0; k < ST::SR * GPR / NTHR; ++k) {
                const int srow = (static_cast<int>(threadIdx.x) + k * NTHR) / GPR, trow = (srow >> 5) * FM * 32 + (srow & 31);
                const u32x4 gate = *reinterpret_cast<const u32x4*>(cs + ST::at(srow, cg * 8)),
                            up = *reinterpret_cast<const u32x4*>(cs + ST::at(srow, cg * 8 + 32));
                u32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = pack_bf16(gated(lo(gate[e]), lo(up[e])), gated(hi(gate[e]), hi(up[e])));
                const uint32_t row = static_cast<uint32_t>(trow) * g.N * 2u;
                store16(v, (row + col * 2) | mask, to_c, soff);
                if constexpr (EPI == 5) {
                    store16(gate, (2 * row + col * 2) | mask, to_d, 2 * soff);
                    store16(up, (2 * row + col * 2) | mask, to_d, 2 * soff + g.N * 2u);
                }
            }
            __syncthreads();
        }
    };
    auto store_gated_grad = [&](const Block& bl) {
        const u32x4 to_c = tile_rsrc(g.c, bl, 2 * g.N, 2 * g.N - bl.n0), gu = tile_rsrc(g.d, bl, 2 * g.N, 2 * g.N - bl.n0);
        const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint16_t*>(static_cast<const uint16_t*>(g.d) + static_cast<int64_t>(bl.m0) * 2 * g.N + bl.n0), 0, static_cast<int>(gu[2]), 0x00020000);
        const __amdgpu_buffer_rsrc_t to = __builtin_amdgcn_make_buffer_rsrc(static_cast<uint16_t*>(g.c) + static_cast<int64_t>(bl.m0) * 2 * g.N + bl.n0, 0,
                                                                            static_cast<int>(to_c[2]), 0x00020000);
        const uint32_t mask = bl.n0 + st_ch * 8 < g.N ? 0u : OUTSIDE;
        uint16_t* const cs = reinterpret_cast<uint16_t*>(strip);
        // Gate and up of as many strips as the registers hold are on their way before the first store, and the compiler counts the stores: waits for
        // loads are none for stores (8192 x 1376 x 512 38.8 -> 37.6 us).
        constexpr int AHEAD = BM > 128 ? 1 : FM;
        u32x4 gate[AHEAD][ST::PER_PHASE], up[AHEAD][ST::PER_PHASE];
        const auto ask = [&](int i) {
            const uint32_t soff = static_cast<uint32_t>(i * 32) * g.N * 4u, up_at = soff + g.N * 2u;
#pragma unroll
            for (int k = 0; k < ST::PER_PHASE; ++k) {
                gate[i % AHEAD][k] = __builtin_amdgcn_raw_buffer_load_b128(from, static_cast<int>(coff[k] | mask), static_cast<int>(soff), 0);
                up[i % AHEAD][k] = __builtin_amdgcn_raw_buffer_load_b128(from, static_cast<int>(coff[k] | mask), static_cast<int>(up_at), 0);
            }
        };
#pragma unroll
        for (int i = 0; i < AHEAD - 1; ++i) ask(i);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const uint32_t soff = static_cast<uint32_t>(i * 32) * g.N * 4u, up_at = soff + g.N * 2u;
            if (i + AHEAD - 1 < FM) ask(i + AHEAD - 1);
            write_strip(cs, i);
            __syncthreads();
#pragma unroll
            for (int k = 0; k < ST::PER_PHASE; ++k) {
                const int srow = (static_cast<int>(threadIdx.x) + k * NTHR) / ST::CPR;
                const u32x4 d = *reinterpret_cast<const u32x4*>(cs + ST::at(srow, st_ch * 8));
                u32x4 dg, du;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float a[2], b[2];
                    gated_grad(lo(gate[i % AHEAD][k][e]), lo(up[i % AHEAD][k][e]), lo(d[e]), a[0], b[0]);
                    gated_grad(hi(gate[i % AHEAD][k][e]), hi(up[i % AHEAD][k][e]), hi(d[e]), a[1], b[1]);
                    dg[e] = pack_bf16(a[0], a[1]);
                    du[e] = pack_bf16(b[0], b[1]);
                }
                store16_counted(dg, coff[k] | mask, to, soff);
                store16_counted(du, coff[k] | mask, to, up_at);
            }
            __syncthreads();
        }
    };
    // The product counts as it is stored, rounded. Cosines and sines of all chunks' four pairs are asked for before the first store, behind
    // which they would wait.
    auto store_turned = [&](const Block& bl) {
        const u32x4 to_c = tile_rsrc(g.c, bl, g.N, g.N - bl.n0);
        const int col = bl.n0 + st_ch * 8, pair = max(turned_pair(hd.turn, col), 0), base = bl.m0 - quotient(bl.m0, hd.turn.seq_len) * hd.turn.seq_len;
        const bool turns = turned_pair(hd.turn, col) >= 0;
        const uint32_t mask = col < g.N ? 0u : OUTSIDE;
        uint16_t* const cs = reinterpret_cast<uint16_t*>(strip);
        f32x4 by[FM][ST::PER_PHASE][2];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int k = 0; k < ST::PER_PHASE; ++k) {
                const int srow = (static_cast<int>(threadIdx.x) + k * NTHR) / ST::CPR;
                const int at = turned_position<BM>(hd.turn, base, (srow >> 5) * FM * 32 + (srow & 31) + i * 32);
                const f32x4* const p = reinterpret_cast<const f32x4*>(hd.turn.table + (static_cast<int64_t>(at) * (hd.turn.head_dim / 2) + pair) * 2);
                by[i][k][0] = p[0], by[i][k][1] = p[1];
            }
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            write_strip(cs, i);
            __syncthreads();
            const uint32_t soff = static_cast<uint32_t>(i * 32) * g.N * 2u;
#pragma unroll
            for (int k = 0; k < ST::PER_PHASE; ++k) {
                const int srow = (static_cast<int>(threadIdx.x) + k * NTHR) / ST::CPR;
                u32x4 v = *reinterpret_cast<const u32x4*>(cs + ST::at(srow, st_ch * 8));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x0 = lo(v[e]), x1 = hi(v[e]), c = by[i][k][e / 2][e % 2 * 2], s = by[i][k][e / 2][e % 2 * 2 + 1];
                    const uint32_t t = pack_bf16(x0 * c - x1 * s, x0 * s + x1 * c);
                    v[e] = turns ? t : v[e];
                }
                store16(v, coff[k] | mask, to_c, soff);
            }
            __syncthreads();
        }
    };
    // The tile's result, through the strip. One body adds and one does not: with a condition around the loads and another around their use the
    // compiler also waits for them in the contraction (two wavefront sets: a third longer).
    auto store_result_as = [&](auto adding, const Block& bl) {
        constexpr bool adds = decltype(adding)::value;
        // descriptor of C from the tile's first element on (rows past the matrix are dropped by the range check,
        // columns past it by the lane's offset)
        const Prob cp = prob(bl);
        CT* ctile = static_cast<CT*>(cp.c) + (g.part_stride ? static_cast<int64_t>(bl.z) * g.part_stride : 0) +
                    static_cast<int64_t>(bl.m0) * cp.ldc + bl.n0;
        const int64_t cleft = (static_cast<int64_t>(cp.M - bl.m0 - 1) * cp.ldc + (cp.N - bl.n0)) * ES;
        const uint32_t crec = cleft > 0x7ffffff0 ? 0x7ffffff0u : static_cast<uint32_t>(cleft);
        const uint64_t ca = reinterpret_cast<uint64_t>(ctile);
        const u32x4 crs = {static_cast<uint32_t>(ca), static_cast<uint32_t>(ca >> 32) & 0xffffu, crec, 0x00020000u};
        CT* dtile = g.d ? static_cast<CT*>(const_cast<void*>(g.d)) + static_cast<int64_t>(bl.m0) * cp.ldc + bl.n0 : ctile;
        const __amdgpu_buffer_rsrc_t crs_b = __builtin_amdgcn_make_buffer_rsrc(dtile, 0, static_cast<int>(crec), 0x00020000);
        const __amdgpu_buffer_rsrc_t crs_c = __builtin_amdgcn_make_buffer_rsrc(ctile, 0, static_cast<int>(crec), 0x00020000);
        const uint32_t cmask = bl.n0 + st_ch * ST::EPC < cp.N ? 0u : OUTSIDE;
        // What the product is added to: asked for AHEAD stores ahead, and the sums stored where the compiler counts them. Asked for in front of
        // each store it is a round trip to memory 8 to 32 times a tile, and each waits for the store before it as well. In a d 512 model of 8192 tokens:
        // the tied head's [32000, 512] += over 4096 rows 123.6 -> 114.0 us, a block's weight gradients 77.2 -> 74.1, the products that end in a
        // residual 14.25 -> 12.9.
        const auto place = [&](int k) -> uint32_t {
            if (!GROUPED) return coff[k] | cmask;
            const int srow = (static_cast<int>(threadIdx.x) + k * NTHR) / ST::CPR, trow = CF32 ? srow : (srow >> 5) * FM * 32 + (srow & 31);
            return ((static_cast<uint32_t>(trow) * static_cast<uint32_t>(cp.ldc) + st_ch * ST::EPC) * ES) | cmask;  // the row pitch is the problem's
        };
        // rows of C that a strip holds start at tile row (ws FM + i) 32 (fp32) or i 32 (bf16, plus the lane's part)
        const auto strip_at = [&](int ph) { return static_cast<uint32_t>((CF32 ? ph % G::WGM * FM + ph / G::WGM : ph) * 32) * static_cast<uint32_t>(cp.ldc) * ES; };
        constexpr int FIT = BM == 128 ? 8 : !CF32 ? 4 : TA && TB ? 2 : 3, AHEAD = FIT < ST::NST ? FIT : ST::NST;  // what the registers hold
        u32x4 old[AHEAD];
        const auto ask = [&](int q) {
            old[q % AHEAD] =
                __builtin_amdgcn_raw_buffer_load_b128(crs_b, static_cast<int>(place(q % ST::PER_PHASE)), static_cast<int>(strip_at(q / ST::PER_PHASE)), 0);
        };
        if constexpr (adds) {
#pragma unroll
            for (int q = 0; q < AHEAD; ++q) ask(q);
        }
        if (KS == 2) {  // set 1 hands its sums to set 0, half of them at a time: [wavefront][16-byte group][lane]
            f32x4* red = reinterpret_cast<f32x4*>(strip) + wq * ((FM / 2) * FN * 4) * 64 + lane;
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                if (ks == 1) {
#pragma unroll
                    for (int i = 0; i < FM / 2; ++i)
#pragma unroll
                        for (int j = 0; j < FN; ++j)
#pragma unroll
                            for (int qd = 0; qd < 4; ++qd) {
                                const f32x16& a = acc[half * (FM / 2) + i][j];
                                const f32x4 v = {a[qd * 4], a[qd * 4 + 1], a[qd * 4 + 2], a[qd * 4 + 3]};
                                red[((i * FN + j) * 4 + qd) * 64] = v;
                            }
                }
                __syncthreads();
                if (ks == 0) {
#pragma unroll
                    for (int i = 0; i < FM / 2; ++i)
#pragma unroll
                        for (int j = 0; j < FN; ++j)
#pragma unroll
                            for (int qd = 0; qd < 4; ++qd) {
                                const f32x4 v = red[((i * FN + j) * 4 + qd) * 64];
#pragma unroll
                                for (int e = 0; e < 4; ++e) acc[half * (FM / 2) + i][j][qd * 4 + e] += v[e];
                            }
                }
                __syncthreads();
            }
        }
        CT* cs = reinterpret_cast<CT*>(strip);
#pragma unroll
        for (int ph = 0; ph < ST::PHASES; ++ph) {
            const int i = CF32 ? ph / G::WGM : ph, ws = CF32 ? ph % G::WGM : 0;
            if (ks == 0 && (!CF32 || wm == ws)) {  // wavefront-uniform: the wavefronts that hold this strip's sums
#pragma unroll
                for (int j = 0; j < FN; ++j)
#pragma unroll
                    for (int qd = 0; qd < 4; ++qd) {
                        const int row = (CF32 ? 0 : wm * 32) + c32, col = (wn * FN + j) * 32 + qd * 8 + gh * 4;
                        if (CF32) {
                            const f32x4 v = {acc[i][j][qd * 4], acc[i][j][qd * 4 + 1], acc[i][j][qd * 4 + 2], acc[i][j][qd * 4 + 3]};
                            *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(cs) + ST::at(row, col)) = v;
                        } else {
                            const u32x2 v = {pack_bf16(acc[i][j][qd * 4], acc[i][j][qd * 4 + 1]),
                                             pack_bf16(acc[i][j][qd * 4 + 2], acc[i][j][qd * 4 + 3])};
                            *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(cs) + ST::at(row, col)) = v;
                        }
                    }
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < ST::PER_PHASE; ++k) {
                u32x4 v = *reinterpret_cast<const u32x4*>(cs + ST::at((static_cast<int>(threadIdx.x) + k * NTHR) / ST::CPR, st_ch * ST::EPC));
                if constexpr (adds) {
                    const int q = ph * ST::PER_PHASE + k;
                    const u32x4 o = old[q % AHEAD];
                    if (CF32) {
                        const f32x4 sum = *reinterpret_cast<const f32x4*>(&o) + *reinterpret_cast<const f32x4*>(&v);
                        v = *reinterpret_cast<const u32x4*>(&sum);
                    } else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) v[e] = pack_bf16(lo(o[e]) + lo(v[e]), hi(o[e]) + hi(v[e]));
                    }
                    if (q + AHEAD < ST::NST) ask(q + AHEAD);
                    store16_counted(v, place(k), crs_c, strip_at(ph));
                } else {
                    store16<SPILLED>(v, place(k), crs, strip_at(ph));
                }
            }
            __syncthreads();
        }
    };
    auto store_result = [&](const Block& bl) {
        if ((EPI == 0 || EPI == 3) && g.beta)
            store_result_as(std::integral_constant<bool, EPI == 0 || EPI == 3>{}, bl);
        else
            store_result_as(std::false_type{}, bl);
    };

    // ---- the stream ----
    // Rotated by a k-chunk: a chunk's matrix instructions run while the next chunk's fragments are read, and a slice's last chunk runs
    // behind the barrier that hands out the next slice, whose first fragments are read meanwhile and whose slot's successor is asked
    // for (half of its loads there, half beside the next slice's first chunk). Left to itself the compiler reads a chunk's fragments
    // right in front of its matrix instructions, and a barrier drains both wavefronts of a SIMD. Microseconds so | now, whole launches:
    // 4096^3 115 | 103, [32000, 512] over 4096 137 | 132, [4096, 512] over 32000 134 | 124, the head's first pass over 4096 x 32000 x 512
    // 134 | 126, [8192, 1536] over 512 20.1 | 19.5. What is left is the loads' way into LDS and the clock: without them 4096^3 takes 82,
    // with operands of zeros (no lower clock) 77, without the fragment reads 103 to 111. Not ahead: 256 x 256 tiles of four wavefronts,
    // 128 x 128 each (half the fragment reads: level), slices of 32 in rings of 3 and 4 slots (117 | 107).
    constexpr int NF = FM + FN, NM = FM * FN, HALF = PERTOT / 2;
    static_assert(KPW % 2 == 0, "fragments of even and odd chunks in registers of their own");
    bf16x8 fra[2][FM], frb[2][FN];
    auto read_frag = [&](auto qc, auto kqc, const uint8_t* As) {  // fragment Q of chunk KQ, in the order the matrix instructions need them
        constexpr int Q = decltype(qc)::value, KQ = decltype(kqc)::value, L = FM < FN ? FM : FN;
        const uint8_t* Bs = As + OA::BYTES;
        const int kk = ks * KPW + KQ;
        if constexpr (Q < 2 * L && Q % 2 == 0)
            frb[KQ & 1][Q / 2] = read_b(Bs, Q / 2, KQ, kk);
        else if constexpr (Q < 2 * L)
            fra[KQ & 1][Q / 2] = read_a(As, Q / 2, KQ, kk);
        else if constexpr (FM > FN)
            fra[KQ & 1][Q - L] = read_a(As, Q - L, KQ, kk);
        else
            frb[KQ & 1][Q - L] = read_b(Bs, Q - L, KQ, kk);
    };
    // the matrix instructions of chunk KQ, each behind a fragment of chunk KN (of the slice at `next`) and before a load of its share
    auto chunk = [&](auto kqc, auto knc, const uint8_t* next, auto first, auto count) {
        constexpr int KQ = decltype(kqc)::value, F = decltype(first)::value, N = decltype(count)::value;
        static_for<0, NM>([&](auto mc) {
            constexpr int Q = decltype(mc)::value, PERQ = (NF + NM - 1) / NM;
            static_for<Q * PERQ, (Q + 1) * PERQ < NF ? (Q + 1) * PERQ : NF>([&](auto fc) { read_frag(fc, knc, next); });
            acc[Q / FN][Q % FN] = mfma32(frb[KQ & 1][Q % FN], fra[KQ & 1][Q / FN], acc[Q / FN][Q % FN]);
            static_for<F + Q * N / NM, F + (Q + 1) * N / NM>([&](auto pc) { fetch_piece(pc); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    const auto keep_here = []() { asm volatile("" ::: "memory"); };  // reads above are not to move behind the branch below
    open();
    {
        int slot = 0;
        for (int s = 0; s < NS - 1; ++s) fetch(slot++);
    }
    fetch_begin(NS - 1);
    static_for<0, HALF>([&](auto pc) { fetch_piece(pc); });
    Block cb;  // compute side: the block in hand
    int cv = next_block(static_cast<int>(blockIdx.x), cb);
    int c_slice = 0, c_nslices = (cb.k_end - cb.k_begin + BK - 1) / BK;
    int since_store = NS;  // waits since the last tile's stores were issued; below NS - 2 they are still counted
    zero_acc();
    wait_loads<(NS - 2) * PERTOT + HALF>();
    barrier();
    static_for<0, NF>([&](auto fc) { read_frag(fc, std::integral_constant<int, 0>{}, lds); });
    for (;;) {
        bool done = false;
#pragma unroll
        for (int u = 0; u < NS; ++u) {
            const uint8_t* const slice = lds + u * SLOT;
            // the second half of the loads that the slice before began
            chunk(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{}, slice, std::integral_constant<int, HALF>{},
                  std::integral_constant<int, PERTOT - HALF>{});
            keep_here();
            fetch_end();
            static_for<1, KPW - 1>([&](auto kc) {
                constexpr int KQ = decltype(kc)::value;
                chunk(kc, std::integral_constant<int, KQ + 1>{}, slice, std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{});
            });
            // The next slice landed: everything this wavefront issued after that slice's loads may still be in flight -- the loads of
            // NS - 2 later slices and, for the slices asked for before the last tile's stores, those stores (memory operations
            // complete in order). This slice's last fragments are in registers, so behind the barrier its slot is free.
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (NS > 2 && since_store < NS - 2)
                wait_loads<(NS - 2) * PERTOT + NST>();
            else
                wait_loads<(NS - 2) * PERTOT>();
            since_store = min(since_store + 1, NS);
            barrier();
            fetch_begin(u);
            chunk(std::integral_constant<int, KPW - 1>{}, std::integral_constant<int, 0>{}, lds + (u + 1) % NS * SLOT, std::integral_constant<int, 0>{},
                  std::integral_constant<int, HALF>{});
            keep_here();
            if (++c_slice == c_nslices) {  // wavefront-uniform
                if constexpr (EPI == 1) {
                    head_stats(cb);
                } else {
                    if constexpr (EPI == 2 || EPI == 4) head_dlogits(cb);
                    if constexpr (GATE)
                        store_gated(cb);
                    else if constexpr (GATE_GRAD)
                        store_gated_grad(cb);
                    else if (TURN && (cb.n0 < hd.turn.cols || (cb.n0 < hd.turn.d + hd.turn.cols && cb.n0 + BN > hd.turn.d)))
                        store_turned(cb);
                    else
                        store_result(cb);
                    since_store = 0;
                }
                // the next slice's first fragments once more, not kept over the end of a tile whose gate and up take their registers
                if constexpr (GATE_GRAD && BM > 128)
                    static_for<0, NF>([&](auto fc) { read_frag(fc, std::integral_constant<int, 0>{}, lds + (u + 1) % NS * SLOT); });
                cv = next_block(cv + stride, cb);
                if (cv >= V) {
                    done = true;
                    break;
                }
                c_slice = 0;
                c_nslices = (cb.k_end - cb.k_begin + BK - 1) / BK;
                zero_acc();
            }
        }
        if (done) break;
    }
    wait_loads<0>();  // the zero-filling loads past the end write LDS: they must have landed before the workgroup ends
}

__global__ void sum_slices(const float* part, void* dst, int nparts, int64_t part_stride, int M, int N, int64_t ldc, int beta,
                           int c_f32) {
    const int64_t n4 = static_cast<int64_t>(M) * N / 4;
    for (int64_t i = blockIdx.x * 256LL + threadIdx.x; i < n4; i += static_cast<int64_t>(gridDim.x) * 256) {
        const int64_t e = i * 4, m = e / N, n = e % N;
        f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int p = 0; p < nparts; ++p) s += *reinterpret_cast<const f32x4*>(part + p * part_stride + e);
        if (c_f32) {
            f32x4* d = reinterpret_cast<f32x4*>(static_cast<float*>(dst) + m * ldc + n);
            *d = beta ? *d + s : s;
        } else {
            u32x2* d = reinterpret_cast<u32x2*>(static_cast<uint16_t*>(dst) + m * ldc + n);
            if (beta) {
                const u32x2 o = *d;
                s[0] += __uint_as_float(o[0] << 16);
                s[1] += __uint_as_float(o[0] & 0xffff0000u);
                s[2] += __uint_as_float(o[1] << 16);
                s[3] += __uint_as_float(o[1] & 0xffff0000u);
            }
            const u32x2 v = {pack_bf16(s[0], s[1]), pack_bf16(s[2], s[3])};
            *d = v;
        }
    }
}

// Joins a row's span statistics of the head's first pass, in span order: the row's maximum M, 1 / sum_j exp(z_j - M)
// and its loss -log(max(P_target, 1e-12)) (src/ops.cpp:360-368). 16 rows x 16 groups of spans per block.
__global__ __launch_bounds__(256) void head_rows(const float2* stats, const float* zt, int spans, int M, float* row_max,
                                                 float* row_inv, float* nll) {
    __shared__ float sh_m[16][16], sh_s[16][16];
    const int lr = threadIdx.x & 15, grp = threadIdx.x >> 4, r = blockIdx.x * 16 + lr;
    auto join = [](float& m, float& s, float m2, float s2) {
        const float nm = fmaxf(m, m2), ref = nm == -INFINITY ? 0.0f : nm;
        s = s * __builtin_amdgcn_exp2f((m - ref) * LOG2E) + s2 * __builtin_amdgcn_exp2f((m2 - ref) * LOG2E);
        m = nm;
    };
    float m = -INFINITY, s = 0.0f;
    if (r < M) {
        int p = grp;
        for (; p + 48 < spans; p += 64) {  // four loads in flight, joined in span order
            float2 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = stats[static_cast<int64_t>(p + 16 * u) * M + r];
#pragma unroll
            for (int u = 0; u < 4; ++u) join(m, s, v[u].x, v[u].y);
        }
        for (; p < spans; p += 16) {
            const float2 v = stats[static_cast<int64_t>(p) * M + r];
            join(m, s, v.x, v.y);
        }
    }
    sh_m[grp][lr] = m;
    sh_s[grp][lr] = s;
    __syncthreads();
    if (grp == 0 && r < M) {
        for (int q = 1; q < 16; ++q) join(m, s, sh_m[q][lr], sh_s[q][lr]);
        const float inv = 1.0f / s;
        row_max[r] = m;
        row_inv[r] = inv;
        nll[r] = -logf(fmaxf(__builtin_amdgcn_exp2f((zt[r] - m) * LOG2E) * inv, 1e-12f));
    }
}

template <typename G, bool CF32>
void launch_form(bool tA, bool tB, const GemmArgs& g, dim3 grid, hipStream_t st) {
    if (!tA && !tB) hipLaunchKernelGGL((gemm_bf16<G, false, false, CF32>), grid, dim3(G::NTHR), 0, st, g);
    if (!tA && tB) hipLaunchKernelGGL((gemm_bf16<G, false, true, CF32>), grid, dim3(G::NTHR), 0, st, g);
    if (tA && !tB) hipLaunchKernelGGL((gemm_bf16<G, true, false, CF32>), grid, dim3(G::NTHR), 0, st, g);
    if (tA && tB) hipLaunchKernelGGL((gemm_bf16<G, true, true, CF32>), grid, dim3(G::NTHR), 0, st, g);
}
template <typename G, bool CF32, int NS>
void launch_ring_form(bool tA, bool tB, const GemmArgs& g, dim3 grid, hipStream_t st) {
    if (!tA && !tB) hipLaunchKernelGGL((gemm_ring<G, false, false, CF32, NS>), grid, dim3(G::NTHR), 0, st, g, HeadArgs{}, GroupArgs{});
    if (!tA && tB) hipLaunchKernelGGL((gemm_ring<G, false, true, CF32, NS>), grid, dim3(G::NTHR), 0, st, g, HeadArgs{}, GroupArgs{});
    if (tA && !tB) hipLaunchKernelGGL((gemm_ring<G, true, false, CF32, NS>), grid, dim3(G::NTHR), 0, st, g, HeadArgs{}, GroupArgs{});
    if (tA && tB) hipLaunchKernelGGL((gemm_ring<G, true, true, CF32, NS>), grid, dim3(G::NTHR), 0, st, g, HeadArgs{}, GroupArgs{});
}
int cu_count() {
    static const int n = [] {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            cus <= 0)
            return 256;
        return cus;
    }();
    return n;
}
template <typename G, int NS>
void launch_ring(bool tA, bool tB, GemmArgs g, int S, bool c_f32, hipStream_t st) {
    g.tiles_m = (g.M + G::BM - 1) / G::BM;
    g.tiles_n = (g.N + G::BN - 1) / G::BN;
    g.splits = S;
    // persistent: as many workgroups as the chip holds at once (a multiple of 8, one XCD's share each), or fewer
    const int64_t vblocks = (static_cast<int64_t>(g.tiles_m) * g.tiles_n * S + 7) / 8 * 8;
    const int64_t slots = static_cast<int64_t>(cu_count()) / 8 * 8 * RingLds<G, NS>::PER_CU;
    const unsigned gx = static_cast<unsigned>(std::min(vblocks, slots));
    if (c_f32)
        launch_ring_form<G, true, NS>(tA, tB, g, dim3(gx), st);
    else
        launch_ring_form<G, false, NS>(tA, tB, g, dim3(gx), st);
    hip_check(hipGetLastError(), "gemm_ring launch");
}
template <typename G>
void launch_geo(bool tA, bool tB, GemmArgs g, int S, bool c_f32, hipStream_t st) {
    g.tiles_m = (g.M + G::BM - 1) / G::BM;
    g.tiles_n = (g.N + G::BN - 1) / G::BN;
    const unsigned gx = static_cast<unsigned>((g.tiles_m * g.tiles_n + 7) / 8 * 8);
    if (c_f32)
        launch_form<G, true>(tA, tB, g, dim3(gx, 1, static_cast<unsigned>(S)), st);
    else
        launch_form<G, false>(tA, tB, g, dim3(gx, 1, static_cast<unsigned>(S)), st);
    hip_check(hipGetLastError(), "gemm_bf16 launch");
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

int g_force_geo = -1;  // -1: choose by shape; 0 / 1: small / large tiles always (measurement)

}  // namespace

void gemm_mfma_force_tiles(int which) { g_force_geo = which; }

namespace {
// How a product is run: tile geometry and kernel form, and into how many slices the contraction is cut.
struct Plan {
    bool large;  // 256 x 256 tiles
    int ring;    // 0: gemm_bf16 (register-staged tiles); otherwise a gemm_ring form (the numbers of pk_set_gemm_backend)
    int S;       // slices of the contraction, each multiplied into an fp32 partial product of its own
    int kps;     // contraction elements per slice (a multiple of BK)
};
Plan make_plan(bool tA, bool tB, int64_t M, int64_t N, int64_t K, int64_t lda, int64_t ldb, int64_t ldc) {
    Plan p;
    // Which tiles (measured on the Linear shapes of a d = 512 block and of a 32000-word tied head). 256 x 256 where
    // the output gives nearly every CU a tile of its own and the contraction is long enough to pay for the larger
    // prologue, or where there are tiles for two rounds; 128 x 128 otherwise, two workgroups per CU -- except that an
    // output of at most one such tile per CU with a long contraction takes the two-set form with a deep ring, since
    // no second workgroup would come to share the CU.
    const int64_t tiles_large = ((M + 255) / 256) * ((N + 255) / 256);
    p.large = g_force_geo >= 0 ? (g_force_geo == 1 || g_force_geo == 8) : tiles_large >= 240 && (K >= 1024 || tiles_large >= 512);
    int64_t ntiles = p.large ? tiles_large : ((M + 127) / 128) * ((N + 127) / 128);
    // the ring kernels keep offsets and extents in 32 bits
    const int64_t ext_a = (tA ? K : M) * lda * 2, ext_b = (tB ? N : K) * ldb * 2;
    const int64_t ext_max = (int64_t{1} << 30) - 8192;
    const bool ring_ok = ext_a < ext_max && ext_b < ext_max && lda < (1 << 21) && ldb < (1 << 21) && ldc < (1 << 20);
    p.ring = 0;
    if (ring_ok && g_force_geo >= 5) p.ring = g_force_geo;
    if (ring_ok && g_force_geo < 0) p.ring = p.large ? 8 : (ntiles <= 256 && K >= 1024) ? 11 : 6;
    // Split the contraction when the tiles alone would leave most of the chip idle and the contraction is long: as
    // many slices as give every workgroup the chip holds at once one (tile, slice) -- a second round costs more than
    // longer slices -- but none shorter than 1024, since every slice is another partial product to write and add
    // (measured on [512, 1536], [512, 512], [512, 2752] and [1376, 512] outputs over 8192 tokens and on
    // [2048, 512] over 32000). Split products take 128 x 128 tiles: fewer than 64 of them in the two-set form, one
    // workgroup of eight wavefronts per CU, otherwise two workgroups of four per CU.
    p.S = 1;
    if (ntiles < 192 && K >= 2048) {
        if (ring_ok && g_force_geo < 0) p.ring = ntiles < 64 ? 11 : 6;
        // ... unless 256 x 256 tiles times slices of 1024 or more fill the chip by themselves (dh of a 4096-row head
        // chunk, [4096, 512] over 32000: 144 us against 162)
        const int64_t s_large = std::min<int64_t>({cu_count() / tiles_large, K / 1024, 16});
        if (ring_ok && g_force_geo < 0 && tiles_large * s_large >= 240) {
            p.large = true;
            p.ring = 8;
            ntiles = tiles_large;
        }
        const bool one_per_cu = p.ring == 5 || p.ring == 7 || p.ring == 8 || p.ring == 10 || p.ring == 11;
        const int64_t s = std::min<int64_t>({(one_per_cu ? cu_count() : 2 * cu_count()) / ntiles, K / 1024, 16});
        p.S = static_cast<int>(std::max<int64_t>(s, 1));
    }
    p.kps = static_cast<int>(((K + p.S - 1) / p.S + BK - 1) / BK * BK);
    p.S = static_cast<int>((K + p.kps - 1) / p.kps);
    return p;
}
void run_plan(const Plan& p, bool tA, bool tB, const GemmArgs& ga, int splits, bool f32, hipStream_t st) {
    switch (p.ring) {
        case 5: launch_ring<GeoSmall, 4>(tA, tB, ga, splits, f32, st); break;
        case 6: launch_ring<GeoSmall, 2>(tA, tB, ga, splits, f32, st); break;
        case 7: launch_ring<GeoSmall, 3>(tA, tB, ga, splits, f32, st); break;
        case 8: launch_ring<GeoLarge, 2>(tA, tB, ga, splits, f32, st); break;
        case 9: launch_ring<GeoSmallK2, 2>(tA, tB, ga, splits, f32, st); break;
        case 10: launch_ring<GeoSmallK2, 3>(tA, tB, ga, splits, f32, st); break;
        case 11: launch_ring<GeoSmallK2, 4>(tA, tB, ga, splits, f32, st); break;
        default:
            if (p.large)
                launch_geo<GeoLarge>(tA, tB, ga, splits, f32, st);
            else
                launch_geo<GeoSmall>(tA, tB, ga, splits, f32, st);
    }
}
bool takes(const void* a, bool tA, int64_t lda, const void* b, bool tB, int64_t ldb, int64_t M, int64_t N, int64_t K,
           bool any_n = false) {
    if (M <= 0 || N <= 0 || K <= 0 || M > (1 << 30) || N > (1 << 30) || K > (1 << 30)) return false;
    if (!aligned16(a) || !aligned16(b)) return false;
    if (lda % 8 || ldb % 8 || (N % 8 && !any_n)) return false;
    // a contraction that runs along a row of either operand is read in 16-byte chunks; where it is the row index of both
    // (a weight gradient over the tokens) rows past its end read as zeros and any length goes
    return K % 8 == 0 || (tA && !tB);  // A^T is read in chunks along M, which end inside its rows' pitch
}
GemmArgs gemm_args(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K) {
    GemmArgs g;
    g.a = static_cast<const uint16_t*>(a);
    g.b = static_cast<const uint16_t*>(b);
    g.c = nullptr;
    g.M = static_cast<int>(M), g.N = static_cast<int>(N), g.K = static_cast<int>(K);
    g.lda = lda, g.ldb = ldb, g.ldc = N;
    g.beta = 0;
    g.d = nullptr;
    g.k_per_split = g.K;
    g.part_stride = 0;
    g.tiles_m = g.tiles_n = 0;
    g.splits = 1;
    return g;
}
}  // namespace

// Returns false, having done nothing, for what the kernel does not take (fp32 operands, unaligned rows, sizes
// that are not multiples of 8): the caller then uses the library GEMM.
bool gemm_mfma_bf16(const void* a, bool tA, int64_t lda, const void* b, bool tB, int64_t ldb, void* c, int c_dtype,
                    int64_t M, int64_t N, int64_t K, int64_t ldc, float beta, hipStream_t st, const void* addend) {
    if (beta != 0.0f && beta != 1.0f) return false;
    if (g_force_geo < 0 && gemm_small_is_ahead(tA, tB, M, N, K)) {
        const SmallProduct p{a, lda, b, ldb, c, ldc, addend, M, N, K};
        if (gemm_small(&p, 1, tA, tB, c_dtype, addend ? 0.0f : beta, st)) return true;
    }
    if (!takes(a, tA, lda, b, tB, ldb, M, N, K) || !aligned16(c) || ldc % 8) return false;
    GemmArgs g = gemm_args(a, lda, b, ldb, M, N, K);
    g.c = c;
    g.ldc = ldc;
    g.beta = beta != 0.0f;
    const Plan p = make_plan(tA, tB, M, N, K, lda, ldb, ldc);
    if (addend) {  // C = addend + product: in the epilogue of the ring kernels, whole contractions only
        if (beta != 1.0f || !aligned16(addend) || p.ring == 0 || p.S != 1) return false;
        g.d = addend;
    }
    if (p.S == 1) {
        run_plan(p, tA, tB, g, 1, c_dtype == PK_F32, st);
        return true;
    }
    Buffer part(sizeof(float) * static_cast<size_t>(p.S) * M * N);
    GemmArgs gp = g;
    gp.c = part.p;
    gp.ldc = N;
    gp.beta = 0;
    gp.k_per_split = p.kps;
    gp.part_stride = M * N;
    run_plan(p, tA, tB, gp, p.S, true, st);
    const int64_t n4 = M * N / 4;
    hipLaunchKernelGGL(sum_slices, dim3(static_cast<unsigned>(std::min<int64_t>((n4 + 255) / 256, 4096))), dim3(256), 0, st,
                       static_cast<const float*>(part.p), c, p.S, M * N, static_cast<int>(M), static_cast<int>(N), ldc,
                       g.beta, c_dtype == PK_F32 ? 1 : 0);
    hip_check(hipGetLastError(), "sum_slices launch");
    return true;
}

// The same product left as its fp32 partial products part[s][M][N], s < nparts (one where the contraction is not
// cut), for a caller that adds them itself on the way to where the result goes.
bool gemm_mfma_bf16_parts(const void* a, bool tA, int64_t lda, const void* b, bool tB, int64_t ldb, int64_t M, int64_t N,
                          int64_t K, hipStream_t st, std::unique_ptr<Buffer>& part, int& nparts) {
    if (!takes(a, tA, lda, b, tB, ldb, M, N, K)) return false;
    const Plan p = make_plan(tA, tB, M, N, K, lda, ldb, N);
    part.reset(new Buffer(sizeof(float) * static_cast<size_t>(p.S) * M * N));
    GemmArgs g = gemm_args(a, lda, b, ldb, M, N, K);
    g.c = part->p;
    g.k_per_split = p.kps;
    g.part_stride = p.S > 1 ? M * N : 0;
    run_plan(p, tA, tB, g, p.S, true, st);
    nparts = p.S;
    return true;
}

// ---- the tied head's cross-entropy inside its logits product ----
namespace {
bool head_takes(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K) {
    if (!takes(a, false, lda, b, true, ldb, M, N, K, true)) return false;
    const int64_t ext_max = (int64_t{1} << 30) - 8192;
    return M * lda * 2 < ext_max && N * ldb * 2 < ext_max && lda < (1 << 21) && ldb < (1 << 21) && N < (1 << 20);
}
template <typename G, int EPI>
void launch_head(GemmArgs g, const HeadArgs& hd, hipStream_t st) {
    g.tiles_m = (g.M + G::BM - 1) / G::BM;
    g.tiles_n = (g.N + G::BN - 1) / G::BN;
    g.splits = 1;
    const int64_t vblocks = static_cast<int64_t>((g.tiles_m * g.tiles_n + 7) / 8 * 8);
    const int64_t slots = cu_count() / 8 * 8 * (G::BM > 128 ? 1 : 2);
    const unsigned gx = static_cast<unsigned>(std::min<int64_t>(vblocks, slots));
    hipLaunchKernelGGL((gemm_ring<G, false, true, false, 2, EPI>), dim3(gx), dim3(G::NTHR), 0, st, g, hd, GroupArgs{});
    hip_check(hipGetLastError(), "gemm_ring (head) launch");
}
}  // namespace

// 256 x 256 tiles, one workgroup of eight wavefronts per CU (128 x 128 tiles with two workgroups per CU, whose
// epilogues could overlap each other's matrix work, measured 15 % slower on [2048, 32000] x 512), unless those are fewer
// than three quarters of the CUs.
namespace {
bool head_small(int64_t M, int64_t N) {
    return ((M + GeoLarge::BM - 1) / GeoLarge::BM) * ((N + GeoLarge::BN - 1) / GeoLarge::BN) < cu_count() * 3 / 4;
}
}  // namespace
bool gemm_head_takes(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K) {
    return head_takes(a, lda, b, ldb, M, N, K);
}
int64_t gemm_head_spans(int64_t M, int64_t N) {
    return head_small(M, N) ? (N + GeoSmall::BN - 1) / GeoSmall::BN * GeoSmall::WGN : (N + GeoLarge::BN - 1) / GeoLarge::BN * GeoLarge::WGN;
}

// Pass 1 over logits = A B^T (A [M, K] and B [N, K], bf16), which are formed tile by tile and never stored: per row
// its maximum, 1 / sum exp(z - maximum) and its loss against target[row]. `stats` is scratch of gemm_head_spans(M, N) * M
// pairs of floats, `zt` of M floats. False, with nothing done, for operands the kernel does not take.
bool gemm_head_rows(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K, const int* target,
                    void* stats, float* zt, float* row_max, float* row_inv, float* nll, hipStream_t st) {
    if (!head_takes(a, lda, b, ldb, M, N, K)) return false;
    GemmArgs g = gemm_args(a, lda, b, ldb, M, N, K);
    HeadArgs hd{};
    hd.target = target;
    hd.stats = static_cast<float2*>(stats);
    hd.zt = zt;
    head_small(M, N) ? launch_head<GeoSmall, 1>(g, hd, st) : launch_head<GeoLarge, 1>(g, hd, st);
    hipLaunchKernelGGL(head_rows, dim3(static_cast<unsigned>((M + 15) / 16)), dim3(256), 0, st, hd.stats, zt,
                       static_cast<int>(gemm_head_spans(M, N)), static_cast<int>(M), row_max, row_inv, nll);
    hip_check(hipGetLastError(), "head_rows launch");
    return true;
}

// Pass 2: the same tiles again, stored as dlogits[M, N] (bf16, row pitch ldc) =
// (exp(z - row_max) row_inv - [column == target]) gscale (src/ops.cpp:371-374). N is a multiple of 8 here: a vocabulary
// that is not comes padded with rows of zeros in B, and the columns from `vocab` on come out 0.
bool gemm_head_dlogits(const void* a, int64_t lda, const void* b, int64_t ldb, int64_t M, int64_t N, int64_t K,
                       int64_t vocab, const int* target, const float* row_max, const float* row_inv, float gscale, void* dl,
                       int64_t ldc, hipStream_t st) {
    if (!head_takes(a, lda, b, ldb, M, N, K) || !aligned16(dl) || N % 8 || vocab > N || ldc % 8 || ldc >= (1 << 20)) return false;
    GemmArgs g = gemm_args(a, lda, b, ldb, M, N, K);
    g.c = dl;
    g.ldc = ldc;
    HeadArgs hd{};
    hd.target = target;
    hd.row_max = row_max;
    hd.row_inv = row_inv;
    hd.gscale = gscale;
    hd.vocab = static_cast<int>(vocab);
    if (vocab == N)
        head_small(M, N) ? launch_head<GeoSmall, 2>(g, hd, st) : launch_head<GeoLarge, 2>(g, hd, st);
    else
        head_small(M, N) ? launch_head<GeoSmall, 4>(g, hd, st) : launch_head<GeoLarge, 4>(g, hd, st);
    return true;
}

// ---- SwiGLU inside the products beside it ----
// The gate|up projection's two halves meet in the tile that forms them, and the down projection's dX becomes the two halves'
// gradients where it is formed: no pass reads [tokens, 2 d_ff] to write [tokens, d_ff] or the other way round, and a forward
// pass that keeps nothing for a backward one does not write gate and up at all (8192 tokens, d_ff 1376: those passes are 14 us
// and 21; the 35 M parameter model's step with checkpointing, which makes 18 of them, 5.26 -> 5.08 ms). Whole contractions on
// the two-slot ring.
namespace {
template <typename G, bool TB, int EPI>
void launch_gated_form(GemmArgs g, hipStream_t st) {
    constexpr int BNC = EPI == 7 ? G::BN : G::BN / 2;
    g.tiles_m = (g.M + G::BM - 1) / G::BM;
    g.tiles_n = (g.N + BNC - 1) / BNC;
    const int64_t vblocks = (static_cast<int64_t>(g.tiles_m) * g.tiles_n + 7) / 8 * 8, slots = cu_count() / 8 * 8 * (G::BM > 128 ? 1 : 2);
    hipLaunchKernelGGL((gemm_ring<G, false, TB, false, 2, EPI>), dim3(static_cast<unsigned>(std::min(vblocks, slots))), dim3(G::NTHR), 0,
                       st, g, HeadArgs{}, GroupArgs{});
    hip_check(hipGetLastError(), "gemm_ring (gated) launch");
}
// the plan of the product by itself, where it is one of the two forms that are built
// 128 x 128 tiles take contractions of up to 768. Above, little goes by (two layers forward and backward, ms, SwiGLU in passes of its own | without this
// line: width 896, d_ff 2392, 8192 tokens 1.97 | 1.93; 1024, 512, 8192 1.39 | 1.38; 1024, 2736, 2048 0.91 | 0.91; 2048, 5464, 1024 1.76 | 1.77): most such
// products have 256 x 256 tiles or split their contraction.
bool gated_plan(bool tB, int64_t M, int64_t cols, int64_t K, int64_t ldb, int64_t pitch, bool& large) {
    const Plan p = make_plan(false, tB, M, cols, K, K, ldb, pitch);
    large = p.large;
    return g_force_geo < 0 && p.S == 1 && (p.ring == 8 || (p.ring == 6 && K <= 768)) && M * pitch * 2 < (int64_t{1} << 31) - 4096;
}
}  // namespace
// h = silu(x gate) .* (x up) for w = [gate | up], N columns each; [x gate | x up] to gu unless that is null.
bool gemm_mfma_gated(const void* x, const void* w, void* gu, void* h, int64_t M, int64_t N, int64_t K, hipStream_t st, const Norm* norm) {
    if (g_force_geo < 0 && gemm_small_is_ahead(false, false, M, 2 * N, K) && gemm_small_gated(x, w, gu, h, M, N, K, st, norm)) return true;
    if (norm) return false;
    bool large;
    if (N % 8 || !takes(x, false, K, w, false, 2 * N, M, 2 * N, K) || !aligned16(h) || !aligned16(gu) || !gated_plan(false, M, 2 * N, K, 2 * N, 2 * N, large))
        return false;
    GemmArgs g = gemm_args(x, K, w, 2 * N, M, N, K);
    g.c = h;
    g.d = gu;
    if (gu)
        large ? launch_gated_form<GeoLarge, false, 5>(g, st) : launch_gated_form<GeoSmall, false, 5>(g, st);
    else
        large ? launch_gated_form<GeoLarge, false, 6>(g, st) : launch_gated_form<GeoSmall, false, 6>(g, st);
    return true;
}
// d = dy w^T, the gradient of silu(gate) .* up; dgu = [d gate | d up] for gu = [gate | up], N columns each. w is [N, K].
bool gemm_mfma_gated_grad(const void* dy, const void* w, const void* gu, void* dgu, int64_t M, int64_t N, int64_t K, hipStream_t st) {
    if (g_force_geo < 0 && gemm_small_is_ahead(false, true, M, N, K) && gemm_small_gated_grad(dy, w, gu, dgu, M, N, K, st)) return true;
    bool large;
    if (!takes(dy, false, K, w, true, K, M, N, K) || !aligned16(gu) || !aligned16(dgu) || !gated_plan(true, M, N, K, K, 2 * N, large)) return false;
    GemmArgs g = gemm_args(dy, K, w, K, M, N, K);
    g.c = dgu;
    g.d = gu;
    g.ldc = 2 * N;
    large ? launch_gated_form<GeoLarge, true, 7>(g, st) : launch_gated_form<GeoSmall, true, 7>(g, st);
    return true;
}

// ---- RoPE inside the q|k|v product ----
// On its way out the product turns q and k by the cosines and sines of a table, which a pass of its own over q and k would form anew (8192 x
// 1536 x 512: 19.4 us and 5.0 | 21.6, first head or all 8; a model of 6 such layers with checkpointing, whose step makes 12, all heads,
// 3.84 -> 3.75 ms a step). The small kernels ask for a lane's cosines behind the first chunks (fp32, 512 x 384 x 128: 4.8 us and 3.0 | 5.0).
// Tiles of 128 x 128; not the 256 x 256 ones, which start at 512 tiles of q|k|v and whose ends have no registers left.
bool gemm_mfma_turned(const void* x, const void* w, void* y, int64_t M, int64_t K, const Turn& turn, hipStream_t st, const Norm* norm) {
    const int64_t N = 3 * static_cast<int64_t>(turn.d);
    if (g_force_geo < 0 && gemm_small_is_ahead(false, false, M, N, K) && gemm_small_turned(x, w, y, M, K, turn, st, norm)) return true;
    if (norm) return false;
    if (turn.d % 8 || turn.head_dim % 8 || turn.cols % 8 || !takes(x, false, K, w, false, N, M, N, K) || !aligned16(y) || !aligned16(turn.table)) return false;
    const Plan p = make_plan(false, false, M, N, K, K, N, N);
    if (g_force_geo >= 0 || p.S != 1 || p.ring != 6 || M * N * 2 >= (int64_t{1} << 31) - 4096) return false;
    GemmArgs g = gemm_args(x, K, w, N, M, N, K);
    g.c = y;
    g.tiles_m = (g.M + GeoSmall::BM - 1) / GeoSmall::BM;
    g.tiles_n = (g.N + GeoSmall::BN - 1) / GeoSmall::BN;
    HeadArgs hd{};
    hd.turn = turn;
    const int64_t vblocks = (static_cast<int64_t>(g.tiles_m) * g.tiles_n + 7) / 8 * 8, slots = cu_count() / 8 * 8 * RingLds<GeoSmall, 2>::PER_CU;
    hipLaunchKernelGGL((gemm_ring<GeoSmall, false, false, false, 2, 8>), dim3(static_cast<unsigned>(std::min(vblocks, slots))), dim3(GeoSmall::NTHR), 0,
                       st, g, hd, GroupArgs{});
    hip_check(hipGetLastError(), "gemm_ring (turned) launch");
    return true;
}

// ---- several small weight-gradient products as one launch ----
// C_p += A_p^T B_p, p < count <= GROUP_MAX: A_p [K, M_p] and B_p [K, N_p] bf16 with row pitches lda / ldb, C_p
// [M_p, N_p] fp32 with row pitch ldc, one contraction length K for all. The products of a layer's backward pass
// (X^T dY per weight, K = every token) are each a few dozen 128 x 128 tiles: alone each would cut its contraction into
// slices to fill the chip and add the partial products afterwards; together their tiles fill it with whole
// contractions; narrow layers' tiles do not, and then the launch cuts the common contraction and a second one adds the
// slices. False, with nothing done, when an operand is not what the ring kernel takes or the tiles are too few
// to be worth it (the caller then multiplies them one by one).
namespace {
struct GroupSums {
    int count;
    int end[GROUP_MAX];  // groups of four elements of problems 0 .. p
    float* c[GROUP_MAX];
    int N[GROUP_MAX], ldc[GROUP_MAX];
};
// C_p += the slices' partial products, part[s][problem after problem][M_p][N_p], added in slice order
__global__ void sum_group(const float* part, int nparts, GroupSums gs) {
    const int n4 = gs.end[gs.count - 1];
    for (int i = blockIdx.x * 256 + threadIdx.x; i < n4; i += static_cast<int>(gridDim.x) * 256) {
        int p = 0;
        while (i >= gs.end[p]) ++p;
        const int e = (i - (p > 0 ? gs.end[p - 1] : 0)) * 4, N = gs.N[p];
        f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int k = 0; k < nparts; ++k) s += *reinterpret_cast<const f32x4*>(part + (static_cast<int64_t>(k) * n4 + i) * 4);
        f32x4* const d = reinterpret_cast<f32x4*>(gs.c[p] + static_cast<int64_t>(e / N) * gs.ldc[p] + e % N);
        *d += s;
    }
}
}  // namespace
bool gemm_mfma_grouped_tn(const GroupedProduct* ps, int count, int64_t K, hipStream_t st) {
    if (count < 2 || count > GROUP_MAX) return false;
    GroupArgs gr{};
    gr.count = count;
    int tiles = 0;
    int64_t small = 0;  // tiles of 32 x 32
    const int64_t ext_max = (int64_t{1} << 30) - 8192;
    for (int p = 0; p < count; ++p) {
        const GroupedProduct& q = ps[p];
        if (!takes(q.a, true, q.lda, q.b, false, q.ldb, q.M, q.N, K) || !aligned16(q.c) || q.ldc % 4) return false;
        if (K * q.lda * 2 >= ext_max || K * q.ldb * 2 >= ext_max || q.lda >= (1 << 21) || q.ldb >= (1 << 21) || q.ldc >= (1 << 20))
            return false;
        gr.a[p] = static_cast<const uint16_t*>(q.a);
        gr.b[p] = static_cast<const uint16_t*>(q.b);
        gr.c[p] = q.c;
        gr.M[p] = static_cast<int>(q.M);
        gr.N[p] = static_cast<int>(q.N);
        gr.lda[p] = static_cast<int>(q.lda);
        gr.ldb[p] = static_cast<int>(q.ldb);
        gr.ldc[p] = static_cast<int>(q.ldc);
        gr.tiles_n[p] = static_cast<int>((q.N + 127) / 128);
        tiles += static_cast<int>((q.M + 127) / 128) * gr.tiles_n[p];
        small += ((q.M + 31) / 32) * ((q.N + 31) / 32);
        gr.tile_end[p] = tiles;
    }
    for (int p = count; p < GROUP_MAX; ++p) gr.tile_end[p] = tiles;
    // Slices of the contraction: as many as give every CU a (tile, slice), none shorter than 512. Microseconds of whole contractions and
    // of slices with their sum, against the kernel of few tiles (a block's weights of width 192, d_ff 512, 5940 tokens: 36.2 us
    // there, 17.5 + 4.9 in six slices; width 128, d_ff 344, 6754 tokens 24.5 and 12.3 + 5.9).
    int64_t elements = 0;
    for (int p = 0; p < count; ++p) elements += ps[p].M * ps[p].N;
    int S = static_cast<int>(std::min<int64_t>({cu_count() / tiles, K / 512, 16}));
    const int kps = S > 1 ? static_cast<int>(((K + S - 1) / S + BK - 1) / BK * BK) : static_cast<int>(K);
    if (S > 1) S = static_cast<int>((K + kps - 1) / kps);
    const double whole = (4.0 + 0.0105 * K) * ((tiles + cu_count() - 1) / cu_count());
    const double sliced = S > 1 && elements < (int64_t{1} << 28) ? 7.5 + 0.0105 * kps + elements * (8.0 * S + 8.0) / 4.5e6 : 1e30;
    if (g_force_geo < 0 && gemm_small_us(true, false, small, K) < std::min(whole, sliced)) {
        SmallProduct sp[GROUP_MAX];
        for (int p = 0; p < count; ++p)
            sp[p] = SmallProduct{ps[p].a, ps[p].lda, ps[p].b, ps[p].ldb, ps[p].c, ps[p].ldc, nullptr, ps[p].M, ps[p].N, K};
        if (gemm_small(sp, count, true, false, PK_F32, 1.0f, st)) return true;
    }
    // worth it from about 3/8 of the CUs busy with whole contractions (measured: 196 tiles x 8192 in 69 us against 132
    // for the same four products one by one), and with any number of tiles where the contraction is short: a product of its
    // own is 10 us or more there, with a pass over its partial sums, and the grouped launch takes about 0.4 us for 64 tokens
    const bool slices = g_force_geo < 0 && sliced < whole;
    if (!slices && tiles < cu_count() * 3 / 8 && K > 640 * count) return false;
    GemmArgs g = gemm_args(ps[0].a, ps[0].lda, ps[0].b, ps[0].ldb, ps[0].M, ps[0].N, K);
    g.beta = 1;
    g.splits = 1;
    g.tiles_m = g.tiles_n = 0;
    if (slices) {
        Buffer part(sizeof(float) * static_cast<size_t>(S) * elements);
        GroupSums gs{};
        gs.count = count;
        int64_t at = 0;
        for (int p = 0; p < count; ++p) {
            gs.c[p] = ps[p].c;
            gs.N[p] = gr.N[p];
            gs.ldc[p] = gr.ldc[p];
            gr.c[p] = static_cast<float*>(part.p) + at;
            gr.ldc[p] = gr.N[p];
            at += ps[p].M * ps[p].N;
            gs.end[p] = static_cast<int>(at / 4);
        }
        g.beta = 0;
        g.splits = S;
        g.k_per_split = kps;
        g.part_stride = elements;
        const int64_t vblocks = (static_cast<int64_t>(tiles) * S + 7) / 8 * 8;
        hipLaunchKernelGGL((gemm_ring<GeoSmallK2, true, false, true, 4, 3>),
                           dim3(static_cast<unsigned>(std::min<int64_t>(vblocks, cu_count() / 8 * 8))), dim3(GeoSmallK2::NTHR), 0, st, g, HeadArgs{}, gr);
        hip_check(hipGetLastError(), "gemm_ring (grouped) launch");
        hipLaunchKernelGGL(sum_group, dim3(static_cast<unsigned>(std::min<int64_t>((elements / 4 + 255) / 256, 4096))), dim3(256), 0, st,
                           static_cast<const float*>(part.p), S, gs);
        hip_check(hipGetLastError(), "sum_group launch");
        return true;
    }
    const int64_t vblocks = (static_cast<int64_t>(tiles) + 7) / 8 * 8;
    if (tiles <= cu_count()) {
        const unsigned gx = static_cast<unsigned>(std::min<int64_t>(vblocks, cu_count() / 8 * 8));
        hipLaunchKernelGGL((gemm_ring<GeoSmallK2, true, false, true, 4, 3>), dim3(gx), dim3(GeoSmallK2::NTHR), 0, st, g,
                           HeadArgs{}, gr);
    } else {
        const unsigned gx = static_cast<unsigned>(std::min<int64_t>(vblocks, cu_count() / 8 * 8 * 2));
        hipLaunchKernelGGL((gemm_ring<GeoSmall, true, false, true, 2, 3>), dim3(gx), dim3(GeoSmall::NTHR), 0, st, g,
                           HeadArgs{}, gr);
    }
    hip_check(hipGetLastError(), "gemm_ring (grouped) launch");
    return true;
}

}  // namespace pk
