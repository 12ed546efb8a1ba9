// Projections around the attention path: y = W·x for one decoded token
// (bf16 or fp32 out) and y[t] = W·x[t] for a prefill batch.
//
// W is [M][N] bf16 row-major (one output per row, as the reference stores
// its projection weights), x is [T][N] bf16, y is [T][M].  Every product is
// accumulated in fp32 and rounded once at the store.
//
//  * gemv_kernel: HBM-bound.  A workgroup of 256 lanes owns RB output rows
//    and TB tokens; each lane walks 16-byte chunks of the rows (chunk c =
//    lane + 256 j), loads the token chunk once and reuses it for all RB rows,
//    and keeps TB x RB fp32 partials.  Partials are reduced in the wave
//    (DPP rows, then v_permlane16/32_swap) and across the four waves in LDS.
//    Buffer loads with an exact range return zeros past the last row or
//    token, so the tails need no branches.  The weight rows, read once per
//    call, carry the non-temporal hint (the lm-head's 1.24 GB then streams
//    at 6.95 TB/s where plain loads reach 6.2).
//  * gemm_kernel: MFMA-bound (prefill, T > kGemvMaxTokens, but for the small
//    products of a few tokens, which proj_skinny.hip has).  K in 64-wide slices
//    through a ring of two to four LDS stages by buffer-load DMA,
//    v_mfma_f32_32x32x16_bf16 on 32 x 32 blocks.  Nine tile sizes from 64 x 64
//    to 256 x 256, picked by a cost model of tiles, rounds and slices.  Tiles
//    are ordered in 8 x 8 groups and the groups are dealt to XCDs in
//    contiguous runs, so the blocks resident on one XCD share W and x slices
//    in that XCD's L2.  The results leave through LDS as whole 16-byte chunks
//    of token rows.
#include <cmath>
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"

namespace tiattn {
namespace {

// ------------------------------------------------------------------ GEMV

constexpr int kGvThreads = 256;
constexpr uint32_t kOob = 0xF0000000u;  // a byte offset past every range below

// E bf16 values per load: 8 (16-byte chunks), 2 (bf16 pairs) or 1.
template <int E>
struct GvChunk {
    static constexpr int WORDS = E == 8 ? 4 : 1;
    uint32_t w[WORDS];
};

// POL: the loads' cache-policy bits (kGvStream for the weight rows, which
// one call reads exactly once).
constexpr int kGvStream = 2;  // nt

template <int E, int POL = 0>
__device__ __forceinline__ GvChunk<E> gv_load(__amdgpu_buffer_rsrc_t r, uint32_t off) {
    GvChunk<E> c;
    if constexpr (E == 8) {
        const uint4 v = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, POL));
        c.w[0] = v.x; c.w[1] = v.y; c.w[2] = v.z; c.w[3] = v.w;
    } else if constexpr (E == 2) {
        c.w[0] = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, POL);
    } else {
        c.w[0] = __builtin_amdgcn_raw_buffer_load_b16(r, off, 0, POL);
    }
    return c;
}

template <int E>
__device__ __forceinline__ float gv_dot(const GvChunk<E>& w, const GvChunk<E>& x, float acc) {
    if constexpr (E == 1) {
        return fmaf(bf16_lo(w.w[0]), bf16_lo(x.w[0]), acc);
    } else {
#pragma unroll
        for (int i = 0; i < GvChunk<E>::WORDS; ++i)
            acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w.w[i]),
                                                  __builtin_bit_cast(bf16x2_t, x.w[i]), acc, false);
        return acc;
    }
}

__device__ __forceinline__ void gv_store(uint16_t* y, size_t i, float v) { y[i] = f32_to_bf16(v); }
__device__ __forceinline__ void gv_store(float* y, size_t i, float v) { y[i] = v; }

template <int E, int RB, int TB, typename OutT>
__global__ __launch_bounds__(kGvThreads) void gemv_kernel(const uint16_t* __restrict__ W,
                                                          const uint16_t* __restrict__ x,
                                                          OutT* __restrict__ y, uint32_t T,
                                                          uint32_t M, uint32_t N) {
    const uint32_t r0 = blockIdx.x * RB, t0 = blockIdx.y * TB;
    const uint32_t nrows = min((uint32_t)RB, M - r0), ntok = min((uint32_t)TB, T - t0);
    const uint32_t row_bytes = 2 * N;
    const auto rw = make_rsrc(W + (size_t)r0 * N, nrows * row_bytes);
    const auto rx = make_rsrc(x + (size_t)t0 * N, ntok * row_bytes);
    const uint32_t nchunk = N / E;

    float acc[TB][RB];
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int r = 0; r < RB; ++r) acc[t][r] = 0.0f;

    // Two chunks per lane per trip; the second one's offset is pushed out of
    // range (zeros) when it is past the row.
    for (uint32_t c = threadIdx.x; c < nchunk; c += 2 * kGvThreads) {
        const uint32_t c2 = c + kGvThreads;
        const uint32_t off[2] = {c * 2 * E, c2 < nchunk ? c2 * 2 * E : kOob};
        GvChunk<E> xv[2][TB], wv[2][RB];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int t = 0; t < TB; ++t) xv[u][t] = gv_load<E>(rx, t * row_bytes + off[u]);
#pragma unroll
            for (int r = 0; r < RB; ++r) wv[u][r] = gv_load<E, kGvStream>(rw, r * row_bytes + off[u]);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int t = 0; t < TB; ++t)
#pragma unroll
                for (int r = 0; r < RB; ++r) acc[t][r] = gv_dot<E>(wv[u][r], xv[u][t], acc[t][r]);
    }

    __shared__ float red[kGvThreads / 64][TB * RB];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const float s = wave_sum(acc[t][r]);
            if (lane == 0) red[wave][t * RB + r] = s;
        }
    __syncthreads();
    if (threadIdx.x < TB * RB) {
        const uint32_t t = threadIdx.x / RB, r = threadIdx.x % RB;
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < kGvThreads / 64; ++w) s += red[w][threadIdx.x];
        if (t < ntok && r < nrows) gv_store(y, (size_t)(t0 + t) * M + r0 + r, s);
    }
}

template <int E, int RB, int TB, typename OutT>
hipError_t gemv_launch(const uint16_t* W, const uint16_t* x, OutT* y, uint32_t T, uint32_t M,
                       uint32_t N, hipStream_t stream) {
    const dim3 grid((M + RB - 1) / RB, (T + TB - 1) / TB);
    gemv_kernel<E, RB, TB, OutT><<<grid, kGvThreads, 0, stream>>>(W, x, y, T, M, N);
    return hipGetLastError();
}

// Rows per workgroup: enough workgroups (about two per CU) for small M,
// more reuse of each token chunk for large M.
template <int E, int TB, typename OutT>
hipError_t gemv_rows(const uint16_t* W, const uint16_t* x, OutT* y, uint32_t T, uint32_t M,
                     uint32_t N, hipStream_t stream) {
    if constexpr (E != 8) {
        return gemv_launch<E, 4, TB>(W, x, y, T, M, N, stream);
    } else {
        if (M >= 4096) return gemv_launch<E, 8, TB>(W, x, y, T, M, N, stream);
        if (M >= 2048) return gemv_launch<E, 4, TB>(W, x, y, T, M, N, stream);
        if (M >= 1024) return gemv_launch<E, 2, TB>(W, x, y, T, M, N, stream);
        return gemv_launch<E, 1, TB>(W, x, y, T, M, N, stream);
    }
}

template <int TB, typename OutT>
hipError_t gemv_any(const uint16_t* W, const uint16_t* x, OutT* y, uint32_t T, uint32_t M,
                    uint32_t N, hipStream_t stream) {
    const uintptr_t a = (uintptr_t)W | (uintptr_t)x;
    if (N % 8 == 0 && a % 16 == 0) return gemv_rows<8, TB>(W, x, y, T, M, N, stream);
    if (N % 2 == 0 && a % 4 == 0) return gemv_rows<2, TB>(W, x, y, T, M, N, stream);
    return gemv_rows<1, TB>(W, x, y, T, M, N, stream);
}

// ------------------------------------------------------------------ GEMM

constexpr int kGmBK = 64;    // K granularity every GEMM configuration handles
constexpr int kGmGroup = 8;  // tile groups of 8 x 8

// Block tile BM (tokens) x BN (outputs) on a WGM x WGN grid of waves; each
// wave owns IM x JN blocks of 32 x 32.  K advances in slices of kGmBK
// through a ring of ST LDS stages.
template <int BM_, int BN_, int WGM_, int WGN_, int MINB_, int ST_>
struct GmCfg {
    static constexpr int BM = BM_, BN = BN_, WGM = WGM_, WGN = WGN_, MINB = MINB_, ST = ST_;
    static constexpr int BK = kGmBK;
    static constexpr int WAVES = WGM * WGN, THREADS = 64 * WAVES;
    static constexpr int IM = BM / WGM / 32, JN = BN / WGN / 32;
    static constexpr int RPB = 8;  // rows per DMA instruction
    static constexpr int A_ELEMS = BM * BK, B_ELEMS = BN * BK;
    static constexpr int A_BLOCKS = BM / RPB;                  // DMA instructions per slice of A
    static constexpr int BLOCKS = (BM + BN) / RPB;             // and in all
    static constexpr int DMAS = (BLOCKS + WAVES - 1) / WAVES;  // of them per wave, rounded up
    static_assert(ST >= 2 && ST <= 4 && (ST - 2) * DMAS < 64, "ring depth");
    static_assert(32 * IM * WGM == BM && 32 * JN * WGN == BN, "wave grid");
    static_assert(A_BLOCKS % WAVES == 0, "a wave's j-th DMA is of A or of B for every wave");
};
// The configurations, smallest tile first, each with its cost model (us):
// `fixed` + rounds * (`round` + slices * (`slice` + `load` * u)), rounds =
// ceil(tiles / CUs), u = the share of the rounds' CU slots that hold a tile.
// slice is the time of a K slice while the rest of the chip idles (DMA and
// operand reads for the small tiles, MFMAs for the large), load what a full
// chip adds (shared caches, and the clock the power limit leaves).  Fitted
// to 830 measured problems with the weights in HBM (T 5-4096, the
// projections of 512- to 5120-wide layers, outputs from 64 to 65536, N from
// 64): within 11-19 % rms of every configuration's time, and the configuration
// it picks is on average 0.5 % and at most 23 % slower than the fastest.  (A
// fit to 136 problems of two layers, caches warm, took 64 x 64 tiles at N =
// 128, T = 2000, 4096 outputs, 15.1 us, where 192 x 192 take 8.5.)
struct GmCost {
    float fixed, round, slice, load;
};
struct GmMini : GmCfg<64, 64, 2, 2, 2, 4> {  // 4 waves of 32 x 32, two workgroups per CU
    static constexpr GmCost COST{2.33f, 0.53f, 0.223f, 0.060f};
};
struct GmSix : GmCfg<96, 64, 3, 2, 1, 4> {  // 6 waves of 32 x 32
    static constexpr GmCost COST{1.45f, 1.62f, 0.240f, 0.082f};
};
struct GmFlat : GmCfg<128, 64, 4, 2, 1, 4> {  // 8 waves of 32 x 32
    static constexpr GmCost COST{0.95f, 2.67f, 0.244f, 0.111f};
};
struct GmDeep : GmCfg<128, 128, 2, 4, 1, 4> {  // 8 waves of 64 x 32
    static constexpr GmCost COST{0.71f, 2.85f, 0.352f, 0.225f};
};
struct GmTall : GmCfg<192, 128, 2, 4, 1, 3> {  // 8 waves of 96 x 32
    static constexpr GmCost COST{0.33f, 3.48f, 0.473f, 0.277f};
};
struct GmHalf : GmCfg<256, 128, 4, 2, 1, 3> {  // 8 waves of 64 x 64
    static constexpr GmCost COST{0.0f, 4.66f, 0.529f, 0.404f};
};
struct GmWide : GmCfg<192, 192, 2, 6, 1, 3> {  // 12 waves of 96 x 32
    static constexpr GmCost COST{0.0f, 4.46f, 0.572f, 0.450f};
};
struct GmBroad : GmCfg<256, 192, 4, 2, 1, 2> {  // 8 waves of 64 x 96
    static constexpr GmCost COST{0.28f, 4.60f, 0.849f, 0.583f};
};
struct GmLarge : GmCfg<256, 256, 2, 4, 1, 2> {  // 8 waves of 128 x 64
    static constexpr GmCost COST{0.01f, 5.92f, 0.972f, 0.734f};
};

// LDS rows of BK bf16 (128 bytes, eight 16-byte chunks); chunk c of row r
// sits at c ^ gm_swz(r).  A 16-byte LDS read serves 16 lanes per cycle from 64
// banks (256 bytes), and the MFMA operand reads put 16 consecutive rows on 16
// consecutive lanes, all at one logical chunk: rows r and r + 1 share a
// 256-byte bank line (r & 1 picks its half), so the 8 rows of each parity need
// different chunks.  (A swizzle r & 7 had rows r and r + 8 meet on the same
// banks: 4 conflict cycles per read.)
__device__ __forceinline__ uint32_t gm_swz(uint32_t row) { return (row >> 1) & 7; }

struct GmTile {
    uint32_t tt, tm;  // token tile, output tile
};

// Grouped order (8 output tiles x 8 token tiles per group, token-major
// inside a group), and consecutive group positions on one XCD: hardware
// deals workgroup b to XCD b % 8, so b -> (b % 8) * (n / 8) + b / 8 gives
// XCD x the run [x n / 8, (x + 1) n / 8) when n % 8 == 0.
__device__ __forceinline__ GmTile gm_tile(uint32_t b, uint32_t n_tt, uint32_t n_tm) {
    const uint32_t n = n_tt * n_tm;
    const uint32_t g = n % 8 == 0 ? (b % 8) * (n / 8) + b / 8 : b;
    const uint32_t per_group = kGmGroup * n_tt;
    const uint32_t first_tm = (g / per_group) * kGmGroup;
    const uint32_t gsize = min((uint32_t)kGmGroup, n_tm - first_tm);
    const uint32_t in = g % per_group;
    return {in / gsize, first_tm + in % gsize};
}

// Output tiles of one launch: BN columns of the stacked segments, or with
// the SwiGLU epilogue BN / 2 columns of the gate/up pair.
template <typename C, bool SW>
__device__ __host__ __forceinline__ uint32_t gm_out_tiles(const GemmArgs& g) {
    if (SW) return (g.rows[0] + C::BN / 2 - 1) / (C::BN / 2);
    uint32_t n = 0;
    for (int sg = 0; sg < g.nseg; ++sg) n += (g.rows[sg] + C::BN - 1) / C::BN;
    return n;
}

// Epilogue staging: chunk c of staged row t (CR 16-byte chunks per row)
// sits at ep_chunk<CR>(c, t), its two 8-byte halves swapped when
// ep_swap<CR>(t).  An 8-byte LDS write serves 16 lanes per cycle from 32
// banks (128 bytes), and the staging writes put 16 consecutive rows on 16
// lanes at one logical half chunk, so those 16 (chunk, half) positions must
// differ modulo 128 bytes: with 128-byte rows (CR 8) every row starts on the
// same banks, the chunk takes bits 1-3 of t and the half bit 0; with 64- or
// 192-byte rows (CR 4, 12) bit 0 of t picks the 64-byte half of the bank
// line, the chunk takes bits 1-2 (within its aligned group of four) and the
// half bit 3; with 32- or 96-byte rows (CR 2, 6) bits 0-1 pick the quarter,
// the chunk takes bit 2 (within its pair) and the half bit 3.  The 16-byte
// read-back (16 lanes per cycle from 64 banks) of consecutive chunks of a
// row stays a permutation of the row's banks.
template <int CR>
__device__ __forceinline__ int ep_chunk(int c, int t) {
    return CR == 8 ? c ^ ((t >> 1) & 7) : (CR % 4 ? c ^ ((t >> 2) & 1) : c ^ ((t >> 1) & 3));
}
template <int CR>
__device__ __forceinline__ int ep_swap(int t) {
    return CR == 8 ? t & 1 : (t >> 3) & 1;
}

// Epilogue LDS accesses in asm: to the compiler they are not LDS accesses,
// which it would make wait for every buffer load that writes LDS (it cannot
// tell the ring slot they use from the others).  A wave's LDS operations run
// in order, so its staging writes need no wait before its reads; ep_read
// waits for its own reads.
__device__ __forceinline__ uint32_t lds_addr(const uint16_t* p) {
    return (uint32_t)(size_t)(const __attribute__((address_space(3))) void*)p;
}
__device__ __forceinline__ void ep_write(uint16_t* p, uint32_t lo, uint32_t hi) {
    typedef unsigned v2u_t __attribute__((ext_vector_type(2)));
    const v2u_t v = {lo, hi};
    asm volatile("ds_write_b64 %0, %1" ::"v"(lds_addr(p)), "v"(v) : "memory");
}
template <int N>
__device__ __forceinline__ void ep_read(uint4 (&x)[N], const uint32_t (&a)[N]) {
    typedef unsigned v4u_t __attribute__((ext_vector_type(4)));
    v4u_t v[N];
    if constexpr (N == 1) {
        asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(v[0])
                     : "v"(a[0])
                     : "memory");
    } else if constexpr (N == 2) {
        asm volatile("ds_read_b128 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(v[0]), "=&v"(v[1])
                     : "v"(a[0]), "v"(a[1])
                     : "memory");
    } else if constexpr (N == 4) {
        asm volatile(
            "ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %6\n\t"
            "ds_read_b128 %3, %7\n\ts_waitcnt lgkmcnt(0)"
            : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
            : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3])
            : "memory");
    } else if constexpr (N == 6) {
        asm volatile(
            "ds_read_b128 %0, %6\n\tds_read_b128 %1, %7\n\tds_read_b128 %2, %8\n\t"
            "ds_read_b128 %3, %9\n\tds_read_b128 %4, %10\n\tds_read_b128 %5, %11\n\t"
            "s_waitcnt lgkmcnt(0)"
            : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5])
            : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5])
            : "memory");
    } else {
        static_assert(N == 8, "ep_read sizes");
        asm volatile(
            "ds_read_b128 %0, %8\n\tds_read_b128 %1, %9\n\tds_read_b128 %2, %10\n\t"
            "ds_read_b128 %3, %11\n\tds_read_b128 %4, %12\n\tds_read_b128 %5, %13\n\t"
            "ds_read_b128 %6, %14\n\tds_read_b128 %7, %15\n\ts_waitcnt lgkmcnt(0)"
            : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3]), "=&v"(v[4]), "=&v"(v[5]),
              "=&v"(v[6]), "=&v"(v[7])
            : "v"(a[0]), "v"(a[1]), "v"(a[2]), "v"(a[3]), "v"(a[4]), "v"(a[5]), "v"(a[6]),
              "v"(a[7])
            : "memory");
    }
#pragma unroll
    for (int k = 0; k < N; ++k) x[k] = make_uint4(v[k].x, v[k].y, v[k].z, v[k].w);
}

// Eight packed bf16 pairs: bf16(a + b) each, the sums in fp32.
__device__ __forceinline__ uint4 add_bf16x8(uint4 a, uint4 b) {
    const uint32_t x[4] = {a.x, a.y, a.z, a.w}, z[4] = {b.x, b.y, b.z, b.w};
    uint32_t o[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        o[k] = pack_bf16x2(bf16_lo(x[k]) + bf16_lo(z[k]), bf16_hi(x[k]) + bf16_hi(z[k]));
    return make_uint4(o[0], o[1], o[2], o[3]);
}

// DMA instruction `blk` of a slice fills the eight tile rows from 8 blk on
// (the A rows, then the B rows) of the stage at st; lane l loads row l / 8's
// physical chunk l % 8, i.e. logical chunk (l % 8) ^ gm_swz(row).  SW: 16 gate and 16 up rows make a 32-row block of B,
// positions p with bit 3 clear gate, the others up, both of the 16 output
// columns 8 (p / 16) + p % 8, so that a lane's accumulator values 8 q + u
// and 8 q + 4 + u (u < 4) are gate and up of one output; the eight rows of
// a DMA instruction are all of one kind.
template <typename C, bool SW>
__device__ __forceinline__ uint32_t gm_dma_offset(uint32_t blk, int lane, uint32_t row_bytes) {
    const uint32_t r = C::RPB * blk + lane / 8;  // tile row
    const uint32_t logical = (lane % 8) ^ gm_swz(r);
    uint32_t src = r < (uint32_t)C::BM ? r : r - C::BM;
    if (SW && r >= (uint32_t)C::BM)
        src = 16 * (src / 32) + 8 * (src / 16 % 2) + src % 8;
    return src * row_bytes + 16 * logical;
}

// The tile's products: K slices stream through a ring of ST LDS stages by
// buffer-load DMA, ST - 1 slices ahead of the MFMAs.  What bounds it: the
// MFMAs (at the clock the power limit leaves) for 256 x 256, whose two stages
// fill the LDS; for tiles of which a CU runs one, the DMA's latency, which a
// ring of three or four stages covers.  The hand-over from slice to slice
// sits before the last k-step's MFMAs (their operands already in registers)
// and the next slice's first operand reads after it, so that neither the
// barrier nor the LDS latency leaves the matrix cores idle.  Measured against
// two stages with the hand-over between slices and 2-4 tile sizes by rule
// (us, before -> after): 4096 x 4096 x 4096 108.4 -> 102.3 (1343 TFLOP/s); T
// = 1371, 1024-wide layer: q/k/v 16.1 -> 14.5, o 10.8 -> 10.1, gate/up 25.3
// -> 21.4, down 18.5 -> 15.4; T = 37: 6.1 -> 5.3, 9.2 -> 7.0, 12.6 -> 5.3,
// 12.4 -> 8.9; T = 600, 4096-wide: 51 -> 32, 45 -> 26, 194 -> 120, 130 -> 74.
//
// kGmShort: at most ST slices, all requested at once and no ring (N = 64, T =
// 16, 1024 outputs 3.06 -> 2.66 us, where ST - 1 requests past the end held up
// the one slice).
//
// kGmMixed: a stack of which some segments are summed as the few-token kernel
// sums them (proj_uses_skinny), so that each element has the bits it has by
// itself: the slices in that kernel's order (every eighth, from slice 0, then
// from slice 1, ...), its MFMA, and eight partials added one after another.
// One launch of every segment's tiles, where the two kernels in turn cost a
// launch and left CUs idle twice.  Weights from HBM, us, two launches -> one (the
// GEMM of before the few-token kernel): q/k/v of a 1024-wide layer, T = 160 10.8
// -> 8.0 (10.0), T = 320 18.9 -> 9.6 (10.4); 2560-wide, T = 96 23.7 -> 15.3 (20.7),
// T = 256 33.0 -> 22.9 (21.4, on slices of 128); 4096-wide, T = 128 33.1 -> 22.8
// (31.0).  Every segment in the GEMM's own order takes 0.2 us less.
enum GmForm : int { kGmRing, kGmShort, kGmMixed };

template <typename C, bool SW, int FORM>
__global__ __launch_bounds__(C::THREADS, C::MINB) void gemm_kernel(GemmArgs g) {
    constexpr int IM = C::IM, JN = C::JN, BK = C::BK, ST = C::ST;
    const uint32_t T = g.T, N = g.N;
    const uint16_t* __restrict__ x = g.x;
    // One array per stage (A rows, then B rows), so that the compiler can
    // tell the stage being read from those the DMA is filling.
    constexpr int STAGE = C::A_ELEMS + C::B_ELEMS;
    __shared__ __align__(1024) uint16_t s_0[STAGE];
    __shared__ __align__(1024) uint16_t s_1[STAGE];
    __shared__ __align__(1024) uint16_t s_2[ST > 2 ? STAGE : 8];
    __shared__ __align__(1024) uint16_t s_3[ST > 3 ? STAGE : 8];
    // Output tiles run over the segments' rows stacked, each segment
    // starting on a tile boundary.
    const uint32_t n_tm = gm_out_tiles<C, SW>(g);
    const uint32_t n_tt = (T + C::BM - 1) / C::BM;
    const GmTile tile = gm_tile(blockIdx.x, n_tt, n_tm);
    uint32_t tm = tile.tm;
    int seg = 0;
    if (!SW) {
        const uint32_t spans[3] = {(g.rows[0] + C::BN - 1) / C::BN, (g.rows[1] + C::BN - 1) / C::BN,
                                   (g.rows[2] + C::BN - 1) / C::BN};
        seg = segment_of(spans, g.nseg, tm);
    }
    constexpr uint32_t TILE_N = SW ? C::BN / 2 : C::BN;  // output columns per tile
    const uint32_t M = pick3(g.rows, seg);
    uint16_t* __restrict__ y = pick3(g.y, seg);
    const uint32_t t0 = tile.tt * C::BM, m0 = tm * TILE_N;
    const uint32_t row_bytes = 2 * N;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wr = wave / C::WGN, wc = wave % C::WGN;

    // Whether this tile's segment is summed in the few-token kernel's order.
    const bool split = FORM == kGmMixed && proj_uses_skinny(T, M, N);

    f32x16_t acc[IM][JN];
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

    // Every wave issues DMAS instructions per slice, which the vmcnt waits
    // count on: where BLOCKS is not a multiple of the waves, the surplus
    // ones load one of the last two blocks again (the same bytes to the same
    // place, and of the same kind, gate or up: WAVES and BLOCKS are even).
    const uint32_t nk = N / BK;
    const uint32_t wave_s = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t d_off[C::DMAS], d_blk[C::DMAS];
#pragma unroll
    for (int j = 0; j < C::DMAS; ++j) {
        const uint32_t blk = wave_s + C::WAVES * j;
        d_blk[j] = blk < (uint32_t)C::BLOCKS ? blk : C::BLOCKS - 2 + blk % 2;
        d_off[j] = gm_dma_offset<C, SW>(d_blk[j], lane, row_bytes);
    }
    // The next slice to load: its first column in A and in this wave's part
    // of B, and the bytes from there to the tile's end.  Past the last slice
    // the ranges are empty: those loads give zeros, which nothing multiplies.
    const uint16_t* pa = x + (size_t)t0 * N;
    const uint16_t* pb = pick3(g.w, seg) + (size_t)m0 * N;
    if (SW && wave_s % 2) pb = g.w[1] + (size_t)m0 * N;
    uint32_t a_left = min((uint32_t)C::BM, T - t0) * row_bytes;
    uint32_t b_left = min(TILE_N, M - m0) * row_bytes;
    uint32_t k_left = nk;
    auto dma_slice = [&](uint16_t* st) __attribute__((always_inline)) {
        const auto ra = make_rsrc(pa, k_left ? a_left : 0);
        const auto rb = make_rsrc(pb, k_left ? b_left : 0);
#pragma unroll
        for (int j = 0; j < C::DMAS; ++j)
            dma16(C::WAVES * j < C::A_BLOCKS ? ra : rb, st + 512 * d_blk[j], d_off[j]);
    };
    auto advance = [&](int slices) __attribute__((always_inline)) {  // or back
        pa += slices * BK;
        pb += slices * BK;
        a_left -= (uint32_t)(2 * BK * slices);
        b_left -= (uint32_t)(2 * BK * slices);
    };
    // The products of this tile, in blocks of BLK x BLK: k-steps of 512 / BLK,
    // whose operands lane l reads as row l % BLK, k 8 (l / BLK).
    auto products = [&](auto split_order) __attribute__((always_inline)) {
        constexpr bool SPLIT = decltype(split_order)::value;
        constexpr int BLK = SPLIT ? 16 : 32;
        constexpr int STEPS = BK * BLK / 512, AM = 32 / BLK * IM, BN = 32 / BLK * JN;
        // Operand read offsets (elements) inside a stage for block 0, per
        // k-step; block i adds BLK i rows, which the swizzle does not see.
        int a_off[STEPS], b_off[STEPS];
#pragma unroll
        for (int s = 0; s < STEPS; ++s) {
            const int row = lane % BLK, chunk = (64 / BLK * s + lane / BLK) ^ gm_swz(row);
            a_off[s] = (32 * IM * wr + row) * BK + 8 * chunk;
            b_off[s] = C::A_ELEMS + (32 * JN * wc + row) * BK + 8 * chunk;
        }
        f32x4_t part[AM][BN];
        if constexpr (SPLIT) {
#pragma unroll
            for (int i = 0; i < AM; ++i)
#pragma unroll
                for (int j = 0; j < BN; ++j) part[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
        // Operands of k-step s + 1 are read while the MFMAs of k-step s run
        // (two register sets; STEPS is even, so a slice starts on set 0).
        bf16x8_t a[2][AM], b[2][BN];
        auto read = [&](const uint16_t* st, int s) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < AM; ++i)
                a[s & 1][i] = as_bf16x8(*reinterpret_cast<const uint4*>(st + a_off[s] + BLK * BK * i));
#pragma unroll
            for (int j = 0; j < BN; ++j)
                b[s & 1][j] = as_bf16x8(*reinterpret_cast<const uint4*>(st + b_off[s] + BLK * BK * j));
        };
        auto mfmas = [&](int s) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < AM; ++i)
#pragma unroll
                for (int j = 0; j < BN; ++j) {  // W rows first
                    if constexpr (SPLIT)
                        part[i][j] = mfma16x16x32(b[s & 1][j], a[s & 1][i], part[i][j]);
                    else
                        acc[i][j] = mfma32x32x16(b[s & 1][j], a[s & 1][i], acc[i][j]);
                }
        };
        // SPLIT: the next slice is eight on, or the first of the next partial.
        uint32_t slice = 0, partial = 0, partial_left = (nk + 7) / 8;
        auto next_slice = [&]() __attribute__((always_inline)) {
            if constexpr (SPLIT) {
                const uint32_t to = slice + 8 < nk ? slice + 8 : slice % 8 + 1;
                advance((int)to - (int)slice);
                slice = to;
            } else {
                advance(1);
            }
            k_left -= k_left != 0;
        };
        // SPLIT: a finished partial is added to the sums (the 16 x 16 blocks
        // of a 32 x 32 one at values 4 (2 J + I) on, J its half of the outputs, I
        // of the tokens).
        auto slice_done = [&]() __attribute__((always_inline)) {
            if constexpr (SPLIT) {
                if (--partial_left != 0) return;
                partial_left = (nk - ++partial + 7) / 8;
#pragma unroll
                for (int i = 0; i < AM; ++i)
#pragma unroll
                    for (int j = 0; j < BN; ++j)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            acc[i / 2][j / 2][4 * (2 * (j % 2) + i % 2) + v] += part[i][j][v];
                            part[i][j][v] = 0.0f;
                        }
            }
        };
        if constexpr (FORM == kGmShort) {
            uint16_t* const stage[4] = {s_0, s_1, s_2, s_3};
#pragma unroll
            for (int k = 0; k < ST; ++k)
                if (k < (int)nk) {
                    dma_slice(stage[k]);
                    next_slice();
                }
            __builtin_amdgcn_s_waitcnt(kWaitVmLgkm0);
            asm volatile("s_barrier" ::: "memory");
#pragma unroll
            for (int k = 0; k < ST; ++k)
                if (k < (int)nk) {
#pragma unroll
                    for (int s = 0; s < STEPS; ++s) {
                        read(stage[k], s);
                        mfmas(s);
                    }
                }
        } else {
            // Slice kt, in `cur`, its first operands already in registers: the
            // MFMAs of all k-steps but the last; then, with the last k-step's
            // operands in registers too, the hand-over (this wave's reads of cur
            // and its part of slice kt + 1 have landed, then every wave's have),
            // the first operand reads of slice kt + 1 and the DMA of slice kt +
            // ST into cur, all spread over the MFMAs of the last k-step.
            constexpr int DMAS = C::DMAS;
            auto step = [&](uint16_t* cur, const uint16_t* nxt) __attribute__((always_inline)) {
#pragma unroll
                for (int s = 0; s < STEPS - 1; ++s) {
                    read(cur, s + 1);
                    mfmas(s);
                    __builtin_amdgcn_sched_group_barrier(0x100, AM + BN, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, AM * BN, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_s_waitcnt(wait_vmcnt_lgkm0((ST - 2) * DMAS));
                asm volatile("s_barrier" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                read(nxt, 0);
                dma_slice(cur);
                mfmas(STEPS - 1);
                __builtin_amdgcn_sched_group_barrier(0x100, AM + BN, 0);
#pragma unroll
                for (int k = 0; k < AM * BN; ++k) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x020, (DMAS + AM * BN - 1) / (AM * BN), 0);
                }
                __builtin_amdgcn_sched_barrier(0);
                next_slice();
                slice_done();
            };
            dma_slice(s_0);
            next_slice();
            dma_slice(s_1);
            next_slice();
            if constexpr (ST > 2) {
                dma_slice(s_2);
                next_slice();
            }
            if constexpr (ST > 3) {
                dma_slice(s_3);
                next_slice();
            }
            __builtin_amdgcn_s_waitcnt(wait_vmcnt_lgkm0((ST - 1) * DMAS));
            asm volatile("s_barrier" ::: "memory");
            read(s_0, 0);
            // Whole rounds of the ring, then the nk % ST slices left (a further
            // round would multiply zeros: at N = 1024 on three stages 18 slices'
            // time for 16, at N = 128 on four stages 4 for 2).
            uint32_t kt = 0;
            for (; kt + ST <= nk; kt += ST) {
                step(s_0, s_1);
                if constexpr (ST == 2) {
                    step(s_1, s_0);
                } else if constexpr (ST == 3) {
                    step(s_1, s_2);
                    step(s_2, s_0);
                } else {
                    step(s_1, s_2);
                    step(s_2, s_3);
                    step(s_3, s_0);
                }
            }
            if (kt < nk) step(s_0, s_1);
            if (ST > 2 && kt + 1 < nk) step(s_1, s_2);
            if (ST > 3 && kt + 2 < nk) step(s_2, s_3);
        }
    };
    if (FORM == kGmMixed && split)
        products(std::bool_constant<FORM == kGmMixed>{});
    else
        products(std::bool_constant<false>{});
    // The ring is free for the epilogue once every wave's last reads and
    // (empty) DMA are done.
    __builtin_amdgcn_s_waitcnt(kWaitVmLgkm0);
    asm volatile("s_barrier" ::: "memory");

    // Block (i, j), W rows first: lane l value v is output column
    // 32 (JN wc + j) + 8 (v / 4) + 4 (l / 32) + v % 4 (SW: gate v = 8 q + u and
    // up 8 q + 4 + u of column 16 (JN wc + j) + 8 q + 4 (l / 32) + u) of token
    // row 32 (IM wr + i) + l % 32, so v / 4 picks four consecutive outputs of
    // one token (split: column 32 (JN wc + j) + 16 (v / 8) + 4 (l / 16) + v % 4,
    // row 32 (IM wr + i) + 16 (v / 4 % 2) + l % 16).  Each wave stages its bf16 results (rows of OUTC outputs) in
    // its part of the first stage, R token blocks at a time, and writes whole
    // 16-byte chunks of token rows.
    constexpr int OUTC = SW ? 16 * JN : 32 * JN;  // a wave's output columns
    constexpr int CR = OUTC / 8;                  // 16-byte chunks per staged row
    constexpr int AREA = STAGE / C::WAVES / 64 * 64;  // elements per wave
    constexpr int FIT = CR == 2 ? 2 : AREA / (32 * OUTC);
    constexpr int R = IM < FIT ? IM : FIT;
    static_assert(32 * R * OUTC <= AREA, "epilogue area");
    static_assert(R >= 1 && (CR == 2 || CR == 4 || CR == 6 || CR == 8 || CR == 12), "epilogue staging");
    constexpr int PER_LANE = 32 * R * CR / 64;  // chunks a lane moves per round (R CR is even)
    uint16_t* const area = s_0 + wave * AREA;
    const uint32_t col0 = m0 + OUTC * wc;
    const bool residual = !SW && g.residual;
    // Whole 16-byte stores need every row start 16-byte aligned.
    const bool vec = M % 8 == 0 && (reinterpret_cast<uintptr_t>(y) & 15) == 0;
#pragma unroll
    for (int r0 = 0; r0 < IM; r0 += R) {
        const int nb = IM - r0 < R ? IM - r0 : R;  // token blocks this round
        const uint32_t row0 = t0 + 32 * (IM * wr + r0);
        // This round's old values first, so that their latency overlaps
        // the staging.
        uint4 old[PER_LANE];
        if (residual) {
#pragma unroll
            for (int k = 0; k < PER_LANE; ++k) {
                const int idx = lane + 64 * k, t = idx / CR, c = idx % CR;
                const uint32_t tok = row0 + t, m = col0 + 8 * c;
                old[k] = make_uint4(0, 0, 0, 0);
                if (vec && t < 32 * nb && tok < T && m < M)
                    old[k] = *reinterpret_cast<const uint4*>(y + (size_t)tok * M + m);
            }
        }
#pragma unroll
        for (int ii = 0; ii < R; ++ii) {
            if (ii >= nb) break;
            const int i = r0 + ii;
#pragma unroll
            for (int j = 0; j < JN; ++j)
#pragma unroll
                for (int q = 0; q < (SW ? 2 : 4); ++q) {
                    float e[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if constexpr (SW)
                            e[u] = swiglu1(bf16_to_f32(f32_to_bf16(acc[i][j][8 * q + u])),
                                           bf16_to_f32(f32_to_bf16(acc[i][j][8 * q + 4 + u])));
                        else
                            e[u] = acc[i][j][4 * q + u];
                    }
                    int t = 32 * ii + lane % 32, c = (SW ? 2 : 4) * j + q, h = lane / 32;
                    if (FORM == kGmMixed && split) {
                        t = 32 * ii + 16 * (q % 2) + lane % 16;
                        c = 4 * j + 2 * (q / 2) + lane / 32;
                        h = lane / 16 % 2;
                    }
                    ep_write(area + t * OUTC + 8 * ep_chunk<CR>(c, t) + 4 * (h ^ ep_swap<CR>(t)), pack_bf16x2(e[0], e[1]),
                             pack_bf16x2(e[2], e[3]));
                }
        }
        // Every lane reads its PER_LANE chunks (rows below 32 R: inside this
        // wave's area), then stores those of this round's rows.
        uint4 stg[PER_LANE];
        {
            uint32_t a[PER_LANE];
#pragma unroll
            for (int k = 0; k < PER_LANE; ++k) {
                const int idx = lane + 64 * k, t = idx / CR, c = idx % CR;
                a[k] = lds_addr(area + t * OUTC + 8 * ep_chunk<CR>(c, t));
            }
            ep_read<PER_LANE>(stg, a);
        }
#pragma unroll
        for (int k = 0; k < PER_LANE; ++k)
            if (ep_swap<CR>((lane + 64 * k) / CR)) stg[k] = make_uint4(stg[k].z, stg[k].w, stg[k].x, stg[k].y);
        if (vec) {
#pragma unroll
            for (int k = 0; k < PER_LANE; ++k) {
                const int idx = lane + 64 * k, t = idx / CR, c = idx % CR;
                const uint32_t tok = row0 + t, m = col0 + 8 * c;
                if (t < 32 * nb && tok < T && m < M)
                    *reinterpret_cast<uint4*>(y + (size_t)tok * M + m) =
                        residual ? add_bf16x8(old[k], stg[k]) : stg[k];
            }
        } else {
            // Rows not 16-byte aligned or a partial last chunk: element stores.
#pragma unroll
            for (int k = 0; k < PER_LANE; ++k) {
                const int idx = lane + 64 * k, t = idx / CR, c = idx % CR;
                const uint32_t tok = row0 + t, m = col0 + 8 * c;
                if (t >= 32 * nb || tok >= T || m >= M) continue;
                uint16_t* dst = y + (size_t)tok * M + m;
                const uint32_t w[4] = {stg[k].x, stg[k].y, stg[k].z, stg[k].w};
                for (int u = 0; u < 8 && m + u < M; ++u) {
                    const uint16_t val = uint16_t(w[u / 2] >> (16 * (u % 2)));
                    dst[u] = residual ? f32_to_bf16(bf16_to_f32(dst[u]) + bf16_to_f32(val)) : val;
                }
            }
        }
    }
}

template <typename C, bool SW = false>
uint32_t gemm_tiles(const GemmArgs& g) {
    return ((g.T + C::BM - 1) / C::BM) * gm_out_tiles<C, SW>(g);
}

template <typename C, bool SW = false>
hipError_t gemm_launch(const GemmArgs& g, hipStream_t stream) {
    const uint32_t tiles = gemm_tiles<C, SW>(g);
    if (g.N / kGmBK <= C::ST)
        gemm_kernel<C, SW, kGmShort><<<tiles, C::THREADS, 0, stream>>>(g);
    else
        gemm_kernel<C, SW, kGmRing><<<tiles, C::THREADS, 0, stream>>>(g);
    return hipGetLastError();
}

template <typename C>
hipError_t gemm_launch_mixed(const GemmArgs& g, hipStream_t stream) {
    gemm_kernel<C, false, kGmMixed><<<gemm_tiles<C>(g), C::THREADS, 0, stream>>>(g);
    return hipGetLastError();
}

}  // namespace

int gemm_cus() {
    static int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 256;
        return n;
    }();
    return cus;
}

namespace {

template <typename C, bool SW>
float gemm_cost(const GemmArgs& g, uint32_t cus) {
    const float tiles = (float)gemm_tiles<C, SW>(g);
    const float rounds = ceilf(tiles / cus), u = tiles / (rounds * cus);
    const float slices = (float)(g.N / kGmBK);
    return C::COST.fixed + rounds * (C::COST.round + slices * (C::COST.slice + C::COST.load * u));
}

// The configuration of least modelled cost, or the one that the caller names.
// Every one sums K in the same MFMA order, so the choice does not change a
// result bit.
struct GmPick {
    const GemmArgs& g;
    const uint32_t cus = (uint32_t)gemm_cus();
    hipError_t (*best)(const GemmArgs&, hipStream_t) = nullptr;
    float least = 0.0f;
    int tile = 0;
    template <typename C, bool SW>
    void consider(hipError_t (*launch)(const GemmArgs&, hipStream_t)) {
        const float cost = gemm_cost<C, SW>(g, cus);
        if (g.tile ? ++tile == g.tile : best == nullptr || cost < least) {
            least = cost;
            best = launch;
        }
    }
};

template <bool SW>
hipError_t gemm_pick_launch(const GemmArgs& g, hipStream_t stream) {
    GmPick p{g};
    p.consider<GmMini, SW>(gemm_launch<GmMini, SW>);
    p.consider<GmSix, SW>(gemm_launch<GmSix, SW>);
    p.consider<GmFlat, SW>(gemm_launch<GmFlat, SW>);
    p.consider<GmDeep, SW>(gemm_launch<GmDeep, SW>);
    p.consider<GmTall, SW>(gemm_launch<GmTall, SW>);
    p.consider<GmHalf, SW>(gemm_launch<GmHalf, SW>);
    p.consider<GmWide, SW>(gemm_launch<GmWide, SW>);
    p.consider<GmBroad, SW>(gemm_launch<GmBroad, SW>);
    p.consider<GmLarge, SW>(gemm_launch<GmLarge, SW>);
    return p.best(g, stream);
}

// The tiles that few tokens leave in question.
hipError_t gemm_pick_launch_mixed(const GemmArgs& g, hipStream_t stream) {
    GmPick p{g};
    p.consider<GmMini, false>(gemm_launch_mixed<GmMini>);
    p.consider<GmSix, false>(gemm_launch_mixed<GmSix>);
    p.consider<GmFlat, false>(gemm_launch_mixed<GmFlat>);
    p.consider<GmDeep, false>(gemm_launch_mixed<GmDeep>);
    return p.best(g, stream);
}

}  // namespace

hipError_t launch_gemv_bf16(const uint16_t* W, const uint16_t* x, uint16_t* y, uint32_t M,
                            uint32_t N, hipStream_t stream) {
    return gemv_any<1>(W, x, y, 1, M, N, stream);
}

hipError_t launch_gemv_f32(const uint16_t* W, const uint16_t* x, float* y, uint32_t M, uint32_t N,
                           hipStream_t stream) {
    return gemv_any<1>(W, x, y, 1, M, N, stream);
}

bool proj_uses_gemm(uint32_t T, uint32_t N, const void* W, const void* x) {
    return T > kGemvMaxTokens && N % kGmBK == 0 && ((uintptr_t)W | (uintptr_t)x) % 16 == 0;
}

hipError_t launch_batch_proj_bf16(const uint16_t* W, const uint16_t* x, uint16_t* y, uint32_t T,
                                  uint32_t M, uint32_t N, hipStream_t stream) {
    if (T == 1) return gemv_any<1>(W, x, y, T, M, N, stream);
    if (!proj_uses_gemm(T, N, W, x)) return gemv_any<4>(W, x, y, T, M, N, stream);
    GemmArgs g;
    g.x = x;
    g.T = T;
    g.N = N;
    g.w[0] = W;
    g.y[0] = y;
    g.rows[0] = M;
    return launch_gemm(g, stream);
}

hipError_t launch_gemm(const GemmArgs& g, hipStream_t stream) {
    int split = 0;  // segments summed in the few-token kernel's order
    uint64_t blocks = 0;
    for (int s = 0; s < g.nseg; ++s) {
        split += proj_uses_skinny(g.T, g.rows[s], g.N);
        blocks += skinny_tiles(g.T, g.rows[s]);
    }
    if (g.swiglu)
        return split && !g.tile ? launch_gemm_skinny(g, stream) : gemm_pick_launch<true>(g, stream);
    if (split == 0) return gemm_pick_launch<false>(g, stream);
    // A segment alone, or a stack that is one round of the few-token kernel's
    // blocks as well.
    if (!g.tile && (g.nseg == 1 || (split == g.nseg && blocks <= kSkinnyRound)))
        return launch_gemm_skinny(g, stream);
    return gemm_pick_launch_mixed(g, stream);
}

}  // namespace tiattn
