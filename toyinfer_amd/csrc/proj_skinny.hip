// Projections of a few tokens (a short prompt): y[t][m] = sum_n W[m][n] x[t][n]
// where proj_uses_skinny says, with the segments, residual and SwiGLU forms of
// the GEMM (GemmArgs).
//
// What bounds it: with so few tokens a launch is a read of the weights, and
// an output tile walked slice by slice (the GEMM) is a serial chain of N / 64
// load latencies on the few CUs its tiles give work.  Here the eight waves of
// a workgroup split K (64-wide chunk c to wave c % 8), so the chain is N / 512
// chunks with DEPTH of them in flight per wave.  Each wave streams its chunks
// through LDS slots of its own by buffer-load DMA (eight lanes per 128-byte
// row, where operands loaded straight into the MFMA layout put every lane of
// a 16-lane group on a row of its own: measured 13 bytes per clock and CU)
// and waits for its own loads only: no barrier before the eight partial tiles
// are added.  The tiles, 16 JN outputs by 16 IM tokens, are as small as fills
// the CUs.  Each element is the sum of eight fp32 partials in wave order, a
// partial the MFMA chain over its wave's chunks: the same for every tile size.
// Measured against the ring GEMM (us, weights from HBM, T = 37): 1024-wide
// layer q/k/v 7.4 -> 5.5, o 9.0 -> 4.6, gate/up 7.4 -> 6.8, down 15.0 -> 6.5;
// 4096-wide q/k/v 20.5 -> 16.8, o 19.7 -> 12.0, down 54 -> 26.7.
#include <cmath>

#include "common.hpp"
#include "kernels.hpp"

namespace tiattn {
namespace {

constexpr int kSkWaves = 8;
constexpr int kSkThreads = 64 * kSkWaves;
constexpr int kSkChunk = 64;  // K columns per chunk: one 128-byte line of each row

// A wave's LDS slot holds one chunk of its JN + IM 16-row blocks; DEPTH slots
// per wave, at most four and as many as 160 KB hold, are in flight at a time.
constexpr int sk_depth(int jn, int im) { return jn + im <= 2 ? 4 : (jn + im <= 3 ? 3 : 2); }

// 128-byte rows, 16-byte chunk q of row r at q ^ sk_swz(r): the 16 consecutive
// rows an operand read takes at one q then cover all 64 banks (rows r and
// r + 1 share a 256-byte bank line).
__device__ __forceinline__ uint32_t sk_swz(uint32_t row) { return (row >> 1) & 7; }

// SW: JN = 2, the first 16 rows of W the gate's, the others the up's, of the
// same 16 outputs.
template <int JN, int IM, bool SW>
__global__ __launch_bounds__(kSkThreads, 2) void skinny_kernel(GemmArgs g) {
    constexpr int DEPTH = sk_depth(JN, IM);
    constexpr int BLOCK = 16 * kSkChunk;  // elements of a 16-row block
    constexpr int SLOT = (JN + IM) * BLOCK;
    constexpr uint32_t TILE_N = SW ? 16 : 16 * JN;  // outputs per tile
    static_assert(!SW || JN == 2, "gate and up");
    static_assert(JN * IM * 512 <= SLOT, "the partials fit one slot of each wave");
    // One array per slot of the ring, so that the compiler can tell the one
    // being read from those the DMA is filling.
    __shared__ __align__(1024) uint16_t s_0[kSkWaves * SLOT];
    __shared__ __align__(1024) uint16_t s_1[kSkWaves * SLOT];
    __shared__ __align__(1024) uint16_t s_2[DEPTH > 2 ? kSkWaves * SLOT : 8];
    __shared__ __align__(1024) uint16_t s_3[DEPTH > 3 ? kSkWaves * SLOT : 8];
    const uint32_t T = g.T, N = g.N;
    const int lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // The token tiles of one output tile are 8 blocks apart: on one XCD,
    // whose L2 then serves all but the first read of the weights.
    const uint32_t n_tt = (T + 16 * IM - 1) / (16 * IM);
    uint32_t tm = blockIdx.x / (8 * n_tt) * 8 + blockIdx.x % 8;
    const uint32_t tt = blockIdx.x / 8 % n_tt;
    const uint32_t spans[3] = {(g.rows[0] + TILE_N - 1) / TILE_N, (g.rows[1] + TILE_N - 1) / TILE_N,
                               (g.rows[2] + TILE_N - 1) / TILE_N};
    const int seg = SW ? 0 : segment_of(spans, g.nseg, tm);
    if (tm >= (seg == 0 ? spans[0] : (seg == 1 ? spans[1] : spans[2]))) return;  // padding block
    const uint32_t M = pick3(g.rows, seg);
    const uint32_t m0 = tm * TILE_N, t0 = tt * 16 * IM;
    const uint32_t row_bytes = 2 * N;

    // DMA: one instruction fills eight rows; lane l loads row l / 8's
    // physical chunk l % 8.  The ranges end with the last valid row (rows
    // past it read zeros) and are empty for chunks past N (zeros add nothing).
    uint32_t d_off[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t row = 8 * h + lane / 8;
        d_off[h] = row * row_bytes + 16 * ((lane % 8) ^ sk_swz(row));
    }
    const uint16_t* px = g.x + (size_t)t0 * N + wave * kSkChunk;
    const uint16_t* pw = pick3(g.w, seg) + (size_t)m0 * N + wave * kSkChunk;
    const uint16_t* pu = SW ? g.w[1] + (size_t)m0 * N + wave * kSkChunk : pw;
    uint32_t x_left = min(16u * IM, T - t0) * row_bytes - 2 * kSkChunk * wave;
    uint32_t w_left = min(TILE_N, M - m0) * row_bytes - 2 * kSkChunk * wave;
    const uint32_t n_chunks = N / kSkChunk;
    const uint32_t mine = wave < n_chunks ? (n_chunks - wave + kSkWaves - 1) / kSkWaves : 0;
    uint32_t left = mine;
    auto dma = [&](uint16_t* ring) __attribute__((always_inline)) {
        uint16_t* const st = ring + wave * SLOT;
        const auto rw = make_rsrc(pw, left ? w_left : 0);
        const auto ru = make_rsrc(pu, left ? w_left : 0);
        const auto rx = make_rsrc(px, left ? x_left : 0);
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                dma16(SW && j ? ru : rw, st + j * BLOCK + 512 * h, d_off[h] + (SW ? 0 : 16 * j) * row_bytes);
#pragma unroll
        for (int i = 0; i < IM; ++i)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                dma16(rx, st + (JN + i) * BLOCK + 512 * h, d_off[h] + 16 * i * row_bytes);
        pw += kSkWaves * kSkChunk;
        pu += kSkWaves * kSkChunk;
        px += kSkWaves * kSkChunk;
        w_left -= 2 * kSkWaves * kSkChunk;
        x_left -= 2 * kSkWaves * kSkChunk;
        left -= left != 0;
    };
    // Operand reads: lane l takes row l % 16, k 8 (l / 16) of k-step s.
    int r_off[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
        r_off[s] = (lane & 15) * kSkChunk + 8 * ((4 * s + (lane >> 4)) ^ sk_swz(lane & 15));
    f32x4_t acc[JN][IM];
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int i = 0; i < IM; ++i) acc[j][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int DMAS = 2 * (JN + IM);
    // The slot of `ring` (this wave's oldest DMA), then the slot refilled.
    auto consume = [&](uint16_t* ring) __attribute__((always_inline)) {
        const uint16_t* const st = ring + wave * SLOT;
        __builtin_amdgcn_s_waitcnt(wait_vmcnt((DEPTH - 1) * DMAS));
        asm volatile("" ::: "memory");
        bf16x8_t a[JN][2], b[IM][2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int j = 0; j < JN; ++j)
                a[j][s] = as_bf16x8(*reinterpret_cast<const uint4*>(st + j * BLOCK + r_off[s]));
#pragma unroll
            for (int i = 0; i < IM; ++i)
                b[i][s] = as_bf16x8(*reinterpret_cast<const uint4*>(st + (JN + i) * BLOCK + r_off[s]));
        }
        __builtin_amdgcn_s_waitcnt(kWaitLgkm0);  // read before the DMA below writes there
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        dma(ring);
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int j = 0; j < JN; ++j)
#pragma unroll
                for (int i = 0; i < IM; ++i) acc[j][i] = mfma16x16x32(a[j][s], b[i][s], acc[j][i]);
        __builtin_amdgcn_sched_barrier(0);
    };
    dma(s_0);
    dma(s_1);
    if constexpr (DEPTH > 2) dma(s_2);
    if constexpr (DEPTH > 3) dma(s_3);
    for (uint32_t c = 0; c < mine; c += DEPTH) {
        consume(s_0);
        consume(s_1);
        if constexpr (DEPTH > 2) consume(s_2);
        if constexpr (DEPTH > 3) consume(s_3);
    }
    // The partials go where the operands were, once no DMA writes there.
    __builtin_amdgcn_s_waitcnt(kWaitVmLgkm0);
    __syncthreads();
    float4* const s_red = reinterpret_cast<float4*>(s_0);  // [wave][block][lane]

    // Lane l's value v of block (j, i) is output 16 j + 4 (l / 16) + v of
    // token 16 i + l % 16: add the waves' partials, four outputs per lane.
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int i = 0; i < IM; ++i)
            s_red[(wave * JN * IM + j * IM + i) * 64 + lane] =
                make_float4(acc[j][i][0], acc[j][i][1], acc[j][i][2], acc[j][i][3]);
    __syncthreads();
    auto total = [&](int blk, int l) {
        float4 s = s_red[blk * 64 + l];
#pragma unroll
        for (int w = 1; w < kSkWaves; ++w) {
            const float4 p = s_red[(w * JN * IM + blk) * 64 + l];
            s.x += p.x;
            s.y += p.y;
            s.z += p.z;
            s.w += p.w;
        }
        return s;
    };
    uint16_t* __restrict__ y = pick3(g.y, seg);
    const bool vec = M % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 7) == 0;
    constexpr int GROUPS = (SW ? 1 : JN) * IM * 64;  // of four outputs of one token
    for (int f = threadIdx.x; f < GROUPS; f += kSkThreads) {
        const int blk = f / 64, l = f % 64, i = blk % IM, j = blk / IM;
        const uint32_t tok = t0 + 16 * i + l % 16, m = m0 + 16 * j + 4 * (l / 16);
        float4 s = total(blk, l);
        if constexpr (SW) {
            const float4 u = total(IM + blk, l);
            s.x = swiglu1(bf16_to_f32(f32_to_bf16(s.x)), bf16_to_f32(f32_to_bf16(u.x)));
            s.y = swiglu1(bf16_to_f32(f32_to_bf16(s.y)), bf16_to_f32(f32_to_bf16(u.y)));
            s.z = swiglu1(bf16_to_f32(f32_to_bf16(s.z)), bf16_to_f32(f32_to_bf16(u.z)));
            s.w = swiglu1(bf16_to_f32(f32_to_bf16(s.w)), bf16_to_f32(f32_to_bf16(u.w)));
        }
        if (tok >= T || m >= M) continue;
        uint2 v = make_uint2(pack_bf16x2(s.x, s.y), pack_bf16x2(s.z, s.w));
        uint16_t* dst = y + (size_t)tok * M + m;
        const bool residual = !SW && g.residual;
        if (vec) {
            if (residual) {
                const uint2 o = *reinterpret_cast<const uint2*>(dst);
                v.x = pack_bf16x2(bf16_lo(o.x) + bf16_lo(v.x), bf16_hi(o.x) + bf16_hi(v.x));
                v.y = pack_bf16x2(bf16_lo(o.y) + bf16_lo(v.y), bf16_hi(o.y) + bf16_hi(v.y));
            }
            *reinterpret_cast<uint2*>(dst) = v;
        } else {
            const uint32_t w[2] = {v.x, v.y};
            for (int u = 0; u < 4 && m + u < M; ++u) {
                const uint16_t val = uint16_t(w[u / 2] >> (16 * (u % 2)));
                dst[u] = residual ? f32_to_bf16(bf16_to_f32(dst[u]) + bf16_to_f32(val)) : val;
            }
        }
    }
}

template <int JN, bool SW>
constexpr uint32_t kSkTileN = SW ? 16 : 16 * JN;

template <int JN, int IM, bool SW>
uint32_t skinny_blocks(const GemmArgs& g) {
    uint32_t n_tm = 0;
    for (int s = 0; s < (SW ? 1 : g.nseg); ++s)
        n_tm += (g.rows[s] + kSkTileN<JN, SW> - 1) / kSkTileN<JN, SW>;
    return (n_tm + 7) / 8 * 8 * ((g.T + 16 * IM - 1) / (16 * IM));
}

template <int JN, int IM, bool SW>
hipError_t skinny_launch(const GemmArgs& g, hipStream_t stream) {
    skinny_kernel<JN, IM, SW><<<skinny_blocks<JN, IM, SW>(g), kSkThreads, 0, stream>>>(g);
    return hipGetLastError();
}

// The tile of least modelled cost (us): fixed + rounds * (round + N / 1024 *
// (k + load * the rounds' share of CUs in use)), rounds = blocks per CU, one
// at a time.  Fitted to 84 problems (T 16-256, the projections of 1024-,
// 2560- and 4096-wide layers, weights from HBM): 8-13 % rms, and the tile it
// picks is on average 0.5 % and at most 12 % slower than the fastest.
template <bool SW>
hipError_t skinny_pick(const GemmArgs& g, hipStream_t stream) {
    hipError_t (*best)(const GemmArgs&, hipStream_t) = nullptr;
    float least = 0.0f;
    const float cus = (float)gemm_cus();
    auto consider = [&](uint32_t blocks, float fixed, float round, float k, float load,
                        hipError_t (*launch)(const GemmArgs&, hipStream_t)) {
        const float rounds = ceilf(blocks / cus), use = blocks / (cus * rounds);
        const float cost = fixed + rounds * (round + g.N / 1024.0f * (k + load * use));
        if (best == nullptr || cost < least) {
            least = cost;
            best = launch;
        }
    };
    if constexpr (!SW) {
        consider(skinny_blocks<1, 1, SW>(g), 1.6f, 2.1f, 0.89f, 0.0f, skinny_launch<1, 1, SW>);
        consider(skinny_blocks<1, 2, SW>(g), 1.2f, 2.5f, 1.17f, 0.14f, skinny_launch<1, 2, SW>);
        consider(skinny_blocks<1, 3, SW>(g), 1.3f, 2.0f, 1.39f, 0.32f, skinny_launch<1, 3, SW>);
    }
    consider(skinny_blocks<2, 1, SW>(g), 1.6f, 2.4f, 1.42f, 0.0f, skinny_launch<2, 1, SW>);
    consider(skinny_blocks<2, 2, SW>(g), 1.1f, 2.3f, 1.69f, 0.29f, skinny_launch<2, 2, SW>);
    consider(skinny_blocks<2, 3, SW>(g), 1.1f, 2.6f, 2.04f, 0.25f, skinny_launch<2, 3, SW>);
    return best(g, stream);
}

}  // namespace

hipError_t launch_gemm_skinny(const GemmArgs& g, hipStream_t stream) {
    return g.swiglu ? skinny_pick<true>(g, stream) : skinny_pick<false>(g, stream);
}

}  // namespace tiattn
