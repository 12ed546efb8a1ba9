// Top-k / top-p sampling over fp32 logits on the device: the reference's
// Sampler::sample (src/sampler.cpp:18-67), which runs on the host over logits
// copied back every step (src/engine.cpp:183-190, 443-468).  Here the logits
// stay in HBM and the pick is one launch that a hipGraph can hold.
//
// Same arithmetic as the reference, in its order:
//   x_i = logit_i / T                          (src/sampler.cpp:24-27)
//   top-k set of x (k = min(top_k, vocab))     (:29-32, quick select)
//   p_i = exp((x_i - max x) / T) / sum         (:33-44; T enters twice)
//   sort by p descending, keep the shortest prefix whose running sum
//   exceeds top_p                              (:45-57)
//   coin = u * (that prefix's sum); the first kept token whose running sum
//   exceeds the coin                           (:58-67)
// The uniform draw u comes from the caller (a device float) or, in the model
// harness, from a counter-based hash of (seed, position), so a replayed graph
// draws a fresh coin per step without host work.
//
// Layout: G workgroups of 256 threads (G = 64 for k <= 128, else 32).
// Workgroup b takes the contiguous
// chunk b of the logits (at most 8192, held in registers: element j*256 + t
// in thread t's j-th slot), finds its local k-th largest key by a radix
// select (four 8-bit digit passes over per-wave LDS histograms), and writes
// its top k (keys and indices) to the workspace.  The last workgroup to
// finish (an agent-scope ticket) runs the same select over the G*k
// candidates, sorts the k survivors (by rank in one wave for k <= 64,
// in LDS above), and does the softmax, the top-p cut and the coin walk with
// lane or block scans.  Ties at the k-th value keep the lowest indices;
// equal values are ordered by index.
//
// What bounds it is that chain of dependent steps, not the 0.6 MB of logits.
// For small k both selects are therefore replaced by a filter: a lower bound
// of the k-th largest key (from the 256 threads' own maxima) lets through the
// top k and a few more, and the final ranking drops those.  Where a filter
// lets through too many (heavy ties, rows masked to one value) the select
// runs in its place.  With it, the candidates in four-place loads that are
// all out at once, and the ranking in place of a bitonic sort (us, V =
// 151936): k = 2 15.4 -> 11.7, 20 18.2 -> 12.2, 40 21.7 -> 13.2; by select
// k = 41 21.9 -> 18.6, 64 25.2 -> 20.9, 200 37.1 -> 31.4; V = 8192: k = 20
// 15.4 -> 11.5, 200 30.4 -> 24.6.
#include <hip/hip_runtime.h>

#include "../../include/toyinfer_attn.h"
#include "common.hpp"
#include "kernels.hpp"

namespace tiattn {
namespace {

constexpr int kSpThreads = 256, kSpWaves = kSpThreads / 64;
constexpr int kSpPer = 32;                             // keys per thread, held in registers
constexpr uint32_t kSpChunk = kSpPer * kSpThreads;     // logits (or candidates) per workgroup
// 64 workgroups for k <= 128 (half the chunk per workgroup), 32 above, so
// that the merge's blocks * k candidates always fit one workgroup's slots.
constexpr int kSpBlocksSmallK = 64, kSpBlocksLargeK = 32, kSpSmallK = 128;
static_assert(kSampleMaxK <= kSpThreads, "one thread per kept candidate");
static_assert(kSpBlocksSmallK * kSpSmallK <= kSpChunk && kSpBlocksLargeK * kSampleMaxK <= kSpChunk,
              "candidates fit the per-thread key slots");
static_assert(kSpBlocksLargeK * kSpChunk >= kSampleMaxVocab, "every chunk fits one workgroup");
constexpr uint32_t kSpMaxCand = kSpChunk;
// Filtered selection: k up to kSpFilterK and chunks longer than that.  k keys
// spread over 256 threads leave about k^2 / 512 of them beside a larger one
// of the same thread, and the 16-bit bound a few per cent more, so 40 stay
// within 64 places with room, 20 within 32 and 10 within 16 (each place more
// is one more for the merge to read: k = 20 12.2 us, 21 12.9); at k = 50 some
// of the 64 chunks would run over in many calls, which then pay for both forms.
// Short rows leave most threads without a key to bound with (V = 4095, k = 20:
// 13.2 us by select, 11.5 filtered at 8192).
constexpr uint32_t kSpFilterK = 40, kSpFilterMinVocab = 64 * kSpBlocksSmallK;
static_assert(kSpFilterMinVocab / kSpBlocksSmallK > kSpFilterK, "full chunks exceed k");
__device__ __forceinline__ uint32_t sp_width(uint32_t n, uint32_t k) {
    if (k > kSpFilterK || n < kSpFilterMinVocab) return k;
    return k <= 10 ? 16u : (k <= 20 ? 32u : 64u);
}
static_assert(kSpBlocksSmallK * 64 <= kSpMaxCand, "64 places per chunk fit the workspace");
static_assert(kSpBlocksSmallK % 4 == 0 && kSpBlocksLargeK % 4 == 0 && kSpChunk == 32 * kSpThreads,
              "the merge loads four places at a time");

// Workspace: [0, 8) argmax key, [8, 12) argmax ticket, [12, 16) sampler
// ticket, then keys [G][width] and indices [G][width] from byte 256 (width:
// sp_width; places without a candidate hold key 0, index ~0).
constexpr size_t kSpCandOff = 256;

// Order-preserving map of a float to an unsigned key (larger float, larger key).
__device__ __forceinline__ uint32_t sp_key(float x) {
    const uint32_t b = __float_as_uint(x);
    return b ^ ((b >> 31) ? 0xffffffffu : 0x80000000u);
}
__device__ __forceinline__ float sp_val(uint32_t k) {
    return __uint_as_float((k >> 31) ? (k ^ 0x80000000u) : ~k);
}

// Exclusive prefix sum of one value per thread over the workgroup.
template <typename T>
__device__ __forceinline__ T block_scan_excl(T v, T* s_w, T& total) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    T x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const T y = __shfl_up(x, o);
        if (lane >= o) x += y;
    }
    if (lane == 63) s_w[w] = x;
    __syncthreads();
    T base = 0;
    total = 0;
#pragma unroll
    for (int i = 0; i < kSpWaves; ++i) {
        if (i < w) base += s_w[i];
        total += s_w[i];
    }
    __syncthreads();
    return base + x - v;
}

// Inclusive prefix sum over the 64 lanes of a wave with DPP row shifts and
// row broadcasts (no LDS round trips): within each row of 16 lanes by
// shifts of 1, 2, 3, then 4 and 8 on the upper banks; then row 1 and 3 take
// lane 15 of the row before, rows 2 and 3 lane 31.
__device__ __forceinline__ uint32_t wave_scan_incl(uint32_t v) {
    uint32_t s = v;
    s += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true);
    s += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true);
    s += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x113, 0xf, 0xf, true);
    s += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)s, 0x114, 0xf, 0xe, true);
    s += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)s, 0x118, 0xf, 0xc, true);
    s += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)s, 0x142, 0xa, 0xf, true);
    s += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)s, 0x143, 0xc, 0xf, true);
    return s;
}
template <int CTRL, int ROWS, int BANKS>
__device__ __forceinline__ float dpp_f(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, ROWS, BANKS, true));
}
__device__ __forceinline__ float wave_scan_incl(float v) {
    float s = v + dpp_f<0x111, 0xf, 0xf>(v);
    s += dpp_f<0x112, 0xf, 0xf>(v);
    s += dpp_f<0x113, 0xf, 0xf>(v);
    s += dpp_f<0x114, 0xf, 0xe>(s);
    s += dpp_f<0x118, 0xf, 0xc>(s);
    s += dpp_f<0x142, 0xa, 0xf>(s);
    s += dpp_f<0x143, 0xc, 0xf>(s);
    return s;
}
// The value of lane l - 1 (0 for lane 0): DPP wave_shr:1.
__device__ __forceinline__ float lane_before(float x) { return dpp_f<0x138, 0xf, 0xf>(x); }
__device__ __forceinline__ uint32_t read_lane(uint32_t x, int l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)x, l);
}

struct Sel {
    uint32_t thr;   // the k-th largest key
    uint32_t need;  // how many keys equal to thr belong to the top k
    uint32_t eq;    // how many keys equal thr
};

// The k-th largest of the valid keys of the workgroup (1 <= k <= their
// number): thread t holds element j*256 + t in key[j], valid where bit j of
// `valid` is set.  Four 8-bit digit passes; each wave counts into its own
// histogram (two sets, alternating by pass, so one barrier per pass
// suffices), and every wave then finds the digit itself from the four
// histograms with a lane scan, so no result needs broadcasting.
__device__ __forceinline__ Sel select_kth(const uint32_t (&key)[kSpPer], uint32_t valid, uint32_t k,
                          uint32_t* s_hist, int slots) {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t prefix = 0, mask = 0, need = k, eq = 0;
#pragma unroll
    for (int pass = 0; pass < 4; ++pass) {
        const int shift = 24 - 8 * pass;
        uint32_t* set = s_hist + (pass & 1) * kSpWaves * 256;
        uint32_t* own = set + w * 256;
        *reinterpret_cast<uint4*>(own + 4 * lane) = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (int j = 0; j < kSpPer; ++j) {
            if (j >= slots) break;  // workgroup-uniform: slots past the last key are skipped
            if ((valid >> j & 1u) && (key[j] & mask) == prefix)
                atomicAdd(&own[(key[j] >> shift) & 255u], 1u);
        }
        __syncthreads();
        // Lane l: digits 255-4l down to 252-4l, so that the larger digits sit
        // in the lower lanes.  `above` counts larger digits; exactly one digit
        // has above < need <= above + count.
        uint32_t h[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int ww = 0; ww < kSpWaves; ++ww) {
            const uint4 v = *reinterpret_cast<const uint4*>(set + ww * 256 + 252 - 4 * lane);
            h[0] += v.w;
            h[1] += v.z;
            h[2] += v.y;
            h[3] += v.x;
        }
        const uint32_t t = h[0] + h[1] + h[2] + h[3];
        uint32_t above = wave_scan_incl(t) - t;
        int found = -1;
        uint32_t f_need = 0, f_cnt = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (above < need && need <= above + h[i]) {
                found = 255 - 4 * lane - i;
                f_need = need - above;
                f_cnt = h[i];
            }
            above += h[i];
        }
        const int src = __builtin_ctzll(__ballot(found >= 0));
        prefix |= read_lane((uint32_t)found, src) << shift;
        mask |= 255u << shift;
        need = read_lane(f_need, src);
        eq = read_lane(f_cnt, src);
    }
    return {prefix, need, eq};
}

// Bit j set: element j*256 + t is one of the top k.  Keys above thr all are;
// of the keys equal to thr, the `need` with the smallest indices (a second
// select over the complemented indices when there are more).
__device__ __forceinline__ uint32_t top_mask(const uint32_t (&key)[kSpPer], const uint32_t (&idx)[kSpPer],
                             uint32_t valid, const Sel& s, uint32_t* s_hist, int slots) {
    uint32_t take = 0, tie = 0;
    uint32_t nidx[kSpPer];
#pragma unroll
    for (int j = 0; j < kSpPer; ++j) {
        nidx[j] = 0;
        if (j >= slots) break;
        const bool v = valid >> j & 1u;
        take |= (uint32_t)(v && key[j] > s.thr) << j;
        tie |= (uint32_t)(v && key[j] == s.thr) << j;
        nidx[j] = ~idx[j];
    }
    if (s.eq == s.need) return take | tie;  // uniform over the workgroup
    const Sel t = select_kth(nidx, tie, s.need, s_hist, slots);
#pragma unroll
    for (int j = 0; j < kSpPer; ++j) take |= (uint32_t)((tie >> j & 1u) && nidx[j] >= t.thr) << j;
    return take;
}

// Bits FROM .. TO of the k-th largest of the 256 values v holds per wave, below
// the higher bits t (each wave finds them by itself, bit by bit).
template <int FROM, int TO>
__device__ __forceinline__ uint32_t kth_bits(uint4 v, uint32_t k, uint32_t t) {
#pragma unroll
    for (int bit = FROM; bit >= TO; --bit) {
        const uint32_t c = t | 1u << bit;
        const uint32_t n = __popcll(__ballot(v.x >= c)) + __popcll(__ballot(v.y >= c)) +
                           __popcll(__ballot(v.z >= c)) + __popcll(__ballot(v.w >= c));
        if (n >= k) t = c;
    }
    return t;
}

// A lower bound of the k-th largest valid key of the workgroup: the k-th
// largest of the threads' maxima (left in s_max), its upper 16 bits.  0 when
// fewer than k threads hold a key.
__device__ __forceinline__ uint32_t bound_kth(const uint32_t (&key)[kSpPer], uint32_t valid, uint32_t k,
                                              uint32_t* s_max, int slots) {
    uint32_t mx = 0;
#pragma unroll
    for (int j = 0; j < kSpPer; ++j) {
        if (j >= slots) break;
        mx = max(mx, valid >> j & 1u ? key[j] : 0u);
    }
    s_max[threadIdx.x] = mx;
    __syncthreads();
    return kth_bits<31, 16>(reinterpret_cast<const uint4*>(s_max)[threadIdx.x & 63], k, 0);
}

// Emits the valid keys from that bound on, at least the top k with all ties,
// if there are at most `room` of them; returns how many there are.
template <typename F>
__device__ __forceinline__ uint32_t filter_top(const uint32_t (&key)[kSpPer], uint32_t valid, uint32_t room,
                                               uint32_t bound, uint32_t* s_cnt, int slots, F&& emit) {
    uint32_t take = 0;
#pragma unroll
    for (int j = 0; j < kSpPer; ++j) {
        if (j >= slots) break;
        take |= (uint32_t)((valid >> j & 1u) && key[j] >= bound) << j;
    }
    const uint32_t n = __popc(take);
    const uint32_t incl = wave_scan_incl(n);
    uint32_t base = 0;
    if ((threadIdx.x & 63) == 63) base = atomicAdd(s_cnt, incl);
    uint32_t slot = read_lane(base, 63) + incl - n;
    __syncthreads();
    const uint32_t total = *s_cnt;
    if (total <= room) {
#pragma unroll
        for (int j = 0; j < kSpPer; ++j)
            if (j < slots && (take >> j & 1u)) emit(slot++, j);
    }
    return total;
}

// The k-th largest key after a filter that let through too many, without the
// select's four passes where it is among many equals (rows of equal or masked
// keys) or, in a chunk, almost always.
// CHUNK: all bits of the k-th largest of the maxima, if fewer than k keys lie
// above it (then k keys lie at or above it).  Candidates, of which a thread
// holds neighbours, so that one chunk's top keys share few threads: any key with
// the bound's upper 16 bits, if the top k end among its equals.
// V = 151936, k = 20: all equal 38.5 us by the select alone, 40.4 after the filter,
// 28.3 so; 300 tokens allowed 31.5, 30.0, 22.5.  need 0: not found.
template <bool CHUNK>
__device__ __forceinline__ Sel kth_after_filter(const uint32_t (&key)[kSpPer], uint32_t valid, uint32_t k,
                                                uint32_t bound, const uint32_t* s_max, uint32_t* s_cnt,
                                                int slots) {
    uint32_t t;
    if constexpr (CHUNK) {
        t = kth_bits<15, 0>(reinterpret_cast<const uint4*>(s_max)[threadIdx.x & 63], k, bound);
    } else {
#pragma unroll
        for (int j = 0; j < kSpPer; ++j) {
            if (j >= slots) break;
            // (whichever lane's write lands last)
            if ((valid >> j & 1u) && key[j] >> 16 == bound >> 16) s_cnt[1] = key[j];
        }
        __syncthreads();
        t = s_cnt[1];
    }
    uint32_t n = 0;  // keys above t, and equal ones in the upper half (8192 at most)
#pragma unroll
    for (int j = 0; j < kSpPer; ++j) {
        if (j >= slots) break;
        if (valid >> j & 1u) n += key[j] > t ? 1u : (key[j] == t ? 0x10000u : 0u);
    }
    const uint32_t sum = wave_scan_incl(n);
    if ((threadIdx.x & 63) == 63) atomicAdd(s_cnt, sum);
    __syncthreads();
    const uint32_t above = *s_cnt & 0xffffu, eq = *s_cnt >> 16;
    return {t, above < k && above + eq >= k ? k - above : 0u, eq};
}

// Slots 0..k-1 for the set bits of `take` across the workgroup (any order):
// a wave scan of the per-thread counts and one LDS atomic per wave.
template <typename F>
__device__ __forceinline__ void emit_top(uint32_t take, uint32_t k, int slots, uint32_t* s_cnt,
                                         F&& emit) {
    const int lane = threadIdx.x & 63;
    const uint32_t n = __popc(take);
    const uint32_t incl = wave_scan_incl(n);
    uint32_t base = 0;
    if (lane == 63) base = atomicAdd(s_cnt, incl);
    uint32_t slot = read_lane(base, 63) + incl - n;
#pragma unroll
    for (int j = 0; j < kSpPer; ++j)
        if (j < slots && (take >> j & 1u) && slot < k) emit(slot++, j);  // exactly k bits are set
}

// Emits the top k of the workgroup's valid keys, all of them and up to `room`
// keys by the filter, or exactly k; returns how many.  s_cnt: four words, 0.
// Candidates of which the filter passes fewer than half are not equals: select.
template <bool CHUNK, typename F>
__device__ __forceinline__ uint32_t emit_selected(const uint32_t (&key)[kSpPer], const uint32_t (&idx)[kSpPer],
                                                  uint32_t valid, uint32_t k, bool filter, uint32_t room,
                                                  uint32_t* s_max, uint32_t* s_cnt, uint32_t* s_hist,
                                                  int slots, F&& emit) {
    uint32_t n = ~0u, bound = 0;
    if (filter) {
        bound = bound_kth(key, valid, k, s_max, slots);
        n = filter_top(key, valid, room, bound, s_cnt, slots, emit);
        if (n <= room) return n;
    }
    Sel s = {0, 0, 0};
    if (filter && (CHUNK || n >= kSpBlocksSmallK * k / 2))
        s = kth_after_filter<CHUNK>(key, valid, k, bound, s_max, s_cnt + 1, slots);
    if (s.need == 0) s = select_kth(key, valid, k, s_hist, slots);
    emit_top(top_mask(key, idx, valid, s, s_hist, slots), k, slots, s_cnt + 3, emit);
    return k;
}

// SplitMix64 finaliser (Steele, Lea and Flood, "Fast splittable pseudorandom
// number generators", 2014) of seed + (pos + 1) * golden gamma; the top 24
// bits give u in [0, 1).
__device__ __forceinline__ float sp_coin(uint64_t seed, uint32_t pos) {
    uint64_t z = seed + (uint64_t)(pos + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (float)(uint32_t)(z >> 40) * 0x1p-24f;
}

// Writes the picked token (and advances the position) from thread 0.
__device__ __forceinline__ void sp_write(const SampleArgs& a, uint32_t p_out, uint32_t idx,
                                         uint32_t* ticket) {
    *ticket = 0;
    if (a.pos) {
        if (p_out + 1 < a.out_cap) a.out[p_out + 1] = idx;
        *a.pos = p_out + 1;
    } else {
        a.out[0] = idx;
    }
}

__global__ __launch_bounds__(kSpThreads) void sample_kernel(SampleArgs a) {
    __shared__ __align__(16) uint32_t s_hist[2 * kSpWaves * 256];
    __shared__ float s_wf[kSpWaves];
    __shared__ __align__(16) uint32_t s_max[kSpThreads];
    __shared__ uint64_t s_top[kSampleMaxK];
    __shared__ uint64_t s_sorted[64];
    __shared__ float s_acc[kSampleMaxK];
    __shared__ uint32_t s_res[2], s_cnt[8];  // s_cnt: emit_selected's, of either phase
    __shared__ bool s_last;

    const uint32_t k = a.k, tid = threadIdx.x;
    char* ws = static_cast<char*>(a.workspace);
    uint32_t* ticket = reinterpret_cast<uint32_t*>(ws + 12);
    uint32_t* ws_key = reinterpret_cast<uint32_t*>(ws + kSpCandOff);
    const uint32_t G = gridDim.x;
    const uint32_t width = sp_width(a.n, k);
    const bool filter = width != k;
    uint32_t* ws_idx = ws_key + G * width;
    if (tid < 8) s_cnt[tid] = 0;

    // Phase 1: this workgroup's chunk, element j*256 + t in thread t's key[j].
    const uint32_t cs = (a.n + G - 1) / G;
    const uint32_t c0 = min(a.n, blockIdx.x * cs), m = min(a.n, c0 + cs) - c0;
    uint32_t key[kSpPer], idx[kSpPer], valid = 0;
    {
        // Range-checked buffer loads: no branch per slot, zeros past the chunk.
        const __amdgpu_buffer_rsrc_t r = make_rsrc(a.logits + c0, m * 4);
        const int slots = (int)((m + kSpThreads - 1) / kSpThreads);
        float x[kSpPer];
#pragma unroll
        for (int j = 0; j < kSpPer; ++j)
            x[j] = j < slots ? __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(
                                   r, 4 * (j * kSpThreads + tid), 0, 0))
                             : 0.0f;
#pragma unroll
        for (int j = 0; j < kSpPer; ++j) {
            const uint32_t e = j * kSpThreads + tid;
            key[j] = sp_key(x[j] / a.temperature);
            idx[j] = c0 + e;
            valid |= (uint32_t)(e < m) << j;
        }
    }
    uint32_t* bk = ws_key + blockIdx.x * width;
    uint32_t* bi = ws_idx + blockIdx.x * width;
    if (m <= k) {
        // The whole chunk; key 0 pads (below every key of a non-NaN float).
#pragma unroll
        for (int j = 0; j < kSpPer; ++j) {
            const uint32_t e = j * kSpThreads + tid;
            if (e < width) {
                bk[e] = e < m ? key[j] : 0u;
                bi[e] = e < m ? idx[j] : 0xffffffffu;
            }
        }
    } else {
        const int slots = (int)((m + kSpThreads - 1) / kSpThreads);
        auto emit = [&](uint32_t slot, int j) {
            bk[slot] = key[j];
            bi[slot] = idx[j];
        };
        const uint32_t n =
            emit_selected<true>(key, idx, valid, k, filter, width, s_max, s_cnt, s_hist, slots, emit);
        if (tid >= n && tid < width) {
            bk[tid] = 0u;
            bi[tid] = 0xffffffffu;
        }
    }
    // Every wave waits for its own stores to reach the L2, the barrier joins
    // them, and one agent-scope release (not one per wave) publishes the
    // chunk before the ticket; the last workgroup's acquire precedes its reads
    // of the other chunks.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
        __threadfence();
        s_last = atomicAdd(ticket, 1u) == G - 1;
        if (s_last) __threadfence();
    }
    __syncthreads();
    if (!s_last) return;

    // Phase 2 (last workgroup): the top k of the G*width candidates, as
    // (key << 32 | ~index) so that one ordering covers the ties; `found` of
    // them in s_top, the top k among them.
    const uint32_t nc = G * width;
    uint32_t found;
    valid = 0;
    // Four places per load (nc is a multiple of 4), every load out before the
    // first is waited for.
    const int slots = 4 * (int)((nc + 4 * kSpThreads - 1) / (4 * kSpThreads));
    {
        const __amdgpu_buffer_rsrc_t rk = make_rsrc(ws_key, nc * 4), ri = make_rsrc(ws_idx, nc * 4);
#pragma unroll
        for (int j = 0; j < kSpPer; j += 4) {
            if (j >= slots) break;
            const uint32_t e = j * kSpThreads + 4 * tid;
            const uint4 x = buf_load16(rk, 4 * e), y = buf_load16(ri, 4 * e);
            key[j] = x.x, key[j + 1] = x.y, key[j + 2] = x.z, key[j + 3] = x.w;
            idx[j] = y.x, idx[j + 1] = y.y, idx[j + 2] = y.z, idx[j + 3] = y.w;
            valid |= (e < nc ? 15u : 0u) << j;
        }
    }
    {
        auto emit = [&](uint32_t slot, int j) {
            s_top[slot] = ((uint64_t)key[j] << 32) | (uint32_t)~idx[j];
        };
        found = emit_selected<false>(key, idx, valid, k, filter, 64, s_max, s_cnt + 4, s_hist, slots, emit);
    }
    uint32_t p_out = 0;
    if (a.pos) p_out = *a.pos;
    const float u = a.coin ? *a.coin : sp_coin(a.seed, p_out);
    __syncthreads();

    if (k <= 64) {
        // One wave: each lane counts the keys above its own (all differ: the
        // index is part of them) and puts it at that place, then softmax,
        // running sums, the top-p cut and the coin walk with lane scans.
        if (tid >= 64) return;
        const int lane = tid;
        if ((uint32_t)lane >= found) s_top[lane] = 0;
        // The wave's LDS accesses run in order; the fences keep the compiler's.
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const uint64_t own = s_top[lane];
        uint32_t rank = 0;
        for (uint32_t i = 0; i < found; i += 4) {  // places past `found` hold 0
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) rank += s_top[i + u] > own;
        }
        if ((uint32_t)lane < found) s_sorted[rank] = own;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        const uint64_t v = (uint32_t)lane < k ? s_sorted[lane] : 0ull;
        const bool in = (uint32_t)lane < k;
        const float x = sp_val((uint32_t)(v >> 32));
        const float xmax = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
        const float p = in ? expf((x - xmax) / a.temperature) : 0.0f;
        const float sum = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wave_scan_incl(p)), 63));
        const float acc = wave_scan_incl(p / sum);
        const float prev = lane_before(acc);
        const uint64_t cut = __ballot(in && acc > a.top_p && (lane == 0 || !(prev > a.top_p)));
        const uint32_t kept = cut ? (uint32_t)__builtin_ctzll(cut) + 1 : k;
        const float coin = u * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(acc), kept - 1));
        const uint64_t hit = __ballot((uint32_t)lane < kept && acc > coin &&
                                      (lane == 0 || !(prev > coin)));
        const int pick = hit ? __builtin_ctzll(hit) : (int)kept - 1;
        const uint64_t chosen = __shfl(v, pick);
        if (lane == 0) sp_write(a, p_out, ~(uint32_t)chosen, ticket);
        return;
    }

    // k > 64: bitonic sort in LDS over the workgroup, block scans.
    if (tid >= k && tid < kSampleMaxK) s_top[tid] = 0;
    uint32_t n2 = 1;
    while (n2 < k) n2 <<= 1;
    for (uint32_t size = 2; size <= n2; size <<= 1) {
        for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
            __syncthreads();
            const uint32_t j = tid ^ stride;
            if (tid < n2 && j > tid) {
                const uint64_t x = s_top[tid], y = s_top[j];
                const bool desc = (tid & size) == 0;
                if ((x < y) == desc) {
                    s_top[tid] = y;
                    s_top[j] = x;
                }
            }
        }
    }
    __syncthreads();
    const float xmax = sp_val((uint32_t)(s_top[0] >> 32));
    const float p = tid < k ? expf((sp_val((uint32_t)(s_top[tid] >> 32)) - xmax) / a.temperature) : 0.0f;
    float sum;
    (void)block_scan_excl(p, s_wf, sum);
    const float q = p / sum;
    float qtot;
    const float acc = block_scan_excl(q, s_wf, qtot) + q;
    if (tid < k) s_acc[tid] = acc;
    if (tid == 0) {
        s_res[0] = k;
        s_res[1] = 0xffffffffu;
    }
    __syncthreads();
    // Kept prefix: through the first running sum above top_p (all k if none).
    if (tid < k && acc > a.top_p && (tid == 0 || !(s_acc[tid - 1] > a.top_p))) s_res[0] = tid + 1;
    __syncthreads();
    const uint32_t kept = s_res[0];
    const float coin = u * s_acc[kept - 1];
    if (tid < kept && acc > coin && (tid == 0 || !(s_acc[tid - 1] > coin))) s_res[1] = tid;
    __syncthreads();
    if (tid == 0) {
        const uint32_t pick = s_res[1] != 0xffffffffu ? s_res[1] : kept - 1;
        sp_write(a, p_out, ~(uint32_t)s_top[pick], ticket);
    }
}

}  // namespace

size_t sample_workspace_bytes() { return kSpCandOff + 2ull * kSpMaxCand * 4; }

int sample_config(uint32_t vocab, float temperature, uint32_t top_k, float top_p, SampleArgs& a) {
    if (vocab == 0 || !(temperature >= 0.0f)) return TOYINFER_ERR_INVALID_ARGUMENT;
    a.n = vocab;
    a.temperature = temperature;
    a.top_p = top_p;
    // src/sampler.cpp:20-22: greedy below 1e-3 or for top_k == 1.
    a.greedy = temperature < 1e-3f || top_k == 1;
    if (a.greedy) {
        a.k = 1;
        return TOYINFER_OK;
    }
    if (top_k == 0) return TOYINFER_ERR_INVALID_ARGUMENT;  // the reference asserts k > 0
    a.k = top_k < vocab ? top_k : vocab;                   // :29-30
    return a.k <= kSampleMaxK && vocab <= kSampleMaxVocab ? TOYINFER_OK : TOYINFER_ERR_UNSUPPORTED;
}

hipError_t launch_sample(const SampleArgs& a, hipStream_t stream) {
    if (a.greedy) {
        char* ws = static_cast<char*>(a.workspace);
        return launch_argmax_wide(a.logits, a.n, a.out, a.pos, a.out_cap,
                                  reinterpret_cast<uint64_t*>(ws), reinterpret_cast<uint32_t*>(ws + 8),
                                  stream);
    }
    sample_kernel<<<a.k <= kSpSmallK ? kSpBlocksSmallK : kSpBlocksLargeK, kSpThreads, 0, stream>>>(a);
    return hipGetLastError();
}

}  // namespace tiattn
