// gfx950 kernels of one EZLDA Gibbs sweep.
//
// Stage order per sweep (reference EZLDA/mainKernel.cu:158-380):
//   begin (clears what the counts add to, moves the sweep counter on)
//   -> topic_hist (n_k), wt_head, wt_tail (WT from z) -> inv_order + word_top
//   (phi top-3) -> dt_build (DT rows + per-token aux) -> sample (three-bucket
//   draw, writes z).
// Every float operation follows the canonical order of the CPU oracle
// (oracle/ezlda_oracle.c); builds use -ffp-contract=off, so the topics agree
// bit for bit.  Wave64: one wavefront owns a doc (dt_build) or a tail word
// (wt_tail, word_top); in the sampler one lane owns a token.
#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>

#include "ezlda_device.h"
#include "ezlda_philox.h"

// Sampler row blocking (16-byte loads per block, checkpoints per lane).
// DT rows are padded to multiples of 32 entries, so blocks up to 8 loads
// never read past a row's padding.
#ifndef EZ_SAMPLE_BLK
#define EZ_SAMPLE_BLK 4
#endif
#ifndef EZ_SAMPLE_CP
#define EZ_SAMPLE_CP 12
#endif
// Largest K whose sampler keeps a table of the Q running sums inside each
// 64-topic slab in LDS (a Q draw then bisects it); above it a Q draw
// recomputes its slab's running sums, which halves the sampler's LDS.
#ifndef EZ_Q_TABLE_MAX_K
#define EZ_Q_TABLE_MAX_K 1024
#endif
static_assert(EZ_Q_TABLE_MAX_K <= 8192, "the Q-table sampler variants assume compact (K <= 8192) DT rows");

namespace ez {

static constexpr float kMargin = 0.998046875f;  // 1 - 2^-9
static constexpr uint32_t kNone = 0xFFFFu;

// ---------------------------------------------------------------- helpers
__device__ __forceinline__ float readlane_f(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}
__device__ __forceinline__ uint32_t readlane_u(uint32_t v, int l) {
    return (uint32_t)__builtin_amdgcn_readlane((int)v, l);
}
__device__ __forceinline__ int first_lane(uint64_t m) { return __ffsll((unsigned long long)m) - 1; }
__device__ __forceinline__ uint64_t lanemask_lt(int lane) { return (1ull << lane) - 1ull; }

// Orders LDS traffic between the phases of one wavefront.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

static int grid_for(size_t n, int bd, int cap) {
    size_t g = (n + (size_t)bd - 1) / (size_t)bd;
    if (g < 1) g = 1;
    if (g > (size_t)cap) g = (size_t)cap;
    return (int)g;
}

static size_t wave_hist_bytes(int K) { return (size_t)((K + 1) >> 1) * sizeof(uint32_t); }
// DT rebuild: 16-bit counts plus a topic bitmap per wavefront
static size_t dt_wave_bytes(int K) { return wave_hist_bytes(K) + (size_t)((K + 31) >> 5) * sizeof(uint32_t); }

// the same without the bitmap, whole 16-byte words
__host__ __device__ static inline size_t scan_wave_bytes(int K) { return ((size_t)((K + 1) >> 1) + 3) / 4 * 16; }

// Launch of a kernel whose wavefronts each own wb bytes of LDS (cleared
// when the wavefront starts) and stride over n units (words, docs).  When
// at least 16 wavefronts' LDS fits on a CU: workgroups of four wavefronts,
// one unit each (up to cap workgroups), which the dispatcher balances.
// Otherwise (large K, where clearing the LDS costs more than a unit):
// persistent one-wavefront workgroups, as many as the CUs' LDS holds.
struct WaveGrid {
    int grid, nwv;
};
static WaveGrid wave_grid(const DevState &s, size_t n, size_t wb, int cap) {
    const size_t fit = wb ? (size_t)s.lds_cu / wb : 32;
    if (fit >= 16) return {grid_for(n, 4, cap), 4};
    return {grid_for(n, 1, s.n_cu * (int)std::max<size_t>(1, fit)), 1};
}

// A DT entry is (topic << 2) | (count << 16): its low half is the byte
// offset of phi[topic] in a float array, so a gather needs one AND.
__device__ __forceinline__ uint32_t dt_topic(uint32_t e) { return (e & 0xFFFFu) >> 2; }
__device__ __forceinline__ float dt_count(uint32_t e) { return (float)(e >> 16); }

// Compact DT rows (K <= 8192): 16-bit entries topic | piece << tb, tb =
// max(10, ceil(log2 K)) topic bits; a count stored in pieces of at most
// 2^(16 - tb) - 1.  Decoders take the low 16 bits of e.
__device__ __forceinline__ float c16_count(uint32_t e, uint32_t tb) { return (float)((e & 0xFFFFu) >> tb); }
__device__ __forceinline__ uint32_t c16_topic(uint32_t e, uint32_t tb) { return e & ((1u << tb) - 1u); }

// phi of a DT entry, its table at LDS address 0 (the sampler's dynamic LDS
// when the kernel has no static LDS, which sampler_static_lds() lets the host
// check): the entry's low half is the address itself, no base to add.
typedef __attribute__((address_space(3))) const float lds_cfloat;
__device__ __forceinline__ float phi_at0(uint32_t e) { return *(lds_cfloat *)(e & 0xFFFCu); }

// 16-bit counters, two per LDS word (counts < 65536 by construction).
__device__ __forceinline__ void h16_add(uint32_t *h, uint32_t k) {
    atomicAdd(&h[k >> 1], 1u << ((k & 1u) << 4));
}

__device__ __forceinline__ uint32_t h16_get(const uint32_t *h, uint32_t k) {
    return (h[k >> 1] >> ((k & 1u) << 4)) & 0xFFFFu;
}

// ------------------------------------------------------------ count reset
__global__ void k_fill_u32(uint32_t *__restrict__ p, size_t n, uint32_t v) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ void k_set_u32(uint32_t *p, uint32_t v) { *p = v; }
__global__ void k_inc_u32(uint32_t *p) { *p = *p + 1u; }

// ------------------------------------------------------- n_k histogram
// Adds the topics of tokens [0, n) of zs to the LDS histogram sh: lanes take
// groups of eight tokens (one 16-byte load) i0, i0 + stride, ..., and add
// each run of equal neighbouring topics among them with one atomic (word-
// major neighbours often share a topic, and equal topics in one LDS
// instruction contend for one address).  The lane with i0 == 0 also adds the
// tokens before the first 16-byte boundary and after the last whole group.
__device__ __forceinline__ void hist_add_tokens(uint32_t *sh, const uint16_t *__restrict__ zs, size_t n, size_t i0,
                                                size_t stride) {
    const size_t mis = ((16u - ((uintptr_t)zs & 15u)) & 15u) >> 1;
    const size_t head = mis < n ? mis : n;
    const size_t n8 = (n - head) >> 3;
    const uint4 *z8 = reinterpret_cast<const uint4 *>(zs + head);
    for (size_t i = i0; i < n8; i += stride) {
        const uint4 v = z8[i];
        const uint32_t t[8] = {v.x & 0xFFFFu, v.x >> 16, v.y & 0xFFFFu, v.y >> 16,
                               v.z & 0xFFFFu, v.z >> 16, v.w & 0xFFFFu, v.w >> 16};
        uint32_t c = 1;
#pragma unroll
        for (int j = 0; j < 7; ++j) {
            if (t[j + 1] != t[j]) {
                atomicAdd(&sh[t[j]], c);
                c = 1;
            } else {
                ++c;
            }
        }
        atomicAdd(&sh[t[7]], c);
    }
    if (i0 == 0) {
        for (size_t i = 0; i < head; ++i) atomicAdd(&sh[zs[i]], 1u);
        for (size_t i = head + (n8 << 3); i < n; ++i) atomicAdd(&sh[zs[i]], 1u);
    }
}

// n_k = column sums of WT (WTDen_Sum_Update_Kernel utility.cu:1104-1126 plus
// the tail's atomicAdd in sparseMatrixAdd :1132-1204): one LDS histogram of
// z per workgroup, flushed with one atomic per nonzero topic.
// (block `blk` of `nblk`; the kernel below, or a role of k_wt_all)
__device__ __forceinline__ void topic_hist_block(uint32_t *sh, const uint16_t *__restrict__ z, uint32_t N, int K,
                                                 int32_t *__restrict__ nk, uint32_t blk, uint32_t nblk) {
    for (int k = threadIdx.x; k < K; k += blockDim.x) sh[k] = 0;
    __syncthreads();
    hist_add_tokens(sh, z, N, (size_t)blk * blockDim.x + threadIdx.x, (size_t)nblk * blockDim.x);
    __syncthreads();
    for (int k = threadIdx.x; k < K; k += blockDim.x) {
        uint32_t c = sh[k];
        if (c) atomicAdd(&nk[k], (int32_t)c);
    }
}
__global__ void k_topic_hist(const uint16_t *__restrict__ z, uint32_t N, int K, int32_t *__restrict__ nk) {
    extern __shared__ uint32_t sh[];
    topic_hist_block(sh, z, N, K, nk, blockIdx.x, gridDim.x);
}

// ------------------------------------------------------------- head WT
// Dense head rows (WTDen_Update_Kernel, utility.cu:1067-1102): one workgroup
// per segment of a head word's tokens, LDS histogram, atomic flush into the
// (pre-zeroed) row; with `fresh`, the only segment of a word writes its whole
// row, which then needs no zeroing: 20,011 words at K = 4096 (328 MB) 125 ->
// 57 us, the time of one pass of writes.
__device__ __forceinline__ void wt_head_block(uint32_t *sh, const uint16_t *__restrict__ z,
                                              const uint4 *__restrict__ segs, int K, int32_t *__restrict__ wt_head,
                                              bool fresh, uint32_t seg) {
    const uint4 sg = segs[seg];
    for (int k = threadIdx.x; k < K; k += blockDim.x) sh[k] = 0;
    __syncthreads();
    hist_add_tokens(sh, z + sg.y, sg.z - sg.y, threadIdx.x, blockDim.x);
    __syncthreads();
    int32_t *row = wt_head + (size_t)sg.x * K;
    if (fresh && sg.w) {
        if ((K & 3) == 0)
            for (int k = threadIdx.x; k < K >> 2; k += blockDim.x)
                reinterpret_cast<uint4 *>(row)[k] = reinterpret_cast<const uint4 *>(sh)[k];
        else
            for (int k = threadIdx.x; k < K; k += blockDim.x) row[k] = (int32_t)sh[k];
        return;
    }
    for (int k = threadIdx.x; k < K; k += blockDim.x) {
        uint32_t c = sh[k];
        if (c) atomicAdd(&row[k], (int32_t)c);
    }
}
__global__ void k_wt_head(const uint16_t *__restrict__ z, const uint4 *__restrict__ segs, int K,
                          int32_t *__restrict__ wt_head, bool fresh) {
    extern __shared__ uint32_t sh[];
    wt_head_block(sh, z, segs, K, wt_head, fresh, blockIdx.x);
}

// ------------------------------------------------------ sorted topics
// Bitonic sort, ascending, of 64 NU topics of a wavefront in registers
// (element 64 u + lane in x[u]): partners 64 or more apart are in the same
// lane, the others are fetched by a lane swizzle.
template <int NU>
__device__ __forceinline__ void sort_topics(uint32_t (&x)[NU], uint32_t lane) {
#pragma unroll
    for (uint32_t k = 2; k <= 64u * NU; k <<= 1) {
#pragma unroll
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
#pragma unroll
            for (uint32_t u = 0; u < (uint32_t)NU; ++u) {
                if (j >= 64) {
                    const uint32_t v = u ^ (j >> 6);
                    if (v > u) {
                        const bool up = ((64u * u) & k) == 0;
                        const uint32_t lo = min(x[u], x[v]), hi = max(x[u], x[v]);
                        x[u] = up ? lo : hi;
                        x[v] = up ? hi : lo;
                    }
                } else {
                    const uint32_t o = __shfl_xor(x[u], (int)j);
                    const bool up = ((64u * u + lane) & k) == 0, first = (lane & j) == 0;
                    x[u] = up == first ? min(x[u], o) : max(x[u], o);
                }
            }
        }
    }
}

// Sorts the n <= 64 NU topics that load(i) gives into key[0, 64 NU) (LDS),
// 0xFFFF past them; NU the power of two that n needs.
template <typename Load>
__device__ __forceinline__ void sort_into(uint16_t *key, uint32_t n, uint32_t lane, Load &&load) {
    auto go = [&](auto nu) {
        constexpr int NU = decltype(nu)::value;
        uint32_t x[NU];
#pragma unroll
        for (int u = 0; u < NU; ++u) x[u] = lane + 64u * u < n ? load(u) : 0xFFFFu;
        sort_topics<NU>(x, lane);
#pragma unroll
        for (int u = 0; u < NU; ++u) key[lane + 64 * u] = (uint16_t)x[u];
    };
    if (n <= 64)
        go(std::integral_constant<int, 1>{});
    else if (n <= 128)
        go(std::integral_constant<int, 2>{});
    else if (n <= 256)
        go(std::integral_constant<int, 4>{});
    else
        go(std::integral_constant<int, 8>{});
    static_assert(kDtShort == 512, "at most eight topics a lane");
}

// Lengths of the runs of equal topics of key[0, n): len(u) of the run that
// starts at 64 u + lane (0: none starts there), hm the heads by 64.
struct TopicRuns {
    uint64_t hm[kDtShort / 64];
    int nu;
    __device__ __forceinline__ TopicRuns(const uint16_t *key, uint32_t n, uint32_t lane) {
        nu = (int)((n + 63u) >> 6);
#pragma unroll
        for (int u = 0; u < (int)(kDtShort / 64); ++u) {
            const uint32_t i = lane + 64u * u;
            hm[u] = __ballot(u < nu && i < n && (i == 0 || key[i - 1] != key[i]));
        }
    }
    __device__ __forceinline__ uint32_t len(int u, uint32_t n, uint32_t lane) const {
        if (!((hm[u] >> lane) & 1ull)) return 0u;
        const uint64_t above = hm[u] & ~((2ull << lane) - 1ull);
        uint32_t nxt = n;  // the first head after it
        if (above) {
            nxt = 64u * u + (uint32_t)first_lane(above);
        } else {
#pragma unroll
            for (int v = (int)(kDtShort / 64) - 1; v >= 0; --v)
                if (v > u && v < nu && hm[v]) nxt = 64u * v + (uint32_t)first_lane(hm[v]);
        }
        return nxt - (64u * u + lane);
    }
};

// ------------------------------------------------------------- tail WT
// Sorted sparse tail rows (WT_Update_Kernel, utility.cu:10-76): one
// wavefront per tail word; a 16-bit LDS histogram and a bitmap of the
// word's topics, then a compaction over the bitmap in ascending topic order
// (lane j owns topics [32j, 32j + 32) of each 64-word chunk and takes its
// place from a wave prefix sum), clearing its counts and bitmap as it goes.
__device__ __forceinline__ void wt_tail_block(uint32_t *sh, const uint16_t *__restrict__ z,
                                              const uint32_t *__restrict__ word_off, int VD, int V, int K,
                                              const uint32_t *__restrict__ tail_off, uint32_t *__restrict__ wt_tail,
                                              uint32_t *__restrict__ tail_nnz, int blk, int nblk) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
    const int KH = (K + 1) >> 1, NW = (K + 31) >> 5;
    uint32_t *h = sh + wv * (KH + NW);  // 16-bit counts
    uint32_t *bm = h + KH;              // bitmap of the word's topics
    for (int k = lane; k < KH + NW; k += 64) h[k] = 0;
    wave_lds_sync();
    const int ntail = V - VD;
    for (int tw = blk * nwv + wv; tw < ntail; tw += nblk * nwv) {
        const int w = VD + tw;
        const uint32_t b = word_off[w], e = word_off[w + 1];
        if (b == e) {
            if (lane == 0) tail_nnz[tw] = 0;
            continue;
        }
        for (uint32_t i = b + lane; i < e; i += 64) {
            const uint32_t t = z[i];
            h16_add(h, t);
            atomicOr(&bm[t >> 5], 1u << (t & 31u));
        }
        wave_lds_sync();
        const uint32_t base = tail_off[tw];
        uint32_t nz = 0;
        for (int j = 0; j < NW; j += 64) {
            const int wi = j + lane;
            const uint32_t word = wi < NW ? bm[wi] : 0u;
            const uint32_t m = (uint32_t)__popc(word);
            uint32_t incl = m;  // inclusive scan over lanes
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t v = __shfl_up(incl, d);
                if (lane >= d) incl += v;
            }
            uint32_t pos = nz + incl - m;
            for (uint32_t x = word; x; x &= x - 1u) {
                const uint32_t k = ((uint32_t)wi << 5) + (uint32_t)__ffs(x) - 1u;
                wt_tail[base + pos++] = k | (h16_get(h, k) << 16);
            }
            for (uint32_t x = word; x; x &= x - 1u) {  // the lane's own 16 count words
                const uint32_t k = ((uint32_t)wi << 5) + (uint32_t)__ffs(x) - 1u;
                h[k >> 1] = 0;
            }
            if (wi < NW) bm[wi] = 0;
            nz += __shfl(incl, 63);
        }
        wave_lds_sync();
        if (lane == 0) tail_nnz[tw] = nz;
    }
}
__global__ void k_wt_tail(const uint16_t *__restrict__ z, const uint32_t *__restrict__ word_off, int VD, int V,
                          int K, const uint32_t *__restrict__ tail_off, uint32_t *__restrict__ wt_tail,
                          uint32_t *__restrict__ tail_nnz) {
    extern __shared__ uint32_t sh[];
    wt_tail_block(sh, z, word_off, VD, V, K, tail_off, wt_tail, tail_nnz, blockIdx.x, gridDim.x);
}

// The rows of tail words of at most kDtShort tokens at large K, where a
// K-sized histogram leaves a CU few wavefronts (seven at K = 10000, 95 us for
// 29,600 words, of which 29,200 take 22 us here): a wavefront sorts its word's
// topics.
__global__ void __launch_bounds__(256) k_wt_sort(const uint16_t *__restrict__ z, const uint32_t *__restrict__ word_off,
                                                 int w0, int VD, int V, const uint32_t *__restrict__ tail_off,
                                                 uint32_t *__restrict__ wt_tail, uint32_t *__restrict__ tail_nnz) {
    __shared__ uint16_t keys[4][kDtShort];
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6;
    uint16_t *key = keys[wv];
    for (int w = w0 + (int)(blockIdx.x * 4u + wv); w < V; w += (int)gridDim.x * 4) {
        const uint32_t b = word_off[w], n = word_off[w + 1] - b, base = tail_off[w - VD];
        sort_into(key, n, lane, [&](int u) { return (uint32_t)z[b + lane + 64 * u]; });
        wave_lds_sync();
        const TopicRuns r(key, n, lane);
        uint32_t nz = 0;
#pragma unroll
        for (int u = 0; u < (int)(kDtShort / 64); ++u) {
            if (u >= r.nu) break;
            const uint32_t len = r.len(u, n, lane);
            const uint32_t pos = nz + (uint32_t)__popcll(r.hm[u] & lanemask_lt((int)lane));
            if (len) wt_tail[base + pos] = (uint32_t)key[lane + 64 * u] | len << 16;
            nz += (uint32_t)__popcll(r.hm[u]);
        }
        if (lane == 0) tail_nnz[w - VD] = nz;
        wave_lds_sync();
    }
}

// The three count builds of a sweep in one launch (they touch disjoint
// outputs): blocks [0, nb_hist) build n_k, the next nb_head the head rows,
// the rest the tail rows, so each role's last blocks overlap the next role's
// instead of draining the device between launches.
__global__ void __launch_bounds__(256) k_wt_all(int nb_hist, int nb_head, const uint16_t *__restrict__ z,
                                                uint32_t N, int K, int32_t *__restrict__ nk,
                                                const uint4 *__restrict__ segs, int32_t *__restrict__ wt_head,
                                                bool fresh, const uint32_t *__restrict__ word_off, int VD, int V,
                                                const uint32_t *__restrict__ tail_off, uint32_t *__restrict__ wt_tail,
                                                uint32_t *__restrict__ tail_nnz) {
    extern __shared__ uint32_t sh[];
    const int b = (int)blockIdx.x;
    if (b < nb_hist)
        topic_hist_block(sh, z, N, K, nk, (uint32_t)b, (uint32_t)nb_hist);
    else if (b < nb_hist + nb_head)
        wt_head_block(sh, z, segs, K, wt_head, fresh, (uint32_t)(b - nb_hist));
    else
        wt_tail_block(sh, z, word_off, VD, V, K, tail_off, wt_tail, tail_nnz, b - nb_hist - nb_head,
                      (int)gridDim.x - nb_hist - nb_head);
}

// ----------------------------------------------------- inv and top-3
// inv, and the same in FP64 (vbeta64) for the log-likelihood
__global__ void k_inv(const int32_t *__restrict__ nk, int K, float vbeta, double vbeta64, float *__restrict__ inv,
                      double *__restrict__ inv64) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= K) return;
    inv[k] = 1.0f / ((float)nk[k] + vbeta);
    inv64[k] = 1.0 / ((double)nk[k] + vbeta64);
}

struct Top3 {
    float v0, v1, v2;
    uint32_t k0, k1, k2;
};

__device__ __forceinline__ bool better(float va, uint32_t ka, float vb, uint32_t kb) {
    return va > vb || (va == vb && ka < kb);
}

// A key whose unsigned order is better()'s: value bits (v >= 0, so their
// order is the value's) above the complemented topic; empty (v < 0) is 0.
__device__ __forceinline__ uint64_t top_key(float v, uint32_t k) {
    return v < 0.0f ? 0ull : ((uint64_t)(__float_as_uint(v) + 1u) << 32) | (uint64_t)(0xFFFFFFFFu - k);
}

__device__ __forceinline__ void top3_insert(Top3 &t, float v, uint32_t k) {
    if (!better(v, k, t.v2, t.k2)) return;
    if (better(v, k, t.v1, t.k1)) {
        t.v2 = t.v1; t.k2 = t.k1;
        if (better(v, k, t.v0, t.k0)) {
            t.v1 = t.v0; t.k1 = t.k0;
            t.v0 = v; t.k0 = k;
        } else {
            t.v1 = v; t.k1 = k;
        }
    } else {
        t.v2 = v; t.k2 = k;
    }
}

// inv, and the topics by beta * inv[k] (the value of a topic a word has no
// count of), largest first, ties to the lower topic.  A workgroup of 16
// wavefronts ranks 64 topics: it computes every topic's value into LDS, lane
// i's topic is compared with a sixteenth of them by each wavefront (four
// values a read, all lanes the same address), and the counts are added in
// LDS.  Topics before the workgroup's own win ties, later ones lose them, so
// only its own 64 need the tie test.  Bound by its K^2 compares: 20 -> 5.7 us at
// K = 1024, 176 -> 19 us at K = 10000 (four wavefronts, a scalar read and the
// tie test for each, inv from a launch before it).
__global__ void __launch_bounds__(1024) k_inv_order(const int32_t *__restrict__ nk, int K, float vbeta, double vbeta64,
                                                    float beta, float *__restrict__ inv, double *__restrict__ inv64,
                                                    uint32_t *__restrict__ zero_order) {
    extern __shared__ float sv[];  // K values padded to whole groups of 4, then 64 ranks
    const int KG = (K + 3) >> 2;
    uint32_t *rank = reinterpret_cast<uint32_t *>(sv + 4 * KG);
    const int own = (int)blockIdx.x * 64;
    for (int k = threadIdx.x; k < 4 * KG; k += blockDim.x) {
        float v = -1.0f;  // padding: below every value
        if (k < K) {
            const float iv = 1.0f / ((float)nk[k] + vbeta);
            v = beta * iv;
            if (k >= own && k < own + 64) {
                inv[k] = iv;
                inv64[k] = 1.0 / ((double)nk[k] + vbeta64);
            }
        }
        sv[k] = v;
    }
    if (threadIdx.x < 64) rank[threadIdx.x] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
    const int k = own + lane;
    const float v = k < K ? sv[k] : 0.0f;
    const float4 *s4 = reinterpret_cast<const float4 *>(sv);
    const int q = (KG + nwv - 1) / nwv, g0 = wv * q, g1 = min(KG, g0 + q);
    const int o0 = own >> 2, o1 = o0 + 16;  // the workgroup's own groups
    uint32_t r = 0;
#pragma unroll 4
    for (int g = g0; g < min(g1, o0); ++g) {
        const float4 x = s4[g];
        r += (x.x >= v) + (x.y >= v) + (x.z >= v) + (x.w >= v);
    }
    for (int g = max(g0, o0); g < min(g1, o1); ++g) {
        const float4 x = s4[g];
        const float y[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
        for (int c = 0; c < 4; ++c) r += better(y[c], (uint32_t)(4 * g + c), v, (uint32_t)k) ? 1u : 0u;
    }
#pragma unroll 4
    for (int g = max(g0, o1); g < g1; ++g) {
        const float4 x = s4[g];
        r += (x.x > v) + (x.y > v) + (x.z > v) + (x.w > v);
    }
    if (k < K) atomicAdd(&rank[lane], r);
    __syncthreads();
    if (wv == 0 && k < K) zero_order[rank[lane]] = (uint32_t)k;
}

// Per word the three largest phi_wk, ties to the lower topic
// (MaxTopicDense/Sparse_Update_Kernel, utility.cu:305-678, :679-1062).  One
// wavefront per word; a tail word's topics are marked in a bitmap in LDS (K
// bits, so it leaves the occupancy alone at every K: with a table of 16-bit
// counts, 20 KB a wavefront at K = 10000, 30,000 words took 104 us, in two
// launches, 59 with the bitmap).  A dense row is read by 16-byte loads where K
// is a multiple of 4, two in flight (20,011 rows at K = 4096 136 -> 100 us; four
// took 74 registers and the tail words of 49.5M tokens at K = 1024 65 -> 74).
// The order is total, so the order in which the lanes' lists are merged does
// not matter.
__global__ void k_word_top(int V, int VD, int K, float beta, const int32_t *__restrict__ wt_head,
                           const uint32_t *__restrict__ tail_off, const uint32_t *__restrict__ wt_tail,
                           const uint32_t *__restrict__ tail_nnz, const float *__restrict__ inv,
                           const uint32_t *__restrict__ zero_order, ushort4 *__restrict__ wtop) {
    extern __shared__ uint32_t sh[];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
    const int NW = (K + 31) >> 5;
    uint32_t *bm = sh + wv * NW;
    if (V > VD) {
        for (int k = lane; k < NW; k += 64) bm[k] = 0;
        wave_lds_sync();
    }
    for (int w = blockIdx.x * nwv + wv; w < V; w += gridDim.x * nwv) {
        Top3 t{-1.f, -1.f, -1.f, kNone, kNone, kNone};
        if (w < VD) {
            // two 16-byte (else four 4-byte) loads of the row and of inv in flight a lane
            const int32_t *row = wt_head + (size_t)w * K;
            if ((K & 3) == 0) {
                const int4 *row4 = reinterpret_cast<const int4 *>(row);
                const float4 *inv4 = reinterpret_cast<const float4 *>(inv);
                const int K4 = K >> 2;
                for (int k0 = lane; k0 < K4; k0 += 128) {
                    int4 c[2];
                    float4 iv[2];
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const int k = k0 + 64 * u;
                        c[u] = k < K4 ? row4[k] : make_int4(0, 0, 0, 0);
                        iv[u] = k < K4 ? inv4[k] : make_float4(0.f, 0.f, 0.f, 0.f);
                    }
#pragma unroll
                    for (int u = 0; u < 2; ++u)
                        if (k0 + 64 * u < K4) {
                            const uint32_t k = 4u * (uint32_t)(k0 + 64 * u);
                            top3_insert(t, ((float)c[u].x + beta) * iv[u].x, k);
                            top3_insert(t, ((float)c[u].y + beta) * iv[u].y, k + 1u);
                            top3_insert(t, ((float)c[u].z + beta) * iv[u].z, k + 2u);
                            top3_insert(t, ((float)c[u].w + beta) * iv[u].w, k + 3u);
                        }
                }
            }
            for (int k0 = lane; (K & 3) != 0 && k0 < K; k0 += 256) {
                int32_t c[4];
                float iv[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int k = k0 + 64 * u;
                    c[u] = k < K ? row[k] : 0;
                    iv[u] = k < K ? inv[k] : 0.0f;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (k0 + 64 * u < K) top3_insert(t, ((float)c[u] + beta) * iv[u], (uint32_t)(k0 + 64 * u));
            }
        } else {
            // the word's topics with a count, then those without one: their
            // value is beta * inv[k], so the first three of zero_order that
            // have no count are the best of them
            const int tw = w - VD;
            const uint32_t b = tail_off[tw], n = tail_nnz[tw];
            for (uint32_t i = lane; i < n; i += 64) {
                const uint32_t e = wt_tail[b + i];
                const uint32_t k = e & 0xFFFFu;
                atomicOr(&bm[k >> 5], 1u << (k & 31u));
                top3_insert(t, ((float)(e >> 16) + beta) * inv[k], k);
            }
            wave_lds_sync();
            uint32_t got = 0;  // wavefront-uniform
            for (int j0 = 0; j0 < K && got < 3u; j0 += 64) {
                const int j = j0 + lane;
                const uint32_t k = j < K ? zero_order[j] : 0u;
                const bool free_k = j < K && !((bm[k >> 5] >> (k & 31u)) & 1u);
                const uint64_t m = __ballot(free_k);
                if (free_k && got + (uint32_t)__popcll(m & lanemask_lt(lane)) < 3u)
                    top3_insert(t, ((float)0u + beta) * inv[k], k);
                got += (uint32_t)__popcll(m);
            }
            wave_lds_sync();
            for (uint32_t i = lane; i < n; i += 64) bm[(wt_tail[b + i] & 0xFFFFu) >> 5] = 0;
            wave_lds_sync();
        }
        // the wavefront's best three: three max-reductions of the lanes'
        // list heads, the winner's lane popping its head each time (a lane's
        // topics are its own, so the winner is one lane)
        uint64_t a0 = top_key(t.v0, t.k0), a1 = top_key(t.v1, t.k1), a2 = top_key(t.v2, t.k2);
        uint32_t best[3];
#pragma unroll
        for (int r = 0; r < 3; ++r) {
            uint64_t m = a0;
#pragma unroll
            for (int off = 32; off >= 1; off >>= 1) {
                const uint64_t o = __shfl_xor(m, off);
                m = o > m ? o : m;
            }
            best[r] = m ? 0xFFFFFFFFu - (uint32_t)m : kNone;
            if (a0 == m) {
                a0 = a1;
                a1 = a2;
                a2 = 0;
            }
        }
        if (lane == 0)
            wtop[w] = make_ushort4((unsigned short)best[0], (unsigned short)best[1], (unsigned short)best[2], 0);
    }
}

// Doc-slot copy of z from z (after a layout change: slots of words that
// were tail words hold stale topics there).
__global__ void k_z_to_doc(uint32_t N, const uint32_t *__restrict__ slot_tok, const uint16_t *__restrict__ z,
                           uint16_t *__restrict__ z_doc) {
    for (uint32_t p = blockIdx.x * blockDim.x + threadIdx.x; p < N; p += gridDim.x * blockDim.x)
        z_doc[p] = z[slot_tok[p]];
}

hipError_t launch_z_to_doc(const DevState &s, hipStream_t st) {
    if (s.N == 0) return hipSuccess;
    hipLaunchKernelGGL(k_z_to_doc, dim3(grid_for(s.N, 256, 1 << 16)), dim3(256), 0, st, s.N, s.slot_tok, s.z, s.z_doc);
    return hipGetLastError();
}

// Topics in the corpus' own (doc-major) order, straight into pinned host
// memory: eight positions a lane, one 16-byte store.  Bound by the gathers (a
// 2-byte read of z fills a line) and then by the copy out of the pinned pieces:
// 3.8 ms for 49.5M tokens with its host side; the host loop it replaced (one
// thread, a random read a token) took 188 ms.
__global__ void __launch_bounds__(256) k_topics_out(uint32_t b, uint32_t n, const uint32_t *__restrict__ doc_tok,
                                                    const uint16_t *__restrict__ z, uint16_t *__restrict__ out) {
    const uint32_t i = (blockIdx.x * 256u + threadIdx.x) * 8u;
    if (i >= n) return;
    const uint32_t *dt = doc_tok + b + i;
    if (i + 8u <= n) {
        const uint4 p = *reinterpret_cast<const uint4 *>(dt), q = *reinterpret_cast<const uint4 *>(dt + 4);
        const uint32_t t[8] = {p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w};
        uint32_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = z[t[u]];
        *reinterpret_cast<uint4 *>(out + i) =
            make_uint4(v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16);
    } else {
        for (uint32_t u = 0; i + u < n; ++u) out[i + u] = z[dt[u]];
    }
}

hipError_t launch_topics_out(const DevState &s, uint32_t b, uint32_t n, uint16_t *out, hipStream_t st) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_topics_out, dim3((n + 2047u) / 2048u), dim3(256), 0, st, b, n, s.doc_tok, s.z, out);
    return hipGetLastError();
}

// A chunk's runs and slot words from the short form that its image carries
// over the host link (run_slot and run_len, runs in token order), one
// wavefront an item: a counting sort by length puts the runs in the order of
// the sampler (longest first, then by token), a prefix sum of the lengths
// numbers their tokens, and the doc of a run is searched by its first slot.
// The link bounds a sweep over chunks, not the kernels: 5 bytes a run over it
// instead of 16, and neither the word of each slot (4 bytes a token), nor its
// token (4, not needed on the device), nor z beside z_doc (2, each way).
// 6.6M tokens in 4 chunks, K = 1024: 29 us a chunk of 1.65M tokens alone, 75
// on average beside the other stream's kernels and an upload of 160-225 us (was
// 480); a sweep 4.0 -> 1.95 ms with the first
// uploads begun before the last sweep ends.
// TOPICS: z of z_doc instead, which the first sweep counts.
template <bool TOPICS>
__global__ __launch_bounds__(256) void k_chunk_runs(const uint4 *__restrict__ items, uint32_t n_items, ChunkRuns R,
                                                    uint32_t D, const uint32_t *__restrict__ soff,
                                                    const uint2 *__restrict__ doc_info, uint4 *__restrict__ runs,
                                                    uint32_t *__restrict__ slot_wrd,
                                                    const uint16_t *__restrict__ z_doc, uint16_t *__restrict__ z,
                                                    uint32_t *__restrict__ counters, uint32_t n_queues,
                                                    uint32_t sweep) {
    __shared__ uint32_t bins[TOPICS ? 1 : 4][64];  // run_cap is at most 32
    const uint32_t lane = threadIdx.x & 63u, wv = threadIdx.x >> 6, gid = blockIdx.x * 256u + threadIdx.x;
    if (!TOPICS) {
        if (gid == 0) counters[1] = sweep;
        if (gid < n_queues) counters[kQueueStride * (gid + 1)] = 0u;
    }
    uint32_t *bin = bins[TOPICS ? 0 : wv];
    for (uint32_t i = blockIdx.x * 4u + wv; i < n_items; i += gridDim.x * 4u) {
        const uint4 it = items[i];
        if (it.x == 0xFFFFFFFFu) continue;
        if (!TOPICS) {  // bin[n]: place of the next run of n tokens
            bin[lane] = 0u;
            wave_lds_sync();
            for (uint32_t r = it.y + lane; r < it.z; r += 64) atomicAdd(&bin[R.run_len[r]], 1u);
            wave_lds_sync();
            const uint32_t c = bin[63u - lane];
            uint32_t incl = c;
            for (uint32_t d = 1; d < 64; d <<= 1) {
                const uint32_t v = __shfl_up(incl, d);
                if (lane >= d) incl += v;
            }
            wave_lds_sync();
            bin[63u - lane] = it.y + incl - c;
            wave_lds_sync();
        }
        uint32_t tok = R.item_tok[i];
        for (uint32_t b = it.y; b < it.z; b += 64) {
            const uint32_t r = b + lane;
            const bool have = r < it.z;
            const uint32_t n = have ? R.run_len[r] : 0u, slot = have ? R.run_slot[r] : 0u;
            uint32_t incl = n;
            for (uint32_t d = 1; d < 64; d <<= 1) {
                const uint32_t v = __shfl_up(incl, d);
                if (lane >= d) incl += v;
            }
            const uint32_t t0 = tok + incl - n;
            tok += __shfl(incl, 63);
            if (TOPICS) {
                for (uint32_t j = 0; j < n; ++j) z[t0 + j] = z_doc[slot + j];
                continue;
            }
            uint32_t q = 0;  // the last doc whose first slot is not after this one
            for (uint32_t lo = 1, hi = D; lo < hi;) {
                const uint32_t mid = (lo + hi) >> 1;
                if (soff[mid] <= slot)
                    q = mid, lo = mid + 1;
                else
                    hi = mid;
            }
            const uint32_t row = doc_info[q].x, len = soff[q + 1] - soff[q];
            uint32_t at = 0;
            for (uint64_t left = __ballot(have); left;) {
                const uint32_t ln = __shfl(n, __ffsll((unsigned long long)left) - 1);
                const uint64_t same = __ballot(have && n == ln);
                const uint32_t first = bin[ln];
                if (n == ln) at = first + (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
                wave_lds_sync();
                if (lane == 0) bin[ln] = first + (uint32_t)__popcll(same);
                wave_lds_sync();
                left &= ~same;
            }
            if (have) runs[at] = make_uint4(t0, slot, row, n | len << 16);
            for (uint32_t j = 0; j < n; ++j) slot_wrd[slot + j] = it.x;
        }
    }
}

template <bool TOPICS>
static hipError_t chunk_runs(const DevState &s, const ChunkRuns &r, uint32_t sweep, hipStream_t st) {
    if (s.n_smp_segs == 0) return hipSuccess;
    hipLaunchKernelGGL((k_chunk_runs<TOPICS>), dim3(grid_for((size_t)s.n_smp_segs, 4, 1 << 14)), dim3(256), 0, st,
                       s.smp_segs, (uint32_t)s.n_smp_segs, r, (uint32_t)s.D, s.soff, s.doc_info, s.runs, s.slot_wrd,
                       s.z_doc, s.z, s.counters, (uint32_t)s.n_queues, sweep);
    return hipGetLastError();
}

hipError_t launch_chunk_runs(const DevState &s, const ChunkRuns &r, uint32_t sweep, hipStream_t st) {
    return chunk_runs<false>(s, r, sweep, st);
}

hipError_t launch_chunk_topics(const DevState &s, const ChunkRuns &r, hipStream_t st) {
    return chunk_runs<true>(s, r, 0, st);
}

// --------------------------------------------------- DT rows and aux
// DT_Update_Kernel (utility.cu:79-284), on the doc-major copy of z: doc q
// (docs in descending length order) owns slots [soff[q], soff[q+1]), its
// tokens grouped by word, and the sampler keeps z_doc in step with z, so
// every read and write here is a coalesced stream.  One wavefront per doc
// builds a 16-bit LDS histogram, compacts the row in ascending topic order
// (:183-238), and writes each slot's record: n_dk1 at its word's top topic
// with the row's length (the sampler's), or with n_dk2 = n_dk at its word's
// second topic (the re-pack of :125-161, for the getter).  A row starts on a
// 128-byte boundary and is zero-padded to a multiple of 32 entries.
// Up to this K the row is compacted from the counts themselves, two topics a
// lane and 128 a step, and no bitmap is kept: that costs K / 128 short steps,
// the bitmap three loops over the topics of the fullest 32 (and, before, a
// division a topic).  us a sweep: 1M tokens at K = 64 29 -> 14, 1.7M at K = 300
// 34 -> 27, 18,000 at K = 20 11.5 -> 7, 49.5M at K = 1024 338 -> 331; equal at K
// = 2048 (161), at K = 4096 160 -> 250.
static constexpr int kScanMaxK = 1024;
static constexpr int kDtU = 8;  // slots per lane per chunk in k_dt_build

template <bool COMPACT, bool N_DK2, bool SCAN>
__global__ void k_dt_build(int q0, int q1, int K, int VD, uint32_t tb, const uint32_t *__restrict__ soff,
                           const uint32_t *__restrict__ slot_wrd, const uint32_t *__restrict__ slot_tok,
                           const uint16_t *__restrict__ z, const uint16_t *__restrict__ z_doc,
                           const ushort4 *__restrict__ wtop,
                           uint32_t *__restrict__ aux_doc, uint2 *__restrict__ doc_info, uint32_t *__restrict__ dt) {
    extern __shared__ uint32_t sh[];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
    const int KH = SCAN ? (int)(scan_wave_bytes(K) / 4) : (K + 1) >> 1, NW = SCAN ? 0 : (K + 31) >> 5;
    const uint32_t piece = (1u << (16u - tb)) - 1u;  // compact rows: largest count of one entry
    uint32_t *h = sh + wv * (KH + NW);  // 16-bit counts
    uint32_t *bm = h + KH;              // bitmap of the doc's topics
    for (int k = lane; k < KH + NW; k += 64) h[k] = 0;
    wave_lds_sync();
    for (int q = q0 + blockIdx.x * nwv + wv; q < q1; q += gridDim.x * nwv) {
        const uint32_t b = soff[q], e = soff[q + 1];
        // The doc in chunks of kDtU slots per lane, every load of a chunk
        // issued before the first is used.  A doc of one chunk keeps its
        // words' top topics in registers for the aux pass.
        const bool one = e - b <= 64u * kDtU;
        uint32_t tp[kDtU];  // top-1 | top-2 << 16 of each slot's word (one-chunk docs)
        for (uint32_t c = b; c < e; c += 64u * kDtU) {
            uint32_t w[kDtU], t[kDtU];
#pragma unroll
            for (int u = 0; u < kDtU; ++u) {
                const uint32_t i = c + lane + 64u * u;
                w[u] = i < e ? slot_wrd[i] : 0u;
                t[u] = i < e ? z_doc[i] : 0u;
            }
#pragma unroll
            for (int u = 0; u < kDtU; ++u) {
                const uint32_t i = c + lane + 64u * u;
                if (i < e && w[u] >= (uint32_t)VD) t[u] = z[slot_tok[i]];
            }
            if (one) {
#pragma unroll
                for (int u = 0; u < kDtU; ++u) {
                    const ushort4 x = wtop[w[u]];
                    tp[u] = x.x | ((uint32_t)x.y << 16);
                }
            }
#pragma unroll
            for (int u = 0; u < kDtU; ++u) {
                if (c + lane + 64u * u < e) {
                    h16_add(h, t[u]);
                    if (!SCAN) atomicOr(&bm[t[u] >> 5], 1u << (t[u] & 31u));
                }
            }
        }
        wave_lds_sync();
        // Compaction over the bitmap: lane j owns topics [32j, 32j + 32) of
        // each 64-word chunk, counts its entries, takes its place from a
        // wave prefix sum and writes them in ascending topic order.  Cost
        // follows the doc's topics, not K.
        const uint32_t base = doc_info[q].x;
        uint32_t nz = 0;
        auto put = [&](uint32_t at, uint32_t k, uint32_t c) {
            if (COMPACT)
                (reinterpret_cast<uint16_t *>(dt) + base)[at] = (uint16_t)(k | (c << tb));
            else
                dt[base + at] = (k << 2) | (c << 16);
        };
        // SCAN: the counts themselves, two topics a lane
        for (int j = 0; SCAN && j < KH; j += 64) {
            const uint32_t k = 2u * (uint32_t)(j + lane), cc = j + lane < KH ? h[j + lane] : 0u;
            const uint32_t c0 = cc & 0xFFFFu, c1 = cc >> 16;
            if (COMPACT && __ballot(max(c0, c1) > piece)) {  // entries of several pieces
                const uint32_t m = (c0 + piece - 1u) / piece + (c1 + piece - 1u) / piece;
                uint32_t incl = m;
                for (int d = 1; d < 64; d <<= 1) {
                    const uint32_t v = __shfl_up(incl, d);
                    if (lane >= d) incl += v;
                }
                uint32_t pos = nz + incl - m;
                for (uint32_t c = c0; c; c -= min(c, piece)) put(pos++, k, min(c, piece));
                for (uint32_t c = c1; c; c -= min(c, piece)) put(pos++, k + 1u, min(c, piece));
                nz += __shfl(incl, 63);
            } else {
                const uint64_t m0 = __ballot(c0 != 0u), m1 = __ballot(c1 != 0u), lt = lanemask_lt(lane);
                const uint32_t pos = nz + (uint32_t)(__popcll(m0 & lt) + __popcll(m1 & lt));
                if (c0) put(pos, k, c0);
                if (c1) put(pos + (c0 ? 1u : 0u), k + 1u, c1);
                nz += (uint32_t)(__popcll(m0) + __popcll(m1));
            }
        }
        for (int j = 0; j < NW; j += 64) {
            const int wi = j + lane;
            const uint32_t word = wi < NW ? bm[wi] : 0u;
            uint32_t m = 0;  // entries of this lane's topics
            if (COMPACT) {
                for (uint32_t x = word; x; x &= x - 1u) {
                    const uint32_t k = ((uint32_t)wi << 5) + (uint32_t)__ffs(x) - 1u;
                    const uint32_t c = h16_get(h, k);
                    m += c <= piece ? 1u : (c + piece - 1u) / piece;
                }
            } else {
                m = (uint32_t)__popc(word);
            }
            uint32_t incl = m;  // inclusive scan over lanes
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t v = __shfl_up(incl, d);
                if (lane >= d) incl += v;
            }
            uint32_t pos = nz + incl - m;
            for (uint32_t x = word; x; x &= x - 1u) {
                const uint32_t k = ((uint32_t)wi << 5) + (uint32_t)__ffs(x) - 1u;
                uint32_t c = h16_get(h, k);
                if (COMPACT) {
                    uint16_t *dt16 = reinterpret_cast<uint16_t *>(dt) + base;
                    for (; c > piece; c -= piece) dt16[pos++] = (uint16_t)(k | (piece << tb));
                    dt16[pos++] = (uint16_t)(k | (c << tb));
                } else {
                    dt[base + pos++] = (k << 2) | (c << 16);
                }
            }
            nz += __shfl(incl, 63);
        }
        // zero entries up to the next 128 bytes: the sampler reads rows in
        // 128-byte blocks and a zero entry adds nothing
        if (e > b) {
            if (COMPACT) {
                uint16_t *dt16 = reinterpret_cast<uint16_t *>(dt) + base;
                if ((uint32_t)lane < ((64u - (nz & 63u)) & 63u)) dt16[nz + lane] = 0;
            } else {
                if ((uint32_t)lane < ((32u - (nz & 31u)) & 31u)) dt[base + nz + lane] = 0u;
            }
        }
        if (lane == 0) doc_info[q].y = nz | ((e - b) << 16);
        // each slot's record: n_dk1 and the row's length (a tail word's run
        // is in a random doc, whose doc_info would cost a cache line of its
        // own), or n_dk1 and n_dk2
        if (one) {
#pragma unroll
            for (int u = 0; u < kDtU; ++u) {
                const uint32_t i = b + lane + 64u * u;
                if (i < e) {
                    const uint32_t k2 = tp[u] >> 16;
                    const uint32_t hi = N_DK2 ? (k2 != kNone ? h16_get(h, k2) : 0u) : nz;
                    aux_doc[i] = h16_get(h, tp[u] & 0xFFFFu) | (hi << 16);
                }
            }
        } else {
            for (uint32_t c = b; c < e; c += 64u * kDtU) {
                uint32_t x[kDtU];
#pragma unroll
                for (int u = 0; u < kDtU; ++u) {
                    const uint32_t i = c + lane + 64u * u;
                    x[u] = i < e ? slot_wrd[i] : 0u;
                }
#pragma unroll
                for (int u = 0; u < kDtU; ++u) {
                    const ushort4 y = wtop[x[u]];
                    x[u] = y.x | ((uint32_t)y.y << 16);
                }
#pragma unroll
                for (int u = 0; u < kDtU; ++u) {
                    const uint32_t i = c + lane + 64u * u;
                    if (i < e) {
                        const uint32_t k2 = x[u] >> 16;
                        const uint32_t hi = N_DK2 ? (k2 != kNone ? h16_get(h, k2) : 0u) : nz;
                        aux_doc[i] = h16_get(h, x[u] & 0xFFFFu) | (hi << 16);
                    }
                }
            }
        }
        wave_lds_sync();
        if (SCAN)
            for (int k = lane; k < KH >> 2; k += 64) reinterpret_cast<uint4 *>(h)[k] = make_uint4(0u, 0u, 0u, 0u);
        // each lane clears its own count words and bitmap words
        for (int wi = lane; wi < NW; wi += 64) {
            for (uint32_t x = bm[wi]; x; x &= x - 1u) {
                const uint32_t k = ((uint32_t)wi << 5) + (uint32_t)__ffs(x) - 1u;
                h[k >> 1] = 0;
            }
            bm[wi] = 0;
        }
        wave_lds_sync();
    }
}

// The same DT rows and aux for short documents (n <= kDtShort slots) at
// large K, where a K-sized LDS histogram per wavefront limits a CU to a few
// wavefronts: one wavefront per doc sorts its topics in registers, reads the
// runs of equal topics off the sorted keys in LDS (ascending topic, as the
// histogram's compaction writes them) and finds each slot's (n_dk1, n_dk2)
// by bisection.  Rows, pieces, padding and aux are those of k_dt_build.
// 50,000 documents of 90 tokens at K = 10000: 120 -> 86 us (sorted in LDS
// before, two reads and a barrier a pass).
template <bool COMPACT, bool N_DK2>
__global__ void __launch_bounds__(256) k_dt_sort(int q0, int q1, int VD, uint32_t tb,
                                                 const uint32_t *__restrict__ soff, const uint32_t *__restrict__ slot_wrd,
                                                 const uint32_t *__restrict__ slot_tok, const uint16_t *__restrict__ z,
                                                 const uint16_t *__restrict__ z_doc, const ushort4 *__restrict__ wtop,
                                                 uint32_t *__restrict__ aux_doc,
                                                 uint2 *__restrict__ doc_info, uint32_t *__restrict__ dt) {
    extern __shared__ uint32_t sh[];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
    uint16_t *key = reinterpret_cast<uint16_t *>(sh + wv * kDtShort);  // kDtShort sorted topics
    uint16_t *run = key + kDtShort;                                      // run length at each run's first key
    const uint32_t piece = (1u << (16u - tb)) - 1u;
    constexpr int kU = kDtShort / 64;
    for (int q = q0 + blockIdx.x * nwv + wv; q < q1; q += gridDim.x * nwv) {
        const uint32_t b = soff[q], e = soff[q + 1], n = e - b;  // n <= kDtShort
        const int nu = (int)((n + 63u) >> 6);
        uint32_t wrd[kU];
        // topics (the doc-slot copy for head words, z by token id for tail
        // words), padded with 0xFFFF, which sorts last
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const uint32_t i = (uint32_t)lane + 64u * u;
            wrd[u] = i < n ? slot_wrd[b + i] : 0u;
        }
        sort_into(key, n, (uint32_t)lane, [&](int u) {
            const uint32_t i = b + lane + 64u * u;
            return (uint32_t)(wrd[u] < (uint32_t)VD ? z_doc[i] : z[slot_tok[i]]);
        });
        wave_lds_sync();
        const TopicRuns runs(key, n, (uint32_t)lane);
        const uint32_t base = doc_info[q].x;
        uint32_t nz = 0;
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            if (u >= nu) break;
            const uint32_t i = (uint32_t)lane + 64u * u;
            const uint32_t len = runs.len(u, n, (uint32_t)lane), m = COMPACT ? (len + piece - 1u) / piece : len ? 1u : 0u;
            const bool head = len != 0u;
            if (head) run[i] = (uint16_t)len;
            uint32_t incl = m;  // inclusive scan over lanes
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t v = __shfl_up(incl, d);
                if (lane >= d) incl += v;
            }
            uint32_t pos = nz + incl - m;
            if (head) {
                const uint32_t k = key[i];
                if (COMPACT) {
                    uint16_t *dt16 = reinterpret_cast<uint16_t *>(dt) + base;
                    uint32_t c = len;
                    for (; c > piece; c -= piece) dt16[pos++] = (uint16_t)(k | (piece << tb));
                    dt16[pos++] = (uint16_t)(k | (c << tb));
                } else {
                    dt[base + pos] = (k << 2) | (len << 16);
                }
            }
            nz += __shfl(incl, 63);
        }
        // zero entries up to the next 128 bytes, as k_dt_build
        if (n > 0) {
            if (COMPACT) {
                uint16_t *dt16 = reinterpret_cast<uint16_t *>(dt) + base;
                if ((uint32_t)lane < ((64u - (nz & 63u)) & 63u)) dt16[nz + lane] = 0;
            } else {
                if ((uint32_t)lane < ((32u - (nz & 31u)) & 31u)) dt[base + nz + lane] = 0u;
            }
        }
        if (lane == 0) doc_info[q].y = nz | (n << 16);
        wave_lds_sync();  // run lengths visible
        // (n_dk1, n_dk2) of each slot's word: its top topics' runs, found by
        // bisection of the sorted keys
#pragma unroll
        for (int u = 0; u < kU; ++u) {
            const uint32_t i = (uint32_t)lane + 64u * u;
            if (u < nu && i < n) {
                const ushort4 tp = wtop[wrd[u]];
                uint32_t cnt[2] = {0u, 0u};
                const uint32_t want[2] = {tp.x, tp.y};
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    if (want[h] == kNone) continue;
                    uint32_t lo = 0, hi = n;
                    while (lo < hi) {
                        const uint32_t mid = (lo + hi) >> 1;
                        if (key[mid] < want[h]) lo = mid + 1; else hi = mid;
                    }
                    if (lo < n && key[lo] == want[h]) cnt[h] = run[lo];
                }
                aux_doc[b + i] = cnt[0] | ((N_DK2 ? cnt[1] : nz) << 16);
            }
        }
        wave_lds_sync();  // the next doc reuses the keys
    }
}

// ------------------------------------------------------------- sampler
// Checkpoints of the S running sum kept per lane: one per block of kBlkU4
// 16-byte loads (4 * kBlkU4 entries of 32 bits, 8 * kBlkU4 of 16) for the
// first CP blocks, and with kHalfCp, in 16-bit rows, one more in the middle of
// each, so the S-bucket search re-reads half a block (6.09 -> 5.98 ms a sweep
// on the 99M-token corpus at K = 1024; with 32-bit rows it cost 1.5 ms of 63.6
// at K = 10000, so they search whole blocks).  A wavefront with a longer row
// keeps CF more, m blocks apart (m the same for its lanes), so the search
// past the first CP reads at most m blocks again: walking them from the
// CP-th took most of the sampler on heavy-tailed documents (8.9M tokens of
// up to 20,000 a document at K = 2048: 2.63 -> 1.67 ms a sweep with 8 + 8,
// 1.72 with 9 + 6, 1.78 with 12 + 4; 49.5M tokens at K = 1024 2.92 -> 2.90
// with 12 + 4, 2.92 with 9 + 6).  The counts are what fits 128 registers
// (MULTI, whose lanes each have their own word's values: 6 + 2, rows at most 512
// topics).
template <bool COMPACT, bool QTAB, bool MULTI>
struct Checkpoints {
    static constexpr int CP = MULTI ? 6 : !QTAB && COMPACT ? 8 : EZ_SAMPLE_CP;
    static constexpr int CF = MULTI ? 2 : !QTAB && COMPACT ? 8 : 4;
};
static constexpr int kBlkU4 = EZ_SAMPLE_BLK;
#ifndef EZ_SAMPLE_HALF_CP
#define EZ_SAMPLE_HALF_CP 1
#endif
static constexpr bool kHalfCp = EZ_SAMPLE_HALF_CP != 0 && kBlkU4 % 2 == 0;
// Uniforms kept in registers per run between the shortcut test and the draw
// (tokens past them draw theirs again).
// (32-bit rows keep one: at K > 8192 the registers of four cost more than the
// draws they save, 63.9 against 63.5 ms a sweep on 180M tokens at K = 10000)
static constexpr int kUKeep = 4;    // 16-bit rows
static constexpr int kUKeep32 = 1;  // 32-bit rows

// Running FMA sum over one block of a DT row: kBlkU4 16-byte loads issued
// together, then the entries in order.
struct RowBlock {
    uint4 e[kBlkU4];
};

__device__ __forceinline__ RowBlock load_block(const uint4 *__restrict__ p) {
    RowBlock r;
#pragma unroll
    for (int i = 0; i < kBlkU4; ++i) r.e[i] = p[i];
    return r;
}

// The sampler's phi table in LDS, for compact rows, holds phi * 2^24: an
// entry's count, moved to the low bits of its half-word, is a subnormal f16 of
// value count * 2^-24, so one v_fma_mix_f32 takes it as it is and the products
// (hence the rounded sums) are those of count * phi.  Both scalings are exact.
static constexpr float kPhiUp = 16777216.0f, kPhiDown = 5.9604644775390625e-08f;

// The two compact entries of a dword (low half first) decoded together: both
// counts by one packed 16-bit shift, both topics by one mask (tm2 = the topic
// mask in each half), each phi address (topic * 4) by one shift that reads
// its half of the word (SDWA word select; the compiler forms it for the high
// half by itself, the low half is written out).  With the sum that is three
// VALU operations an entry (four with a conversion of each count); the scan
// keeps the VALU busy 66% of the cycles on the 49.5M-token corpus at K = 1024
// and 85% on rows of up to 2,700 entries (2.96 -> 2.92 and 2.81 -> 2.63 ms).
typedef unsigned short ez_us2 __attribute__((ext_vector_type(2)));
typedef _Float16 ez_h2 __attribute__((ext_vector_type(2)));
struct C16x2 {
    _Float16 c0, c1;  // count * 2^-24
    uint32_t a0, a1;
};
__device__ __forceinline__ uint32_t lo16_times4(uint32_t t) {
    uint32_t r;
    asm("v_lshlrev_b32_sdwa %0, %1, %2 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:WORD_0"
        : "=v"(r)
        : "v"(2u), "v"(t));
    return r;
}
// topic * 4 + base of the low / high half of t in one operation
__device__ __forceinline__ uint32_t lo16_times4_plus(uint32_t t, uint32_t base) {
    uint32_t r;
    asm("v_mad_u32_u16 %0, %1, 4, %2" : "=v"(r) : "v"(t), "v"(base));
    return r;
}
__device__ __forceinline__ uint32_t hi16_times4_plus(uint32_t t, uint32_t base) {
    uint32_t r;
    asm("v_mad_u32_u16 %0, %1, 4, %2 op_sel:[1,0,0,0]" : "=v"(r) : "v"(t), "v"(base));
    return r;
}
// MULTI: the lane's phi table starts at LDS address lb (else at 0)
template <bool MULTI>
__device__ __forceinline__ C16x2 c16_x2(uint32_t w, uint32_t tb, uint32_t tm2, uint32_t lb) {
    const ez_us2 c = __builtin_bit_cast(ez_us2, w) >> (ez_us2)((unsigned short)tb);
    const ez_h2 h = __builtin_bit_cast(ez_h2, c);
    const uint32_t t = w & tm2;
    if (MULTI) return C16x2{h.x, h.y, lo16_times4_plus(t, lb), hi16_times4_plus(t, lb)};
    return C16x2{h.x, h.y, lo16_times4(t), (t >> 16) << 2};
}
// s + count * phi in one rounding (v_fma_mix_f32)
__device__ __forceinline__ float fma_count(_Float16 c, float phi, float s) { return __builtin_fmaf((float)c, phi, s); }
__device__ __forceinline__ float phi_a(uint32_t a) { return *(lds_cfloat *)a; }

// A word's phi as the topics without a count, which its workgroup's words
// share (at LDS address 0), and the word's own values: by topic word (32
// topics) the bits of the topics it has and the LDS float index of the first
// one's value (uint2 at LDS address lb + 8 * (k / 32)).
typedef __attribute__((address_space(3))) const uint32_t lds_cu32;
__device__ __forceinline__ float phi_own(uint32_t k, uint32_t lb) {
    lds_cu32 *p = (lds_cu32 *)(lb + ((k >> 2) & ~7u));
    const uint32_t bits = p[0], first = p[1];
    const uint32_t i = first + (uint32_t)__popc(bits & ((1u << (k & 31u)) - 1u));
    return phi_a(((bits >> (k & 31u)) & 1u ? i : k) << 2);
}

// Where a lane's phi is: one table at LDS address 0, its word's table at LDS
// address lb, or the two of phi_own.
enum PhiAt { kPhiOne, kPhiGroup, kPhiOwn };

// The entries of one 16-byte load, in order.
template <bool COMPACT, PhiAt P>
__device__ __forceinline__ float sum_u4(const uint4 &e, float s, uint32_t tb, uint32_t lb) {
    constexpr bool MULTI = P == kPhiGroup;
    static_assert(P != kPhiOwn || !COMPACT, "phi_own is for 32-bit rows");
    if (P == kPhiOwn) {
        s = __builtin_fmaf(dt_count(e.x), phi_own(dt_topic(e.x), lb), s);
        s = __builtin_fmaf(dt_count(e.y), phi_own(dt_topic(e.y), lb), s);
        s = __builtin_fmaf(dt_count(e.z), phi_own(dt_topic(e.z), lb), s);
        return __builtin_fmaf(dt_count(e.w), phi_own(dt_topic(e.w), lb), s);
    }
    if (COMPACT) {  // two 16-bit entries per dword, low half first
        const uint32_t w[4] = {e.x, e.y, e.z, e.w};
        const uint32_t tm2 = ((1u << tb) - 1u) * 0x10001u;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const C16x2 d = c16_x2<MULTI>(w[q], tb, tm2, lb);
            s = fma_count(d.c0, phi_a(d.a0), s);
            s = fma_count(d.c1, phi_a(d.a1), s);
        }
    } else {
        s = __builtin_fmaf(dt_count(e.x), phi_at0(e.x), s);
        s = __builtin_fmaf(dt_count(e.y), phi_at0(e.y), s);
        s = __builtin_fmaf(dt_count(e.z), phi_at0(e.z), s);
        s = __builtin_fmaf(dt_count(e.w), phi_at0(e.w), s);
    }
    return s;
}

// The block's entries in order; `half` gets the running sum after its
// first kBlkU4 / 2 loads.
template <bool COMPACT, PhiAt P>
__device__ __forceinline__ float sum_block(const RowBlock &r, float s, uint32_t tb, uint32_t lb,
                                           float &half) {
#pragma unroll
    for (int i = 0; i < kBlkU4; ++i) {
        s = sum_u4<COMPACT, P>(r.e[i], s, tb, lb);
        if (i == kBlkU4 / 2 - 1) half = s;
    }
    return s;
}

// S-bucket search over n consecutive 16-byte pieces of a row from running
// sum `run`: the first entry whose running sum exceeds t2 (running sums never
// decrease).
template <bool COMPACT, PhiAt P, int N>
__device__ __forceinline__ void search_u4(const uint4 (&blk)[N], float &run, float t2, uint32_t tb, uint32_t lb,
                                          uint32_t &newz, bool &found) {
    constexpr bool MULTI = P == kPhiGroup;
    auto at32 = [&](uint32_t e) { return P == kPhiOwn ? phi_own(dt_topic(e), lb) : phi_at0(e); };
#pragma unroll
    for (int gi = 0; gi < N; ++gi) {
        const uint4 e = blk[gi];
        if (COMPACT) {
            const uint32_t w[4] = {e.x, e.y, e.z, e.w};
            const uint32_t tm2 = ((1u << tb) - 1u) * 0x10001u;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const C16x2 d = c16_x2<MULTI>(w[q], tb, tm2, lb);
                const float ra = fma_count(d.c0, phi_a(d.a0), run);
                const float rb = fma_count(d.c1, phi_a(d.a1), ra);
                if (!found && ra > t2) {
                    newz = (d.a0 - (MULTI ? lb : 0u)) >> 2;
                    found = true;
                } else if (!found && rb > t2) {
                    newz = (d.a1 - (MULTI ? lb : 0u)) >> 2;
                    found = true;
                }
                run = rb;
            }
        } else if (!found) {
            const float r0 = __builtin_fmaf(dt_count(e.x), at32(e.x), run);
            const float r1 = __builtin_fmaf(dt_count(e.y), at32(e.y), r0);
            const float r2 = __builtin_fmaf(dt_count(e.z), at32(e.z), r1);
            const float r3 = __builtin_fmaf(dt_count(e.w), at32(e.w), r2);
            if (r3 > t2) {
                newz = dt_topic(r0 > t2 ? e.x : r1 > t2 ? e.y : r2 > t2 ? e.z : e.w);
                found = true;
            }
            run = r3;
        }
    }
}

// Sampler work item: a word, or a doc tile / token segment of a head word,
// given as a range of runs, and the offset from the layout's token ids to
// the corpus-wide ones that key the draws (0 unless the corpus is chunked).  A run is up to run_cap consecutive tokens of the
// word in one document (tokens of a word are numbered by document, so the
// repeats of a word in a document are adjacent); its tokens share n_d, the
// max-topic counts and the DT row, hence the S sum and its checkpoints.  One
// lane per run: the shortcut test of each token, then, if any token needs
// the full draw, one pass over the doc's DT row (16 bytes per load) for S and
// the checkpoints, and per such token the bucket choice and either a re-read
// of one row block to the first running sum above the target (S) or a
// bisection of the monotone Q running sums (Q).  Every token's draw is the
// one it would get on its own; only the row scan is shared.
// Replaces UpdateProbKernelTrainD1 (utility.cu:2680-3312), LDAKernelTrainD
// (:1625-2103) and LDAKernelTrain (:1217-1611); one kernel serves head and
// tail words, which differ only in how phi_w is staged.
struct SampleArgs {
    const uint4 *segs;
    const uint4 *runs;  // (first token, first doc slot, the doc's DT row offset, tokens | doc length << 16)
    uint32_t n_items;
    uint32_t first_item;  // k_sample_own: its first
    int VD, K;
    float alpha, beta;
    const int32_t *wt_head;
    const uint32_t *tail_off, *wt_tail, *tail_nnz;
    const float *inv;
    const ushort4 *wtop;
    const uint32_t *aux_doc;  // by doc slot: n_dk1 | the doc's row length (nnz) << 16
    const uint32_t *dt;
    uint16_t *z, *z_doc;      // by token (word-major) and by doc slot
    const uint32_t *counters;  // [0]: the sweep drawn (DevState's counters, or from their [1] on where it was begun)
    uint32_t *queue;  // persistent mode: queue q's item counter at queue[q * kQueueStride]
    uint32_t n_queues;
    uint32_t tb;  // compact rows: topic bits
    unsigned long long *stats;
    uint64_t seed;
    uint32_t mode;  // kSampleHead | kSampleTail: which words' items; | kShortcutOnly: no full draws
    uint32_t word_stride;  // MULTI: LDS floats of one word's tables
};

// phi (scaled by `up`) of a word's dense counts (COUNTS), or of no counts, into
// LDS, zero past K up to whole slabs.  Every lane has four 16-byte loads of
// each input in flight (eight scalar ones where K is no multiple of 4): one
// load at a time was a chain of K / blockDim latencies an item.  Sampler ms a
// sweep: 4.5M tokens K = 10000 1.36 -> 1.11, 9M K = 4096 0.84 -> 0.70, heavy-
// tailed K = 2048 1.71 -> 1.57, 49.5M K = 1024 2.90 -> 2.87.
template <bool COUNTS>
__device__ __forceinline__ void stage_phi(float *phi, const int32_t *__restrict__ row, const float *__restrict__ inv,
                                          int K, int NS, float beta, float up) {
    const int tid = threadIdx.x, bd = blockDim.x;
    auto value = [&](int32_t c, float iv) { return COUNTS ? ((float)c + beta) * iv * up : beta * iv * up; };
    if ((K & 3) == 0) {
        const int n4 = NS * 16, K4 = K >> 2;
        const int4 *row4 = reinterpret_cast<const int4 *>(row);
        const float4 *inv4 = reinterpret_cast<const float4 *>(inv);
        float4 *phi4 = reinterpret_cast<float4 *>(phi);
        for (int k0 = tid; k0 < n4; k0 += 4 * bd) {
            int4 c[4];
            float4 iv[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = k0 + u * bd;
                c[u] = COUNTS && k < K4 ? row4[k] : make_int4(0, 0, 0, 0);
                iv[u] = k < K4 ? inv4[k] : make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int k = k0 + u * bd;
                if (k < n4)
                    phi4[k] = make_float4(value(c[u].x, iv[u].x), value(c[u].y, iv[u].y), value(c[u].z, iv[u].z),
                                          value(c[u].w, iv[u].w));
            }
        }
    } else {
        for (int k0 = tid; k0 < NS * 64; k0 += 8 * bd) {
            int32_t c[8];
            float iv[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int k = k0 + u * bd;
                c[u] = COUNTS && k < K ? row[k] : 0;
                iv[u] = k < K ? inv[k] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (k0 + u * bd < NS * 64) phi[k0 + u * bd] = value(c[u], iv[u]);
        }
    }
}

// A group item's tables: G words of few tokens (all dense or all sparse),
// word g's phi, Q running sums and totals at g * ST, after them f1, f2 and k1.
// As for one word, but every phase works on all of them at once: small words
// are a chain of latencies each, and fill few of a wavefront's lanes.
template <bool COMPACT>
__device__ __forceinline__ void stage_group(const SampleArgs &A, int w, int G, int ST, float *smf) {
    const int K = A.K, NS = (K + 63) >> 6, tid = threadIdx.x, bd = blockDim.x;
    const float alpha = A.alpha, beta = A.beta;
    constexpr float up = COMPACT ? kPhiUp : 1.0f, down = COMPACT ? kPhiDown : 1.0f;
    const bool head = w < A.VD;
    const int32_t *rows = A.wt_head + (size_t)w * K;
    auto value = [&](int32_t c, float iv) { return ((float)c + beta) * iv * up; };
    if ((K & 3) == 0) {  // slab s of the group: 16 loads of 4 topics
        const int n = G * NS * 16;
        for (int i0 = tid; i0 < n; i0 += 4 * bd) {
            int4 c[4];
            float4 iv[4];
            int at[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int i = i0 + u * bd, sl = i >> 4, g = sl / NS, k = (sl - g * NS) * 64 + (i & 15) * 4;
                at[u] = i < n ? g * ST + k : -1;
                const bool in = i < n && k < K;
                c[u] = in && head ? *reinterpret_cast<const int4 *>(rows + (size_t)g * K + k) : make_int4(0, 0, 0, 0);
                iv[u] = in ? *reinterpret_cast<const float4 *>(A.inv + k) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (at[u] >= 0)
                    *reinterpret_cast<float4 *>(smf + at[u]) =
                        make_float4(value(c[u].x, iv[u].x), value(c[u].y, iv[u].y), value(c[u].z, iv[u].z),
                                    value(c[u].w, iv[u].w));
        }
    } else {
        const int n = G * NS * 64;
        for (int i0 = tid; i0 < n; i0 += 8 * bd) {
            int32_t c[8];
            float iv[8];
            int at[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int i = i0 + u * bd, sl = i >> 6, g = sl / NS, k = (sl - g * NS) * 64 + (i & 63);
                at[u] = i < n ? g * ST + k : -1;
                const bool in = i < n && k < K;
                c[u] = in && head ? rows[(size_t)g * K + k] : 0;
                iv[u] = in ? A.inv[k] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (at[u] >= 0) smf[at[u]] = value(c[u], iv[u]);
        }
    }
    __syncthreads();
    if (!head) {  // four words' nonzeros at a time
        for (int g0 = 0; g0 < G; g0 += 4) {
            uint32_t b[4], n[4], most = 0;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                b[u] = g0 + u < G ? A.tail_off[w - A.VD + g0 + u] : 0u;
                n[u] = g0 + u < G ? A.tail_nnz[w - A.VD + g0 + u] : 0u;
                most = max(most, n[u]);
            }
            for (uint32_t i = tid; i < most; i += bd) {
                uint32_t e[4];
                float iv[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) e[u] = i < n[u] ? A.wt_tail[b[u] + i] : 0u;
#pragma unroll
                for (int u = 0; u < 4; ++u) iv[u] = A.inv[e[u] & 0xFFFFu];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (i < n[u]) smf[(g0 + u) * ST + (int)(e[u] & 0xFFFFu)] = value((int32_t)(e[u] >> 16), iv[u]);
            }
        }
        __syncthreads();
    }
    const int qo = NS * 64, to = 2 * NS * 64;  // a word's Q running sums, slab totals
    for (int g = tid; g < G; g += bd) {
        const ushort4 tp = A.wtop[w + g];
        float *p = smf + g * ST, *wc = p + to + 2 * NS;
        wc[0] = p[tp.x] * down;
        wc[1] = tp.y != kNone ? p[tp.y] * down : 0.0f;
        wc[2] = __uint_as_float((uint32_t)tp.x);
        p[tp.x] = 0.0f;
    }
    __syncthreads();
    for (int i = tid; i < G * NS; i += bd) {  // one slab a lane
        const int g = i / NS, j = i - g * NS;
        const float4 *p4 = reinterpret_cast<const float4 *>(smf + g * ST + j * 64);
        float4 *q4 = reinterpret_cast<float4 *>(smf + g * ST + qo + j * 64);
        float4 v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = p4[u];
        float run = 0.0f;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            run = run + alpha * (v[u].x * down);
            v[u].x = run;
            run = run + alpha * (v[u].y * down);
            v[u].y = run;
            run = run + alpha * (v[u].z * down);
            v[u].z = run;
            run = run + alpha * (v[u].w * down);
            v[u].w = run;
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) q4[u] = v[u];
        smf[g * ST + to + j] = run;
    }
    __syncthreads();
    for (int g = tid; g < G; g += bd) {
        float acc = 0.0f;
        float *qt = smf + g * ST + to;
        for (int j = 0; j < NS; ++j) {
            acc = acc + qt[j];
            qt[NS + j] = acc;
        }
    }
    __syncthreads();
}

// LDS floats of k_sample_own: of what all words of a workgroup share (phi of
// the topics without a count, its slab totals), and of one word (its topics'
// bits and first values, its values, its slabs' running sums, the list of the
// slabs with topics of its own).
__host__ __device__ __forceinline__ int own_shared(int NS) { return (NS * 65 + 3) & ~3; }
__host__ __device__ __forceinline__ int own_stride(int NS) {
    return NS * 4 + (int)kOwnMax + 4 + ((NS + 3) & ~3) + (int)kOwnMax / 4 + 4;
}

// The tables of a tail word of at most kOwnMax tokens, by half a wavefront:
// see phi_own.  f1 and f2 as in sample_item.
__device__ __forceinline__ void stage_own(const SampleArgs &A, int w, ushort4 tp, float *phi0, float *mine, float &f1,
                                          float &f2) {
    const int K = A.K, NS = (K + 63) >> 6, NW = NS * 2, l = threadIdx.x & 31;
    const uint32_t half = threadIdx.x & 32u;
    const float alpha = A.alpha, beta = A.beta;
    constexpr int U = kOwnMax / 32;
    const float *qt_shared = phi0 + NS * 64;
    uint2 *bp = reinterpret_cast<uint2 *>(mine);
    float *val = mine + 2 * NW, *qacc = val + kOwnMax + 4;
    uint8_t *touched = reinterpret_cast<uint8_t *>(qacc + ((NS + 3) & ~3));
    const uint32_t lb = 4u * (uint32_t)(mine - phi0), at0 = (uint32_t)(val - phi0);
    wave_lds_sync();  // the words before are done with them
    for (int i = l; i < NS; i += 32) reinterpret_cast<uint4 *>(bp)[i] = make_uint4(0u, 0u, 0u, 0u);
    // the word's topics: four a lane
    const uint32_t b = A.tail_off[w - A.VD], n = A.tail_nnz[w - A.VD];
    uint32_t e[U];
    float v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) e[u] = (uint32_t)(l + 32 * u) < n ? A.wt_tail[b + l + 32 * u] : 0u;
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = A.inv[e[u] & 0xFFFFu];
    wave_lds_sync();
    // bits of its topics and of its top one, then the index of each 32's first value
    const uint32_t k1 = tp.x;
#pragma unroll
    for (int u = 0; u < U; ++u)
        if ((uint32_t)(l + 32 * u) < n) atomicOr(&bp[(e[u] & 0xFFFFu) >> 5].x, 1u << (e[u] & 31u));
    if (l == 0) atomicOr(&bp[k1 >> 5].x, 1u << (k1 & 31u));
    wave_lds_sync();
    {
        const int per = (NW + 31) >> 5, i0 = l * per, i1 = min(NW, i0 + per);
        uint32_t m = 0;
        for (int i = i0; i < i1; ++i) m += (uint32_t)__popc(bp[i].x);
        uint32_t incl = m;
        for (int d = 1; d < 32; d <<= 1) {
            const uint32_t x = __shfl_up(incl, d, 32);
            if (l >= d) incl += x;
        }
        uint32_t at = at0 + incl - m;
        for (int i = i0; i < i1; ++i) {
            bp[i].y = at;
            at += (uint32_t)__popc(bp[i].x);
        }
    }
    wave_lds_sync();
    auto index = [&](uint32_t k) {
        const uint2 x = bp[k >> 5];
        return x.y + (uint32_t)__popc(x.x & ((1u << (k & 31u)) - 1u));
    };
    if (l == 0) phi0[index(k1)] = phi0[k1];  // it may have no count
    wave_lds_sync();
#pragma unroll
    for (int u = 0; u < U; ++u)
        if ((uint32_t)(l + 32 * u) < n) phi0[index(e[u] & 0xFFFFu)] = ((float)(e[u] >> 16) + beta) * v[u];
    wave_lds_sync();
    f1 = phi_own(k1, lb);
    f2 = tp.y != kNone ? phi_own(tp.y, lb) : 0.0f;
    wave_lds_sync();
    if (l == 0) phi0[index(k1)] = 0.0f;
    wave_lds_sync();
    // slab totals: the shared ones, and those of the slabs with topics of the
    // word's own, summed in the order of sample_item; then their running sums
    uint32_t nt = 0;
    for (int j0 = 0; j0 < ((NS + 3) & ~3); j0 += 32) {
        const int j = j0 + l;
        const bool t = j < NS && (bp[2 * j].x | bp[2 * j + 1].x) != 0u;
        if (j < ((NS + 3) & ~3) && !t) qacc[j] = j < NS ? qt_shared[j] : 0.0f;
        const uint32_t m = (uint32_t)(__ballot(t) >> half);
        if (t) touched[nt + (uint32_t)__popc(m & ((1u << l) - 1u))] = (uint8_t)j;
        nt += (uint32_t)__popc(m);
    }
    wave_lds_sync();
    for (uint32_t i = l; i < nt; i += 32) {
        const int j = (int)touched[i];
        const float4 *p4 = reinterpret_cast<const float4 *>(phi0 + j * 64);
        const uint4 b4 = reinterpret_cast<const uint4 *>(bp)[j];
        const uint32_t bits[2] = {b4.x, b4.z};
        uint32_t at = b4.y;
        float run = 0.0f;
#pragma unroll
        for (int i4 = 0; i4 < 16; i4 += 4) {
            float4 x4[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) x4[u] = p4[i4 + u];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                float x[4] = {x4[u].x, x4[u].y, x4[u].z, x4[u].w};
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if ((bits[i4 >> 3] >> (((4 * i4) & 31) + 4 * u + c)) & 1u) x[c] = phi0[at++];
                    run = run + alpha * x[c];
                }
            }
        }
        qacc[j] = run;
    }
    wave_lds_sync();
    float acc = 0.0f;
    float4 *q4 = reinterpret_cast<float4 *>(qacc);
    for (int j0 = 0; j0 < ((NS + 3) >> 2); j0 += 4) {  // by every lane, the half's first one writes
        float4 x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = j0 + i < ((NS + 3) >> 2) ? q4[j0 + i] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            x[i].x = acc = acc + x[i].x;
            x[i].y = acc = acc + x[i].y;
            x[i].z = acc = acc + x[i].z;
            x[i].w = acc = acc + x[i].w;
        }
        if (l == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (j0 + i < ((NS + 3) >> 2)) q4[j0 + i] = x[i];
        }
    }
    wave_lds_sync();
}

// (kPhiOwn: the item and its tables f123 are those of the lane's half
// wavefront; without `any`, it draws nothing)
template <bool SHORTCUT, bool COMPACT, bool QTAB, PhiAt P>
__device__ __forceinline__ void sample_item(const SampleArgs &A, uint32_t item, float *smf, float *f123,
                                            uint32_t sweep, uint32_t &n_full, uint32_t &n_scanned, bool any = true) {
    const int K = A.K, NS = (K + 63) >> 6;
    const float alpha = A.alpha, beta = A.beta;
    const int tid = threadIdx.x, lane = P == kPhiOwn ? tid & 31 : tid & 63, wv = P == kPhiOwn ? 0 : tid >> 6,
              nwv = P == kPhiOwn ? 1 : blockDim.x >> 6;
    constexpr bool qtab = QTAB;  // K <= EZ_Q_TABLE_MAX_K
    constexpr bool MULTI = P == kPhiGroup;
    constexpr bool OWN = P == kPhiOwn;
    const uint32_t own = OWN ? 4u * (uint32_t)(f123 - smf) : 0u;
    constexpr int CP = Checkpoints<COMPACT, QTAB, MULTI>::CP, CF = Checkpoints<COMPACT, QTAB, MULTI>::CF;
    constexpr float up = COMPACT ? kPhiUp : 1.0f, down = COMPACT ? kPhiDown : 1.0f;
    float *phi0 = smf;                         // NS*64
    float *qs0 = phi0 + NS * 64;                // NS*64 when qtab: running sums inside each slab
    float *qt0 = qs0 + (qtab ? NS * 64 : 0);    // NS: slab totals
    float *qacc0 = OWN ? f123 + NS * 4 + kOwnMax + 4 : qt0 + NS;                    // NS: running sum of the slab totals
    const uint4 sg = A.segs[item];
    if (sg.x == 0xFFFFFFFFu) return;  // padding item (uniform over the block)
    // MULTI: the item's words are w .. w + G - 1, word g's tables at g * ST
    const uint32_t gw = MULTI ? (uint32_t)__builtin_amdgcn_readfirstlane((int)sg.x) : sg.x;
    const int w = MULTI ? (int)(gw & kGroupWord) : (int)gw, G = MULTI ? 1 + (int)(gw >> kGroupShift) : 1;
    const int ST = MULTI ? (int)A.word_stride : 0;
    if (!(A.mode & (w < A.VD ? kSampleHead : kSampleTail))) return;  // the other words' stage
    const bool sc_only = (A.mode & kShortcutOnly) != 0;
    const ushort4 tp = MULTI ? make_ushort4(0, 0, 0, 0) : A.wtop[w];
    float fo1 = 0.0f, fo2 = 0.0f;
    if (MULTI) {
        stage_group<COMPACT>(A, w, G, ST, smf);
    } else if (OWN) {
        stage_own(A, w, tp, smf, f123, fo1, fo2);
    } else {
        if (w < A.VD) {
            stage_phi<true>(phi0, A.wt_head + (size_t)w * K, A.inv, K, NS, beta, up);
        } else {
            // the word's row is on its way while the topics without a count are staged
            const int tw = w - A.VD;
            const uint32_t b = A.tail_off[tw], n = A.tail_nnz[tw];
            stage_phi<false>(phi0, nullptr, A.inv, K, NS, beta, up);
            __syncthreads();
            for (uint32_t i0 = tid; i0 < n; i0 += 4u * blockDim.x) {
                uint32_t e[4];
                float iv[4];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) e[u] = i0 + u * blockDim.x < n ? A.wt_tail[b + i0 + u * blockDim.x] : 0u;
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u) iv[u] = A.inv[e[u] & 0xFFFFu];
#pragma unroll
                for (uint32_t u = 0; u < 4; ++u)
                    if (i0 + u * blockDim.x < n) phi0[e[u] & 0xFFFFu] = ((float)(e[u] >> 16) + beta) * iv[u] * up;
            }
        }
        __syncthreads();
        if (tid == 0) {
            f123[0] = phi0[tp.x] * down;
            f123[1] = tp.y != kNone ? phi0[tp.y] * down : 0.0f;
            f123[2] = tp.z != kNone ? phi0[tp.z] * down : 0.0f;
            phi0[tp.x] = 0.0f;
        }
        __syncthreads();
        // Q: the running sums inside each 64-topic slab, left to right (phi0 is 0
        // past K, which leaves the sum unchanged); the slab's 64 values are
        // loaded at once, then summed in order.  With qtab the running sums are
        // kept; else only the slab total, and a Q draw recomputes its slab's
        // running sums in the same order
        for (int j = tid; j < NS; j += blockDim.x) {
            const float4 *p4 = reinterpret_cast<const float4 *>(phi0 + j * 64);
            float4 v[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) v[i] = p4[i];
            float run = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                run = run + alpha * (v[i].x * down);
                v[i].x = run;
                run = run + alpha * (v[i].y * down);
                v[i].y = run;
                run = run + alpha * (v[i].z * down);
                v[i].z = run;
                run = run + alpha * (v[i].w * down);
                v[i].w = run;
            }
            if (qtab) {
                float4 *q4 = reinterpret_cast<float4 *>(qs0 + j * 64);
#pragma unroll
                for (int i = 0; i < 16; ++i) q4[i] = v[i];
            }
            qt0[j] = run;
        }
        __syncthreads();
        if (tid == 0) {
            float acc = 0.0f;
            for (int j0 = 0; j0 < NS; j0 += 16) {
                float v[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) v[i] = j0 + i < NS ? qt0[j0 + i] : 0.0f;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    if (j0 + i < NS) {
                        acc = acc + v[i];
                        qacc0[j0 + i] = acc;
                    }
                }
            }
        }
        __syncthreads();
    }
    const float Q1 = MULTI ? 0.0f : qacc0[NS - 1], f11 = MULTI ? 0.0f : OWN ? fo1 : f123[0],
                f21 = MULTI ? 0.0f : OWN ? fo2 : f123[1];
    // head words also write the doc-slot copy of z (their items share a doc
    // tile, so the copy's lines fill in L2); tail tokens, in random docs,
    // are read back by token id in the DT rebuild instead
    const bool head = w < A.VD;
    const uint32_t tb = A.tb;

    if (OWN && !any) return;
    for (uint32_t base = sg.y + (uint32_t)wv * 64u; base < sg.z; base += OWN ? 32u : (uint32_t)nwv * 64u) {
        const uint32_t r = base + (uint32_t)lane;
        if (r >= sg.z) break;
        const uint4 rn = A.runs[r];
        const uint32_t t0 = rn.x, p0 = rn.y, nd = rn.w >> 16;
        uint32_t len = rn.w & (MULTI ? 0xFFu : 0xFFFFu);
        // the run's word: its tables and what the draws need of it
        const uint32_t go = MULTI ? ((rn.w >> 8) & 0xFFu) * (uint32_t)ST : 0u, lb = MULTI ? 4u * go : own;
        const float *phi = phi0 + go, *qs = qs0 + go, *qt = qt0 + go, *qacc = qacc0 + go;
        const float *wc = qacc + NS;  // MULTI: f1, f2, k1
        const float Q = MULTI ? qacc[NS - 1] : Q1, f1 = MULTI ? wc[0] : f11, f2 = MULTI ? wc[1] : f21;
        const uint32_t k1 = MULTI ? __float_as_uint(wc[2]) : tp.x;
        // (the empty asm hides len's bound from the optimizer, whose
        // rewrites of the token loops from it otherwise cost a spill)
        asm volatile("" : "+v"(len));
        // n_dk1 and the row's length in one load (a tail word's docs are
        // random ones: a per-doc record would cost a cache line of its own);
        // the row's offset and the doc's length come with the run
        const uint32_t a = A.aux_doc[p0];
        const uint2 di = make_uint2(rn.z, a >> 16);  // row offset, nnz
        const uint32_t n1 = a & 0xFFFFu;
        const float P1 = ((float)n1 + alpha) * f1;
        // tokens of the run that need the full draw; shortcut tokens take k1.
        // The uniforms of the first kUKeep tokens are kept for the draw.
        uint32_t need = 0;
        constexpr int UK = COMPACT ? kUKeep : kUKeep32;
        float uk[UK];
        // S <= (n_d - n_dk1) * phi_k2: every other topic's phi is at most the
        // second largest.  Any bound >= S leaves every draw as the full path
        // makes it (the margin covers the rounding), so the shortcut only
        // skips work; this one needs no n_dk2.
        const float maxS = (float)(nd - n1) * f2;
        const float B = (P1 + maxS) + Q;
#pragma unroll
        for (uint32_t j = 0; j < (uint32_t)UK; ++j) {
            uk[j] = 0.0f;
            if (j < len) {
                const float u = ez_u24(ez_philox_x0(A.seed, t0 + j + sg.w, sweep, EZ_TAG_SAMPLE));
                uk[j] = u;
                if (!SHORTCUT || !(u * B < P1 * kMargin)) {
                    need |= 1u << j;
                } else {
                    A.z[t0 + j] = (uint16_t)k1;
                    if (head) A.z_doc[p0 + j] = (uint16_t)k1;
                }
            }
        }
        for (uint32_t j = UK; j < len; ++j) {
            bool full = true;
            if (SHORTCUT) {
                const float u = ez_u24(ez_philox_x0(A.seed, t0 + j + sg.w, sweep, EZ_TAG_SAMPLE));
                full = !(u * B < P1 * kMargin);
            }
            if (full) {
                need |= 1u << j;
            } else {
                A.z[t0 + j] = (uint16_t)k1;
                if (head) A.z_doc[p0 + j] = (uint16_t)k1;
            }
        }
        if (!need || sc_only) continue;
        // the row: 32-bit entries, or 16-bit entries at a 16-bit offset
        const uint4 *rp = COMPACT ? reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(A.dt) + di.x)
                                  : reinterpret_cast<const uint4 *>(A.dt + di.x);
        const uint32_t nnz = di.y & 0xFFFFu;
        constexpr uint32_t kEPB = (COMPACT ? 8u : 4u) * kBlkU4;  // entries per block
        const uint32_t nb = (nnz + kEPB - 1u) / kEPB;            // blocks of the row
        n_full += (uint32_t)__popc(need);
        n_scanned += nnz;
        // S: one FMA per entry, left to right; cp[b] = running sum at the
        // end of block b (the first CP blocks), so the S-bucket search
        // re-reads one block instead of the row up to the target
        // Block b + 1 is loaded before block b is summed (only by lanes
        // whose row has it, so a wavefront stops loading at its longest row).
        float cp[CP], ch[CP];  // running sum at the end / the middle of block b
        float S = 0.0f;
        RowBlock cur = load_block(rp);
#pragma unroll
        for (int b = 0; b < CP; ++b) {
            RowBlock nxt;
            if ((uint32_t)b + 1u < nb) nxt = load_block(rp + kBlkU4 * (b + 1));
            ch[b] = S;
            if ((uint32_t)b < nb) S = sum_block<COMPACT, P>(cur, S, tb, lb, ch[b]);
            cp[b] = S;
            cur = nxt;
        }
        // past them, CF more checkpoints m blocks apart
        float cf[CF];
#pragma unroll
        for (int i = 0; i < CF; ++i) cf[i] = 0.0f;
        uint32_t m = 0;
        while (__ballot(nb > (uint32_t)(CP + CF * m))) ++m;
        for (uint32_t i = 0, b = CP; m != 0 && i < (uint32_t)CF; ++i) {
            for (const uint32_t e = b + m; b < e; ++b) {
                RowBlock nxt;
                if (b + 1u < nb) nxt = load_block(rp + kBlkU4 * (b + 1u));
                float unused;
                if (b < nb) S = sum_block<COMPACT, P>(cur, S, tb, lb, unused);
                cur = nxt;
            }
#pragma unroll
            for (int q = 0; q < CF; ++q)
                if (i == (uint32_t)q) cf[q] = S;
        }
        const float Aa = P1 + S;
        const float total = Aa + Q;
        while (need) {
            const uint32_t j = (uint32_t)__ffs(need) - 1u;
            need &= need - 1u;
            const uint32_t t = t0 + j;
            float u = uk[0];
#pragma unroll
            for (int i = 1; i < UK; ++i)
                if (j == (uint32_t)i) u = uk[i];
            if (j >= (uint32_t)UK) u = ez_u24(ez_philox_x0(A.seed, t + sg.w, sweep, EZ_TAG_SAMPLE));
            const float target = u * total;
            uint32_t newz = k1;
            // P1 below, S up to Aa, Q above.  The S bucket's loads are issued
            // before the Q lanes search their running sums in LDS, which hides
            // part of their latency.
            const bool in_s = target >= P1 && target < Aa;
            const float t2s = target - P1;
            int bs = -1;
            float run = 0.0f;
            constexpr int NH = kHalfCp && COMPACT ? kBlkU4 / 2 : kBlkU4;  // loads of one search
            uint4 blk[NH];
            if (in_s) {
#pragma unroll
                for (int b = CP - 1; b >= 0; --b)
                    if (cp[b] > t2s) bs = b;
                if (bs >= 0) {
                    // the checkpointed block that holds the target: from the
                    // running sum before it, or with kHalfCp from the one in
                    // its middle, half the block's loads
                    float mid = ch[0];
#pragma unroll
                    for (int b = 0; b < CP - 1; ++b)
                        if (b + 1 == bs) {
                            run = cp[b];
                            mid = ch[b + 1];
                        }
                    uint32_t at = kBlkU4 * (uint32_t)bs;
                    if (NH < kBlkU4 && !(mid > t2s)) {
                        run = mid;
                        at += NH;
                    }
#pragma unroll
                    for (int i = 0; i < NH; ++i) blk[i] = rp[at + i];
                }
            }
            asm volatile("" ::: "memory");  // the loads stay above the Q search
            if (!(target < Aa)) {
                const float t2 = target - Aa;
                int lo = 0, hi = NS;  // first slab whose running sum exceeds t2
                while (lo < hi) {
                    const int mid = (lo + hi) >> 1;
                    if (qacc[mid] > t2) hi = mid; else lo = mid + 1;
                }
                int js = lo < NS ? lo : -1;
                if (js < 0 && OWN)  // the last slab with mass
                    for (int k = K - 1; k >= 0; --k)
                        if (alpha * (phi_own((uint32_t)k, lb) * down) > 0.0f) {
                            js = k >> 6;
                            break;
                        }
                if (js < 0 && !OWN)
                    for (int jj = NS - 1; jj >= 0; --jj)
                        if (qt[jj] > 0.0f) {
                            js = jj;
                            break;
                        }
                if (js >= 0) {
                    const float t3 = t2 - (js > 0 ? qacc[js - 1] : 0.0f);
                    const int k0 = js * 64, ke = min(k0 + 64, K);
                    lo = ke;
                    if (qtab) {  // first running sum above t3, by bisection
                        lo = k0;
                        hi = ke;
                        while (lo < hi) {
                            const int mid = (lo + hi) >> 1;
                            if (qs[mid] > t3) hi = mid; else lo = mid + 1;
                        }
                    }
                    // else the slab's running sums, recomputed in the order
                    // its total was summed: the first above t3
                    const float4 *p4 = reinterpret_cast<const float4 *>(phi + k0);
                    float run = 0.0f;
                    uint32_t bits[2] = {0u, 0u}, own_at = 0;  // the word's own topics of the slab, their next value
                    if (P == kPhiOwn) {
                        lds_cu32 *p = (lds_cu32 *)(lb + 16u * (uint32_t)js);
                        bits[0] = p[0], bits[1] = p[2], own_at = 4u * p[1];
                    }
                    for (int i4 = 0; i4 < 16 && !qtab && lo == ke; i4 += 4) {
                        float4 v[4];
#pragma unroll
                        for (int u = 0; u < 4; ++u) v[u] = p4[i4 + u];
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            float x[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
                            for (int c = 0; c < 4; ++c) {
                                const int k = k0 + 4 * (i4 + u) + c;
                                if (P == kPhiOwn && ((bits[i4 >> 3] >> (((4 * i4) & 31) + 4 * u + c)) & 1u)) {
                                    x[c] = phi_a(own_at);
                                    own_at += 4u;
                                }
                                run = run + alpha * (x[c] * down);
                                if (lo == ke && k < ke && run > t3) lo = k;
                            }
                        }
                    }
                    if (lo < ke) {
                        newz = (uint32_t)lo;
                    } else {
                        for (int k = ke - 1; k >= k0; --k)
                            if (alpha * ((P == kPhiOwn ? phi_own((uint32_t)k, lb) : phi[k]) * down) > 0.0f) {
                                newz = (uint32_t)k;
                                break;
                            }
                    }
                }
            }
            if (in_s) {
                bool found = false;
                if (bs >= 0) {
                    search_u4<COMPACT, P, NH>(blk, run, t2s, tb, lb, newz, found);
                } else if (nb > (uint32_t)CP) {
                    // past them: the blocks of the far checkpoint that holds
                    // the target, in order
                    uint32_t g0 = CP;
                    run = cp[CP - 1];
#pragma unroll
                    for (int i = 0; i < CF - 1; ++i)
                        if (!(cf[i] > t2s)) {
                            g0 = CP + m * (uint32_t)(i + 1);
                            run = cf[i];
                        }
                    for (uint32_t gb = g0; gb < nb && !found; ++gb)
                        search_u4<COMPACT, P, kBlkU4>(load_block(rp + kBlkU4 * gb).e, run, t2s, tb, lb, newz,
                                                            found);
                }
                if (!found) {  // rounding left every running sum at or below t2
                    if (COMPACT) {
                        const uint16_t *rr = reinterpret_cast<const uint16_t *>(A.dt) + di.x;
                        for (uint32_t i = 0; i < nnz; ++i)
                            if (c16_count(rr[i], tb) > 0.0f && phi[c16_topic(rr[i], tb)] > 0.0f) newz = c16_topic(rr[i], tb);
                    } else {
                        const uint32_t *rr = A.dt + di.x;
                        for (uint32_t i = 0; i < nnz; ++i)
                            if (dt_count(rr[i]) > 0.0f &&
                                (P == kPhiOwn ? phi_own(dt_topic(rr[i]), lb) : phi_at0(rr[i])) > 0.0f)
                                newz = dt_topic(rr[i]);
                    }
                }
            }
            A.z[t] = (uint16_t)newz;
            if (head) A.z_doc[p0 + j] = (uint16_t)newz;
        }
    }
}

// Workgroups that take items in turn (item = workgroup, then + grid: n_queues
// 0), or persistent ones that pull
// items from n_queues counters: queue q holds the items with index = q mod
// n_queues (the items of one XCD when items are dealt round-robin to XCDs),
// a workgroup drains its own queue (blockIdx mod n_queues) and then the
// others.  Every workgroup leaves once every queue is past its last item.
template <bool SHORTCUT, bool COMPACT, bool QTAB, bool MULTI>
__global__ void __launch_bounds__(1024) k_sample(const SampleArgs A) {
    // the only LDS of the kernel, so phi starts at address 0 and a DT entry's
    // low half is directly the LDS address of its phi value
    extern __shared__ float smf[];
    const int NS = (A.K + 63) >> 6;
    float *f123 = smf + (QTAB ? 2 : 1) * NS * 64 + 2 * NS;  // after phi, qs, qt, qacc
    // MULTI: the item number before the words' tables end (the last word of
    // the pad of its stride)
    uint32_t &s_item = *reinterpret_cast<uint32_t *>(MULTI ? smf + A.word_stride - 1 : f123 + 3);
    const uint32_t sweep = A.counters[0];
    uint32_t n_full = 0, n_scanned = 0;
    const bool own = A.n_queues == 0;  // items dealt in turn
    const uint32_t nq = own ? 1u : A.n_queues, x0 = blockIdx.x % nq;
    for (uint32_t h = 0; h < nq; ++h) {
        const uint32_t q = (x0 + h) % nq;
        for (uint32_t i = 0;; ++i) {
            uint64_t item = (uint64_t)blockIdx.x + (uint64_t)i * gridDim.x;
            if (!own) {
                __syncthreads();  // the previous item is done with s_item and LDS
                if (threadIdx.x == 0) s_item = atomicAdd(&A.queue[q * kQueueStride], 1u);
                __syncthreads();
                item = (uint64_t)q + (uint64_t)s_item * nq;
            }
            if (item >= A.n_items) break;
            if (own && i) __syncthreads();
            sample_item<SHORTCUT, COMPACT, QTAB, MULTI ? kPhiGroup : kPhiOne>(A, (uint32_t)item, smf, f123, sweep, n_full, n_scanned);
        }
    }
    // per-wavefront totals of the counters
    const int lane = threadIdx.x & 63;
    for (int off = 32; off >= 1; off >>= 1) {
        n_full += __shfl_xor(n_full, off);
        n_scanned += __shfl_xor(n_scanned, off);
    }
    if (lane == 0 && n_full) {
        atomicAdd(&A.stats[0], (unsigned long long)n_full);
        atomicAdd(&A.stats[1], (unsigned long long)n_scanned);
    }
}

// Tail words of at most kOwnMax tokens (32-bit rows), two a wavefront: what
// their phi has in common is staged once for the whole launch and a word adds
// its own few values (phi_own), so a CU works on 32 words at a time, without
// barriers, where three workgroups with a table each fit (K = 10000) and wait
// for memory in 78% of their cycles.  Bound by the VALU (a lookup is 11
// operations where one table takes one) and by lanes without a run: a word a
// wavefront took 412 us where two take 312.  Sampler ms a sweep, with a table
// a word / with this: 4.5M tokens in short documents at K = 10000 1.11 / 0.74,
// 16383 1.84 / 0.90; 3.2M heavy-tailed at K = 10000 7.57 / 3.80; 3M tokens of
// 60,000 equally frequent words at K = 8200 2.42 / 1.14, 10000 3.06 / 1.16.
// In 16-bit rows (K <= 8192) an entry takes 3.5 operations and 4 to 16 tables
// fit: there it lost (a word a wavefront at K = 4096: 0.96 / 1.63 and, heavy-
// tailed, 1.76 / 4.84; K = 7000 0.80 / 0.72).  Items from first_item on, in
// pairs from a queue an XCD (dealt in turn, 320 us and 4.29 ms heavy-tailed).
// A workgroup drains the queue of its number modulo kQueues and no other, so
// the grid is at least kQueues workgroups.
template <bool SHORTCUT>
__global__ void __launch_bounds__(1024) k_sample_own(const SampleArgs A) {
    extern __shared__ float smf[];  // the only LDS: phi at address 0
    const int NS = (A.K + 63) >> 6, wv = threadIdx.x >> 6, nwv = blockDim.x >> 6;
    const uint32_t sweep = A.counters[0];
    uint32_t n_full = 0, n_scanned = 0;
    stage_phi<false>(smf, nullptr, A.inv, A.K, NS, A.beta, 1.0f);
    __syncthreads();
    for (int j = threadIdx.x; j < NS; j += blockDim.x) {
        const float *p = smf + j * 64;
        float run = 0.0f;
        for (int i = 0; i < 64; ++i) run = run + A.alpha * p[i];
        smf[NS * 64 + j] = run;
    }
    __syncthreads();
    const uint32_t h = (threadIdx.x >> 5) & 1u;
    float *mine = smf + own_shared(NS) + (2 * wv + (int)h) * own_stride(NS);
    // queue q: the pairs of items with index = q mod kQueues, of which a
    // wavefront claims its next one while it draws the last
    const uint32_t q = blockIdx.x % kQueues, n_pairs = (A.n_items - A.first_item + 1u) / 2u;
    uint32_t *head = A.queue + kQueueStride * (kQueues + q);
    auto claim = [&]() {
        uint32_t c = 0;
        if ((threadIdx.x & 63u) == 0) c = atomicAdd(head, 1u);
        return c;
    };
    uint32_t next = claim();
    for (;;) {
        const uint32_t pair = q + kQueues * (uint32_t)__builtin_amdgcn_readfirstlane((int)next);
        if (pair >= n_pairs) break;
        next = claim();
        const uint32_t at = A.first_item + 2u * pair;
        const bool any = at + h < A.n_items;
        sample_item<SHORTCUT, false, false, kPhiOwn>(A, at + (any ? h : 0u), smf, mine, sweep, n_full, n_scanned, any);
    }
    const int lane = threadIdx.x & 63;
    for (int off = 32; off >= 1; off >>= 1) {
        n_full += __shfl_xor(n_full, off);
        n_scanned += __shfl_xor(n_scanned, off);
    }
    if (lane == 0 && n_full) {
        atomicAdd(&A.stats[0], (unsigned long long)n_full);
        atomicAdd(&A.stats[1], (unsigned long long)n_scanned);
    }
}

// ------------------------------------------------ FP64 log-likelihood
// sum_t log( sum_k (n_dk + alpha)/(n_d + K alpha) * (n_wk + beta)/(n_k + V beta) )
// per token, the term of profilePerp/utility.cu:2398,2810 reduced in FP64
// (profilePerp/utility.cu:2858-2928).  One workgroup per sampler item (phi_w
// in FP64 in LDS), one lane per run; the per-item partials are summed in
// fixed order by k_ll_final.  Bound by the latencies of an item (most have
// fewer than 64 runs: workgroups are as small as the LDS lets a CU hold 12
// wavefronts of) and by the row scan: 9.9M tokens at K = 1024 1.40 -> 0.67 ms
// (256 threads an item, an FP64 division a phi, one 16-byte load of the row in
// flight).  Workgroups with further items keep beta * inv64 in phi between
// tail words, so such a word stages only its nonzeros.
template <bool COMPACT, bool MULTI>
__global__ void __launch_bounds__(1024) k_ll(uint32_t n_items, const uint4 *__restrict__ segs, const uint4 *__restrict__ runs, int VD,
                                             int K, double alpha, double beta,
                                             const int32_t *__restrict__ wt_head,
                                             const uint32_t *__restrict__ tail_off,
                                             const uint32_t *__restrict__ wt_tail,
                                             const uint32_t *__restrict__ tail_nnz, const double *__restrict__ inv64,
                                             const uint32_t *__restrict__ aux_doc, const uint32_t *__restrict__ dt,
                                             uint32_t tb, double *__restrict__ part) {
    extern __shared__ double smd[];
    __shared__ double red[16];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, nwv = blockDim.x >> 6;
    double *phi = smd;
    __shared__ double qg[MULTI ? kGroupMax : 1];
    // sum over the workgroup, in wavefront order
    auto block_total = [&](double v) {
        for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off);
        if (nwv == 1) return v;
        __syncthreads();  // the previous total is read
        if (lane == 0) red[wv] = v;
        __syncthreads();
        v = 0.0;
        for (int i = 0; i < nwv; ++i) v += red[i];
        return v;
    };
    bool base = false;  // phi holds beta * inv64, their sum in qbase
    double qbase = 0.0;
    for (uint32_t item = blockIdx.x; item < n_items; item += gridDim.x) {
        const uint4 sg = segs[item];
        if (sg.x == 0xFFFFFFFFu) {  // padding item
            if (tid == 0) part[item] = 0.0;
            continue;
        }
        const int w = MULTI ? (int)(sg.x & kGroupWord) : (int)sg.x;
        uint32_t tb0 = 0, tn = 0;
        double q = 0.0;
        if (MULTI) {  // word g's phi at g * K, its Q mass after the words' tables
            const int G = 1 + (int)(sg.x >> kGroupShift);
            for (int i = tid; i < G * K; i += blockDim.x) {
                const int g = i / K, k = i - g * K;
                phi[i] = ((w < VD ? (double)wt_head[(size_t)w * K + i] : 0.0) + beta) * inv64[k];
            }
            __syncthreads();
            if (w >= VD)
                for (int g = 0; g < G; ++g) {
                    const uint32_t b = tail_off[w - VD + g], n = tail_nnz[w - VD + g];
                    for (uint32_t i = tid; i < n; i += blockDim.x) {
                        const uint32_t e = wt_tail[b + i], k = e & 0xFFFFu;
                        phi[(uint32_t)(g * K) + k] = ((double)(e >> 16) + beta) * inv64[k];
                    }
                }
            __syncthreads();
            for (int g = wv; g < G; g += nwv) {
                double x = 0.0;
                for (int k = lane; k < K; k += 64) x += phi[g * K + k];
                for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off);
                if (lane == 0) qg[g] = x * alpha;
            }
        } else if (w < VD) {
            const int32_t *row = wt_head + (size_t)w * K;
            for (int k = tid; k < K; k += blockDim.x) {
                const double v = ((double)row[k] + beta) * inv64[k];
                phi[k] = v;
                q += v;
            }
            q = block_total(q);
            base = false;
        } else {
            if (!base) {
                qbase = 0.0;
                for (int k = tid; k < K; k += blockDim.x) {
                    const double v = beta * inv64[k];
                    phi[k] = v;
                    qbase += v;
                }
                qbase = block_total(qbase);
                base = true;
                __syncthreads();
            }
            tb0 = tail_off[w - VD];
            tn = tail_nnz[w - VD];
            for (uint32_t i = tid; i < tn; i += blockDim.x) {
                const uint32_t e = wt_tail[tb0 + i], k = e & 0xFFFFu;
                const double c = (double)(e >> 16), iv = inv64[k];
                phi[k] = (c + beta) * iv;
                q += c * iv;
            }
            q = qbase + block_total(q);
        }
        q *= alpha;
        __syncthreads();
        // one lane per run (a word's tokens in one doc share the term): its DT
        // row in blocks of kBlkU4 16-byte loads, the next one loaded while one is
        // summed (rows are 128-byte aligned and zero padded; a zero entry adds
        // nothing)
        double acc = 0.0;
        const double kalpha = (double)K * alpha;
        const uint32_t tmask = (1u << tb) - 1u;
        for (uint32_t r = sg.y + (uint32_t)tid; r < sg.z; r += (uint32_t)blockDim.x) {
            const uint4 rn = runs[r];
            const uint32_t g = MULTI ? (rn.w >> 8) & 0xFFu : 0u;
            const double *ph = phi + g * (uint32_t)K;
            if (MULTI) q = qg[g];
            const uint2 di = make_uint2(rn.z, aux_doc[rn.y] >> 16);  // row offset, nnz
            const uint32_t nnz = di.y & 0xFFFFu;
            const uint4 *rp = COMPACT ? reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(dt) + di.x)
                                      : reinterpret_cast<const uint4 *>(dt + di.x);
            constexpr uint32_t kEPB = (COMPACT ? 8u : 4u) * kBlkU4;  // entries per block
            const uint32_t nb = (nnz + kEPB - 1u) / kEPB;
            double s = 0.0;
            RowBlock cur = load_block(rp);
            for (uint32_t b = 0; b < nb; ++b) {
                RowBlock nxt;
                if (b + 1u < nb) nxt = load_block(rp + kBlkU4 * (b + 1u));
    #pragma unroll
                for (int i = 0; i < kBlkU4; ++i) {
                    const uint4 v = cur.e[i];
                    const uint32_t e[4] = {v.x, v.y, v.z, v.w};
    #pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        if (COMPACT) {
                            const uint32_t x = e[u] & 0xFFFFu, y = e[u] >> 16;
                            s = __builtin_fma((double)(x >> tb), ph[x & tmask], s);
                            s = __builtin_fma((double)(y >> tb), ph[y & tmask], s);
                        } else {
                            s = __builtin_fma((double)(e[u] >> 16), ph[dt_topic(e[u])], s);
                        }
                    }
                }
                cur = nxt;
            }
            acc += (double)(rn.w & 0xFFu) * log((s + q) / ((double)(rn.w >> 16) + kalpha));
        }
        acc = block_total(acc);
        if (tid == 0) part[item] = acc;
        if (!MULTI && w >= VD && item + gridDim.x < n_items) {  // the base again (every lane is past its reads of phi)
            for (uint32_t i = tid; i < tn; i += blockDim.x) {
                const uint32_t k = wt_tail[tb0 + i] & 0xFFFFu;
                phi[k] = beta * inv64[k];
            }
        }
        __syncthreads();  // the next item's phi
    }
}

// One workgroup of 1024 threads, eight partials in flight a thread (one by
// one in 256 threads: 101 us for 140,000 partials, 16 now).
__global__ void __launch_bounds__(1024) k_ll_final(const double *__restrict__ part, int n, double *__restrict__ out) {
    __shared__ double red[1024];
    double s[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int i = threadIdx.x; i < n; i += 8 * 1024) {
#pragma unroll
        for (int u = 0; u < 8; ++u) s[u] += i + 1024 * u < n ? part[i + 1024 * u] : 0.0;
    }
    red[threadIdx.x] = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    __syncthreads();
    for (int h = 512; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = red[0];
}

// --------------------------------------------------------------- fold-in
// Frozen-model tables for fold-in (no reference counterpart): per word the
// phi row and the Q bucket's running sums (inside 64-topic slabs, and over the
// slab totals), from the counts of the model at freezing time.
__global__ void __launch_bounds__(256) k_foldin_tables(int V, int VD, int K, float alpha, float beta,
                                                       const int32_t *__restrict__ wt_head,
                                                       const uint32_t *__restrict__ tail_off,
                                                       const uint32_t *__restrict__ wt_tail,
                                                       const uint32_t *__restrict__ tail_nnz,
                                                       const float *__restrict__ inv, float *__restrict__ phi_out,
                                                       float *__restrict__ qs_out, float *__restrict__ qacc_out) {
    extern __shared__ float ph[];
    const int NS = (K + 63) >> 6;
    const int tid = threadIdx.x;
    for (int w = blockIdx.x; w < V; w += gridDim.x) {
        if (w < VD) {
            const int32_t *row = wt_head + (size_t)w * K;
            for (int k = tid; k < K; k += blockDim.x) ph[k] = ((float)row[k] + beta) * inv[k];
        } else {
            for (int k = tid; k < K; k += blockDim.x) ph[k] = beta * inv[k];
            __syncthreads();
            const int tw = w - VD;
            const uint32_t b = tail_off[tw], n = tail_nnz[tw];
            for (uint32_t i = tid; i < n; i += blockDim.x) {
                const uint32_t e = wt_tail[b + i];
                const uint32_t k = e & 0xFFFFu;
                ph[k] = ((float)(e >> 16) + beta) * inv[k];
            }
        }
        __syncthreads();
        float *po = phi_out + (size_t)w * K;
        for (int k = tid; k < K; k += blockDim.x) po[k] = ph[k];
        float *qo = qs_out + (size_t)w * K;
        __shared__ float qt[1024];  // slab totals (NS <= 256 for K <= 16383)
        for (int j = tid; j < NS; j += blockDim.x) {
            const int k0 = j * 64, ke = min(k0 + 64, K);
            float run = 0.0f;
            for (int k = k0; k < ke; ++k) {
                run = run + alpha * ph[k];
                qo[k] = run;
            }
            qt[j] = run;
        }
        __syncthreads();
        if (tid == 0) {
            float acc = 0.0f;
            for (int j = 0; j < NS; ++j) {
                acc = acc + qt[j];
                qacc_out[(size_t)w * NS + j] = acc;
            }
        }
        __syncthreads();
    }
}

static constexpr int kFB = 8, kFCP = 16;     // fold-in S blocks and checkpoints
static constexpr uint32_t kFoldSeg = 256;     // tokens per big fold-in work item at most
static constexpr uint32_t kFoldHot = 2048;    // word ranks counted in LDS before the global atomics
static constexpr uint32_t kFoldStageQ = 64;   // tokens of a word in a step that make big items

// A fold-in step runs in word-major order, as the training sweep does: the
// resident documents' rows are built (k_fi_rows), their tokens are bucketed
// by word (k_fi_count, the three-pass scan, k_fi_scatter), and persistent
// workgroups take one (word, segment) item at a time, stage the frozen phi
// row and Q running sums in LDS and draw its tokens (k_fi_sample); documents
// finishing their last sweep get their topics packed for one copy to the host
// (k_fi_final), where they are counted.  Steps of few tokens are drawn
// without buckets (k_fi_few).  The order tokens are drawn in never
// changes a draw, which is keyed by (seed, request id, position, sweep).
// Slots are (request id, pool offset, tokens, sweep); pool offsets are
// multiples of 8, and a document's row lives in the row pool at its offset
// (at most min(n, K) entries, zero padded to a multiple of 8 <= round8(n)).

// Copies admitted documents' words from the upload buffer into the pool:
// records (source offset, pool offset, tokens, 0).
__global__ void __launch_bounds__(256) k_fi_admit(const uint4 *__restrict__ adm, int nadm,
                                                  const uint32_t *__restrict__ src, uint32_t *__restrict__ wpool) {
    for (int a = blockIdx.x; a < nadm; a += gridDim.x) {
        const uint4 r = adm[a];
        for (uint32_t i = threadIdx.x; i < r.z; i += blockDim.x) wpool[r.y + i] = src[r.x + i];
    }
}

// f(value, i) for every i < n of a document's pool range, eight loads per
// thread issued before their uses (long documents would otherwise chain one
// load latency per 256 tokens).
template <class T, class F>
__device__ __forceinline__ void for_doc_tokens(const T *__restrict__ p, uint32_t n, F f) {
    constexpr int U = 8;
    for (uint32_t i0 = threadIdx.x; i0 < n; i0 += U * blockDim.x) {
        T v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + (uint32_t)u * blockDim.x;
            v[u] = i < n ? p[i] : T(0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t i = i0 + (uint32_t)u * blockDim.x;
            if (i < n) f(v[u], i);
        }
    }
}

// Rows of the resident documents (one workgroup per slot): topics drawn from
// the init stream on sweep 0, a 16-bit LDS histogram, a row of topic | count
// << 16 in ascending topic order, zero padded to a multiple of kFB.
// With `group` tokens a workgroup set, also lists the workgroups of k_fi_few:
// slot << 16 | part, from the slot's place in goff.
__global__ void __launch_bounds__(256) k_fi_rows(const uint4 *__restrict__ slots, int nslots, int K, uint64_t seed,
                                                 uint16_t *__restrict__ zpool, uint32_t *__restrict__ rows,
                                                 uint32_t *__restrict__ row_nnz, uint32_t group,
                                                 const uint32_t *__restrict__ goff, uint32_t *__restrict__ groups) {
    extern __shared__ uint32_t shr[];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, bd = blockDim.x;
    const int KH = (K + 1) >> 1;
    uint32_t *h = shr;
    for (int k = tid; k < KH; k += bd) h[k] = 0;
    __syncthreads();
    for (int j = blockIdx.x; j < nslots; j += gridDim.x) {
        const uint4 sl = slots[j];
        const uint32_t rid = sl.x, off = sl.y, n = sl.z, sweep = sl.w;
        uint16_t *z = zpool + off;
        if (group)
            for (uint32_t p = tid; p * group < n; p += bd) groups[goff[j] + p] = ((uint32_t)j << 16) | p;
        if (sweep == 0) {
            for (uint32_t i = tid; i < n; i += bd)
                z[i] = (uint16_t)(ez_philox_x0(seed, ((uint64_t)rid << 32) | i, 0u, EZ_TAG_FOLDIN_INIT) % (uint32_t)K);
            __syncthreads();
        }
        for_doc_tokens(z, n, [&](uint16_t t, uint32_t) { h16_add(h, t); });
        __syncthreads();
        if (wv == 0) {  // one wavefront compacts the row (and clears the counts)
            uint32_t *row = rows + off;
            uint32_t nz = 0;
            for (int c0 = 0; c0 < K; c0 += 64) {
                const int k = c0 + lane;
                const uint32_t c = k < K ? h16_get(h, (uint32_t)k) : 0u;
                const uint64_t m = __ballot(c != 0);
                if (c) row[nz + __popcll(m & lanemask_lt(lane))] = (uint32_t)k | (c << 16);
                nz += (uint32_t)__popcll(m);
                wave_lds_sync();
                if (k < K && !(k & 1)) h[k >> 1] = 0;
            }
            // zero entries up to the next block: count 0 adds exactly nothing
            if ((uint32_t)lane < ((kFB - (nz % kFB)) % kFB)) row[nz + lane] = 0u;
            if (lane == 0) row_nnz[j] = nz;
        }
        __syncthreads();
    }
}

// Tokens per word of the resident documents; the most frequent ranks are
// summed in LDS first so they take one global atomic per workgroup.
__global__ void __launch_bounds__(256) k_fi_count(const uint4 *__restrict__ slots, int nslots,
                                                  const uint32_t *__restrict__ wpool, uint32_t *__restrict__ wcount) {
    __shared__ uint32_t hc[kFoldHot];
    const int tid = threadIdx.x, bd = blockDim.x;
    for (uint32_t k = tid; k < kFoldHot; k += bd) hc[k] = 0;
    __syncthreads();
    for (int j = blockIdx.x; j < nslots; j += gridDim.x) {
        const uint4 sl = slots[j];
        for_doc_tokens(wpool + sl.y, sl.z, [&](uint32_t w, uint32_t) {
            if (w < kFoldHot) atomicAdd(&hc[w], 1u);
            else atomicAdd(&wcount[w], 1u);
        });
    }
    __syncthreads();
    for (uint32_t k = tid; k < kFoldHot; k += bd)
        if (hc[k]) atomicAdd(&wcount[k], hc[k]);
}

// Exclusive scan of M values per thread over a workgroup of up to 1024
// threads; the totals go to tot.  sh holds 16 * M words.
template <int M>
__device__ __forceinline__ void block_scan(uint32_t (&v)[M], uint32_t *sh, uint32_t (&tot)[M]) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    uint32_t inc[M];
#pragma unroll
    for (int m = 0; m < M; ++m) inc[m] = v[m];
    for (int d = 1; d < 64; d <<= 1) {
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const uint32_t x = __shfl_up(inc[m], d);
            if (lane >= d) inc[m] += x;
        }
    }
    if (lane == 63)
#pragma unroll
        for (int m = 0; m < M; ++m) sh[16 * m + wv] = inc[m];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < M; ++m) {
        uint32_t o = 0, t = 0;
        for (int w = 0; w < nw; ++w) {
            const uint32_t x = sh[16 * m + w];
            if (w < wv) o += x;
            t += x;
        }
        tot[m] = t;
        v[m] = o + inc[m] - v[m];
    }
    __syncthreads();
}

// A word with at least kFoldStageQ tokens in the step is big: its tokens
// form items of at most kFoldSeg tokens, a workgroup each, with its phi
// row staged in LDS.  The other words' tokens follow all big words' tokens
// in the bucketed list and are drawn one lane per token straight from the
// tables.
__device__ __forceinline__ uint32_t fold_big(uint32_t c) { return c >= kFoldStageQ ? (c + kFoldSeg - 1u) / kFoldSeg : 0u; }

// Scan pass 1: per 1024 words, their big-word tokens, big items and
// small-word tokens.
__global__ void __launch_bounds__(1024) k_fi_bsum(int V, const uint32_t *__restrict__ wcount,
                                                  uint32_t *__restrict__ bsum) {
    __shared__ uint32_t sh[48];
    const uint32_t w = blockIdx.x * 1024u + threadIdx.x;
    const uint32_t c = w < (uint32_t)V ? wcount[w] : 0u;
    const bool bg = c >= kFoldStageQ;
    uint32_t v[3] = {bg ? c : 0u, fold_big(c), bg ? 0u : c}, t[3];
    block_scan<3>(v, sh, t);
    if (threadIdx.x == 0)
        for (int m = 0; m < 3; ++m) bsum[3 * blockIdx.x + m] = t[m];
}

// Scan pass 2 (one workgroup): exclusive offsets of the per-block sums; ctr
// = [big items, big-word tokens, small-word tokens, 0].
__global__ void __launch_bounds__(1024) k_fi_btop(int nb, uint32_t *__restrict__ bsum, uint32_t *__restrict__ ctr) {
    __shared__ uint32_t sh[48];
    uint32_t carry[3] = {0u, 0u, 0u};
    for (int c0 = 0; c0 < nb; c0 += 1024) {
        const int i = c0 + (int)threadIdx.x;
        uint32_t v[3], t[3];
        for (int m = 0; m < 3; ++m) v[m] = i < nb ? bsum[3 * i + m] : 0u;
        block_scan<3>(v, sh, t);
        for (int m = 0; m < 3; ++m) {
            if (i < nb) bsum[3 * i + m] = carry[m] + v[m];
            carry[m] += t[m];
        }
    }
    if (threadIdx.x == 0) {
        ctr[0] = carry[1];
        ctr[1] = carry[0];
        ctr[2] = carry[2];
        ctr[3] = 0u;
    }
}

// Scan pass 3: bucket starts (the scatter's cursors: big words first, then
// small words, each in word order) and the big items (word, first, end, 0).
__global__ void __launch_bounds__(1024) k_fi_bfin(int V, const uint32_t *__restrict__ wcount,
                                                  const uint32_t *__restrict__ bsum, const uint32_t *__restrict__ ctr,
                                                  uint32_t *__restrict__ wcursor, uint4 *__restrict__ big) {
    __shared__ uint32_t sh[48];
    const uint32_t w = blockIdx.x * 1024u + threadIdx.x;
    const uint32_t c = w < (uint32_t)V ? wcount[w] : 0u;
    const bool bg = c >= kFoldStageQ;
    uint32_t v[3] = {bg ? c : 0u, fold_big(c), bg ? 0u : c}, t[3];
    block_scan<3>(v, sh, t);
    if (w >= (uint32_t)V) return;
    if (bg) {
        const uint32_t base = bsum[3 * blockIdx.x] + v[0];
        wcursor[w] = base;
        uint32_t ib = bsum[3 * blockIdx.x + 1] + v[1];
        for (uint32_t x = 0; x < c; x += kFoldSeg) big[ib++] = make_uint4(w, base + x, base + min(c, x + kFoldSeg), 0u);
    } else {
        wcursor[w] = ctr[1] + bsum[3 * blockIdx.x + 2] + v[2];
    }
}

// Token references (slot << 16 | position) bucketed by word.  Ranks below
// kFoldHot are counted in LDS, reserve one range per workgroup and fill it
// through LDS cursors; the rest take a global cursor per token.
__global__ void __launch_bounds__(256) k_fi_scatter(const uint4 *__restrict__ slots, int nslots,
                                                    const uint32_t *__restrict__ wpool, uint32_t *__restrict__ wcursor,
                                                    uint32_t *__restrict__ tokw) {
    __shared__ uint32_t hc[kFoldHot];
    const int tid = threadIdx.x, bd = blockDim.x;
    for (uint32_t k = tid; k < kFoldHot; k += bd) hc[k] = 0;
    __syncthreads();
    for (int j = blockIdx.x; j < nslots; j += gridDim.x) {
        const uint4 sl = slots[j];
        for_doc_tokens(wpool + sl.y, sl.z, [&](uint32_t w, uint32_t i) {
            if (w < kFoldHot) atomicAdd(&hc[w], 1u);
            else tokw[atomicAdd(&wcursor[w], 1u)] = ((uint32_t)j << 16) | i;
        });
    }
    __syncthreads();
    {  // one range per hot word of the workgroup; the atomics issued together
        constexpr uint32_t U = kFoldHot / 256;
        uint32_t c[U], b[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) c[u] = tid + u * bd < kFoldHot ? hc[tid + u * bd] : 0u;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) b[u] = c[u] ? atomicAdd(&wcursor[tid + u * bd], c[u]) : 0u;
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (c[u]) hc[tid + u * bd] = b[u];
        for (uint32_t k = tid + U * bd; k < kFoldHot; k += bd) {  // block sizes below 256
            const uint32_t cc = hc[k];
            if (cc) hc[k] = atomicAdd(&wcursor[k], cc);
        }
    }
    __syncthreads();
    for (int j = blockIdx.x; j < nslots; j += gridDim.x) {
        const uint4 sl = slots[j];
        for_doc_tokens(wpool + sl.y, sl.z, [&](uint32_t w, uint32_t i) {
            if (w < kFoldHot) tokw[atomicAdd(&hc[w], 1u)] = ((uint32_t)j << 16) | i;
        });
    }
}

__device__ __forceinline__ float fi_sum8(const uint4 &a, const uint4 &b, const float *ph, float s) {
    const uint32_t e[kFB] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int u = 0; u < kFB; ++u) s = __builtin_fmaf((float)(e[u] >> 16), ph[e[u] & 0xFFFFu], s);
    return s;
}

// The entry of a block (zero padded) at which the running sum from `run`
// first exceeds the target; -1 if none does.  Zero entries add exactly
// nothing, so they never cross the target first.
__device__ __forceinline__ int fi_scan8(const uint4 &a, const uint4 &b, const float *ph, float run, float target) {
    const uint32_t e[kFB] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    int zz = -1;
#pragma unroll
    for (int q = 0; q < kFB; ++q) {
        run = __builtin_fmaf((float)(e[q] >> 16), ph[e[q] & 0xFFFFu], run);
        if (zz < 0 && run > target) zz = (int)(e[q] & 0xFFFFu);
    }
    return zz;
}

// First index in [k0, ke) whose running sum exceeds t, ke if none: the
// running sums are nondecreasing, so this is the index a bisection finds.
// Rounds of 8 independent loads: the last entries of up to 8 groups of 8,
// then the entries of the first group whose last one exceeds t.
__device__ __forceinline__ int first_above(const float *q, int k0, int ke, float t) {
    for (int c0 = k0; c0 < ke; c0 += 64) {
        const int c1 = min(c0 + 64, ke);
        int grp = -1;
#pragma unroll
        for (int g = 7; g >= 0; --g) {
            const int s0 = c0 + 8 * g;
            if (s0 < c1 && q[min(s0 + 7, c1 - 1)] > t) grp = g;
        }
        if (grp >= 0) {
            const int g0 = c0 + 8 * grp, g1 = min(g0 + 8, c1);
            int lo = g1;
#pragma unroll
            for (int u = 7; u >= 0; --u)
                if (g0 + u < g1 && q[g0 + u] > t) lo = g0 + u;
            return lo;
        }
    }
    return ke;
}

// The Q bucket's topic at t2 (a word's phi row ph and running sums qa over the
// slab totals, qw within slabs): the first whose running sum exceeds it, else
// the last of positive mass; -1 if there is none.
__device__ __forceinline__ int fi_q_topic(float t2, const float *ph, const float *qa, const float *qw, int K, int NS,
                                          float alpha) {
    const int lo = first_above(qa, 0, NS, t2);
    int js = lo < NS ? lo : -1;
    if (js < 0)
        for (int jj = NS - 1; jj >= 0; --jj)
            if (qa[jj] > (jj > 0 ? qa[jj - 1] : 0.0f)) {
                js = jj;
                break;
            }
    if (js < 0) return -1;
    const float t3 = t2 - (js > 0 ? qa[js - 1] : 0.0f);
    const int k0 = js * 64, ke = min(k0 + 64, K);
    const int kq = first_above(qw, k0, ke, t3);
    if (kq < ke) return kq;
    for (int k = ke - 1; k >= k0; --k)
        if (alpha * ph[k] > 0.0f) return k;
    return -1;
}

// One fold-in draw: token i of slot sl (its row of nz entries at pool
// offset sl.y) for a word whose phi row (ph) and Q running sums (qa over
// the slab totals, qw within slabs) are given, in LDS or in the tables.  S
// over the row in blocks of kFB entries, four blocks' loads issued together
// (the first kFCP block sums kept), then the S entry or the Q topic whose
// running sum first exceeds the target.
__device__ __forceinline__ void fi_draw(const uint4 sl, uint32_t i, uint32_t nz, const uint32_t *__restrict__ rows,
                                        const float *ph, const float *qa, const float *qw, int K, int NS, float alpha,
                                        uint64_t seed, uint16_t *__restrict__ zpool) {
    const uint32_t *row = rows + sl.y;
    const float u = ez_u24(ez_philox_x0(seed, ((uint64_t)sl.x << 32) | i, sl.w, EZ_TAG_FOLDIN));
    const uint32_t nb = (nz + kFB - 1) / kFB;
    float cp[kFCP];
    float S = 0.0f;
#pragma unroll
    for (int g = 0; g < kFCP; g += 4) {
        uint4 e[8];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            e[2 * q] = e[2 * q + 1] = make_uint4(0u, 0u, 0u, 0u);
            if ((uint32_t)(g + q) < nb) {
                e[2 * q] = *(const uint4 *)(row + kFB * (g + q));
                e[2 * q + 1] = *(const uint4 *)(row + kFB * (g + q) + 4);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if ((uint32_t)(g + q) < nb) S = fi_sum8(e[2 * q], e[2 * q + 1], ph, S);
            cp[g + q] = S;
        }
    }
    for (uint32_t b = kFCP; b < nb; b += 4) {
        uint4 e[8];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            e[2 * q] = e[2 * q + 1] = make_uint4(0u, 0u, 0u, 0u);
            if (b + q < nb) {
                e[2 * q] = *(const uint4 *)(row + kFB * (b + q));
                e[2 * q + 1] = *(const uint4 *)(row + kFB * (b + q) + 4);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (b + q < nb) S = fi_sum8(e[2 * q], e[2 * q + 1], ph, S);
    }
    const float target = u * (S + qa[NS - 1]);
    int zz = -1;
    if (target < S) {
        // the first block whose running sum exceeds the target (one exists:
        // the last running sum is S), then its entries in order
        int bs = -1;
#pragma unroll
        for (int b = kFCP - 1; b >= 0; --b)
            if (cp[b] > target) bs = b;
        float run = 0.0f;
        if (bs >= 0) {
#pragma unroll
            for (int b = 0; b < kFCP - 1; ++b)
                if (b + 1 == bs) run = cp[b];
            const uint32_t g0 = (uint32_t)bs * kFB;
            zz = fi_scan8(*(const uint4 *)(row + g0), *(const uint4 *)(row + g0 + 4), ph, run, target);
        } else {
            // past the checkpoints: blocks four at a time until the block
            // whose running sum exceeds the target, then its entries
            run = cp[kFCP - 1];
            for (uint32_t b = kFCP; b < nb && zz < 0; b += 4) {
                uint4 e[8];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    e[2 * q] = e[2 * q + 1] = make_uint4(0u, 0u, 0u, 0u);
                    if (b + q < nb) {
                        e[2 * q] = *(const uint4 *)(row + kFB * (b + q));
                        e[2 * q + 1] = *(const uint4 *)(row + kFB * (b + q) + 4);
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (zz < 0 && b + q < nb) {
                        const float r2 = fi_sum8(e[2 * q], e[2 * q + 1], ph, run);
                        if (r2 > target) zz = fi_scan8(e[2 * q], e[2 * q + 1], ph, run, target);
                        else run = r2;
                    }
                }
            }
        }
        if (zz < 0)  // not reached: kept as the canonical fallback
            for (uint32_t g = 0; g < nz; ++g)
                if ((row[g] >> 16) && ph[row[g] & 0xFFFFu] > 0.0f) zz = (int)(row[g] & 0xFFFFu);
    } else {
        zz = fi_q_topic(target - S, ph, qa, qw, K, NS, alpha);
    }
    zpool[sl.y + i] = (uint16_t)(zz < 0 ? 0 : zz);
}

// Workgroups of 4 wavefronts.  First the big items, assigned by striding
// (each is one pass of similar cost; a shared queue head would serialize on
// one address): phi_w, the slab running sums and the running sums of the
// slab totals staged in LDS, one lane per token.  Then the small words'
// tokens, one lane each, the word read from the pool and its tables from
// HBM (their phi rows are touched by few tokens each, and staging them
// would leave most lanes idle).
__global__ void __launch_bounds__(256) k_fi_sample(const uint4 *__restrict__ slots, int K, float alpha,
                                                   const float *__restrict__ phi, const float *__restrict__ qs,
                                                   const float *__restrict__ qacc, const uint32_t *__restrict__ wpool,
                                                   const uint32_t *__restrict__ rows,
                                                   const uint32_t *__restrict__ row_nnz,
                                                   const uint32_t *__restrict__ tokw, const uint4 *__restrict__ big,
                                                   const uint32_t *__restrict__ ctr, uint16_t *__restrict__ zpool,
                                                   uint64_t seed) {
    extern __shared__ float shs[];
    const int NS = (K + 63) >> 6, tid = threadIdx.x, bd = blockDim.x;
    const uint32_t n_big = ctr[0], t_big = ctr[1], t_all = ctr[1] + ctr[2];
    float *ph = shs;      // K: phi_w
    float *qa = ph + K;   // NS: running sums of the slab totals
    float *ql = qa + NS;  // K: slab running sums
    for (uint32_t it = blockIdx.x; it < n_big; it += gridDim.x) {
        __syncthreads();  // the previous item's reads are done
        const uint4 item = big[it];
        const size_t w = item.x;
        for (int k = tid; k < K; k += bd) {
            ph[k] = phi[w * K + k];
            ql[k] = qs[w * K + k];
        }
        for (int j = tid; j < NS; j += bd) qa[j] = qacc[w * NS + j];
        __syncthreads();
        for (uint32_t t = item.y + tid; t < item.z; t += bd) {
            const uint32_t ref = tokw[t], j = ref >> 16;
            fi_draw(slots[j], ref & 0xFFFFu, row_nnz[j], rows, ph, qa, ql, K, NS, alpha, seed, zpool);
        }
    }
    for (uint32_t t = t_big + blockIdx.x * (uint32_t)bd + tid; t < t_all; t += gridDim.x * (uint32_t)bd) {
        const uint32_t ref = tokw[t], j = ref >> 16, i = ref & 0xFFFFu;
        const uint4 sl = slots[j];
        const uint32_t nz = row_nnz[j];
        const size_t w = wpool[sl.y + i];
        fi_draw(sl, i, nz, rows, phi + w * K, qacc + w * NS, qs + w * K, K, NS, alpha, seed, zpool);
    }
}

// ---- few tokens: one wavefront draws T tokens of a document
// One lane a token leaves most of the chip idle when there are few tokens,
// and one document's gathers of phi all pass through one CU's L1 (64 lines an
// instruction): 18.7 us a sweep for 217 tokens.  Here a wavefront gathers the
// phi values of T tokens for a piece of the row (lane = entry, every load of
// the piece in flight at once) into LDS, lane t then runs token t's FMA chain
// over it in order, keeping the running sums in place, and bisects them; the
// document's tokens are spread over workgroups of four wavefronts.
static constexpr uint32_t kPiece = 256, kPieceRow = kPiece + 4;  // entries; LDS floats a token (padded)
static constexpr uint32_t kMaxPieces = 64;                       // of a row (K <= 16383)

// LDS floats of one wavefront: T rows of running sums, T lists of piece ends
static constexpr uint32_t wave_draw_floats(int T) { return (uint32_t)T * (kPieceRow + kMaxPieces); }

// What a wavefront's tokens [i0, i0 + T) of a document (those below n) need
// besides the row, loaded before the row is there: lane t's word and uniform,
// and (qv) the running sums of each token's slab totals, lane = slab (past the
// 64th a token reads them itself).
template <int T>
struct WaveTokens {
    uint32_t nt, w;
    float u, qv[T];
};
template <int T>
__device__ __forceinline__ WaveTokens<T> fi_wave_tokens(uint32_t i0, uint32_t n, const uint32_t *__restrict__ words,
                                                        uint32_t rid, uint32_t sweep, const float *__restrict__ qacc,
                                                        int NS, uint64_t seed) {
    const int lane = threadIdx.x & 63;
    const uint32_t i = i0 + (uint32_t)lane;
    WaveTokens<T> W;
    W.nt = i0 < n ? min((uint32_t)T, n - i0) : 0u;
    W.w = (uint32_t)lane < W.nt ? words[i] : 0u;
#pragma unroll
    for (int t = 0; t < T; ++t) W.qv[t] = qacc[(size_t)readlane_u(W.w, t) * NS + min(lane, NS - 1)];
    W.u = ez_u24(ez_philox_x0(seed, ((uint64_t)rid << 32) | i, sweep, EZ_TAG_FOLDIN));
    return W;
}

// Draws them: row = the document's nz entries in LDS, 16-byte aligned and
// zero padded to a multiple of 4; lane t writes its topic to z[t].
template <int T>
__device__ __forceinline__ void fi_draw_wave(const uint32_t *row, uint32_t nz, const WaveTokens<T> &W,
                                             const float *__restrict__ phi, const float *__restrict__ qs,
                                             const float *__restrict__ qacc, int K, int NS, float alpha,
                                             float *pv, uint16_t *__restrict__ z) {
    const int lane = threadIdx.x & 63;
    const uint32_t w = W.w;
    const bool mine = (uint32_t)lane < W.nt;
    float *pe = pv + T * kPieceRow + lane * kMaxPieces;  // this lane's piece ends
    float *run = pv + lane * kPieceRow;                  // this lane's running sums
    const uint32_t np = (nz + kPiece - 1u) / kPiece;
    // phi of token t at piece c's entries, into its LDS row
    auto gather = [&](const uint32_t (&e)[4], uint32_t c, int t, float (&v)[4]) {
        const float *base = phi + (size_t)readlane_u(w, t) * K;
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = c * kPiece + 64u * u < nz ? base[e[u] & 0xFFFFu] : 0.0f;
    };
    auto load_entries = [&](uint32_t c, uint32_t (&e)[4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t x = c * kPiece + (uint32_t)lane + 64u * u;
            e[u] = x < nz ? row[x] : 0u;
        }
    };
    // this lane's chain over piece c from s, the running sums kept in place
    auto chain = [&](uint32_t c, float s) {
        const uint32_t ng = (min(kPiece, nz - c * kPiece) + 3u) >> 2;
        const uint4 *r4 = reinterpret_cast<const uint4 *>(row + c * kPiece);
        float4 *v4 = reinterpret_cast<float4 *>(run);
#pragma unroll 4
        for (uint32_t g = 0; g < ng; ++g) {
            const uint4 e = r4[g];
            float4 v = v4[g];
            v.x = __builtin_fmaf((float)(e.x >> 16), v.x, s);
            v.y = __builtin_fmaf((float)(e.y >> 16), v.y, v.x);
            v.z = __builtin_fmaf((float)(e.z >> 16), v.z, v.y);
            s = v.w = __builtin_fmaf((float)(e.w >> 16), v.w, v.z);
            v4[g] = v;
        }
        return s;
    };
    float S = 0.0f;
    for (uint32_t c = 0; c < np; ++c) {
        uint32_t e[4];
        load_entries(c, e);
        float v[T][4];
#pragma unroll
        for (int t = 0; t < T; ++t) gather(e, c, t, v[t]);
#pragma unroll
        for (int t = 0; t < T; ++t)
#pragma unroll
            for (int u = 0; u < 4; ++u) pv[t * kPieceRow + lane + 64 * u] = v[t][u];
        wave_lds_sync();
        if (mine) {
            S = chain(c, S);
            pe[c] = S;
        }
        wave_lds_sync();
    }
    const float *qa = qacc + (size_t)w * NS;
    float qlast = 0.0f;  // the Q mass: the running sum of the last slab
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const float x = readlane_f(W.qv[t], min(NS - 1, 63));
        if (lane == t) qlast = x;
    }
    if (NS > 64 && mine) qlast = qa[NS - 1];
    const float target = W.u * (S + qlast), t2 = target - S;
    const bool in_q = mine && !(target < S);
    int zz = -1;
    uint32_t pc = 0xFFFFFFFFu;  // the piece that holds the target
    if (mine && !in_q) {
        uint32_t lo = 0, hi = np - 1u;  // the last piece's end is S
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (pe[mid] > target) hi = mid; else lo = mid + 1u;
        }
        pc = lo;
    }
    // Q: the whole wavefront looks for each token's slab, then its topic; what
    // rounding leaves above every running sum goes the general way
    uint64_t todo = __ballot(in_q);
    if (NS <= 64) {
#pragma unroll
        for (int t = 0; t < T; ++t) {
            if (!((todo >> t) & 1ull)) continue;
            const float x = readlane_f(t2, t);
            const uint64_t ms = __ballot(lane < NS && W.qv[t] > x);
            if (!ms) continue;
            const int js = first_lane(ms), k0 = js * 64;
            const float t3 = x - (js > 0 ? readlane_f(W.qv[t], js - 1) : 0.0f);
            const bool in = k0 + lane < K;
            const float q = in ? qs[(size_t)readlane_u(w, t) * K + k0 + lane] : 0.0f;
            const uint64_t mk = __ballot(in && q > t3);
            if (!mk) continue;
            if (lane == t) zz = k0 + first_lane(mk);
            todo &= ~(1ull << t);
        }
    }
    if ((todo >> lane) & 1ull)
        zz = fi_q_topic(t2, phi + (size_t)w * K, qa, qs + (size_t)w * K, K, NS, alpha);
    if (np > 1) {  // the piece's running sums once more (LDS holds the last piece's)
        for (int t = 0; t < T; ++t) {
            const uint32_t c = readlane_u(pc, t);
            if (c == 0xFFFFFFFFu) continue;
            uint32_t e[4];
            load_entries(c, e);
            float v[4];
            gather(e, c, t, v);
#pragma unroll
            for (int u = 0; u < 4; ++u) pv[t * kPieceRow + lane + 64 * u] = v[u];
        }
        wave_lds_sync();
        if (pc != 0xFFFFFFFFu) chain(pc, pc ? pe[pc - 1u] : 0.0f);
    }
    if (pc != 0xFFFFFFFFu) {
        uint32_t lo = 0, hi = min(kPiece, nz - pc * kPiece) - 1u;  // the piece's last running sum exceeds the target
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (run[mid] > target) hi = mid; else lo = mid + 1u;
        }
        zz = (int)(row[pc * kPiece + lo] & 0xFFFFu);
    }
    if (mine) z[lane] = (uint16_t)(zz < 0 ? 0 : zz);
}

// One fold-in sweep of the resident documents when they have few tokens:
// each workgroup takes 4 T tokens of a slot (groups: slot << 16 | part), copies
// its row into LDS and draws T of them with each wavefront.  Measured for one
// document of 217 tokens at K = 1024: a step of 18 us, against 48 us with its
// tokens bucketed by word (nine launches, k_fi_sample of 17 us and the others
// of about 4).
template <int T>
__global__ void __launch_bounds__(256) k_fi_few(const uint4 *__restrict__ slots, int K, float alpha,
                                                const float *__restrict__ phi, const float *__restrict__ qs,
                                                const float *__restrict__ qacc, const uint32_t *__restrict__ wpool,
                                                const uint32_t *__restrict__ rows, const uint32_t *__restrict__ row_nnz,
                                                const uint32_t *__restrict__ groups, uint32_t row_cap,
                                                uint16_t *__restrict__ zpool, uint64_t seed) {
    extern __shared__ __align__(16) uint32_t shd[];
    const int NS = (K + 63) >> 6, tid = threadIdx.x, wv = tid >> 6;
    const uint32_t grp = groups[blockIdx.x], j = grp >> 16;
    const uint4 sl = slots[j];
    const uint32_t i0 = ((grp & 0xFFFFu) * 4u + (uint32_t)wv) * T;
    uint32_t *row = shd;  // row_cap entries, padded to 4
    float *pv = reinterpret_cast<float *>(row + ((row_cap + 3u) & ~3u)) + wv * wave_draw_floats(T);
    const WaveTokens<T> W = fi_wave_tokens<T>(i0, sl.z, wpool + sl.y, sl.x, sl.w, qacc, NS, seed);
    const uint32_t nz = row_nnz[j];
    for (uint32_t x = tid; x < ((nz + 3u) & ~3u); x += 256) row[x] = rows[sl.y + x];  // rows are zero padded to 8
    __syncthreads();
    if (i0 < sl.z) fi_draw_wave<T>(row, nz, W, phi, qs, qacc, K, NS, alpha, pv, zpool + sl.y + i0);
}

// The plain fold-in path: one sweep of one document a launch (n tokens; the
// topics go from zin to zout, so every workgroup may read them all).  Each
// workgroup builds the document's row in LDS (a 16-bit histogram and a
// bitmap of its topics, compacted by one wavefront in ascending topic order)
// and draws 4 T tokens against it.  On sweep 0 with zin null the topics are
// those of the init stream.  One launch of one workgroup for all sweeps took
// 373 us for 217 tokens and 20 sweeps at K = 1024 and 29.4 ms for 4,098; this
// takes 175 us (10 us a launch, a chain of latencies: topics, histogram, phi
// gathers, sums, Q) and 0.66 ms.
template <int T>
__global__ void __launch_bounds__(256) k_fi_doc(const uint32_t *__restrict__ words, uint32_t n, uint32_t rid,
                                                uint32_t sweep, int K, float alpha, const float *__restrict__ phi,
                                                const float *__restrict__ qs, const float *__restrict__ qacc,
                                                uint64_t seed, const uint16_t *__restrict__ zin,
                                                uint16_t *__restrict__ zout) {
    extern __shared__ __align__(16) uint32_t shd[];
    const int NS = (K + 63) >> 6, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int KH4 = (((K + 1) >> 1) + 3) & ~3, NW4 = (((K + 31) >> 5) + 3) & ~3;
    uint32_t *h = shd;                                 // KH4 words: 16-bit counts
    uint32_t *bm = h + KH4;                            // NW4 words: bitmap of the topics
    uint32_t *s_nz = bm + NW4;                         // 4 words: the row's entries
    uint32_t *row = s_nz + 4;                          // min(n, K) entries, padded to 4
    float *pv = reinterpret_cast<float *>(row + ((min(n, (uint32_t)K) + 3u) & ~3u)) + wv * wave_draw_floats(T);
    const uint32_t i0 = (blockIdx.x * 4u + (uint32_t)wv) * T;
    const WaveTokens<T> W = fi_wave_tokens<T>(i0, n, words, rid, sweep, qacc, NS, seed);
    for (int k = tid; k < KH4 + NW4; k += 256) h[k] = 0;
    __syncthreads();
    auto add = [&](uint32_t t) {
        h16_add(h, t);
        atomicOr(&bm[t >> 5], 1u << (t & 31u));
    };
    if (zin)
        for_doc_tokens(zin, n, [&](uint16_t t, uint32_t) { add(t); });
    else
        for (uint32_t i = tid; i < n; i += 256)
            add(ez_philox_x0(seed, ((uint64_t)rid << 32) | i, 0u, EZ_TAG_FOLDIN_INIT) % (uint32_t)K);
    __syncthreads();
    if (wv == 0) {
        uint32_t nz = 0;
        for (int j = 0; j < NW4; j += 64) {
            const int wi = j + lane;
            const uint32_t word = wi < NW4 ? bm[wi] : 0u;
            const uint32_t m = (uint32_t)__popc(word);
            uint32_t incl = m;  // inclusive scan over lanes
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t v = __shfl_up(incl, d);
                if (lane >= d) incl += v;
            }
            uint32_t pos = nz + incl - m;
            for (uint32_t x = word; x; x &= x - 1u) {
                const uint32_t k = ((uint32_t)wi << 5) + (uint32_t)__ffs(x) - 1u;
                row[pos++] = k | (h16_get(h, k) << 16);
            }
            nz += __shfl(incl, 63);
        }
        if ((uint32_t)lane < ((4u - (nz & 3u)) & 3u)) row[nz + lane] = 0u;
        if (lane == 0) *s_nz = nz;
    }
    __syncthreads();
    if (i0 < n) fi_draw_wave<T>(row, *s_nz, W, phi, qs, qacc, K, NS, alpha, pv, zout + i0);
}

// Topics of the init stream (documents too long for every workgroup of
// k_fi_doc to draw them itself).
__global__ void __launch_bounds__(256) k_fi_init(uint32_t n, uint32_t rid, int K, uint64_t seed,
                                                 uint16_t *__restrict__ z) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i < n) z[i] = (uint16_t)(ez_philox_x0(seed, ((uint64_t)rid << 32) | i, 0u, EZ_TAG_FOLDIN_INIT) % (uint32_t)K);
}

// LDS of k_fi_doc for a document of n tokens.
static size_t foldin_doc_lds(int K, uint32_t n, int T) {
    const size_t kh4 = (((size_t)K + 1) / 2 + 3) & ~(size_t)3, nw4 = (((size_t)K + 31) / 32 + 3) & ~(size_t)3;
    return (kh4 + nw4 + 4 + ((std::min<size_t>(n, (size_t)K) + 3) & ~(size_t)3) + 4 * wave_draw_floats(T)) *
           sizeof(uint32_t);
}

// Tokens a wavefront draws in k_fi_doc: one while the workgroups fit the
// chip's CUs, more for longer documents (each workgroup builds the row).
static int foldin_doc_t(uint32_t n) { return n <= 1024 ? 1 : n <= 2048 ? 2 : 4; }

hipError_t launch_foldin_doc(const uint32_t *words, uint32_t n, uint32_t rid, int sweeps, int K, float alpha,
                             const float *phi, const float *qs, const float *qacc, uint64_t seed, uint16_t *z,
                             uint16_t *z2, hipStream_t st) {
    if (n == 0) return hipSuccess;
    uint16_t *buf[2] = {z, z2};  // the last sweep writes z
    const int T = foldin_doc_t(n);
    const unsigned grid = (n + 4u * (unsigned)T - 1u) / (4u * (unsigned)T);
    const size_t lds = foldin_doc_lds(K, n, T);
    const bool inline_init = n <= 1024;
    if (!inline_init)
        hipLaunchKernelGGL(k_fi_init, dim3((n + 255u) / 256u), dim3(256), 0, st, n, rid, K, seed, buf[sweeps & 1]);
    for (int sw = 0; sw < sweeps; ++sw) {
        const uint16_t *zin = sw == 0 && inline_init ? nullptr : buf[(sweeps - sw) & 1];
        uint16_t *zout = buf[(sweeps - 1 - sw) & 1];
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), lds, st, words, n, rid, (uint32_t)sw, K, alpha, phi, qs,
                               qacc, seed, zin, zout);
        };
        if (T == 1) go(k_fi_doc<1>);
        else if (T == 2) go(k_fi_doc<2>);
        else go(k_fi_doc<4>);
    }
    return hipGetLastError();
}

// Documents that just drew their last sweep (fin[j] = (output index, topic
// offset), output index ~0 for the others): their topics packed into zout at
// the offset, for one copy to the host (which counts them).
__global__ void __launch_bounds__(256) k_fi_final(const uint4 *__restrict__ slots, const uint2 *__restrict__ fin,
                                                  int nslots, const uint16_t *__restrict__ zpool,
                                                  uint16_t *__restrict__ zout) {
    for (int j = blockIdx.x; j < nslots; j += gridDim.x) {
        const uint2 f = fin[j];
        if (f.x == 0xFFFFFFFFu) continue;  // uniform over the workgroup
        const uint4 sl = slots[j];
        for_doc_tokens(zpool + sl.y, sl.z, [&](uint16_t t, uint32_t i) { zout[f.y + i] = t; });
    }
}

hipError_t launch_foldin_tables(const DevState &s, float *phi, float *qs, float *qacc, hipStream_t st) {
    hipLaunchKernelGGL(k_foldin_tables, dim3(grid_for(s.V, 1, 1 << 16)), dim3(256), (size_t)s.K * sizeof(float), st,
                       s.V, s.VD, s.K, s.alpha, s.beta, s.wt_head, s.tail_off, s.wt_tail, s.tail_nnz, s.inv, phi, qs,
                       qacc);
    return hipGetLastError();
}

static size_t foldin_sample_lds(int K) { return (2 * (size_t)K + (size_t)((K + 63) >> 6)) * sizeof(float); }

size_t foldin_lds_bytes(int K) {
    return std::max(foldin_sample_lds(K) + 16, (size_t)((K + 1) >> 1) * sizeof(uint32_t));
}

uint32_t foldin_max_items(int V, uint32_t max_tokens) { return (uint32_t)V + max_tokens / kFoldSeg + 1u; }

hipError_t launch_foldin_admit(const uint4 *adm, int nadm, const uint32_t *src, uint32_t *wpool, hipStream_t st) {
    if (nadm <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_fi_admit, dim3(std::min(nadm, 1024)), dim3(256), 0, st, adm, nadm, src, wpool);
    return hipGetLastError();
}

// Steps of few tokens are drawn by k_fi_few, straight from the tables: no
// buckets by word, whose six more launches cost more than they save until big
// words gather enough tokens to share a staged phi row.  What a token costs
// there follows its document's row, about min(n / 3, K) entries of which the
// first few hundred count; what buckets save follows V, whose few frequent
// words hold more of the tokens where it is small.  Measured, ms to drain a
// batch of documents (20 sweeps) bucketed / few, on both sides of the line:
//   K = 1024, mean 300, V = 1,000: 120K tokens 2.70 / 2.29, 160K 2.83 / 2.76,
//     200K 3.15 / 3.61; V = 102,660: 150K 3.12 / 2.65, 260K 4.43 / 4.36
//   K = 1024, mean 600: 80K 2.50 / 2.26, 118K 2.65 / 2.94 (V = 2,000),
//     3.13 / 2.91 (V = 102,660)
//   K = 1024, mean 2,000: 59K 3.76 / 3.12, 78K 3.65 / 3.73 (V = 2,000), 77K
//     4.01 / 3.42, 115K 4.15 / 4.67 (V = 102,660)
//   K = 300, mean 2,000: 78K 1.80 / 1.61, 116K 2.15 / 2.31 (V = 2,000)
//   K = 64 to 16,383, mean 60: few up to 150K-200K and more
//   K = 16,383, V = 2,000: mean 300 80K 3.61 / 2.99, 120K 4.16 / 4.16; mean
//     2,000 59K 7.66 / 6.68, 78K 7.43 / 7.75
// Rows of thousands of topics cost more again (K = 16,383, 34K tokens in short
// documents and one, two, three of 16,000: 9.6 / 6.1, 10.0 / 9.6, 10.1 / 13.2).
static constexpr uint32_t kFewTokens = 196608, kFewRow = 430;
static constexpr uint64_t kFewCost = 45000000, kFewCostLargeV = 56000000;

uint64_t foldin_few_cost(uint32_t n, int K) {
    const uint32_t row = std::min(n, (uint32_t)K);
    return (uint64_t)n * (160u + std::min(std::min(n / 3u, kFewRow), (uint32_t)K) +
                          (row > kFewShortRow ? (row - kFewShortRow) / 16u : 0u));
}

uint32_t foldin_few_group(uint32_t ntok, uint64_t cost, int V) {
    if (ntok > kFewTokens || cost > (V >= 16384 ? kFewCostLargeV : kFewCost)) return 0u;
    return ntok <= 4096 ? 4u : ntok <= 8192 ? 8u : 16u;
}

static size_t foldin_few_lds(uint32_t row_cap, uint32_t group) {
    return (((size_t)row_cap + 3) / 4 * 4 + 4 * wave_draw_floats((int)group / 4)) * sizeof(uint32_t);
}

// A step's longest row sizes the LDS of every workgroup of a launch.  Where
// that leaves a CU one or two of them, and there are many, the documents of
// long rows get a launch of their own.  K = 16,383, ms to drain 83K tokens in
// short documents (alone 3.0) and one long document, in one launch / two /
// bucketed: 16,000 tokens 10.3 / 7.2 / 9.8, 9,000 5.3 / 4.8 / 7.3.  Few
// workgroups are better off in one: 34K short tokens and one document of 9,000
// 3.4 / 3.7, 4K and one of 16,000 5.0 / 5.2.
bool foldin_few_split(uint32_t ngroups, uint32_t group, uint32_t max_n, int K, int n_cu, int lds_cu) {
    const uint32_t cap = std::min(max_n, (uint32_t)K);
    const size_t fit = std::max<size_t>(1, (size_t)lds_cu / foldin_few_lds(cap, group));
    return cap > kFewShortRow && fit < 3 && ngroups > 8u * (uint32_t)(n_cu * fit);
}

hipError_t launch_foldin_step(const FoldinBatch &fb, const uint4 *slots, const uint2 *fin, const uint32_t *goff,
                              const FoldinFew &few, int nslots, uint32_t ntok, bool any_fin, int V, int K,
                              float alpha, const float *phi, const float *qs, const float *qacc,
                              const uint32_t *wpool, uint16_t *zpool, uint64_t seed, hipStream_t st) {
    if (nslots <= 0) return hipSuccess;
    const unsigned gs = (unsigned)std::min(nslots, 1 << 16);
    const size_t lds_rows = (size_t)((K + 1) >> 1) * sizeof(uint32_t);
    hipLaunchKernelGGL(k_fi_rows, dim3(gs), dim3(256), lds_rows, st, slots, nslots, K, seed, zpool, fb.rows,
                       fb.row_nnz, few.group, goff, fb.tokw);
    if (few.group) {
        const uint32_t *groups = fb.tokw;
        for (int h = 0; h < 2; ++h) {
            if (!few.groups[h]) continue;
            auto go = [&](auto kernel) {
                hipLaunchKernelGGL(kernel, dim3(few.groups[h]), dim3(256), foldin_few_lds(few.row_cap[h], few.group), st,
                                   slots, K, alpha, phi, qs, qacc, wpool, fb.rows, fb.row_nnz, groups, few.row_cap[h],
                                   zpool, seed);
            };
            if (few.group == 4) go(k_fi_few<1>);
            else if (few.group == 8) go(k_fi_few<2>);
            else go(k_fi_few<4>);
            groups += few.groups[h];
        }
        if (any_fin) hipLaunchKernelGGL(k_fi_final, dim3(gs), dim3(256), 0, st, slots, fin, nslots, zpool, fb.zout);
        return hipGetLastError();
    }
    // count and scatter: one workgroup per CU (fb.grid is 8 per CU), each
    // flushing its LDS table of the most frequent words once for many slots
    const unsigned gc = (unsigned)std::max(1, std::min(nslots, std::max(1, fb.grid / 8)));
    const unsigned nb = (unsigned)((V + 1023) / 1024);
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for((size_t)V, 256, 4096)), dim3(256), 0, st, fb.wcount, (size_t)V, 0u);
    hipLaunchKernelGGL(k_fi_count, dim3(gc), dim3(256), 0, st, slots, nslots, wpool, fb.wcount);
    hipLaunchKernelGGL(k_fi_bsum, dim3(nb), dim3(1024), 0, st, V, fb.wcount, fb.bsum);
    hipLaunchKernelGGL(k_fi_btop, dim3(1), dim3(1024), 0, st, (int)nb, fb.bsum, fb.ctr);
    hipLaunchKernelGGL(k_fi_bfin, dim3(nb), dim3(1024), 0, st, V, fb.wcount, fb.bsum, fb.ctr, fb.wcursor,
                       fb.items);
    hipLaunchKernelGGL(k_fi_scatter, dim3(gc), dim3(256), 0, st, slots, nslots, wpool, fb.wcursor, fb.tokw);
    // no more workgroups than a lane per token could use
    const unsigned gsmp = (unsigned)std::max<int64_t>(1, std::min<int64_t>(fb.grid, ((int64_t)ntok + 255) / 256));
    hipLaunchKernelGGL(k_fi_sample, dim3(gsmp), dim3(256), foldin_sample_lds(K), st, slots, K, alpha, phi, qs, qacc,
                       wpool, fb.rows, fb.row_nnz, fb.tokw, fb.items, fb.ctr, zpool, seed);
    if (any_fin) hipLaunchKernelGGL(k_fi_final, dim3(gs), dim3(256), 0, st, slots, fin, nslots, zpool, fb.zout);
    return hipGetLastError();
}

// ------------------------------------------------------------ self-tests
__global__ void k_selftest_philox(const uint4 *__restrict__ ctr, const uint2 *__restrict__ key,
                                  uint4 *__restrict__ out, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint4 c = ctr[i];
    const ez_u4 o = ez_philox4x32_10(ez_u4{c.x, c.y, c.z, c.w}, key[i].x, key[i].y);
    out[i] = make_uint4(o.x, o.y, o.z, o.w);
}

// Plain streaming copy (16 B per lane per step): the known-size reference
// for scaling HBM counters.
__global__ void k_copy_u4(const uint4 *__restrict__ src, uint4 *__restrict__ dst, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

// Scattered 64-byte reads (the sampler's row-block pattern: each lane loads
// four 16-byte pieces of one 64-byte block at an address no neighbouring lane
// shares), n_reads of them over a buffer of nblk = 2^m 64-byte blocks: read i
// takes block (i * an odd constant) mod nblk, a bijection, so n_reads <= nblk
// reads touch n_reads distinct blocks, each once (64 * n_reads bytes, none of
// them cached by an earlier read).  The known-size workload that scales the
// traffic counters for that request mix.  Nothing is written unless the data
// holds an impossible value (the loads cannot be removed).
__global__ void k_gather64(const uint4 *__restrict__ src, uint64_t blk_mask, uint64_t n_reads,
                           uint32_t *__restrict__ sink) {
    uint32_t acc = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n_reads;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t blk = (i * 0x9E3779B97F4A7C15ull) & blk_mask;
        const uint4 *p = src + blk * 4u;
        const uint4 a = p[0], b = p[1], c = p[2], d = p[3];
        acc ^= a.x ^ a.w ^ b.y ^ c.z ^ d.x ^ d.w;
    }
    if (acc == 0x9E3779B9u) sink[threadIdx.x & 63u] = acc;
}

hipError_t launch_gather64(const void *src, size_t bytes, uint64_t n_reads, uint32_t *sink, hipStream_t st) {
    uint64_t nblk = 1;
    while (nblk * 2 * 64 <= bytes) nblk *= 2;
    if (bytes < 64 || n_reads > nblk) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_gather64, dim3(grid_for((size_t)n_reads, 256, 8192)), dim3(256), 0, st,
                       reinterpret_cast<const uint4 *>(src), nblk - 1, n_reads, sink);
    return hipGetLastError();
}

hipError_t launch_copy(const void *src, void *dst, size_t bytes, hipStream_t st) {
    const size_t n = bytes / 16;
    hipLaunchKernelGGL(k_copy_u4, dim3(grid_for(n, 256, 8192)), dim3(256), 0, st,
                       reinterpret_cast<const uint4 *>(src), reinterpret_cast<uint4 *>(dst), n);
    return hipGetLastError();
}

// ------------------------------------ allocation-free log-likelihood memory
// The device memory of ezlda_loglik_noalloc: kLLScratchItems per-item
// log-likelihood partials, then the result.  A file-scope array, so the call
// needs no allocation; every GPU holds its own copy (8 MiB) until the process
// ends, and every call on a GPU shares it.  Host code never passes the
// array's name to a kernel (on the host it is only a stand-in for the
// symbol): scratch_address() returns the device address, once per device.
static __device__ __align__(256) double scratch[kLLScratchItems + 1];

hipError_t scratch_address(double **p) {
    *p = nullptr;
    return hipGetSymbolAddress(reinterpret_cast<void **>(p), HIP_SYMBOL(scratch));
}

hipError_t launch_selftest_philox(const uint32_t *ctr, const uint32_t *key, uint32_t *out, int n, hipStream_t st) {
    hipLaunchKernelGGL(k_selftest_philox, dim3((n + 255) / 256), dim3(256), 0, st,
                       reinterpret_cast<const uint4 *>(ctr), reinterpret_cast<const uint2 *>(key),
                       reinterpret_cast<uint4 *>(out), n);
    return hipGetLastError();
}

// ------------------------------------------------------------ launchers

hipError_t launch_set_u32(uint32_t *p, uint32_t v, hipStream_t st) {
    hipLaunchKernelGGL(k_set_u32, dim3(1), dim3(1), 0, st, p, v);
    return hipGetLastError();
}

// One launch clears what a sweep starts from: the dense head rows, n_k and,
// for a whole sweep, the sampler's queue heads, and moves the sweep counter on
// (counters[1] = the sweep that begins, counters[0] = the next one).  As four
// launches (three fills, an increment after the sampler) these took 12-18 us
// of every sweep, nearly all of it the launches: 43.2 -> 38.7 us a sweep on 18,000
// tokens.
__global__ void __launch_bounds__(256) k_begin(uint32_t *__restrict__ wt, size_t n, uint32_t *__restrict__ nk, int K,
                                               uint32_t *__restrict__ counters) {
    const size_t gid = (size_t)blockIdx.x * 256u + threadIdx.x, stride = (size_t)gridDim.x * 256u;
    uint4 *w4 = reinterpret_cast<uint4 *>(wt);
    for (size_t i = gid; i < n / 4; i += stride) w4[i] = make_uint4(0u, 0u, 0u, 0u);
    if (gid < (n & 3u)) wt[(n & ~(size_t)3u) + gid] = 0u;
    for (size_t i = gid; i < (size_t)K; i += stride) nk[i] = 0u;
    if (counters) {
        if (gid < 2 * kQueues) counters[kQueueStride * (gid + 1)] = 0u;
        if (gid == 0) {
            const uint32_t sweep = counters[0];
            counters[1] = sweep;
            counters[0] = sweep + 1u;
        }
    }
}

// (fresh: head rows of one segment are about to be written whole)
static hipError_t begin(const DevState &s, bool fresh, uint32_t *counters, hipStream_t st) {
    const size_t nh = (size_t)(fresh ? s.n_cut_rows : s.VD) * s.K;
    hipLaunchKernelGGL(k_begin, dim3(grid_for(std::max(nh / 4, (size_t)s.K), 256, 4096)), dim3(256), 0, st,
                       reinterpret_cast<uint32_t *>(s.wt_head), nh, reinterpret_cast<uint32_t *>(s.nk), s.K, counters);
    return hipGetLastError();
}

hipError_t launch_zero_counts(const DevState &s, hipStream_t st) { return begin(s, false, nullptr, st); }

static hipError_t count_topics(const DevState &s, bool fresh, hipStream_t st);

hipError_t launch_begin_sweep(const DevState &s, hipStream_t st) {
    hipError_t e = begin(s, true, s.counters, st);
    if (e != hipSuccess) return e;
    return count_topics(s, true, st);
}

hipError_t launch_build_wt(const DevState &s, hipStream_t st) {
    hipError_t e = begin(s, true, nullptr, st);
    if (e != hipSuccess) return e;
    return count_topics(s, true, st);
}

hipError_t launch_accumulate_wt(const DevState &s, hipStream_t st) { return count_topics(s, false, st); }

// n_k: about a workgroup a CU, as each adds up to K counts to the same K
// addresses in memory (2,048 of them before: 9M tokens at K = 4096 55 -> 10
// us, 4.5M at K = 10000 53 -> 9, and as a role of k_wt_all, which then took
// 49.5M at K = 1024 111 -> 81 us, 8.9M at K = 2048 90 -> 49).
static void topic_hist(const DevState &s, hipStream_t st) {
    const size_t least = std::max<size_t>(4096, 4 * (size_t)s.K);
    hipLaunchKernelGGL(k_topic_hist, dim3(grid_for(s.N, (int)least, s.n_cu)), dim3(1024), (size_t)s.K * sizeof(uint32_t),
                       st, s.z, s.N, s.K, s.nk);
}

static hipError_t count_topics(const DevState &s, bool fresh, hipStream_t st) {
    const size_t ldsK = (size_t)s.K * sizeof(uint32_t);
    const int ntail = s.V - s.VD;
    if (s.N && s.n_wt_segs && ntail > 0 && (size_t)s.lds_cu / dt_wave_bytes(s.K) >= 16) {
        // one launch of 256-thread blocks (the tail rows' four wavefronts a
        // block, as their own launch takes when 16 wavefronts' tables fit a CU)
        const int nb_hist = (int)grid_for(s.N, 256 * 16, std::max(s.n_cu, (int)(s.N >> 18)));
        const int nb_tail = (int)grid_for((size_t)ntail, 4, 1 << 16);
        const size_t lds = std::max(ldsK, 4 * dt_wave_bytes(s.K));
        hipLaunchKernelGGL(k_wt_all, dim3(nb_hist + s.n_wt_segs + nb_tail), dim3(256), lds, st, nb_hist, s.n_wt_segs,
                           s.z, s.N, s.K, s.nk, s.wt_segs, s.wt_head, fresh, s.word_off, s.VD, s.V, s.tail_off, s.wt_tail,
                           s.tail_nnz);
        return hipGetLastError();
    }
    if (s.N) topic_hist(s, st);
    if (s.n_wt_segs)
        hipLaunchKernelGGL(k_wt_head, dim3(s.n_wt_segs), dim3(256), ldsK, st, s.z, s.wt_segs, s.K, s.wt_head, fresh);
    // (at small K there is no head word or no tail word; the rows are then
    // built by histograms at every length)
    int w1 = (size_t)s.lds_cu / dt_wave_bytes(s.K) < 16 ? std::max(s.VD, std::min(s.V, s.w_short)) : s.V;
    // Where longer words are counted in any case, few short ones are too: a
    // second launch costs 10 us.  The counts take a time like K a word on a number
    // of wavefronts like 1 / K, hence the square (sorted / counted: 2,938 words at
    // K = 4900 59.7 / 45.4, 19,943 56.4 / 53.8, 5,939 at K = 8000 65.8 / 59.1, 3,649
    // at K = 12000 97.4 / 91.9, 1,936 at K = 16383 94.7 / 84.8; beyond the line 9,942
    // at K = 8000 72.3 / 72.8, 9,942 at K = 12000 88.2 / 88.5, 5,939 at K = 16383
    // 101.9 / 105.7, some 3,800 at K = 15099 60.0 / 68.7).
    if (w1 > s.VD && (uint64_t)(s.V - w1) * (uint64_t)s.K * (uint64_t)s.K <= (uint64_t)s.n_cu << 31) w1 = s.V;
    if (w1 > s.VD) {
        const WaveGrid g = wave_grid(s, (size_t)(w1 - s.VD), dt_wave_bytes(s.K), 1 << 16);
        hipLaunchKernelGGL(k_wt_tail, dim3(g.grid), dim3(64 * g.nwv), g.nwv * dt_wave_bytes(s.K), st,
                           s.z, s.word_off, s.VD, w1, s.K, s.tail_off, s.wt_tail, s.tail_nnz);
    }
    if (s.V > w1)
        hipLaunchKernelGGL(k_wt_sort, dim3(grid_for((size_t)(s.V - w1), 4, 1 << 16)), dim3(256), 0, st, s.z, s.word_off,
                           w1, s.VD, s.V, s.tail_off, s.wt_tail, s.tail_nnz);
    return hipGetLastError();
}

hipError_t launch_head_rows(const DevState &s, hipStream_t st) {
    const size_t nh = (size_t)s.n_cut_rows * s.K;
    if (nh) hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(nh, 256, 4096)), dim3(256), 0, st,
                               reinterpret_cast<uint32_t *>(s.wt_head), nh, 0u);
    if (s.n_wt_segs)
        hipLaunchKernelGGL(k_wt_head, dim3(s.n_wt_segs), dim3(256), (size_t)s.K * sizeof(uint32_t), st, s.z, s.wt_segs,
                           s.K, s.wt_head, true);
    return hipGetLastError();
}

hipError_t launch_topic_hist(const DevState &s, hipStream_t st) {
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(s.K, 256, 64)), dim3(256), 0, st, reinterpret_cast<uint32_t *>(s.nk),
                       (size_t)s.K, 0u);
    if (s.N) topic_hist(s, st);
    return hipGetLastError();
}

hipError_t launch_topk(const DevState &s, hipStream_t st) {
    if (s.V > s.VD)
        hipLaunchKernelGGL(k_inv_order, dim3(grid_for(s.K, 64, 1 << 16)), dim3(1024),
                           ((size_t)((s.K + 3) & ~3) + 64) * sizeof(float), st, s.nk, s.K, s.vbeta,
                           (double)s.V * (double)s.beta, s.beta, s.inv, s.inv64, s.zero_order);
    else
        hipLaunchKernelGGL(k_inv, dim3(grid_for(s.K, 256, 1 << 16)), dim3(256), 0, st, s.nk, s.K, s.vbeta,
                           (double)s.V * (double)s.beta, s.inv, s.inv64);
    if (s.V > 0) {
        const size_t lds = s.V > s.VD ? 4 * (size_t)((s.K + 31) >> 5) * sizeof(uint32_t) : 0;
        hipLaunchKernelGGL(k_word_top, dim3(grid_for((size_t)s.V, 4, 1 << 16)), dim3(256), lds, st, s.V, s.VD, s.K,
                           s.beta, s.wt_head, s.tail_off, s.wt_tail, s.tail_nnz, s.inv, s.zero_order, s.wtop);
    }
    return hipGetLastError();
}

template <bool COMPACT, bool N_DK2>
static void build_dt_kernels(const DevState &s, hipStream_t st) {
    // where a K-sized histogram per wavefront leaves fewer than 16 on a CU,
    // the short documents (the last ones: docs come longest first) are sorted
    // instead
    const bool sort_short = (size_t)s.lds_cu / dt_wave_bytes(s.K) < 16;
    const int q1 = sort_short ? s.D_long : s.D;
    if (q1 > 0) {
        const size_t wb = s.K <= kScanMaxK ? scan_wave_bytes(s.K) : dt_wave_bytes(s.K);
        const WaveGrid g = wave_grid(s, (size_t)q1, wb, 1 << 18);
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(g.grid), dim3(64 * g.nwv), g.nwv * wb, st, 0, q1, s.K, s.VD, s.topic_bits,
                               s.soff, s.slot_wrd, s.slot_tok, s.z, s.z_doc, s.wtop, s.aux_doc, s.doc_info, s.dt);
        };
        s.K <= kScanMaxK ? go(k_dt_build<COMPACT, N_DK2, true>) : go(k_dt_build<COMPACT, N_DK2, false>);
    }
    if (q1 < s.D) {
        const size_t lds = 4 * kDtShort * sizeof(uint32_t);  // four wavefronts, 2 KB each
        const unsigned grid = (unsigned)grid_for((size_t)(s.D - q1), 4, 1 << 18);
        hipLaunchKernelGGL((k_dt_sort<COMPACT, N_DK2>), dim3(grid), dim3(256), lds, st, q1, s.D, s.VD, s.topic_bits,
                           s.soff, s.slot_wrd, s.slot_tok, s.z, s.z_doc, s.wtop, s.aux_doc, s.doc_info, s.dt);
    }
}

hipError_t launch_build_dt(const DevState &s, hipStream_t st, bool n_dk2) {
    if (s.D == 0) return hipSuccess;
    if (s.compact) {
        if (n_dk2) build_dt_kernels<true, true>(s, st);
        else build_dt_kernels<true, false>(s, st);
    } else {
        if (n_dk2) build_dt_kernels<false, true>(s, st);
        else build_dt_kernels<false, false>(s, st);
    }
    return hipGetLastError();
}

// LDS floats of one word of a group item: phi and the Q running sums (whole
// slabs), slab totals and their running sums, f1, f2, k1, the item number;
// 4 more than a multiple of 8, so that lanes reading different words' slabs
// start at different banks.
int group_stride(int K) {
    const int NS = (K + 63) >> 6;
    int st = 2 * NS * 64 + 2 * NS + 4;
    while ((st & 7) != 4) ++st;
    return st;
}

size_t sample_lds_bytes(int K, int bd) {
    const int NS = (K + 63) >> 6;
    (void)bd;
    const size_t tab = K <= EZ_Q_TABLE_MAX_K ? 2 : 1;  // phi (and the slab running sums)
    return (tab * (size_t)NS * 64 + 2 * (size_t)NS + 4) * sizeof(float);  // + qt, qacc, f123[3], item
}

size_t sampler_static_lds() {
    // a property of the code: looked up until it is known, once a process
    static std::atomic<size_t> known{(size_t)-1};
    if (known != (size_t)-1) return known;
    const void *fs[] = {reinterpret_cast<const void *>(&k_sample<true, true, true, true>),
                         reinterpret_cast<const void *>(&k_sample<true, true, true, false>),
                         reinterpret_cast<const void *>(&k_sample<true, true, false, false>),
                         reinterpret_cast<const void *>(&k_sample<true, false, false, false>),
                         reinterpret_cast<const void *>(&k_sample<false, true, true, true>),
                         reinterpret_cast<const void *>(&k_sample<false, true, true, false>),
                         reinterpret_cast<const void *>(&k_sample<false, true, false, false>),
                         reinterpret_cast<const void *>(&k_sample<false, false, false, false>),
                         reinterpret_cast<const void *>(&k_sample_own<true>),
                         reinterpret_cast<const void *>(&k_sample_own<false>)};
    size_t m = 0;
    for (const void *f : fs) {
        hipFuncAttributes a;
        if (hipFuncGetAttributes(&a, f) != hipSuccess) return (size_t)-1;
        m = std::max(m, a.sharedSizeBytes);
    }
    known = m;
    return m;
}

size_t max_lds_bytes(int K, int bd) {
    size_t m = sample_lds_bytes(K, bd);
    m = std::max(m, 4 * dt_wave_bytes(K));                           // WT tail, top-3, DT build
    m = std::max(m, (size_t)K * sizeof(double));                     // log-likelihood
    m = std::max(m, (size_t)K * sizeof(float) + 1024 * sizeof(float));  // fold-in tables
    m = std::max(m, foldin_lds_bytes(K));
    m = std::max(m, foldin_doc_lds(K, 65535, 4));
    return m;
}

hipError_t launch_sample(const DevState &s, bool shortcut, hipStream_t st, uint32_t mode, bool begun) {
    if (s.n_smp_segs == 0) return hipSuccess;
    const int bd = s.block_dim;
    size_t lds = sample_lds_bytes(s.K, bd);
    SampleArgs A;
    A.word_stride = 0;
    A.segs = s.smp_segs;
    A.runs = s.runs;
    // the items from first_own on by k_sample_own, where enough wavefronts' tables fit
    const int NS = (s.K + 63) >> 6;
    const long room = (long)s.lds_cu / 4 - own_shared(NS);
    const int own_wv = room > 0 ? (int)std::min<long>(16, room / (2 * own_stride(NS))) : 0;
    // and where there are enough of these items: the launch takes 80 to 110 us
    // however few, as many items a CU as 32 take in k_sample where four of its
    // tables fit a CU, 14 where three do, 10 where two do (without it / with it: 0
    // to 2,500 items at K > 8192 0.36 to 1.0; 6,500 at K = 8348 0.76, 11,000 at K =
    // 8661 0.9 to 1.1, 15,000 at K = 8867 1.4; 2,784 at K = 11709 0.83, 3,151 at K =
    // 11287 0.8 to 0.9, 3,600 to 7,700 at K > 9,950 1.0 to 2.7; 2,568 at K = 13463
    // 1.0, 3,458 at K = 13358 1.4, 2,627 at K = 15552 1.1 to 1.2)
    const int fit = (int)((size_t)s.lds_cu / lds);
    const int line = fit >= 4 ? 32 : fit == 3 ? 14 : 10;
    const bool own = s.n_smp_segs - s.first_own >= s.n_cu * line && own_wv >= 4;
    const int32_t n_first = own ? s.first_own : s.n_smp_segs;
    A.first_item = (uint32_t)n_first;
    A.n_items = (uint32_t)n_first;
    A.VD = s.VD;
    A.K = s.K;
    A.alpha = s.alpha;
    A.beta = s.beta;
    A.wt_head = s.wt_head;
    A.tail_off = s.tail_off;
    A.wt_tail = s.wt_tail;
    A.tail_nnz = s.tail_nnz;
    A.inv = s.inv;
    A.wtop = s.wtop;
    A.aux_doc = s.aux_doc;
    A.dt = s.dt;
    A.z = s.z;
    A.z_doc = s.z_doc;
    A.counters = s.counters + (begun ? 1 : 0);
    A.queue = s.counters + kQueueStride;
    // Queues only where a workgroup has many items to take: the claims, and
    // the failed ones of all workgroups at every queue's end, cost more than
    // the balance gains with a few.  Measured, sampler us a sweep in turn /
    // from queues: 250 items 19 / 64 (as 2,212), 10,215 items (2.5 a
    // workgroup) at K = 64 126 / 152, 10,113 at K = 300 159 / 169; 27,680
    // items (13 a workgroup) at K = 4096 767 / 672, 98,189 (24) at K = 2048
    // 2,277 / 1,564, 126,191 (31) at K = 1024 3,519 / 2,884.
    unsigned grid = (unsigned)n_first;
    // At K > 8192 fewer workgroups fit the CUs than the grid has and an item's
    // tables take long: a resident corpus takes from queues as soon as there are
    // more items than fit (in turn / from queues: 5,392 items at K = 12368 700 /
    // 586, 4,948 at K = 10383 763 / 730, 5,292 at K = 8924 371 / 335).  A chunk,
    // whose first_own is past its items, does not: its many words of few tokens go
    // faster in turn (a sweep of 14,552 items in 4 chunks at K = 15063 2,810 /
    // 3,177, of 17,582 in 5 at K = 15854 3,076 / 3,442, of 13,970 in 3 at K = 9061
    // 2,153 / 1,910 first and 1,336 / 1,369 later).
    const bool resident = s.first_own <= s.n_smp_segs;
    const int32_t many = s.compact || !resident ? 4 * s.grid_dim : std::min(s.grid_dim, s.n_cu * std::max(1, fit) + 1);
    A.n_queues = s.grid_dim > 0 && n_first >= many ? (uint32_t)s.n_queues : 0u;
    if (s.grid_dim > 0 && A.n_queues == 0) grid = (unsigned)std::min(n_first, s.grid_dim);
    A.stats = s.stats;
    A.seed = s.seed;
    A.tb = s.topic_bits;
    A.mode = mode;
    // queue heads start at zero (a fill kernel, so a captured sweep replays it)
    if (!begun && (A.n_queues || own))
        hipLaunchKernelGGL(k_fill_u32, dim3(1), dim3(256), 0, st, A.queue, (size_t)kQueueStride * 2 * kQueues, 0u);
    if (A.n_queues) {
        grid = (unsigned)s.grid_dim;
    }
    const bool qtab = s.K <= EZ_Q_TABLE_MAX_K;  // implies compact rows
    const bool multi = s.group_words > 1;       // implies qtab
    if (multi) {
        A.word_stride = (uint32_t)group_stride(s.K);
        lds = (size_t)s.group_words * A.word_stride * sizeof(float);
    }
    auto go = [&](auto kernel) {
        if (n_first) hipLaunchKernelGGL(kernel, dim3(grid), dim3(bd), lds, st, A);
    };
    if (shortcut && multi)
        go(k_sample<true, true, true, true>);
    else if (shortcut && qtab)
        go(k_sample<true, true, true, false>);
    else if (shortcut && s.compact)
        go(k_sample<true, true, false, false>);
    else if (shortcut)
        go(k_sample<true, false, false, false>);
    else if (multi)
        go(k_sample<false, true, true, true>);
    else if (qtab)
        go(k_sample<false, true, true, false>);
    else if (s.compact)
        go(k_sample<false, true, false, false>);
    else
        go(k_sample<false, false, false, false>);
    if (own && (mode & kSampleTail)) {
        A.n_items = (uint32_t)s.n_smp_segs;
        lds = (size_t)(own_shared(NS) + 2 * own_wv * own_stride(NS)) * sizeof(float);
        // a workgroup drains one queue: each of the kQueues needs one
        const unsigned g = (unsigned)std::max(s.n_cu, kQueues);
        auto go_own = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(g), dim3(64 * own_wv), lds, st, A); };
        shortcut ? go_own(k_sample_own<true>) : go_own(k_sample_own<false>);
    }
    return hipGetLastError();
}

hipError_t launch_advance_sweep(const DevState &s, hipStream_t st) {
    hipLaunchKernelGGL(k_inc_u32, dim3(1), dim3(1), 0, st, s.counters);
    return hipGetLastError();
}

hipError_t launch_loglik(const DevState &s, hipStream_t st) {
    if (s.n_smp_segs > 0) {
        const size_t lds = (size_t)s.K * (size_t)std::max(1, s.group_words) * sizeof(double);
        const int fit = std::max(1, (int)((size_t)s.lds_cu / (lds + 16 * sizeof(double))));
        int bd = 64;
        while (bd < 1024 && fit * (bd / 64) < 12) bd *= 2;
        // K > 4096: as many workgroups as the CUs hold (at most 16 wavefronts
        // each; a multiple of 8, so that an item stays on the XCD it was dealt
        // to), so that most tail words find the base phi in LDS (K = 10000,
        // 4.5M tokens: 1.30 -> 1.08 ms).  Below, a workgroup an item, which
        // the dispatcher balances (K = 2048, heavy-tailed documents: 2.92
        // against 3.65 ms; K = 1024: 0.81 against 0.88).
        const int per_cu = std::max(1, std::min(fit, 16 / (bd / 64)));
        const int grid = s.K > 4096 ? std::min(s.n_smp_segs, std::max(8, s.n_cu * per_cu / 8 * 8)) : s.n_smp_segs;
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(bd), lds, st, (uint32_t)s.n_smp_segs, s.smp_segs, s.runs, s.VD, s.K,
                               (double)s.alpha, (double)s.beta, s.wt_head, s.tail_off, s.wt_tail, s.tail_nnz,
                               s.inv64, s.aux_doc, s.dt, s.topic_bits, s.ll_part);
        };
        if (s.group_words > 1) go(k_ll<true, true>);
        else if (s.compact) go(k_ll<true, false>);
        else go(k_ll<false, false>);
    }
    hipLaunchKernelGGL(k_ll_final, dim3(1), dim3(1024), 0, st, s.ll_part, std::max(s.n_smp_segs, 0), s.ll_out);
    return hipGetLastError();
}

}  // namespace ez
