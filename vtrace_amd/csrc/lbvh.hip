// lbvh.hip — GPU-built LBVH over instance boxes (replaces lib/raytrace.c's one-AABB BLAS,
// lib/raytrace.c:20-96, which the reference builds but never binds or writes).
//
// Up to kOneMax instances one workgroup prepares them and builds the tree in LDS (k_lbvh_one): the
// update of a small scene is one launch.  Above, the steps are launches of their own (one stream, no
// host round trip):
//   k_instance_prep   ABI record (src/render.rs:74-78: column-major mat4, texture id bits
//                     in m[3][3], shaders/trace.vert:37-40) -> M, inverse(M) (FP64, rounded),
//                     padded world AABB of the unit proxy cube (lib/memory.c:22-40), centroid,
//                     centroid bounds of each workgroup;
//   k_rank_sort       30-bit Morton codes of the normalized centroids, sorted by counting the codes
//                     before each; above kRankMax instances k_bounds, k_morton and k_sort_*, a stable
//                     LSD radix sort (4 x 8-bit digits), one workgroup per 1024-key chunk: per-wave
//                     digit match by ballots, per-wave counts, prefix;
//   k_karras          leaves, internal nodes (Karras, HPG 2012), parent links;
//   k_refit_one       bottom-up AABB union and the tree's depth, in one workgroup's LDS; above
//                     kRefitOneMax instances k_refit (second arrival at a node continues, with
//                     agent-scope atomics and loads, so no stale L1 data is read) and k_depth.
// Integer parts (codes, order, topology) and the FP32 min/max unions are bit-exact with the
// CPU oracle; the FP32 arithmetic (corner transform, padding, centroid) follows the same
// operation order.
#include <hip/hip_runtime.h>

#include "vt_internal.h"

namespace {

constexpr int kSortThreads = 1024;
constexpr int kSortWaves = kSortThreads / 64;
// One workgroup for everything takes 8 us for 2 instances, 17 for 48, 29 for 256 and 69 for 1000; the
// launches of the next form, gaps included, 42 us for 512, 55 for 1000 and 84 for 4096.
constexpr uint32_t kOneMax = 512;         // one thread per instance
// k_refit_one: the boxes, links and counters of 4096 instances' inner nodes fill 144 of 160 KB of LDS
constexpr uint32_t kRefitOneMax = 4096;
constexpr int kRefitLeaves = 4;           // leaves per thread: kRefitOneMax / 1024
// k_rank_sort compares every pair of codes: an update (codes, tree and boxes) of 8000 instances takes 165 us with it
// and 178 with the radix sort, of 10000 189 and 193, of 12000 212 and 209, of 16384 262 and 248.
constexpr uint32_t kRankMax = 10240;
constexpr uint32_t kRankKeys = 64;        // keys a workgroup ranks
constexpr uint32_t kPrepThreads = 256;
// The mark behind a refit's first launch costs 5 us (of 30 for 16 instances, of 100 for 8000), which a program
// that draws a frame between refits has nothing for; three refits in a row without one take 112 us marked
// late and 92 marked early for 16, 302 and 272 for 8000, 573 and 499 for 20000.
constexpr uint32_t kMarkLateMax = 8192;

__device__ inline float gmin(float x, float y) { return (y < x) ? y : x; }
__device__ inline float gmax(float x, float y) { return (x < y) ? y : x; }
__device__ inline float pad_of(float v) { return fabsf(v) * 9.5367431640625e-07f + 9.5367431640625e-07f; }

// FP64 Laplace-expansion inverse (same formulas as the host vt_inverse4).
__device__ bool inverse4_d(const float* mf, float* out) {
#define A(r, c) ((double)mf[(c) * 4 + (r)])
    double s0 = A(0, 0) * A(1, 1) - A(1, 0) * A(0, 1);
    double s1 = A(0, 0) * A(1, 2) - A(1, 0) * A(0, 2);
    double s2 = A(0, 0) * A(1, 3) - A(1, 0) * A(0, 3);
    double s3 = A(0, 1) * A(1, 2) - A(1, 1) * A(0, 2);
    double s4 = A(0, 1) * A(1, 3) - A(1, 1) * A(0, 3);
    double s5 = A(0, 2) * A(1, 3) - A(1, 2) * A(0, 3);
    double c5 = A(2, 2) * A(3, 3) - A(3, 2) * A(2, 3);
    double c4 = A(2, 1) * A(3, 3) - A(3, 1) * A(2, 3);
    double c3 = A(2, 1) * A(3, 2) - A(3, 1) * A(2, 2);
    double c2 = A(2, 0) * A(3, 3) - A(3, 0) * A(2, 3);
    double c1 = A(2, 0) * A(3, 2) - A(3, 0) * A(2, 2);
    double c0 = A(2, 0) * A(3, 1) - A(3, 0) * A(2, 1);
    double det = s0 * c5 - s1 * c4 + s2 * c3 + s3 * c2 - s4 * c1 + s5 * c0;
    if (!(det != 0.0) || !isfinite(det)) return false;
    double b[16];  // b[r*4 + c]
    b[0] = (A(1, 1) * c5 - A(1, 2) * c4 + A(1, 3) * c3) / det;
    b[1] = (-A(0, 1) * c5 + A(0, 2) * c4 - A(0, 3) * c3) / det;
    b[2] = (A(3, 1) * s5 - A(3, 2) * s4 + A(3, 3) * s3) / det;
    b[3] = (-A(2, 1) * s5 + A(2, 2) * s4 - A(2, 3) * s3) / det;
    b[4] = (-A(1, 0) * c5 + A(1, 2) * c2 - A(1, 3) * c1) / det;
    b[5] = (A(0, 0) * c5 - A(0, 2) * c2 + A(0, 3) * c1) / det;
    b[6] = (-A(3, 0) * s5 + A(3, 2) * s2 - A(3, 3) * s1) / det;
    b[7] = (A(2, 0) * s5 - A(2, 2) * s2 + A(2, 3) * s1) / det;
    b[8] = (A(1, 0) * c4 - A(1, 1) * c2 + A(1, 3) * c0) / det;
    b[9] = (-A(0, 0) * c4 + A(0, 1) * c2 - A(0, 3) * c0) / det;
    b[10] = (A(3, 0) * s4 - A(3, 1) * s2 + A(3, 3) * s0) / det;
    b[11] = (-A(2, 0) * s4 + A(2, 1) * s2 - A(2, 3) * s0) / det;
    b[12] = (-A(1, 0) * c3 + A(1, 1) * c1 - A(1, 2) * c0) / det;
    b[13] = (A(0, 0) * c3 - A(0, 1) * c1 + A(0, 2) * c0) / det;
    b[14] = (-A(3, 0) * s3 + A(3, 1) * s1 - A(3, 2) * s0) / det;
    b[15] = (A(2, 0) * s3 - A(2, 1) * s1 + A(2, 2) * s0) / det;
#undef A
    bool ok = true;
    for (int r = 0; r < 4; ++r)
        for (int c = 0; c < 4; ++c) {
            float v = (float)b[r * 4 + c];
            if (!isfinite(v)) ok = false;
            out[c * 4 + r] = v;
        }
    return ok;
}

// Instance i from its record (16 floats, M4[0..3]) -> instance data, leaf, centroid.
__device__ void prep_instance(const float4* M4, uint32_t i, const VolumeDesc* vols, uint32_t nvol, InstanceGPU* inst,
                              BvhNode* leaves_tmp, float* cen, float c3[3]) {
    float M[16];
    for (int k = 0; k < 4; ++k) {
        const float4 v = M4[k];
        M[4 * k] = v.x; M[4 * k + 1] = v.y; M[4 * k + 2] = v.z; M[4 * k + 3] = v.w;
    }
    uint32_t tex = __float_as_uint(M[15]);
    M[15] = 1.0f;
    float inv[16];
    bool ok = inverse4_d(M, inv);
    InstanceGPU g;
    for (int c = 0; c < 4; ++c)
        for (int r = 0; r < 3; ++r) {
            g.M[c * 3 + r] = M[c * 4 + r];
            g.inv[c * 3 + r] = inv[c * 4 + r];
        }
    g.tex = tex;
    g.valid = (ok && tex < nvol) ? 1u : 0u;
    for (int a = 0; a < 3; ++a) {
        uint32_t d = g.valid ? vols[tex].dim[a] : 1u;
        g.dim[a] = d;
        g.size[a] = (float)d;
    }
    g.pad[0] = g.pad[1] = 0;
    inst[i] = g;
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (int c = 0; c < 8; ++c) {
        float p[3] = {(c & 1) ? 0.5f : -0.5f, (c & 2) ? 0.5f : -0.5f, (c & 4) ? 0.5f : -0.5f};
        for (int a = 0; a < 3; ++a) {
            float w = ((M[0 * 4 + a] * p[0] + M[1 * 4 + a] * p[1]) + M[2 * 4 + a] * p[2]) + M[3 * 4 + a] * 1.0f;
            lo[a] = gmin(lo[a], w);
            hi[a] = gmax(hi[a], w);
        }
    }
    BvhNode L;
    for (int a = 0; a < 3; ++a) {
        L.lo[a] = ok ? lo[a] - pad_of(lo[a]) : 0.0f;
        L.hi[a] = ok ? hi[a] + pad_of(hi[a]) : 0.0f;
        c3[a] = (L.lo[a] + L.hi[a]) * 0.5f;
        cen[3 * (size_t)i + a] = c3[a];
    }
    L.left = i;
    L.right = VT_EMPTY;
    leaves_tmp[i] = L;
}

// The records of instances [first, first + count) into LDS, 16 B per thread and step: they may lie in
// page-locked host memory, which is read once, in whole lines.  (No barrier at the end.)
__device__ __forceinline__ void stage_records(const float* records, uint32_t first, uint32_t count, float4* lds) {
    const float4* src = reinterpret_cast<const float4*>(records) + 4 * (size_t)first;
    for (uint32_t k = threadIdx.x; k < 4u * count; k += blockDim.x) lds[k] = src[k];
}

// Minima b[0..2] and maxima b[3..5] over a wave, in lane 0.  (gmin and gmax never take a NaN into an
// accumulator that starts infinite, so the order of the elements does not matter.)
__device__ __forceinline__ void wave_bounds(float b[6]) {
    for (int s = 32; s > 0; s >>= 1)
        for (int a = 0; a < 3; ++a) {
            b[a] = gmin(b[a], __shfl_down(b[a], s, 64));
            b[3 + a] = gmax(b[3 + a], __shfl_down(b[3 + a], s, 64));
        }
}

// bounds_out (optional): 6 floats per workgroup
__global__ __launch_bounds__(kPrepThreads) void k_instance_prep(const float* records, uint32_t n, const VolumeDesc* vols,
                                                                uint32_t nvol, InstanceGPU* inst, BvhNode* leaves_tmp,
                                                                float* cen, float* bounds_out) {
    __shared__ float4 rec[4 * kPrepThreads];
    __shared__ float wb[kPrepThreads / 64][6];
    const uint32_t first = blockIdx.x * kPrepThreads, tid = threadIdx.x;
    stage_records(records, first, min(kPrepThreads, n - first), rec);
    __syncthreads();
    float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (first + tid < n) {
        float c[3];
        prep_instance(rec + 4 * tid, first + tid, vols, nvol, inst, leaves_tmp, cen, c);
        for (int a = 0; a < 3; ++a) { b[a] = gmin(b[a], c[a]); b[3 + a] = gmax(b[3 + a], c[a]); }
    }
    if (!bounds_out) return;
    wave_bounds(b);
    if ((tid & 63) == 0)
        for (int a = 0; a < 6; ++a) wb[tid >> 6][a] = b[a];
    __syncthreads();
    if (tid < 6) {
        float v = wb[0][tid];
        for (uint32_t w = 1; w < kPrepThreads / 64; ++w) v = tid < 3 ? gmin(v, wb[w][tid]) : gmax(v, wb[w][tid]);
        bounds_out[6 * (size_t)blockIdx.x + tid] = v;
    }
}

__global__ __launch_bounds__(1024) void k_bounds(const float* cen, uint32_t n, float* bounds) {
    __shared__ float smin[3][1024], smax[3][1024];
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x)
        for (int a = 0; a < 3; ++a) {
            float c = cen[3 * (size_t)i + a];
            lo[a] = gmin(lo[a], c);
            hi[a] = gmax(hi[a], c);
        }
    for (int a = 0; a < 3; ++a) { smin[a][threadIdx.x] = lo[a]; smax[a][threadIdx.x] = hi[a]; }
    __syncthreads();
    for (uint32_t s = blockDim.x / 2; s > 0; s >>= 1) {
        if (threadIdx.x < s)
            for (int a = 0; a < 3; ++a) {
                smin[a][threadIdx.x] = gmin(smin[a][threadIdx.x], smin[a][threadIdx.x + s]);
                smax[a][threadIdx.x] = gmax(smax[a][threadIdx.x], smax[a][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x < 3) {
        bounds[threadIdx.x] = smin[threadIdx.x][0];
        bounds[3 + threadIdx.x] = smax[threadIdx.x][0];
    }
}

__device__ inline uint32_t expand10(uint32_t v) {
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

__device__ inline uint32_t morton_code(const float* cen, uint32_t i, const float* bounds) {
    uint32_t q[3];
    for (int a = 0; a < 3; ++a) {
        float ext = bounds[3 + a] - bounds[a];
        float u = ext > 0.0f ? (cen[3 * (size_t)i + a] - bounds[a]) / ext : 0.0f;
        float s = floorf(u * 1024.0f);
        int qi = (int)s;
        qi = qi < 0 ? 0 : (qi > 1023 ? 1023 : qi);
        q[a] = (uint32_t)qi;
    }
    return (expand10(q[0]) << 2) | (expand10(q[1]) << 1) | expand10(q[2]);
}

__global__ void k_morton(const float* cen, uint32_t n, const float* bounds, uint32_t* keys, uint32_t* vals) {
    uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    keys[i] = morton_code(cen, i, bounds);
    vals[i] = i;
}

// How many of the sorted-by (code, index) pairs [j0, j1) come before (c, i); codes in LDS, j0 and j1
// multiples of 4, entries past the last code 0xFFFFFFFF (codes have 30 bits).
__device__ __forceinline__ uint32_t codes_before(const uint32_t* codes, uint32_t j0, uint32_t j1, uint32_t c, uint32_t i) {
    uint32_t r = 0;
#pragma unroll 4
    for (uint32_t j = j0; j < j1; j += 4) {
        const uint4 v = *reinterpret_cast<const uint4*>(codes + j);
        r += (v.x < c || (v.x == c && j < i)) ? 1u : 0u;
        r += (v.y < c || (v.y == c && j + 1u < i)) ? 1u : 0u;
        r += (v.z < c || (v.z == c && j + 2u < i)) ? 1u : 0u;
        r += (v.w < c || (v.w == c && j + 3u < i)) ? 1u : 0u;
    }
    return r;
}

// Morton codes and their stable order for up to kRankMax instances: every workgroup computes all codes
// into LDS (nb_bounds partial bounds from k_instance_prep) and ranks kRankKeys of them, each wave
// against its 16th of the codes.
__global__ __launch_bounds__(1024) void k_rank_sort(const float* cen, uint32_t n, const float* part, uint32_t nb_bounds,
                                                    uint32_t* keys, uint32_t* vals) {
    extern __shared__ __align__(16) unsigned char smem[];
    uint32_t* const codes = reinterpret_cast<uint32_t*>(smem);   // n rounded up to 64
    __shared__ float bounds[6];
    __shared__ uint32_t rank[kRankKeys];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (wave == 0) {
        float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
        for (uint32_t k = lane; k < nb_bounds; k += 64)
            for (int a = 0; a < 3; ++a) {
                b[a] = gmin(b[a], part[6 * k + a]);
                b[3 + a] = gmax(b[3 + a], part[6 * k + 3 + a]);
            }
        wave_bounds(b);
        if (lane == 0)
            for (int a = 0; a < 6; ++a) bounds[a] = b[a];
        rank[lane] = 0u;
    }
    __syncthreads();
    const uint32_t np = (n + 63u) & ~63u;
    for (uint32_t i = tid; i < np; i += 1024) codes[i] = i < n ? morton_code(cen, i, bounds) : 0xFFFFFFFFu;
    __syncthreads();
    const uint32_t i = blockIdx.x * kRankKeys + lane;
    const uint32_t c = i < n ? codes[i] : 0u;
    const uint32_t per = (np / 16u + 3u) & ~3u, j0 = min(np, wave * per), j1 = min(np, j0 + per);
    atomicAdd(&rank[lane], codes_before(codes, j0, j1, c, i));
    __syncthreads();
    if (wave == 0 && i < n) {
        keys[rank[lane]] = c;
        vals[rank[lane]] = i;
    }
}

// Rank of a key among the keys of its 1024-key chunk with the same digit d that come before
// it (a stable counting sort's offset within the digit): the wave's keys of digit d are
// matched by 8 ballots, counted per wave, and the counts prefixed over the waves.  On return
// wcount[w][d] holds the keys of digit d in waves before w; tot[d] (thread d < 256 writes it)
// the chunk's keys of digit d.  Called by every thread of the workgroup.
__device__ __forceinline__ uint32_t chunk_rank(uint32_t d, bool valid, uint32_t (*wcount)[256], uint32_t* tot) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (uint32_t j = tid; j < kSortWaves * 256; j += kSortThreads) (&wcount[0][0])[j] = 0;
    __syncthreads();
    uint64_t peers = __ballot(valid);
    for (int b = 0; b < 8; ++b) {
        uint64_t bal = __ballot((d >> b) & 1u);
        peers &= ((d >> b) & 1u) ? bal : ~bal;
    }
    const uint64_t lower = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    const uint32_t rank = (uint32_t)__popcll(peers & lower);
    if (valid && rank == 0) wcount[wave][d] = (uint32_t)__popcll(peers);
    __syncthreads();
    if (tid < 256) {  // prefix over waves, per digit
        uint32_t acc = 0;
        for (int w = 0; w < kSortWaves; ++w) {
            uint32_t c = wcount[w][tid];
            wcount[w][tid] = acc;
            acc += c;
        }
        tot[tid] = acc;
    }
    __syncthreads();
    return wcount[wave][d] + rank;
}

// Stable LSD radix sort, one workgroup per 1024-key chunk.  k_sort_hist: the chunk's digit counts,
// stored digit-major (ghist[d * nch + c]), so an exclusive scan of ghist gives each chunk's first
// position for each digit, chunks in order.
__global__ __launch_bounds__(kSortThreads) void k_sort_hist(const uint32_t* kin, uint32_t n, uint32_t shift,
                                                            uint32_t* ghist) {
    __shared__ uint32_t hist[256];
    const uint32_t tid = threadIdx.x, c = blockIdx.x, nch = gridDim.x;
    if (tid < 256) hist[tid] = 0;
    __syncthreads();
    const uint32_t i = c * kSortThreads + tid;
    if (i < n) atomicAdd(&hist[(kin[i] >> shift) & 255u], 1u);
    __syncthreads();
    if (tid < 256) ghist[tid * nch + c] = hist[tid];
}

// Exclusive scan of ghist[0, total) in place, one workgroup: each thread sums a contiguous
// segment, the segment sums are scanned in LDS, then each segment is rewritten.
__global__ __launch_bounds__(kSortThreads) void k_sort_scan(uint32_t* ghist, uint32_t total) {
    __shared__ uint32_t part[kSortThreads];
    const uint32_t tid = threadIdx.x;
    const uint32_t per = (total + kSortThreads - 1) / kSortThreads;
    const uint32_t b = min(tid * per, total), e = min(b + per, total);
    uint32_t s = 0;
    for (uint32_t j = b; j < e; ++j) s += ghist[j];
    part[tid] = s;
    __syncthreads();
    for (uint32_t off = 1; off < (uint32_t)kSortThreads; off <<= 1) {
        const uint32_t v = tid >= off ? part[tid - off] : 0u;
        __syncthreads();
        part[tid] += v;
        __syncthreads();
    }
    uint32_t acc = part[tid] - s;
    for (uint32_t j = b; j < e; ++j) {
        const uint32_t c = ghist[j];
        ghist[j] = acc;
        acc += c;
    }
}

// Scatter of chunk c: position = the chunk's first slot for the digit + the key's stable rank.
__global__ __launch_bounds__(kSortThreads) void k_sort_scatter(const uint32_t* kin, const uint32_t* vin, uint32_t* kout,
                                                               uint32_t* vout, uint32_t n, uint32_t shift,
                                                               const uint32_t* ghist) {
    __shared__ uint32_t wcount[kSortWaves][256];
    __shared__ uint32_t tot[256];
    const uint32_t tid = threadIdx.x, c = blockIdx.x, nch = gridDim.x;
    const uint32_t i = c * kSortThreads + tid;
    const bool valid = i < n;
    const uint32_t key = valid ? kin[i] : 0u, val = valid ? vin[i] : 0u;
    const uint32_t d = (key >> shift) & 255u;
    const uint32_t r = chunk_rank(d, valid, wcount, tot);
    if (valid) {
        const uint32_t pos = ghist[d * nch + c] + r;
        kout[pos] = key;
        vout[pos] = val;
    }
}

// Karras' node ranges over sorted codes: code(i) is the i-th; equal codes are told apart by position.
template <typename Code>
__device__ __forceinline__ int delta_k(const Code& code, int i, int j, int n) {
    if (j < 0 || j >= n) return -1;
    uint32_t a = code(i), b = code(j);
    if (a == b) return 32 + __clz((uint32_t)i ^ (uint32_t)j);
    return __clz(a ^ b);
}
// children of inner node i of n > 1 leaves (inner nodes 0..n-2, leaf k is node n - 1 + k)
template <typename Code>
__device__ __forceinline__ void karras_node(const Code& K, int i, int n, uint32_t* left, uint32_t* right) {
    int d = (delta_k(K, i, i + 1, n) - delta_k(K, i, i - 1, n)) >= 0 ? 1 : -1;
    int dmin = delta_k(K, i, i - d, n);
    int lmax = 2;
    while (delta_k(K, i, i + lmax * d, n) > dmin) lmax *= 2;
    int l = 0;
    for (int t = lmax / 2; t >= 1; t /= 2)
        if (delta_k(K, i, i + (l + t) * d, n) > dmin) l += t;
    int j = i + l * d;
    int dnode = delta_k(K, i, j, n);
    int s = 0;
    for (int div = 2;; div *= 2) {
        int tt = (l + div - 1) / div;
        if (delta_k(K, i, i + (s + tt) * d, n) > dnode) s += tt;
        if (tt <= 1) break;
    }
    int gamma = i + s * d + (d < 0 ? d : 0);
    int first = d > 0 ? i : j;
    int last = d > 0 ? j : i;
    *left = (first == gamma) ? (uint32_t)(n - 1 + gamma) : (uint32_t)gamma;
    *right = (last == gamma + 1) ? (uint32_t)(n - 1 + gamma + 1) : (uint32_t)(gamma + 1);
}

__global__ void k_leaves(const uint32_t* order, uint32_t n, const BvhNode* leaves_tmp, BvhNode* nodes) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    nodes[n - 1 + k] = leaves_tmp[order[k]];
}

// Leaves and inner nodes.  LDS: the codes are staged (dynamic LDS of 4 n bytes), so the search's chain
// of dependent reads stays in the CU.
template <bool LDS>
__global__ __launch_bounds__(256) void k_karras(const uint32_t* K, const uint32_t* order, uint32_t n,
                                                const BvhNode* leaves_tmp, BvhNode* nodes, int32_t* parent,
                                                uint32_t* counters) {
    extern __shared__ __align__(16) unsigned char smem[];
    uint32_t* const codes = reinterpret_cast<uint32_t*>(smem);
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (LDS) {
        for (uint32_t j = threadIdx.x; j < n; j += 256u) codes[j] = K[j];
        __syncthreads();
    }
    if (i < n) nodes[n - 1 + i] = leaves_tmp[order[i]];
    if (i == 0) parent[0] = -1;
    if (i + 1 >= n) return;
    counters[i] = 0;
    uint32_t left, right;
    if (LDS) karras_node([&](int k) { return codes[k]; }, (int)i, (int)n, &left, &right);
    else karras_node([&](int k) { return K[k]; }, (int)i, (int)n, &left, &right);
    nodes[i].left = left;
    nodes[i].right = right;
    parent[left] = (int32_t)i;
    parent[right] = (int32_t)i;
}

__device__ inline float load_f32_agent(const float* p) {
    return __uint_as_float(__hip_atomic_load(reinterpret_cast<const uint32_t*>(p), __ATOMIC_RELAXED,
                                             __HIP_MEMORY_SCOPE_AGENT));
}
__device__ inline void store_f32_agent(float* p, float v) {
    __hip_atomic_store(reinterpret_cast<uint32_t*>(p), __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__global__ void k_refit(uint32_t n, BvhNode* nodes, const int32_t* parent, uint32_t* counters) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    int node = parent[n - 1 + k];
    while (node >= 0) {
        uint32_t old = __hip_atomic_fetch_add(&counters[node], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (old == 0) return;  // first arrival: the sibling's thread continues
        BvhNode* N = &nodes[node];
        const uint32_t l = N->left, r = N->right;
        for (int a = 0; a < 3; ++a) {
            float llo = load_f32_agent(&nodes[l].lo[a]), rlo = load_f32_agent(&nodes[r].lo[a]);
            float lhi = load_f32_agent(&nodes[l].hi[a]), rhi = load_f32_agent(&nodes[r].hi[a]);
            store_f32_agent(&N->lo[a], gmin(llo, rlo));
            store_f32_agent(&N->hi[a], gmax(lhi, rhi));
        }
        __atomic_thread_fence(__ATOMIC_RELEASE);
        node = parent[node];
    }
}

__global__ void k_zero_counters(uint32_t* counters, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) counters[i] = 0u;
}

// Depth of the tree (edges on the longest root-leaf path): one thread per leaf walks up.
__global__ void k_depth(uint32_t n, const int32_t* parent, uint32_t* depth_out) {
    uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    uint32_t d = 0;
    int node = parent[n - 1 + k];
    while (node >= 0 && d < 4096u) {
        ++d;
        node = parent[node];
    }
    atomicMax(depth_out, d);
}

// Inner nodes of a tree in one workgroup's LDS: boxes [6][P], children (left | right << 16), arrivals;
// parents of all nodes.  P >= n.
constexpr uint32_t kNoNode = 0xFFFFu;
struct TreeSmem {
    float* box;
    uint32_t *kids, *seen;
    uint16_t* parent;
    uint32_t P;
    __device__ __forceinline__ TreeSmem(unsigned char* smem, uint32_t P_) : P(P_) {
        box = reinterpret_cast<float*>(smem);
        kids = reinterpret_cast<uint32_t*>(box + 6 * (size_t)P);
        seen = kids + P;
        parent = reinterpret_cast<uint16_t*>(seen + P);
    }
};
constexpr size_t kTreeSmemBytes = 36;   // per P: 6 x 4 B boxes, 4 B children, 4 B arrivals, 2 x 2 B parents

// Boxes of the inner nodes bottom-up and the tree's depth; then the nodes to memory.  Thread t holds
// the leaves [PER t, PER t + PER) (and the next one) in registers.  Two sibling leaves are joined by the left one's
// thread (they are neighbours in the order).  Elsewhere the second to arrive at a node joins its
// children and climbs on: a first arrival leaves its height in the counter, an inner child has its box
// in its own slot, and a leaf child puts its box into the node's slot (the node has no other leaf).
template <int PER>
__device__ __forceinline__ void refit_lds(const TreeSmem& S, uint32_t n, BvhNode* nodes, uint32_t* depth_out) {
    const uint32_t tid = threadIdx.x, T = blockDim.x, P = S.P;
    float lb[PER + 1][6];
#pragma unroll
    for (int q = 0; q <= PER; ++q) {
        const uint32_t k = min(PER * tid + (uint32_t)q, n - 1);
        const float4* src = reinterpret_cast<const float4*>(nodes + n - 1 + k);
        const float4 u = src[0], v = src[1];
        lb[q][0] = u.x; lb[q][1] = u.y; lb[q][2] = u.z; lb[q][3] = u.w; lb[q][4] = v.x; lb[q][5] = v.y;
    }
    for (int q = 0; q < PER; ++q) {
        const uint32_t k = PER * tid + (uint32_t)q;
        if (k >= n) break;
        float b[6], nx[6];
        for (int a = 0; a < 6; ++a) { b[a] = lb[0][a]; nx[a] = lb[1][a]; }
        for (int p = 0; p < PER; ++p)
            for (int a = 0; a < 6; ++a) lb[p][a] = lb[p + 1][a];
        uint32_t self = n - 1 + k, node = S.parent[self], h = 0;
        while (node != kNoNode) {
            const uint32_t l = S.kids[node] & 0xFFFFu, r = S.kids[node] >> 16, sib = l == self ? r : l;
            float o[6];
            if (self >= n - 1 && sib >= n - 1) {
                if (self == r) break;
                for (int a = 0; a < 6; ++a) o[a] = nx[a];
                h = 1;
            } else {
                if (self >= n - 1)
                    for (int a = 0; a < 6; ++a) S.box[a * P + node] = b[a];
                const uint32_t other =
                    __hip_atomic_exchange(&S.seen[node], h + 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (other == 0u) break;   // the sibling's thread goes on
                h = max(h + 1u, other);
                const uint32_t at = sib < n - 1 ? sib : node;
                for (int a = 0; a < 6; ++a) o[a] = S.box[a * P + at];
            }
            for (int a = 0; a < 3; ++a) {   // (left, right), as k_refit
                b[a] = l == self ? gmin(b[a], o[a]) : gmin(o[a], b[a]);
                b[3 + a] = l == self ? gmax(b[3 + a], o[3 + a]) : gmax(o[3 + a], b[3 + a]);
            }
            for (int a = 0; a < 6; ++a) S.box[a * P + node] = b[a];
            self = node;
            node = S.parent[node];
        }
        if (node == kNoNode) *depth_out = h;
    }
    __syncthreads();
    for (uint32_t i = tid; i + 1 < n; i += T) {
        const uint32_t kids = S.kids[i];
        float4* dst = reinterpret_cast<float4*>(nodes + i);
        dst[0] = make_float4(S.box[i], S.box[P + i], S.box[2 * P + i], S.box[3 * P + i]);
        dst[1] = make_float4(S.box[4 * P + i], S.box[5 * P + i], __uint_as_float(kids & 0xFFFFu), __uint_as_float(kids >> 16));
    }
}

__global__ __launch_bounds__(1024) void k_refit_one(uint32_t n, uint32_t P, BvhNode* nodes, const int32_t* parent,
                                                    uint32_t* depth_out) {
    extern __shared__ __align__(16) unsigned char smem[];
    const TreeSmem S(smem, P);
    for (uint32_t i = threadIdx.x; i < 2 * n - 1; i += 1024) S.parent[i] = (uint16_t)parent[i];   // (-1: kNoNode)
    for (uint32_t i = threadIdx.x; i + 1 < n; i += 1024) {
        S.kids[i] = nodes[i].left | (nodes[i].right << 16);
        S.seen[i] = 0u;
    }
    __syncthreads();
    refit_lds<kRefitLeaves>(S, n, nodes, depth_out);
}

// All steps in one workgroup for up to kOneMax instances, one thread each; P threads, the power of
// two >= n, at least 64.  The codes are sorted by counting the codes before each.
// Bound by latency (chains of dependent LDS steps on one CU).  As 8 to 11 launches of their own the
// steps took 33 us for one instance and 48 us for 48, the gaps between them not counted; this kernel
// takes 6 and 17 us.
__global__ __launch_bounds__(kOneMax) void k_lbvh_one(const float* records, uint32_t n, const VolumeDesc* vols,
                                                      uint32_t nvol, InstanceGPU* inst, BvhNode* leaves_tmp, float* cen,
                                                      uint32_t* order, BvhNode* nodes, int32_t* parent_out,
                                                      uint32_t* depth_out) {
    extern __shared__ __align__(16) unsigned char smem[];
    __shared__ float wb[kOneMax / 64][6], bounds[6];
    __shared__ __align__(16) uint32_t codes[kOneMax], sorted[kOneMax];
    const uint32_t tid = threadIdx.x, P = blockDim.x;
    const TreeSmem S(smem, P);
    float4* const rec = reinterpret_cast<float4*>(smem);   // (in the space of the tree)
    stage_records(records, 0, n, rec);
    __syncthreads();
    float b[6] = {INFINITY, INFINITY, INFINITY, -INFINITY, -INFINITY, -INFINITY};
    if (tid < n) {
        float c[3];
        prep_instance(rec + 4 * tid, tid, vols, nvol, inst, leaves_tmp, cen, c);
        for (int a = 0; a < 3; ++a) { b[a] = gmin(b[a], c[a]); b[3 + a] = gmax(b[3 + a], c[a]); }
    }
    if (n == 1) {
        if (tid == 0) {
            order[0] = 0u;
            nodes[0] = leaves_tmp[0];
            *depth_out = 0u;
        }
        return;
    }
    wave_bounds(b);
    if ((tid & 63) == 0)
        for (int a = 0; a < 6; ++a) wb[tid >> 6][a] = b[a];
    __syncthreads();   // (the records are no longer read)
    if (tid < 6) {
        float v = wb[0][tid];
        for (uint32_t w = 1; w < P / 64; ++w) v = tid < 3 ? gmin(v, wb[w][tid]) : gmax(v, wb[w][tid]);
        bounds[tid] = v;
    }
    __syncthreads();
    codes[tid] = tid < n ? morton_code(cen, tid, bounds) : 0xFFFFFFFFu;
    __syncthreads();
    if (tid < n) {
        const uint32_t c = codes[tid], k = codes_before(codes, 0, (n + 3u) & ~3u, c, tid);
        sorted[k] = c;
        order[k] = tid;
        nodes[n - 1 + k] = leaves_tmp[tid];
    }
    if (tid == 0) S.parent[0] = (uint16_t)kNoNode;
    __syncthreads();
    if (tid + 1 < n) {
        uint32_t left, right;
        karras_node([&](int k) { return sorted[k]; }, (int)tid, (int)n, &left, &right);
        S.kids[tid] = left | (right << 16);
        S.seen[tid] = 0u;
        S.parent[left] = (uint16_t)tid;
        S.parent[right] = (uint16_t)tid;
    }
    __syncthreads();
    for (uint32_t i = tid; i < 2 * n - 1; i += P) parent_out[i] = S.parent[i] == kNoNode ? -1 : (int32_t)S.parent[i];
    refit_lds<1>(S, n, nodes, depth_out);
}

}  // namespace

int vt_lbvh_reserve(LbvhWork& w, uint32_t n) {
    if (n <= w.cap && w.inst) return 0;
    vt_lbvh_free(w);
    uint32_t cap = 1;
    while (cap < n) cap *= 2;
    size_t nn = 2 * (size_t)cap;
    bool ok = hipMalloc(&w.inst, cap * sizeof(InstanceGPU)) == hipSuccess &&
              hipMalloc(&w.nodes, nn * sizeof(BvhNode)) == hipSuccess &&
              hipMalloc(&w.cen, 3 * (size_t)cap * sizeof(float) + cap * sizeof(BvhNode)) == hipSuccess &&
              hipMalloc(&w.keys[0], cap * 4) == hipSuccess && hipMalloc(&w.keys[1], cap * 4) == hipSuccess &&
              hipMalloc(&w.vals[0], cap * 4) == hipSuccess && hipMalloc(&w.vals[1], cap * 4) == hipSuccess &&
              hipMalloc(&w.parent, nn * 4) == hipSuccess && hipMalloc(&w.counters, cap * 4) == hipSuccess &&
              hipMalloc(&w.bounds, 6 * 4 * (((size_t)cap + kPrepThreads - 1) / kPrepThreads)) == hipSuccess && hipMalloc(&w.depth, 4) == hipSuccess &&
              hipMalloc(&w.sort_hist, 256 * 4 * ((size_t)(cap + kSortThreads - 1) / kSortThreads)) == hipSuccess;
    if (!ok) {
        vt_lbvh_free(w);
        return -1;
    }
    w.cap = cap;
    return 0;
}

void vt_lbvh_free(LbvhWork& w) {
    hipFree(w.inst); hipFree(w.nodes); hipFree(w.cen);
    hipFree(w.keys[0]); hipFree(w.keys[1]); hipFree(w.vals[0]); hipFree(w.vals[1]);
    hipFree(w.parent); hipFree(w.counters); hipFree(w.bounds); hipFree(w.depth); hipFree(w.sort_hist);
    w = LbvhWork{};
}

// Refit: new records for the same n instances keep the last build's topology (leaf order and
// parents); instance data and leaf boxes are recomputed, internal boxes rebuilt bottom-up.
int vt_lbvh_refit(LbvhWork& w, const float* records_dev, uint32_t n, const VolumeDesc* vols_dev, uint32_t nvol,
                  hipStream_t s, hipEvent_t read) {
    if (n == 0 || n > w.cap || !w.inst) return -1;
    const uint32_t tb = kPrepThreads, nb = (n + tb - 1) / tb;
    BvhNode* leaves_tmp = reinterpret_cast<BvhNode*>(w.cen + 3 * (size_t)w.cap);
    hipLaunchKernelGGL(k_instance_prep, dim3(nb), dim3(tb), 0, s, records_dev, n, vols_dev, nvol, w.inst, leaves_tmp,
                       w.cen, static_cast<float*>(nullptr));
    if (read && n > kMarkLateMax) hipEventRecord(read, s);
    hipLaunchKernelGGL(k_leaves, dim3(nb), dim3(tb), 0, s, w.vals[0], n, leaves_tmp, w.nodes);
    if (n > 1) {
        hipLaunchKernelGGL(k_zero_counters, dim3(nb), dim3(tb), 0, s, w.counters, n - 1);
        hipLaunchKernelGGL(k_refit, dim3(nb), dim3(tb), 0, s, n, w.nodes, w.parent, w.counters);
    }
    if (read && n <= kMarkLateMax) hipEventRecord(read, s);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Codes and order of more than kRankMax instances -> (keys[0], vals[0])
static void radix_sort(LbvhWork& w, uint32_t n, hipStream_t s) {
    const uint32_t tb = kPrepThreads, nb = (n + tb - 1) / tb;
    hipLaunchKernelGGL(k_bounds, dim3(1), dim3(1024), 0, s, w.cen, n, w.bounds);
    hipLaunchKernelGGL(k_morton, dim3(nb), dim3(tb), 0, s, w.cen, n, w.bounds, w.keys[0], w.vals[0]);
    const uint32_t nch = (n + kSortThreads - 1) / kSortThreads;   // 256 * nch <= sort_hist's size
    for (uint32_t pass = 0; pass < 4; ++pass) {   // pass p reads buffer p & 1: the result ends in (keys[0], vals[0])
        const uint32_t a = pass & 1u, b = a ^ 1u, shift = 8 * pass;
        hipLaunchKernelGGL(k_sort_hist, dim3(nch), dim3(kSortThreads), 0, s, w.keys[a], n, shift, w.sort_hist);
        hipLaunchKernelGGL(k_sort_scan, dim3(1), dim3(kSortThreads), 0, s, w.sort_hist, 256 * nch);
        hipLaunchKernelGGL(k_sort_scatter, dim3(nch), dim3(kSortThreads), 0, s, w.keys[a], w.vals[a], w.keys[b],
                           w.vals[b], n, shift, w.sort_hist);
    }
}

// Dynamic LDS of a launch: above the default limit it is allowed first.
template <typename K>
static bool allow_lds(K kernel, size_t lds) {
    return lds <= 49152 || hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) == hipSuccess;
}

int vt_lbvh_build(LbvhWork& w, const float* records_dev, uint32_t n, const VolumeDesc* vols_dev, uint32_t nvol,
                  hipStream_t s, hipEvent_t read) {
    if (n == 0) return 0;
    if (vt_lbvh_reserve(w, n) != 0) return -1;
    const uint32_t tb = kPrepThreads, nb = (n + tb - 1) / tb;
    BvhNode* leaves_tmp = reinterpret_cast<BvhNode*>(w.cen + 3 * (size_t)w.cap);
    if (n <= kOneMax) {
        uint32_t P = 64;
        while (P < n) P *= 2;
        const size_t lds = (size_t)P * 64;   // the records, then the tree
        if (!allow_lds(&k_lbvh_one, lds)) return -1;
        hipLaunchKernelGGL(k_lbvh_one, dim3(1), dim3(P), lds, s, records_dev, n, vols_dev, nvol, w.inst, leaves_tmp,
                           w.cen, w.vals[0], w.nodes, w.parent, w.depth);
        if (read) hipEventRecord(read, s);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    const bool rank = n <= kRankMax;
    hipLaunchKernelGGL(k_instance_prep, dim3(nb), dim3(tb), 0, s, records_dev, n, vols_dev, nvol, w.inst, leaves_tmp,
                       w.cen, rank ? w.bounds : static_cast<float*>(nullptr));
    if (read) hipEventRecord(read, s);
    if (rank) {
        const size_t lds = ((size_t)n + 63) / 64 * 256;
        if (!allow_lds(&k_rank_sort, lds) || !allow_lds(&k_karras<true>, lds)) return -1;
        hipLaunchKernelGGL(k_rank_sort, dim3((n + kRankKeys - 1) / kRankKeys), dim3(1024), lds, s, w.cen, n, w.bounds, nb,
                           w.keys[0], w.vals[0]);
        hipLaunchKernelGGL(k_karras<true>, dim3(nb), dim3(tb), lds, s, w.keys[0], w.vals[0], n, leaves_tmp, w.nodes,
                           w.parent, w.counters);
    } else {
        radix_sort(w, n, s);
        hipLaunchKernelGGL(k_karras<false>, dim3(nb), dim3(tb), 0, s, w.keys[0], w.vals[0], n, leaves_tmp, w.nodes,
                           w.parent, w.counters);
    }
    if (n <= kRefitOneMax) {
        uint32_t P = 64;
        while (P < n) P *= 2;
        const size_t lds = (size_t)P * kTreeSmemBytes;
        if (!allow_lds(&k_refit_one, lds)) return -1;
        hipLaunchKernelGGL(k_refit_one, dim3(1), dim3(1024), lds, s, n, P, w.nodes, w.parent, w.depth);
    } else {
        hipLaunchKernelGGL(k_zero_counters, dim3(1), dim3(64), 0, s, w.depth, 1u);
        hipLaunchKernelGGL(k_refit, dim3(nb), dim3(tb), 0, s, n, w.nodes, w.parent, w.counters);
        hipLaunchKernelGGL(k_depth, dim3(nb), dim3(tb), 0, s, n, w.parent, w.depth);
    }
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
