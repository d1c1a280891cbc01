// upload.hip — dense voxel volume -> 8^3 bricks (the GPU half of add_texture).
//
// Replaces the reference's staging copy into an R8G8B8A8_SRGB 3-D image
// (lib/memory.c:286-385, lib/command.c:132-134).  The dense input is the reference's
// texel order (x fastest).  Voxel v of the bricked volume holds the texel that
// NEAREST/CLAMP sampling at v/size selects (shaders/trace.frag:77, lib/descriptor.c:100-105);
// the per-axis remap tables carry that choice (identity for power-of-two sizes).
//
// Several volumes of one size can be bricked together (the streamed 16^3 terrain chunks):
// their bricks are numbered volume after volume, one scan numbers the non-empty bricks of all
// of them into shared pools, and each volume's map holds ids relative to its first brick in
// the pools, so every volume is laid out exactly as if it had been uploaded alone.
//
// Kernels:
//   k_brick_classify  a workgroup per row of 8 bricks (64 x 8 x 8 voxels), lanes along x: one ballot per
//                     row of voxels gives 8 bricks' bits (alpha > 0, trace.frag:78) -> 8 x u64 mask per
//                     brick and the 2^3-block mask (one bit per 2x2x2 block holding a voxel; zero
//                     for an empty brick);
//   k_scan_*          exclusive scan of the non-empty bricks -> brick ids in brick order;
//   k_dist_x, _y, _z  per empty brick the distance (largest of the axes') to the nearest non-empty brick
//                     of the volume, over all directions (its empty-space radius + 1) and over each
//                     octant alone (the side of the largest empty cube with the brick as its
//                     corner), one axis after another -> its brick map entry;
//   k_brick_scatter   brick map (id, or that entry), masks, block masks and payload of non-empty
//                     bricks into the pools, through LDS so that a brick is written in whole lines;
//                     palette and volume descriptors.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "vt_internal.h"

namespace {

constexpr uint32_t kRowBricks = 8;      // bricks of a workgroup: 64 voxels along x
constexpr uint32_t kRowThreads = 256;   // wave w: z-slices 2 w and 2 w + 1

struct BrickArgs {
    const uint8_t* dense;      // nvol volumes, one after another
    const uint32_t* palette;
    uint32_t dim[3];
    uint32_t bdim[3];
    uint32_t fmt;
    uint32_t nbv;              // bricks per volume
    uint32_t nb;               // bricks of the batch
    uint32_t rows_x;           // rows of kRowBricks bricks along x
    size_t vol_texels;         // texels per volume
};

// Nearest-texel remap of an axis: the texel NEAREST + CLAMP_TO_EDGE sampling of voxel / size selects
// (shaders/trace.frag:77, lib/descriptor.c:100-105), FP32.
__device__ __forceinline__ uint32_t nearest_texel(uint32_t v, uint32_t dim) {
    const float size = (float)dim;
    const float u = (float)v / size;
    const float x = u * size;
    const int t = (int)floorf(x);
    return (uint32_t)(t < 0 ? 0 : (t > (int)dim - 1 ? (int)dim - 1 : t));
}

// The row of bricks of workgroup `row`: its first brick's number in the batch, its bricks, and this
// lane's column of texels (wave w holds the z-slices 2 w and 2 w + 1 of the row).
struct Row {
    uint32_t b0, n, by, bz;
    bool x_in;
    size_t col;   // texel index of this lane's x at y = z = 0
    __device__ __forceinline__ Row(const BrickArgs& a, uint32_t row) {
        const uint32_t rx = row % a.rows_x, rest = row / a.rows_x;
        by = rest % a.bdim[1];
        const uint32_t kz = rest / a.bdim[1], k = kz / a.bdim[2];
        bz = kz % a.bdim[2];
        b0 = k * a.nbv + rx * kRowBricks + a.bdim[0] * (by + a.bdim[1] * bz);
        n = min(kRowBricks, a.bdim[0] - rx * kRowBricks);
        const uint32_t x = rx * kRowBricks * 8u + (threadIdx.x & 63u);
        x_in = x < a.dim[0];
        col = (size_t)k * a.vol_texels + nearest_texel(x_in ? x : 0u, a.dim[0]);
    }
};
// f(z, y, raw) for the 16 voxels of this lane, z in {2 w, 2 w + 1} and y in 0..7 of the row: the texel as
// stored, 0 outside the volume.  (All 16 loads are issued before the first is used.)
template <typename F>
__device__ __forceinline__ void for_voxels(const BrickArgs& a, const Row& R, F&& f) {
    const uint32_t z0 = 2u * (threadIdx.x >> 6);
    uint32_t ty[8], tz[2], raw[2][8];
    bool in[2][8];
#pragma unroll
    for (uint32_t y = 0; y < 8; ++y) ty[y] = nearest_texel(min(R.by * 8 + y, a.dim[1] - 1), a.dim[1]);
#pragma unroll
    for (uint32_t z = 0; z < 2; ++z) tz[z] = nearest_texel(min(R.bz * 8 + z0 + z, a.dim[2] - 1), a.dim[2]);
#pragma unroll
    for (uint32_t z = 0; z < 2; ++z)
#pragma unroll
        for (uint32_t y = 0; y < 8; ++y) {
            in[z][y] = R.x_in && R.by * 8 + y < a.dim[1] && R.bz * 8 + z0 + z < a.dim[2];
            const size_t ti = R.col + (size_t)a.dim[0] * ((size_t)ty[y] + (size_t)a.dim[1] * tz[z]);
            raw[z][y] = 0u;
            if (in[z][y]) raw[z][y] = a.fmt == 0 ? (uint32_t)a.dense[ti] : reinterpret_cast<const uint32_t*>(a.dense)[ti];
        }
#pragma unroll
    for (uint32_t z = 0; z < 2; ++z)
#pragma unroll
        for (uint32_t y = 0; y < 8; ++y) f(z, y, raw[z][y], in[z][y]);
}

// 2x2 footprints of a z-slice's occupancy (bit x + 8y) -> 16 bits, bit bx + 4by for the
// 2x2 column (2bx.., 2by..) of the slice
__device__ inline uint32_t slice_blocks(uint64_t m) {
    uint64_t t = m | (m >> 1);
    t |= t >> 8;
    uint32_t r = 0;
    for (uint32_t by = 0; by < 4; ++by)
        for (uint32_t bx = 0; bx < 4; ++bx) r |= (uint32_t)((t >> (2u * bx + 16u * by)) & 1u) << (bx + 4u * by);
    return r;
}

// Bound by reading the volume once.  (One workgroup per brick with 8-byte segments of a row per load,
// remap tables and a palette load per voxel took 70 us for 256^3 indices; this takes 20 us.)
__global__ __launch_bounds__(kRowThreads) void k_brick_classify(BrickArgs a, uint64_t* masks_all, uint64_t* blocks_all) {
    __shared__ uint64_t alpha[4];   // palette entries with alpha > 0
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (a.fmt == 0) {
        const uint64_t bits = __ballot((a.palette[tid] >> 24) != 0u);
        if (lane == 0) alpha[wave] = bits;
        __syncthreads();
    }
    const Row R(a, blockIdx.x);
    uint64_t m[2] = {0, 0};   // lane b < 8: brick b's slices
    for_voxels(a, R, [&](uint32_t z, uint32_t y, uint32_t raw, bool in) {
        const bool occ = in && (a.fmt == 0 ? ((alpha[raw >> 6] >> (raw & 63u)) & 1ull) != 0ull : (raw >> 24) != 0u);
        const uint64_t bits = __ballot(occ);
        m[z] |= ((bits >> (8u * (lane & 7u))) & 0xFFull) << (8u * y);
    });
    if (lane < R.n) {
        const size_t b = R.b0 + lane;
        masks_all[b * 8 + 2 * wave] = m[0];
        masks_all[b * 8 + 2 * wave + 1] = m[1];
        reinterpret_cast<uint16_t*>(blocks_all)[b * 4 + wave] = (uint16_t)slice_blocks(m[0] | m[1]);
    }
}

// ---- distances ------------------------------------------------------------------------------
// The largest-axis distance to the nearest non-empty brick q is min over q of max(|dx|, |dy|, |dz|), so
// it can be taken one axis after another: along x the nearest in the row, then along y the minimum of
// max(|dy|, that), then along z; the same for the bricks q of one octant alone.  A search along an
// axis ends where its distance reaches what it has found.  Bricks outside the volume are empty.
// (Growing the radii layer by layer took 31 launches and the cubes 7: 160 us and 38 launches for
// 32^3 bricks; these three take 19 us.)
constexpr uint32_t kFar = VT_BRICK_RADIUS_CAP + 1u;   // no non-empty brick nearer: radius VT_BRICK_RADIUS_CAP
// packed: all directions in bits 0..7, octant c in bits 8 + 4 c (at most VT_BRICK_CUBE_CAP)
__device__ __forceinline__ uint32_t oct_dist(uint32_t v, uint32_t c) { return (v >> (8u + 4u * c)) & 15u; }

__global__ __launch_bounds__(256) void k_dist_x(const uint64_t* blocks_all, uint32_t nb, uint32_t bx, uint32_t* out) {
    const uint32_t b = blockIdx.x * 256u + threadIdx.x;
    if (b >= nb) return;
    uint32_t f = 0, g = 0;   // the next non-empty brick up and down the row
    if (blocks_all[b] == 0ull) {
        const uint32_t x = b % bx;
        f = g = kFar;
        for (uint32_t d = 1; d < kFar; ++d) {
            if (f == kFar && x + d < bx && blocks_all[b + d] != 0ull) f = d;
            if (g == kFar && x >= d && blocks_all[b - d] != 0ull) g = d;
            if (min(f, g) <= d && (max(f, g) <= d || d >= VT_BRICK_CUBE_CAP)) break;
        }
    }
    out[b] = min(f, g) | (min(f, VT_BRICK_CUBE_CAP) << 8) | (min(g, VT_BRICK_CUBE_CAP) << 12);
}

// Along an axis of n bricks, `stride` apart: NC octants in, 2 NC out (octant c + NC towards lower indices).
template <uint32_t NC>
__device__ __forceinline__ void dist_axis(const uint32_t* in, uint32_t b, uint32_t at, uint32_t n, uint32_t stride,
                                          uint32_t* r_out, uint32_t (&oct)[2 * NC]) {
    const uint32_t v = in[b];
    uint32_t r = v & 255u, far = 0;
    for (uint32_t c = 0; c < NC; ++c) {
        oct[c] = oct[c + NC] = oct_dist(v, c);
        far = max(far, oct[c]);
    }
    far = max(far, r);
    for (uint32_t d = 1; d < far; ++d) {
        far = 0;
        const uint32_t up = at + d < n ? in[b + (size_t)d * stride] : ~0u;
        const uint32_t down = at >= d ? in[b - (size_t)d * stride] : ~0u;
        if (up != ~0u) r = min(r, max(d, up & 255u));
        if (down != ~0u) r = min(r, max(d, down & 255u));
        for (uint32_t c = 0; c < NC; ++c) {
            if (up != ~0u) oct[c] = min(oct[c], max(d, oct_dist(up, c)));
            if (down != ~0u) oct[c + NC] = min(oct[c + NC], max(d, oct_dist(down, c)));
            far = max(far, max(oct[c], oct[c + NC]));
        }
        far = max(far, r);
    }
    *r_out = r;
}

__global__ __launch_bounds__(256) void k_dist_y(const uint32_t* in, uint32_t nb, uint32_t bx, uint32_t by, uint32_t* out) {
    const uint32_t b = blockIdx.x * 256u + threadIdx.x;
    if (b >= nb) return;
    uint32_t r, oct[4];
    dist_axis<2>(in, b, b / bx % by, by, bx, &r, oct);
    for (uint32_t c = 0; c < 4; ++c) r |= oct[c] << (8u + 4u * c);
    out[b] = r;
}

// -> the brick map's entry of an empty brick (anything for a non-empty one)
__global__ __launch_bounds__(256) void k_dist_z(const uint32_t* in, uint32_t nb, uint32_t bxy, uint32_t bz, uint32_t* entry) {
    const uint32_t b = blockIdx.x * 256u + threadIdx.x;
    if (b >= nb) return;
    uint32_t r, oct[8];
    dist_axis<4>(in, b, b / bxy % bz, bz, bxy, &r, oct);
    uint32_t e = VT_EMPTY_BRICK | ((r - 1u) & 31u) << 24;
    for (uint32_t o = 0; o < 8; ++o) e |= ((oct[o] - 1u) & 7u) << (3u * o);
    entry[b] = e;
}

// ---- pools ----------------------------------------------------------------------------------
struct PoolArgs {
    const uint64_t *masks_all, *blocks_all;
    const uint32_t *ids, *entry;   // ids[nb]: the total
    uint32_t* map;
    uint64_t *masks, *blocks;
    uint8_t* payload;
    uint32_t* palette;             // fmt 0
    VolumeDesc* descs;             // of the batch's volumes
};

// A workgroup per row of bricks, as k_brick_classify; bricks meet in LDS (padded by 16 B, so that the 8
// bricks of a row of voxels lie in different banks) and leave as 16-byte stores: 48 -> 17 us for 256^3.
template <uint32_t BPV>
__global__ __launch_bounds__(kRowThreads) void k_brick_scatter(BrickArgs a, PoolArgs p) {
    constexpr uint32_t kBytes = 512u * BPV, kPitch = kBytes + 16u;
    __shared__ __align__(16) uint8_t tile[kRowBricks * kPitch];
    __shared__ uint32_t any;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    if (BPV == 1 && blockIdx.x == 0) p.palette[tid] = a.palette[tid];
    const Row R(a, blockIdx.x);
    if (tid == 0) any = 0u;
    __syncthreads();
    const uint32_t first = p.ids[R.b0 / a.nbv * a.nbv];   // pool slot of the volume's first brick
    if (tid < R.n) {
        const uint32_t b = R.b0 + tid;
        const bool full = p.blocks_all[b] != 0ull;
        p.map[b] = full ? p.ids[b] - first : p.entry[b];
        if (full) {
            p.blocks[p.ids[b]] = p.blocks_all[b];
            atomicOr(&any, 1u << tid);
        }
    }
    if (tid == 0 && R.b0 % a.nbv == 0u) {
        const uint32_t k = R.b0 / a.nbv, next = (k + 1u) * a.nbv;
        VolumeDesc d;
        for (int c = 0; c < 3; ++c) { d.dim[c] = a.dim[c]; d.bdim[c] = a.bdim[c]; }
        d.fmt = a.fmt;
        d.nbricks = p.ids[next] - first;
        d.brick_map = p.map + (size_t)k * a.nbv;
        d.masks = reinterpret_cast<const uint32_t*>(p.masks + (size_t)first * 8);
        d.payload = p.payload + (size_t)first * kBytes;
        d.palette = p.palette;
        d.blocks = p.blocks + first;
        p.descs[k] = d;
    }
    __syncthreads();
    const uint32_t full = any;
    if (full == 0u) return;
    if (tid < 64u && ((full >> (tid >> 3)) & 1u)) {
        const uint32_t b = R.b0 + (tid >> 3);
        p.masks[(size_t)p.ids[b] * 8 + (tid & 7u)] = p.masks_all[(size_t)b * 8 + (tid & 7u)];
    }
    for_voxels(a, R, [&](uint32_t z, uint32_t y, uint32_t raw, bool) {
        uint8_t* at = tile + (lane >> 3) * kPitch + ((lane & 7u) + 8u * y + 64u * (2u * wave + z)) * BPV;
        if (BPV == 1) *at = (uint8_t)raw;   // the payload keeps the texel as stored
        else *reinterpret_cast<uint32_t*>(at) = raw;
    });
    __syncthreads();
    for (uint32_t c = tid; c < kRowBricks * kBytes / 16u; c += kRowThreads) {
        const uint32_t k = c / (kBytes / 16u), o = c % (kBytes / 16u) * 16u;
        if ((full >> k) & 1u)
            *reinterpret_cast<uint4*>(p.payload + (size_t)p.ids[R.b0 + k] * kBytes + o) =
                *reinterpret_cast<const uint4*>(tile + k * kPitch + o);
    }
}

// ---- exclusive scan of the non-empty bricks ---------------------------------------------
constexpr int kScanBlock = 1024;
// Bricks that one workgroup numbers by itself (4 per thread and step, 19 us for 32768); more: 3
// launches, 1024 per block (14 us for 32768, gaps not counted)
constexpr uint32_t kScanOneMax = 16384;

__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t* total) {
    __shared__ uint32_t wsum[kScanBlock / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t x = v;
    for (int o = 1; o < 64; o <<= 1) {
        uint32_t y = __shfl_up(x, o, 64);
        if (lane >= o) x += y;
    }
    if (lane == 63) wsum[w] = x;
    __syncthreads();
    if (w == 0) {
        uint32_t s = lane < kScanBlock / 64 ? wsum[lane] : 0;
        for (int o = 1; o < 64; o <<= 1) {
            uint32_t y = __shfl_up(s, o, 64);
            if (lane >= o) s += y;
        }
        if (lane < kScanBlock / 64) wsum[lane] = s;
    }
    __syncthreads();
    uint32_t incl = x + (w > 0 ? wsum[w - 1] : 0u);
    *total = wsum[kScanBlock / 64 - 1];
    __syncthreads();
    return incl - v;
}

// ids[0, nb) and the total in ids[nb]; counts (page-locked host memory): ids[k * nbv], k = 0..nvol
__global__ __launch_bounds__(kScanBlock) void k_scan_one(const uint64_t* blocks_all, uint32_t nb, uint32_t* ids,
                                                         uint32_t nbv, uint32_t nvol, uint32_t* counts) {
    uint32_t carry = 0;
    for (uint32_t base = 0; base < nb; base += 4u * kScanBlock) {
        const uint32_t i = base + 4u * threadIdx.x;
        uint32_t f[4], sum = 0, total;
        for (uint32_t q = 0; q < 4; ++q) {
            f[q] = i + q < nb && blocks_all[i + q] != 0ull ? 1u : 0u;
            sum += f[q];
        }
        uint32_t at = carry + block_exclusive_scan(sum, &total);
        for (uint32_t q = 0; q < 4; ++q) {
            if (i + q < nb) ids[i + q] = at;
            at += f[q];
        }
        carry += total;
    }
    if (threadIdx.x == 0) ids[nb] = carry;
    __syncthreads();
    for (uint32_t k = threadIdx.x; k <= nvol; k += kScanBlock) counts[k] = ids[k * nbv];
}

__global__ __launch_bounds__(kScanBlock) void k_scan_reduce(const uint64_t* in, uint32_t n, uint32_t* block_sums) {
    uint32_t i = blockIdx.x * kScanBlock + threadIdx.x;
    uint32_t v = i < n && in[i] != 0ull ? 1u : 0u;
    uint32_t total;
    block_exclusive_scan(v, &total);
    if (threadIdx.x == 0) block_sums[blockIdx.x] = total;
}

__global__ __launch_bounds__(kScanBlock) void k_scan_blocks(uint32_t* block_sums, uint32_t nb, uint32_t* grand_total) {
    __shared__ uint32_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (uint32_t base = 0; base < nb; base += kScanBlock) {
        uint32_t i = base + threadIdx.x;
        uint32_t v = i < nb ? block_sums[i] : 0u;
        uint32_t total;
        uint32_t ex = block_exclusive_scan(v, &total);
        uint32_t c = carry;
        if (i < nb) block_sums[i] = ex + c;
        __syncthreads();
        if (threadIdx.x == 0) carry = c + total;
        __syncthreads();
    }
    if (threadIdx.x == 0) *grand_total = carry;
}

__global__ __launch_bounds__(kScanBlock) void k_scan_apply(const uint64_t* in, uint32_t n, const uint32_t* block_sums,
                                                            uint32_t* out) {
    uint32_t i = blockIdx.x * kScanBlock + threadIdx.x;
    uint32_t v = i < n && in[i] != 0ull ? 1u : 0u;
    uint32_t total;
    uint32_t ex = block_exclusive_scan(v, &total);
    if (i < n) out[i] = ex + block_sums[blockIdx.x];
}

__global__ void k_scan_counts(const uint32_t* ids, uint32_t nbv, uint32_t nvol, uint32_t* counts) {
    for (uint32_t k = blockIdx.x * blockDim.x + threadIdx.x; k <= nvol; k += gridDim.x * blockDim.x) counts[k] = ids[k * nbv];
}

constexpr size_t kKeepWorkspace = (size_t)64 << 20;   // a larger workspace is given back after its upload

}  // namespace

void vt_brick_free(BrickWork& w) {
    hipFree(w.mem);
    hipHostFree(w.counts);
    if (w.counted) hipEventDestroy(w.counted);
    w = BrickWork{};
}

// Brick nvol dense device volumes of one size (packed one after another; fmt 0: palette_host, 256
// entries) and write their descriptors.  One pool for all of them, allocated once the non-empty bricks are
// counted (the GPU works on the distances meanwhile); out[0] owns it.
int vt_brick_volume(BrickWork& w, const uint8_t* dense_dev, uint32_t fmt, const uint32_t* palette_host,
                    const uint32_t dim[3], uint32_t nvol, VolumeStore* out, VolumeDesc* descs, hipStream_t s) {
    if (nvol == 0) return -1;
    BrickArgs a{};
    a.dense = dense_dev;
    for (int k = 0; k < 3; ++k) {
        a.dim[k] = dim[k];
        a.bdim[k] = (dim[k] + 7) / 8;
    }
    a.fmt = fmt;
    const uint64_t nb64 = (uint64_t)a.bdim[0] * a.bdim[1] * a.bdim[2] * nvol;
    if (nb64 >= 0x7FFFFFFFull) return -1;
    a.nbv = a.bdim[0] * a.bdim[1] * a.bdim[2];
    a.nb = (uint32_t)nb64;
    a.rows_x = (a.bdim[0] + kRowBricks - 1) / kRowBricks;
    a.vol_texels = (size_t)dim[0] * dim[1] * dim[2];
    const uint32_t rows = a.rows_x * a.bdim[1] * a.bdim[2] * nvol, tb = (a.nb + 255) / 256;
    const uint32_t nblk = (a.nb + kScanBlock - 1) / kScanBlock;
    // workspace: masks, block masks, ids and total, two distance arrays, scan sums, palette
    const size_t n = a.nb;
    auto up = [](size_t x) { return (x + 255) & ~(size_t)255; };
    const size_t at_blocks = up(n * 64), at_ids = at_blocks + up(n * 8), at_d0 = at_ids + up(n * 4 + 4),
                 at_d1 = at_d0 + up(n * 4), at_sums = at_d1 + up(n * 4), at_pal = at_sums + up((size_t)nblk * 4),
                 need = at_pal + 1024;
    if (need > w.cap) {
        hipFree(w.mem);
        w.mem = nullptr;
        w.cap = 0;
        if (hipMalloc(&w.mem, need) != hipSuccess) return -1;
        w.cap = need;
    }
    if (nvol + 1 > w.counts_cap) {
        hipHostFree(w.counts);
        w.counts = nullptr;
        w.counts_cap = 0;
        const uint32_t cap = std::max(1024u, nvol + 1);
        if (hipHostMalloc(reinterpret_cast<void**>(&w.counts), (size_t)cap * 4, hipHostMallocDefault) != hipSuccess) return -1;
        w.counts_cap = cap;
    }
    if (!w.counted && hipEventCreateWithFlags(&w.counted, hipEventDisableTiming) != hipSuccess) return -1;
    char* const mem = static_cast<char*>(w.mem);
    uint64_t* const masks_all = reinterpret_cast<uint64_t*>(mem);
    uint64_t* const blocks_all = reinterpret_cast<uint64_t*>(mem + at_blocks);
    uint32_t* const ids = reinterpret_cast<uint32_t*>(mem + at_ids);
    uint32_t* const d0 = reinterpret_cast<uint32_t*>(mem + at_d0);
    uint32_t* const d1 = reinterpret_cast<uint32_t*>(mem + at_d1);
    uint32_t* const sums = reinterpret_cast<uint32_t*>(mem + at_sums);
    uint32_t* const pal = reinterpret_cast<uint32_t*>(mem + at_pal);
    if (fmt == 0) {
        if (hipMemcpyAsync(pal, palette_host, 1024, hipMemcpyHostToDevice, s) != hipSuccess) return -1;
        a.palette = pal;
    }
    hipLaunchKernelGGL(k_brick_classify, dim3(rows), dim3(kRowThreads), 0, s, a, masks_all, blocks_all);
    if (a.nb <= kScanOneMax) {
        hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(kScanBlock), 0, s, blocks_all, a.nb, ids, a.nbv, nvol, w.counts);
    } else {
        hipLaunchKernelGGL(k_scan_reduce, dim3(nblk), dim3(kScanBlock), 0, s, blocks_all, a.nb, sums);
        hipLaunchKernelGGL(k_scan_blocks, dim3(1), dim3(kScanBlock), 0, s, sums, nblk, ids + a.nb);
        hipLaunchKernelGGL(k_scan_apply, dim3(nblk), dim3(kScanBlock), 0, s, blocks_all, a.nb, sums, ids);
        hipLaunchKernelGGL(k_scan_counts, dim3(std::min(256u, nvol / 256u + 1u)), dim3(256), 0, s, ids, a.nbv, nvol,
                           w.counts);
    }
    hipError_t e = hipEventRecord(w.counted, s);
    hipLaunchKernelGGL(k_dist_x, dim3(tb), dim3(256), 0, s, blocks_all, a.nb, a.bdim[0], d0);
    hipLaunchKernelGGL(k_dist_y, dim3(tb), dim3(256), 0, s, d0, a.nb, a.bdim[0], a.bdim[1], d1);
    hipLaunchKernelGGL(k_dist_z, dim3(tb), dim3(256), 0, s, d1, a.nb, a.bdim[0] * a.bdim[1], a.bdim[2], d0);
    if (e == hipSuccess) e = hipGetLastError();
    if (e == hipSuccess) e = hipEventSynchronize(w.counted);
    const size_t bpv = fmt == 0 ? 1 : 4;
    char* pool = nullptr;
    size_t cnt = 0, at_masks = 0, at_pblocks = 0, at_payload = 0, at_ppal = 0;
    if (e == hipSuccess) {
        cnt = w.counts[nvol];
        at_masks = up(n * 4);
        at_pblocks = at_masks + up(cnt * 64);
        at_payload = at_pblocks + up(cnt * 8);
        at_ppal = at_payload + up(cnt * 512 * bpv);
        e = hipMalloc(reinterpret_cast<void**>(&pool), at_ppal + 1024);
    }
    PoolArgs p{};
    if (e == hipSuccess) {
        p.masks_all = masks_all;
        p.blocks_all = blocks_all;
        p.ids = ids;
        p.entry = d0;
        p.map = reinterpret_cast<uint32_t*>(pool);
        p.masks = reinterpret_cast<uint64_t*>(pool + at_masks);
        p.blocks = reinterpret_cast<uint64_t*>(pool + at_pblocks);
        p.payload = reinterpret_cast<uint8_t*>(pool + at_payload);
        p.palette = fmt == 0 ? reinterpret_cast<uint32_t*>(pool + at_ppal) : nullptr;
        p.descs = descs;
        if (fmt == 0) hipLaunchKernelGGL(k_brick_scatter<1>, dim3(rows), dim3(kRowThreads), 0, s, a, p);
        else hipLaunchKernelGGL(k_brick_scatter<4>, dim3(rows), dim3(kRowThreads), 0, s, a, p);
        e = hipGetLastError();
    }
    const hipError_t done = hipStreamSynchronize(s);   // (also before the workspace may go)
    if (w.cap > kKeepWorkspace) {
        hipFree(w.mem);
        w.mem = nullptr;
        w.cap = 0;
    }
    if (e != hipSuccess || done != hipSuccess) {
        hipFree(pool);
        return -1;
    }
    for (uint32_t k = 0; k < nvol; ++k) {
        VolumeStore& o = out[k];
        const size_t first = w.counts[k];
        o.owner = k == 0;
        o.pool = pool;
        o.nbricks = w.counts[k + 1] - w.counts[k];
        o.fmt = fmt;
        for (int c = 0; c < 3; ++c) { o.dim[c] = dim[c]; o.bdim[c] = a.bdim[c]; }
        o.brick_map = p.map + (size_t)k * a.nbv;
        o.masks = reinterpret_cast<uint32_t*>(p.masks + first * 8);
        o.payload = p.payload + first * 512 * bpv;
        o.blocks = p.blocks + first;
        o.palette = p.palette;
        o.bytes = (size_t)a.nbv * 4 + (size_t)o.nbricks * (64 + 8 + 512 * bpv);
    }
    return 0;
}

namespace {
__global__ void k_debrick(VolumeDesc v, uint8_t* dense) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t n = (size_t)v.dim[0] * v.dim[1] * v.dim[2];
    if (i >= n) return;
    uint32_t x = (uint32_t)(i % v.dim[0]);
    uint32_t y = (uint32_t)((i / v.dim[0]) % v.dim[1]);
    uint32_t z = (uint32_t)(i / ((size_t)v.dim[0] * v.dim[1]));
    uint32_t b = (x >> 3) + v.bdim[0] * ((y >> 3) + v.bdim[1] * (z >> 3));
    uint32_t e = v.brick_map[b];
    uint32_t li = (x & 7) + 8 * (y & 7) + 64 * (z & 7);
    if (v.fmt == 0) dense[i] = vt_brick_empty(e) ? 0 : v.payload[(size_t)e * 512 + li];
    else reinterpret_cast<uint32_t*>(dense)[i] = vt_brick_empty(e) ? 0u : reinterpret_cast<const uint32_t*>(v.payload)[(size_t)e * 512 + li];
}
}  // namespace

// Bricked -> dense (voxel order, after the texel remap) for round-trip checks.
int vt_debrick(const VolumeDesc& v, uint8_t* dense_dev, hipStream_t s) {
    size_t n = (size_t)v.dim[0] * v.dim[1] * v.dim[2];
    uint32_t blocks = (uint32_t)((n + 255) / 256);
    hipLaunchKernelGGL(k_debrick, dim3(blocks), dim3(256), 0, s, v, dense_dev);
    return hipGetLastError() == hipSuccess ? 0 : -1;
}
