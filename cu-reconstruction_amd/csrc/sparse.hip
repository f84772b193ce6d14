// sparse.hip -- sparse TSDF volume for gfx950: 8x8x8-voxel bricks found
// through a hash table, allocated along each frame's truncation band.
//
// No counterpart on the reference's path: its TSDFVolume is a dense grid
// (tsdf_volume.cu:194-254) and its only sparse structure is an unfinished
// octree prototype (octree.cu).  Here the lattice is the dense volume's --
// voxel v (any int32 triple, |v| < 2^23) has centre ((v + 0.5f) * vs) + off,
// the same float32 operations as tsdf_volume.cu:117-119 -- and a voxel holds
// D and W in the brick b = floor(v / 8) that contains it.  Unallocated voxels
// read as the fill value (D = truncation, W = 0).
//
// One integrate call (recon_sparse_integrate):
//   sparse_alloc_kernel     one lane per pixel with a valid depth d: the
//                           world box of the pixel's frustum slab between
//                           d - trunc and d + trunc (its eight corners), one
//                           voxel wider on every side, and every brick it
//                           meets is inserted (open addressing, linear
//                           probing, bounded, atomicCAS on the key) and
//                           marked new
//   sparse_integrate_kernel one wavefront per allocated brick, one layer of
//                           8 x 8 voxels a step: the dense update rule of
//                           integrate_device.hpp, voxel for voxel; a new
//                           brick starts from (truncation, 0) unread
// Every voxel the dense integrate would update inside the band
// (-trunc <= sdf <= trunc) lies in the slab of the pixel it projects to, so
// its brick is allocated before it is integrated; with every brick already
// allocated the result equals the dense integrate bit for bit.  Voxels of
// unallocated bricks miss only free-space (sdf > trunc) observations.
#pragma clang fp contract(off)

#include "recon_common.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace recon {

constexpr int kBrick = 8;                        // voxels per brick edge
constexpr int kBrickVoxels = kBrick * kBrick * kBrick;
constexpr unsigned long long kEmptySlot = ~0ull;
constexpr int kHalf = kBrick / 2;                // layers a lane holds at a time
constexpr int kMaxBricksPerAxis = 8;             // per pixel slab; more sets the overflow flag
constexpr int kCoordBits = 21;                   // brick coordinate range [-2^20, 2^20)
// Linear probing stops after kMaxProbes slots, on insertion and lookup
// alike, so a key is always within kMaxProbes of its hash.  The table has
// twice the pool's slots and stops taking keys when the pool is full, so it
// stays at most about half full and the bound is almost never reached; when
// it is, the brick is dropped and flagged.
constexpr int kMaxProbes = 128;

struct SparseParams {
    float vs[3], off[3];
    float fx, fy, cx, cy;
    float trunc, maxw, maxd;
    int64_t capacity;                 // bricks in the pool
    uint64_t mask;                    // hash table size - 1 (power of two)
    unsigned long long* keys;         // table keys, kEmptySlot when free
    int32_t* vals;                    // table values: brick index
    int4* coords;                     // brick coordinates, per brick; w = 1 while the brick is
                                      // new (its D and W not yet written)
    float* D;                         // capacity * 512
    float* W;
    unsigned* counter;                // bricks handed out (may exceed capacity)
    unsigned* overflow;               // bit 0: pool full, bit 1: slab too wide, bit 2: coordinate
                                      // range, bit 3: probe limit
    int32_t blo[3], bhi[3];           // allocation bounds in bricks (inclusive)
    float rfx, rfy, rvs[3];           // 1/fx, 1/fy, 1/vs
};

__host__ __device__ inline unsigned long long brick_key(int bx, int by, int bz) {
    const unsigned long long m = (1ull << kCoordBits) - 1ull;
    return (((unsigned long long)bx & m) << (2 * kCoordBits)) |
           (((unsigned long long)by & m) << kCoordBits) | ((unsigned long long)bz & m);
}

__host__ __device__ inline uint64_t hash_key(unsigned long long k) {
    // murmur3 64-bit finaliser
    k ^= k >> 33;
    k *= 0xff51afd7ed558ccdull;
    k ^= k >> 33;
    k *= 0xc4ceb9fe1a85ec53ull;
    k ^= k >> 33;
    return k;
}

__device__ __forceinline__ int floor_div8(int v) { return v >= 0 ? v >> 3 : -((-v + 7) >> 3); }


// Brick index of (bx, by, bz), or -1.
__device__ __forceinline__ int32_t find_brick(const SparseParams& p, int bx, int by, int bz) {
    const unsigned long long key = brick_key(bx, by, bz);
    uint64_t h = hash_key(key) & p.mask;
    for (uint64_t n = 0; n < (uint64_t)kMaxProbes && n <= p.mask; ++n) {
        const unsigned long long k = p.keys[h];
        if (k == key) return p.vals[h];
        if (k == kEmptySlot) return -1;
        h = (h + 1) & p.mask;
    }
    return -1;
}

__device__ __forceinline__ void insert_brick(const SparseParams& p, int bx, int by, int bz) {
    const unsigned long long key = brick_key(bx, by, bz);
    uint64_t h = hash_key(key) & p.mask;
    for (uint64_t n = 0; n < (uint64_t)kMaxProbes && n <= p.mask; ++n) {
        unsigned long long k = p.keys[h];
        if (k == key) return;
        if (k == kEmptySlot) {
            // a full pool takes no more keys (a racing few may still pass)
            if ((int64_t)*p.counter >= p.capacity) {
                atomicOr(p.overflow, 1u);
                return;
            }
            k = atomicCAS(p.keys + h, kEmptySlot, key);
            if (k == kEmptySlot) {
                const unsigned idx = atomicAdd(p.counter, 1u);
                if ((int64_t)idx < p.capacity) {
                    p.vals[h] = (int32_t)idx;
                    p.coords[idx] = make_int4(bx, by, bz, 1);
                } else {
                    p.vals[h] = -1;
                    atomicOr(p.overflow, 1u);
                }
                return;
            }
            if (k == key) return;
        }
        h = (h + 1) & p.mask;
    }
    atomicOr(p.overflow, 8u);
}

// A wavefront takes a patch of 8 x 8 pixels.  Neighbouring pixels mostly
// meet the same bricks, so a lane whose box equals that of the lane to its
// left or above it leaves the insertion to that lane, and the wavefront's
// remaining bricks are spread over its lanes: the probes, chains of dependent
// loads, bound this kernel (a VGA frame at 5 mm: 27 us with every lane
// walking its own box, 24 with the equal boxes dropped, 17 spread out).
// kShort: quotients
// by the reciprocals of fx, fy and vs and div_by_rcp, for parameters whose
// quotients stay normal (sparse_short_forms); else by the divisions.
template <bool kShort>
__global__ __launch_bounds__(256) void sparse_alloc_kernel(const SparseParams p, const FrameParams F,
                                                           int32_t cols, int32_t rows) {
    const int lane = threadIdx.x & 63;
    const int u = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 8 + (lane & 7);
    const int v = blockIdx.y * 8 + (lane >> 3);
    float d = 0.0f;
    if (u < cols && v < rows) d = F.depth[(int64_t)v * F.pitch + u];
    const auto quotient = [](float a, float b, float y) { return kShort ? div_by_rcp(a, b, y) : a / b; };
    const float z0 = d - p.trunc, z1 = d + p.trunc;
    float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const float su = (float)(u + (c & 1)), sv = (float)(v + ((c >> 1) & 1));
        const float z = (c & 4) ? z1 : z0;
        // camera point of pixel corner (su, sv) at depth z, then world = R^T (pc - t)
        const float xc = quotient((su - p.cx) * z, p.fx, p.rfx);
        const float yc = quotient((sv - p.cy) * z, p.fy, p.rfy);
        const float qx = xc - F.t[0], qy = yc - F.t[1], qz = z - F.t[2];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float w = ((F.R[k] * qx + F.R[3 + k] * qy) + F.R[6 + k] * qz);
            lo[k] = fminf(lo[k], w);
            hi[k] = fmaxf(hi[k], w);
        }
    }
    bool ok = d > 0.0f && d <= p.maxd, empty = false;
    unsigned flags = 0;
    int b0[3], b1[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        // voxel index range, one voxel wider on each side (covers rounding)
        const float a = floorf(quotient(lo[k] - p.off[k], p.vs[k], p.rvs[k])) - 1.0f;
        const float b = floorf(quotient(hi[k] - p.off[k], p.vs[k], p.rvs[k])) + 1.0f;
        const bool in = a > -8388608.0f && b < 8388608.0f;  // |v| < 2^23
        // as one axis after the other: an axis out of range ends the lane
        if (ok && !in) flags |= 4u;
        ok = ok && in;
        b0[k] = floor_div8(ok ? (int)a : 0);
        b1[k] = floor_div8(ok ? (int)b : 0);
        if (b1[k] - b0[k] >= kMaxBricksPerAxis) {
            flags |= 2u;
            b1[k] = b0[k] + kMaxBricksPerAxis - 1;
        }
        // allocation bounds (recon_sparse_set_bounds)
        b0[k] = max(b0[k], p.blo[k]);
        b1[k] = min(b1[k], p.bhi[k]);
        empty = empty || b0[k] > b1[k];
    }
    ok = ok && !empty;
    if (flags) atomicOr(p.overflow, flags);
    // the box in three words, the third -1 for a lane without one
    const unsigned long long key = brick_key(b0[0], b0[1], b0[2]);
    const int w0 = (int)(unsigned)key, w1 = (int)(key >> 32);
    const int n0 = b1[0] - b0[0] + 1, n1 = b1[1] - b0[1] + 1, n2 = b1[2] - b0[2] + 1;  // <= 8 each
    const int w2 = ok ? n0 | (n1 << 4) | (n2 << 8) : -1;
    const int left = max(lane - 1, 0), up = max(lane - 8, 0);
    const bool same_left = __shfl(w0, left, 64) == w0 && __shfl(w1, left, 64) == w1 && __shfl(w2, left, 64) == w2;
    const bool same_up = __shfl(w0, up, 64) == w0 && __shfl(w1, up, 64) == w1 && __shfl(w2, up, 64) == w2;
    const int n = !ok || (lane > 0 && same_left) || (lane > 7 && same_up) ? 0 : n0 * n1 * n2;
    // the remaining lanes' bricks, one per lane and round
    int incl = n;
#pragma unroll
    for (int s = 1; s < 64; s <<= 1) {
        const int o = __shfl_up(incl, s, 64);
        if (lane >= s) incl += o;
    }
    const int excl = incl - n, total = __shfl(incl, 63, 64);
    for (int k0 = 0; k0 < total; k0 += 64) {
        const int k = k0 + lane;
        int owner = 0;  // the number of lanes with incl <= k
#pragma unroll
        for (int s = 32; s >= 1; s >>= 1)
            if (__shfl(incl, owner + s - 1, 64) <= k) owner += s;
        owner = min(owner, 63);
        const int i = k - __shfl(excl, owner, 64), m = __shfl(w2, owner, 64);
        const int ox = __shfl(b0[0], owner, 64), oy = __shfl(b0[1], owner, 64), oz = __shfl(b0[2], owner, 64);
        const int m0 = m & 15, m1 = (m >> 4) & 15;
        if (k < total) insert_brick(p, ox + i % m0, oy + (i / m0) % m1, oz + i / (m0 * m1));
    }
}

// Whether the alloc kernel's quotients stay normal numbers (or zero) for
// every depth up to maxd: then the short forms equal the divisions.
static bool sparse_short_forms(const SparseParams& p, const FrameParams& F, int cols, int rows) {
    const auto mid = [](double v, double lo, double hi) { return std::fabs(v) >= lo && std::fabs(v) <= hi; };
    bool ok = mid(p.fx, 1e-3, 1e9) && mid(p.fy, 1e-3, 1e9) && std::fabs(p.cx) < 1e9 && std::fabs(p.cy) < 1e9 &&
              mid(p.trunc, 1e-6, 1e6) && p.maxd < 1e6f && cols < (1 << 24) && rows < (1 << 24);
    for (int k = 0; k < 3; ++k)
        ok = ok && mid(p.vs[k], 1e-6, 1e6) && std::fabs(p.off[k]) < 1e9 && std::fabs(F.t[k]) < 1e9;
    for (int k = 0; k < 9; ++k) ok = ok && std::fabs(F.R[k]) < 1e6;
    return ok;
}

// New bricks := (truncation, 0), one wavefront per brick (recon_sparse_allocate_box;
// an integrate call starts its new bricks itself).
__global__ __launch_bounds__(256) void sparse_init_kernel(const SparseParams p) {
    const int lane = threadIdx.x & 63;
    const unsigned n = (unsigned)min((int64_t)*p.counter, p.capacity);
    const unsigned waves = gridDim.x * 4;
    for (unsigned b = blockIdx.x * 4 + (threadIdx.x >> 6); b < n; b += waves) {
        if (p.coords[b].w == 0) continue;
        for (int i = lane; i < kBrickVoxels; i += 64) {
            p.D[(int64_t)b * kBrickVoxels + i] = p.trunc;
            p.W[(int64_t)b * kBrickVoxels + i] = 0.0f;
        }
        if (lane == 0) p.coords[b].w = 0;
    }
}

// Conservative visibility of a brick for one frame (wave-uniform result).
// Lanes 0..7 take the brick's corner voxel centres to the camera; a voxel
// can only pass the per-voxel tests when its camera point p satisfies
//   z > 0,  fx*x + (cx+1)*z > 0,  (cols-cx)*z - fx*x > 0,
//   fy*y + (cy+1)*z > 0,  (rows-cy)*z - fy*y > 0,  z <= maxd + trunc,
// all linear in p, so when every corner violates one of them by more than a
// relative 1e-3 every voxel centre of the brick (inside the corners' hull)
// does too, and the brick is skipped.
__device__ __forceinline__ bool brick_may_update(const SparseParams& p, const FrameParams& F,
                                                 const int4 bc, float fcols, float frows, int lane) {
    unsigned out = 0;  // bit k: this corner violates constraint k
    if (lane < 8) {
        const int v[3] = {bc.x * kBrick + ((lane & 1) ? kBrick - 1 : 0),
                          bc.y * kBrick + ((lane & 2) ? kBrick - 1 : 0),
                          bc.z * kBrick + ((lane & 4) ? kBrick - 1 : 0)};
        float c[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) c[k] = voxel_centre(v[k], p.vs[k], p.off[k]);
        float q[3];
#pragma unroll
        for (int k = 0; k < 3; ++k)
            q[k] = ((F.R[3 * k] * c[0] + F.R[3 * k + 1] * c[1]) + F.R[3 * k + 2] * c[2]) + F.t[k];
        const float x = q[0], y = q[1], z = q[2];
        const float ax = fabsf(p.fx * x), ay = fabsf(p.fy * y), az = fabsf(z);
        const float e = 1e-3f;
        if (z < -e * (az + 1e-6f)) out |= 1u;
        if (p.fx * x + (p.cx + 1.0f) * z < -e * (ax + fabsf(p.cx + 1.0f) * az + 1e-6f)) out |= 2u;
        if ((fcols - p.cx) * z - p.fx * x < -e * (ax + fabsf(fcols - p.cx) * az + 1e-6f)) out |= 4u;
        if (p.fy * y + (p.cy + 1.0f) * z < -e * (ay + fabsf(p.cy + 1.0f) * az + 1e-6f)) out |= 8u;
        if ((frows - p.cy) * z - p.fy * y < -e * (ay + fabsf(frows - p.cy) * az + 1e-6f)) out |= 16u;
        if (z > (p.maxd + p.trunc) * (1.0f + e)) out |= 32u;
    } else {
        out = 63u;
    }
    // a constraint every corner violates
    unsigned all = out;
#pragma unroll
    for (int d = 1; d < 8; d <<= 1) all &= __shfl_xor(all, d, 64);
    return __builtin_amdgcn_readfirstlane(all) == 0u;
}

// One wavefront per brick (grid-stride over the allocated bricks); at step z
// lane l holds voxel (l % 8, l / 8, z) of the brick, so a step's D and W
// accesses are 256 contiguous bytes and its depth taps neighbours.  The
// arithmetic is integrate_tile's: recip() and div_by_rcp, with `guard` (0, or
// infinity when the short forms do not cover the call) and the residuals
// sending a brick to the divisions.
__global__ __launch_bounds__(256) void sparse_integrate_kernel(const SparseParams p,
                                                               const FrameParams F, float fcols,
                                                               float frows) {
    const int lane = threadIdx.x & 63;
    const unsigned n = (unsigned)min((int64_t)__builtin_amdgcn_readfirstlane(*p.counter), p.capacity);
    const unsigned waves = gridDim.x * 4;
    for (unsigned b = blockIdx.x * 4 + (threadIdx.x >> 6); b < n; b += waves) {
        const int4 bc = p.coords[b];
        const bool fresh = __builtin_amdgcn_readfirstlane(bc.w) != 0;
        const bool seen = brick_may_update(p, F, bc, fcols, frows, lane);
        if (!seen && !fresh) continue;
        float* __restrict__ Db = p.D + (int64_t)b * kBrickVoxels + lane;
        float* __restrict__ Wb = p.W + (int64_t)b * kBrickVoxels + lane;
        if (fresh && lane == 0) p.coords[b].w = 0;
        if (!seen) {
#pragma unroll
            for (int j = 0; j < kBrick; ++j) {
                Db[64 * j] = p.trunc;
                Wb[64 * j] = 0.0f;
            }
            continue;
        }
        const float cx = voxel_centre(bc.x * kBrick + (lane & 7), p.vs[0], p.off[0]);
        const float cy = voxel_centre(bc.y * kBrick + (lane >> 3), p.vs[1], p.off[1]);
#pragma unroll 1
        for (int z0 = 0; z0 < kBrick; z0 += kHalf, Db += 64 * kHalf, Wb += 64 * kHalf) {
            float pz[kHalf], rz[kHalf], cz[kHalf], dep[kHalf];
            bool ok[kHalf];
            float bad = F.guard, most = 0.0f;
#pragma unroll
            for (int j = 0; j < kHalf; ++j) {
                cz[j] = voxel_centre(bc.z * kBrick + z0 + j, p.vs[2], p.off[2]);
                pz[j] = ((F.R[6] * cx + F.R[7] * cy) + F.R[8] * cz[j]) + F.t[2];
                rz[j] = recip(pz[j], bad);
                most = fmaxf(most, rz[j]);
            }
            const bool exact = __builtin_expect(__ballot((bad > kRecipBad) | (most > kRecipMax)) != 0, 0);
            uint32_t at[kHalf];
#pragma unroll
            for (int j = 0; j < kHalf; ++j) {
                const float px = ((F.R[0] * cx + F.R[1] * cy) + F.R[2] * cz[j]) + F.t[0];
                const float py = ((F.R[3] * cx + F.R[4] * cy) + F.R[5] * cz[j]) + F.t[1];
                if (exact) {
                    int u = 0, v = 0;
                    ok[j] = pz[j] > 0.0f && pixel_index(px, p.fx, pz[j], p.cx, fcols, u) &&
                            pixel_index(py, p.fy, pz[j], p.cy, frows, v);
                    dep[j] = F.depth[ok[j] ? (int64_t)v * F.pitch + u : 0];
                } else {
                    const int u = to_int_sat(div_by_rcp(px * p.fx, pz[j], rz[j]) + p.cx);
                    const int v = to_int_sat(div_by_rcp(py * p.fy, pz[j], rz[j]) + p.cy);
                    ok[j] = (pz[j] > 0.0f) & ((uint32_t)u < (uint32_t)(int)fcols) &
                            ((uint32_t)v < (uint32_t)(int)frows);
                    const uint32_t off = mul24((uint32_t)v, 4u * (uint32_t)F.pitch) + 4u * (uint32_t)u;
                    at[j] = ok[j] ? off : 0u;
                }
            }
            if (!exact) {
#pragma unroll
                for (int j = 0; j < kHalf; ++j) dep[j] = load_float((GlobalBytes)F.depth, at[j]);
            }
            bool pass[kHalf];
            float d[kHalf], w[kHalf];
#pragma unroll
            for (int j = 0; j < kHalf; ++j) {
                const float sdf = dep[j] - pz[j];
                pass[j] = ok[j] & (dep[j] > 0.0f) & (dep[j] <= p.maxd) & (sdf >= -p.trunc);
                d[j] = p.trunc;
                w[j] = 0.0f;
                if (pass[j] && !fresh) {
                    d[j] = Db[64 * j];
                    w[j] = Wb[64 * j];
                }
            }
            float nd[kHalf], badw = exact ? INFINITY : 0.0f;
#pragma unroll
            for (int j = 0; j < kHalf; ++j) {
                // tsdf_volume.cu:178-186 with the weight cap, as the dense path
                const float num = (d[j] * w[j]) + min_bound(p.trunc, dep[j] - pz[j]);
                const float nw = w[j] + 1.0f;
                nd[j] = div_by_rcp(num, nw, recip_sum(nw, badw));
            }
            if (__builtin_expect(__ballot(!(badw < kRecipBad)) != 0, 0)) {
#pragma unroll
                for (int j = 0; j < kHalf; ++j)
                    nd[j] = ((d[j] * w[j]) + min_bound(p.trunc, dep[j] - pz[j])) / (w[j] + 1.0f);
            }
#pragma unroll
            for (int j = 0; j < kHalf; ++j)
                if (pass[j] || fresh) {
                    Db[64 * j] = pass[j] ? nd[j] : d[j];
                    Wb[64 * j] = pass[j] ? min_bound(p.maxw, w[j] + 1.0f) : w[j];
                }
        }
    }
}

__global__ __launch_bounds__(256) void sparse_alloc_box_kernel(const SparseParams p, int4 b0, int4 nb) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    const int64_t total = (int64_t)nb.x * nb.y * nb.z;
    if (i >= total) return;
    const int bx = b0.x + (int)(i % nb.x), by = b0.y + (int)((i / nb.x) % nb.y),
              bz = b0.z + (int)(i / ((int64_t)nb.x * nb.y));
    insert_brick(p, bx, by, bz);
}

// Dense box [o, o + size) of the sparse volume; unallocated voxels give the
// fill value.  A wavefront takes a column of four bricks in x: lane l looks up
// the brick of its x once, then writes rows of 32 voxels, two a step, of the
// bricks' 8 x 8 rows.  One thread and one lookup per voxel took 219 us for
// both outputs of a 384^3 box (453 MB); this takes 87, near the 66 of a fill.
__global__ __launch_bounds__(256) void sparse_export_kernel(const SparseParams p, int4 o, int4 size,
                                                            int4 b0, int4 nb, float* __restrict__ D,
                                                            float* __restrict__ W) {
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int nc = (nb.x + 3) / 4;  // columns along x
    if (i >= (int64_t)nc * nb.y * nb.z) return;
    const int cx = (int)(i % nc), by = b0.y + (int)((i / nc) % nb.y), bz = b0.z + (int)(i / ((int64_t)nc * nb.y));
    const int x = (b0.x + 4 * cx) * kBrick + (lane & 31);  // the lane's voxel in x
    const int32_t b = find_brick(p, floor_div8(x), by, bz);
    const int64_t src = (int64_t)b * kBrickVoxels + (x & 7);
    const bool in_x = x >= o.x && x - o.x < size.x;
#pragma unroll 4
    for (int k = 0; k < 32; ++k) {
        const int r = 2 * k + (lane >> 5);  // row of the brick: y + 8 z
        const int y = by * kBrick + (r & 7) - o.y, z = bz * kBrick + (r >> 3) - o.z;
        if (!in_x || y < 0 || y >= size.y || z < 0 || z >= size.z) continue;
        const int64_t j = (x - o.x) + (int64_t)size.x * (y + (int64_t)size.y * z);
        if (D) D[j] = b >= 0 ? p.D[src + 8 * r] : p.trunc;
        if (W) W[j] = b >= 0 ? p.W[src + 8 * r] : 0.0f;
    }
}

__global__ __launch_bounds__(256) void sparse_clear_kernel(unsigned long long* __restrict__ keys,
                                                           uint64_t n, unsigned* counters) {
    const uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) keys[i] = kEmptySlot;
    if (i < 2) counters[i] = 0u;
}

}  // namespace recon

using namespace recon;

struct recon_sparse {
    recon_tsdf_info info;
    recon_tsdf_config cfg;
    SparseParams p;
    void* mem = nullptr;  // one allocation: table, bricks, counters
    int num_cus = 256;
};

extern "C" int recon_sparse_create(const recon_tsdf_config* cfg, int64_t brick_capacity,
                                   recon_sparse** out) {
    clear_error();
    const char* fn = "recon_sparse_create";
    if (!out) return fail(RECON_ERR_NULL, "%s: out is NULL", fn);
    *out = nullptr;
    recon_tsdf_info info;
    int rc = describe(cfg, &info);
    if (rc) return rc;
    if (info.weight_type != RECON_WEIGHT_BY_DEPTH)
        return fail(RECON_ERR_CONFIG, "%s: sparse volumes integrate with WEIGHT_BY_DEPTH only", fn);
    if (brick_capacity < 1 || brick_capacity > (int64_t(1) << 24))
        return fail(RECON_ERR_RANGE, "%s: brick capacity %lld outside 1..2^24", fn,
                    (long long)brick_capacity);
    rc = require_gfx950();
    if (rc) return rc;
    uint64_t table = 1;
    while (table < 2 * (uint64_t)brick_capacity) table <<= 1;
    const size_t bytes_keys = 8 * table, bytes_vals = 4 * table;
    const size_t bytes_coords = 16 * (size_t)brick_capacity;
    const size_t bytes_vox = 4 * (size_t)kBrickVoxels * (size_t)brick_capacity;
    auto a256 = [](size_t b) { return (b + 255) / 256 * 256; };
    const size_t o_vals = a256(bytes_keys), o_coords = o_vals + a256(bytes_vals),
                 o_D = o_coords + a256(bytes_coords), o_W = o_D + a256(bytes_vox),
                 o_cnt = o_W + a256(bytes_vox), total = o_cnt + 256;
    recon_sparse* h = new recon_sparse();
    h->cfg = *cfg;
    h->info = info;
    if (hipMalloc(&h->mem, total) != hipSuccess) {
        delete h;
        return fail(RECON_ERR_DEVICE, "%s: cannot allocate %zu bytes", fn, total);
    }
    char* m = static_cast<char*>(h->mem);
    SparseParams& p = h->p;
    for (int k = 0; k < 3; ++k) {
        p.vs[k] = info.voxel_size[k];
        p.off[k] = info.global_offset[k];
    }
    p.fx = cfg->focal_x;
    p.fy = cfg->focal_y;
    p.cx = cfg->cx;
    p.cy = cfg->cy;
    p.trunc = info.truncation;
    p.maxw = cfg->max_weight;
    p.maxd = info.max_depth;
    p.capacity = brick_capacity;
    p.mask = table - 1;
    p.keys = reinterpret_cast<unsigned long long*>(m);
    p.vals = reinterpret_cast<int32_t*>(m + o_vals);
    p.coords = reinterpret_cast<int4*>(m + o_coords);
    p.D = reinterpret_cast<float*>(m + o_D);
    p.W = reinterpret_cast<float*>(m + o_W);
    for (int k = 0; k < 3; ++k) {
        p.blo[k] = -(1 << (kCoordBits - 1));
        p.bhi[k] = (1 << (kCoordBits - 1)) - 1;
    }
    p.counter = reinterpret_cast<unsigned*>(m + o_cnt);
    p.overflow = p.counter + 1;
    p.rfx = 1.0f / p.fx;
    p.rfy = 1.0f / p.fy;
    for (int k = 0; k < 3; ++k) p.rvs[k] = 1.0f / p.vs[k];
    int dev = 0;
    if (hipGetDevice(&dev) == hipSuccess) {
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, dev) == hipSuccess) h->num_cus = prop.multiProcessorCount;
    }
    hipLaunchKernelGGL(sparse_clear_kernel, dim3((unsigned)((table + 255) / 256)), dim3(256), 0,
                       nullptr, p.keys, table, p.counter);
    if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) {
        (void)hipFree(h->mem);
        delete h;
        return fail(RECON_ERR_DEVICE, "%s: clear failed", fn);
    }
    *out = h;
    return RECON_OK;
}

extern "C" void recon_sparse_destroy(recon_sparse* h) {
    if (!h) return;
    if (h->mem) (void)hipFree(h->mem);
    delete h;
}

extern "C" int recon_sparse_reset(recon_sparse* h, recon_stream_t stream) {
    clear_error();
    if (!h) return fail(RECON_ERR_NULL, "recon_sparse_reset: handle is NULL");
    const uint64_t table = h->p.mask + 1;
    hipLaunchKernelGGL(sparse_clear_kernel, dim3((unsigned)((table + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, h->p.keys, table, h->p.counter);
    RECON_HIP_TRY(hipGetLastError(), "sparse_clear_kernel launch");
    return RECON_OK;
}

extern "C" int recon_sparse_integrate(recon_sparse* h, const recon_depth_view* depth,
                                      const double camera_pose[7], recon_stream_t stream) {
    clear_error();
    const char* fn = "recon_sparse_integrate";
    if (!h) return fail(RECON_ERR_NULL, "%s: handle is NULL", fn);
    if (!depth || !depth->data) return fail(RECON_ERR_NULL, "%s: depth is NULL", fn);
    if (depth->rows <= 0 || depth->cols <= 0)
        return fail(RECON_ERR_SIZE, "%s: depth size %dx%d must be positive", fn, depth->cols,
                    depth->rows);
    if (depth->step < 4 * (size_t)depth->cols || depth->step % 4 != 0)
        return fail(RECON_ERR_SIZE, "%s: depth step %zu invalid", fn, depth->step);
    if ((depth->step / 4) * (size_t)depth->rows >= (size_t(1) << 31) || depth->rows >= (1 << 18))
        return fail(RECON_ERR_RANGE, "%s: depth image too large", fn);
    if (!camera_pose) return fail(RECON_ERR_NULL, "%s: pose is NULL", fn);
    if (!pose_is_finite(camera_pose)) return fail(RECON_ERR_CONFIG, "%s: non-finite pose", fn);
    hipStream_t s = (hipStream_t)stream;
    FrameParams F;
    pose_to_matrix_f32(camera_pose, F.R, F.t);
    F.depth = depth->data;
    F.pitch = (int32_t)(depth->step / 4);
    // the integrate kernel's short forms: as frame_planes, over |v| < 2^23
    double coord = 0.0, rabs = 0.0, tabs = 0.0;
    for (int k = 0; k < 3; ++k) {
        coord += 8388608.0 * h->p.vs[k] + std::fabs(h->p.off[k]);
        tabs += std::fabs(F.t[k]);
    }
    for (int k = 0; k < 9; ++k) rabs += std::fabs(F.R[k]);
    const bool easy = (rabs * coord + tabs) * ((double)h->p.fx + h->p.fy + 1.0) < kProductMax &&
                      std::fabs(h->p.cx) + std::fabs(h->p.cy) < 1e30 && h->p.trunc < kProductMax &&
                      F.pitch < (1 << 22) &&
                      depth->cols < (1 << 24) && 4.0 * (double)F.pitch * depth->rows < 4294967296.0;
    F.guard = easy ? 0.0f : INFINITY;
    const auto alloc = sparse_short_forms(h->p, F, depth->cols, depth->rows) ? sparse_alloc_kernel<true>
                                                                             : sparse_alloc_kernel<false>;
    hipLaunchKernelGGL(alloc, dim3((depth->cols + 31) / 32, (depth->rows + 7) / 8), dim3(256), 0, s, h->p, F,
                       depth->cols, depth->rows);
    RECON_HIP_TRY(hipGetLastError(), "sparse_alloc_kernel launch");
    hipLaunchKernelGGL(sparse_integrate_kernel, dim3((unsigned)(h->num_cus * 8)), dim3(256), 0, s,
                       h->p, F, (float)depth->cols, (float)depth->rows);
    RECON_HIP_TRY(hipGetLastError(), "sparse_integrate_kernel launch");
    return RECON_OK;
}

extern "C" int recon_sparse_allocate_box(recon_sparse* h, const int32_t lo[3], const int32_t hi[3],
                                         recon_stream_t stream) {
    clear_error();
    const char* fn = "recon_sparse_allocate_box";
    if (!h || !lo || !hi) return fail(RECON_ERR_NULL, "%s: null argument", fn);
    int b0[3], nb[3];
    int64_t total = 1;
    for (int k = 0; k < 3; ++k) {
        if (hi[k] <= lo[k]) return fail(RECON_ERR_SIZE, "%s: empty box", fn);
        if (lo[k] < -(1 << 23) || hi[k] > (1 << 23)) return fail(RECON_ERR_RANGE, "%s: box beyond 2^23", fn);
        const int a = lo[k] >= 0 ? lo[k] / 8 : -((-lo[k] + 7) / 8);
        const int hm = hi[k] - 1;
        const int b = hm >= 0 ? hm / 8 : -((-hm + 7) / 8);
        b0[k] = a;
        nb[k] = b - a + 1;
        total *= nb[k];
    }
    if (total > h->p.capacity)
        return fail(RECON_ERR_CAPACITY, "%s: %lld bricks exceed the capacity %lld", fn,
                    (long long)total, (long long)h->p.capacity);
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(sparse_alloc_box_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s,
                       h->p, make_int4(b0[0], b0[1], b0[2], 0), make_int4(nb[0], nb[1], nb[2], 0));
    RECON_HIP_TRY(hipGetLastError(), "sparse_alloc_box_kernel launch");
    hipLaunchKernelGGL(sparse_init_kernel, dim3((unsigned)(h->num_cus * 8)), dim3(256), 0, s, h->p);
    RECON_HIP_TRY(hipGetLastError(), "sparse_init_kernel launch");
    return RECON_OK;
}

extern "C" int recon_sparse_set_bounds(recon_sparse* h, const int32_t lo[3], const int32_t hi[3]) {
    clear_error();
    const char* fn = "recon_sparse_set_bounds";
    if (!h) return fail(RECON_ERR_NULL, "%s: handle is NULL", fn);
    for (int k = 0; k < 3; ++k) {
        if (!lo || !hi) {
            h->p.blo[k] = -(1 << (kCoordBits - 1));
            h->p.bhi[k] = (1 << (kCoordBits - 1)) - 1;
            continue;
        }
        if (hi[k] <= lo[k]) return fail(RECON_ERR_SIZE, "%s: empty box", fn);
        if (lo[k] < -(1 << 23) || hi[k] > (1 << 23)) return fail(RECON_ERR_RANGE, "%s: box beyond 2^23", fn);
    }
    if (lo && hi)
        for (int k = 0; k < 3; ++k) {
            h->p.blo[k] = lo[k] >= 0 ? lo[k] / 8 : -((-lo[k] + 7) / 8);
            const int hm = hi[k] - 1;
            h->p.bhi[k] = hm >= 0 ? hm / 8 : -((-hm + 7) / 8);
        }
    return RECON_OK;
}

extern "C" int recon_sparse_stats(recon_sparse* h, int64_t* num_bricks, uint32_t* overflow,
                                  recon_stream_t stream) {
    clear_error();
    if (!h) return fail(RECON_ERR_NULL, "recon_sparse_stats: handle is NULL");
    unsigned c[2] = {0, 0};
    hipStream_t s = (hipStream_t)stream;
    RECON_HIP_TRY(hipMemcpyAsync(c, h->p.counter, sizeof c, hipMemcpyDeviceToHost, s), "sparse stats");
    RECON_HIP_TRY(hipStreamSynchronize(s), "sparse stats synchronize");
    if (num_bricks) *num_bricks = std::min<int64_t>(c[0], h->p.capacity);
    if (overflow) *overflow = c[1];
    return RECON_OK;
}

extern "C" int recon_sparse_export(recon_sparse* h, const int32_t origin[3], const int32_t size[3],
                                   float* D, float* W, recon_stream_t stream) {
    clear_error();
    const char* fn = "recon_sparse_export";
    if (!h || !origin || !size) return fail(RECON_ERR_NULL, "%s: null argument", fn);
    if (!D && !W) return fail(RECON_ERR_NULL, "%s: no output", fn);
    int64_t total = 1;
    for (int k = 0; k < 3; ++k) {
        if (size[k] < 1) return fail(RECON_ERR_SIZE, "%s: size[%d] < 1", fn, k);
        if ((int64_t)origin[k] < -(1 << 23) || (int64_t)origin[k] + size[k] > (1 << 23))
            return fail(RECON_ERR_RANGE, "%s: box beyond 2^23", fn);
        total *= size[k];
    }
    if (total >= (int64_t(1) << 31)) return fail(RECON_ERR_RANGE, "%s: box too large", fn);
    int b0[3], nb[3];
    for (int k = 0; k < 3; ++k) {
        const int last = origin[k] + size[k] - 1;
        b0[k] = origin[k] >= 0 ? origin[k] / 8 : -((-origin[k] + 7) / 8);
        nb[k] = (last >= 0 ? last / 8 : -((-last + 7) / 8)) - b0[k] + 1;
    }
    const int64_t columns = (int64_t)((nb[0] + 3) / 4) * nb[1] * nb[2];
    hipLaunchKernelGGL(sparse_export_kernel, dim3((unsigned)((columns + 3) / 4)), dim3(256), 0,
                       (hipStream_t)stream, h->p, make_int4(origin[0], origin[1], origin[2], 0),
                       make_int4(size[0], size[1], size[2], 0), make_int4(b0[0], b0[1], b0[2], 0),
                       make_int4(nb[0], nb[1], nb[2], 0), D, W);
    RECON_HIP_TRY(hipGetLastError(), "sparse_export_kernel launch");
    return RECON_OK;
}

extern "C" int recon_sparse_download_bricks(recon_sparse* h, int32_t* coords, float* D, float* W,
                                            int64_t capacity, int64_t* num_bricks,
                                            recon_stream_t stream) {
    clear_error();
    const char* fn = "recon_sparse_download_bricks";
    if (!h || !num_bricks) return fail(RECON_ERR_NULL, "%s: null argument", fn);
    int64_t n = 0;
    int rc = recon_sparse_stats(h, &n, nullptr, stream);
    if (rc) return rc;
    *num_bricks = n;
    if (!coords && !D && !W) return RECON_OK;
    if (n > capacity) return fail(RECON_ERR_CAPACITY, "%s: %lld bricks do not fit", fn, (long long)n);
    hipStream_t s = (hipStream_t)stream;
    if (coords && n) {
        std::vector<int4> c((size_t)n);
        RECON_HIP_TRY(hipMemcpyAsync(c.data(), h->p.coords, 16 * (size_t)n, hipMemcpyDeviceToHost, s),
                      "brick coordinates");
        RECON_HIP_TRY(hipStreamSynchronize(s), "brick coordinates synchronize");
        for (int64_t i = 0; i < n; ++i) {
            coords[3 * i] = c[i].x;
            coords[3 * i + 1] = c[i].y;
            coords[3 * i + 2] = c[i].z;
        }
    }
    const size_t bytes = 4 * (size_t)kBrickVoxels * (size_t)n;
    if (D && n) RECON_HIP_TRY(hipMemcpyAsync(D, h->p.D, bytes, hipMemcpyDeviceToHost, s), "brick D");
    if (W && n) RECON_HIP_TRY(hipMemcpyAsync(W, h->p.W, bytes, hipMemcpyDeviceToHost, s), "brick W");
    RECON_HIP_TRY(hipStreamSynchronize(s), "brick download synchronize");
    return RECON_OK;
}
