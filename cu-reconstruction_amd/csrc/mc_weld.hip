// mc_weld.hip -- welded marching cubes for gfx950: shared vertices, per-vertex
// normals, and the soup's triangles as indices.
//
// No counterpart in the reference, whose generate_triangular_surface emits a
// soup (the per-triangle vert_remap of marching_cubes.cu:171-179 never shares
// a vertex).  Here one vertex per grid edge whose end values differ in sign
// (v < 0 against not), owned by its lower end voxel and numbered in the order
// (voxel x + gx*(y + gy*z), axis x, y, z); triangles are the soup's, in the
// soup's order (cube z, y, x, table slot).
//
// Numbering without a per-voxel table: the voxels of an x-row are cut into
// 64-voxel chunks; a 64-bit word holds a chunk's signs (v < 0), whose XORs
// with the next voxel's, the next row's and the next layer's are the masks of
// its sign-changing x, y and z edges, and an exclusive scan over the chunk
// totals gives each chunk's first vertex.  The index of edge (voxel, axis) is
//   base[chunk] + popc of the three masks below the voxel's lane
//               + the voxel's own set bits of the axes before `axis`,
// which the vertex writer and the triangle writer both evaluate: 16 B of
// signs and counts per 64 voxels.  The field is read whole once, by
// weld_sign_kernel; weld_count_kernel counts vertices and triangles from the
// signs, and after a scan of its block sums weld_write_kernel classifies the
// cubes from the signs again and reads the field at the vertices.
//
// Vertex: from the negative end N to the other end M, r = (-dN)/(dM - dN),
// p = sN + r*(sM - sN) per component.  This is the soup's own formula
// (marching_cubes.cu:23-51) whenever the soup orients the edge from N,
// i.e. except when dM is exactly +-0 and the cube lists M first (there the
// soup's bits already differ between the cubes sharing the edge).
// Normal: the TSDF gradient, central differences over (vs + vs) inside the
// grid and one-sided over vs on its border, lerped from N to M with r and
// normalised; (0,0,0) where the gradient vanishes.
#pragma clang fp contract(off)

#include "mc_device.hpp"

#include <algorithm>
#include <cmath>

namespace recon {

// A group is 16 consecutive chunks (of one voxel row or several): the unit of
// a wavefront in the count and write passes, lane 4i + q holding voxels and
// cubes 16q .. 16q+15 of chunk i.  kBlockGroups groups are a workgroup of the
// count pass; a chunk's first vertex is its block's plus its place in it.
constexpr int kGroupChunks = 16;
constexpr int kBlockGroups = 16, kBlockChunks = kBlockGroups * kGroupChunks;
// A unit of the write pass is up to kUnitRounds rounds of 64 elements of a
// group: its vertices first, then its triangles (<= 48 + 80 rounds, so <= 32
// units).  The list holds group << kUnitBits | unit (group < 2^31 / 16).
constexpr int kUnitRounds = 4, kUnitBits = 5;
static_assert((16 * 64 * 3 + 16 * 64 * 5) / 64 <= kUnitRounds << kUnitBits, "a group's units fit the bits");
constexpr int kSignChunks = 8;  // chunks per wavefront of the sign pass
constexpr int kWeldWaves = 4;   // wavefronts per workgroup of the other passes

struct WeldParams {
    McParams mc;
    int32_t cpr;      // 64-voxel chunks per x-row
    int32_t nchunks;  // cpr * gy * gz
    uint32_t mul_cpr, mul_gy;  // div31's of cpr and gy
    int32_t sh_cpr, sh_gy;
};

// n / d for n < 2^31: ceil(2^(31 + l) / d), l = ceil(log2 d), errs by less
// than 2^-31 of n / d, too little to reach the next whole number.
static void div31_make(uint32_t d, uint32_t& mul, int32_t& sh) {
    int l = 0;
    while ((1ull << l) < d) ++l;
    mul = (uint32_t)((((1ull << 31) << l) + d - 1) / d);
    sh = l;
}
__device__ __forceinline__ uint32_t div31(uint32_t n, uint32_t mul, int32_t sh) {
    return (uint32_t)(((uint64_t)n * mul) >> 31) >> sh;
}

// Bits 0 .. n-1 (none for n <= 0, all for n >= 64).
__device__ __forceinline__ unsigned long long low_bits(int n) {
    return n <= 0 ? 0ull : (n >= 64 ? ~0ull : (1ull << n) - 1ull);
}

// Masks of the sign-changing x, y, z edges owned by the voxels of chunk j of
// row (y, z), from its signs s and those after it (sn: the next chunk's), in
// the next row (sy) and in the next layer (sz); a neighbour past the grid may
// hold anything.
__device__ __forceinline__ void weld_edges(const McParams& p, int j, int y, int z, unsigned long long s,
                                           unsigned long long sn, unsigned long long sy,
                                           unsigned long long sz, unsigned long long m[3]) {
    const unsigned long long in = low_bits(p.gx - 64 * j);
    m[0] = (s ^ ((s >> 1) | (sn << 63))) & low_bits(p.gx - 1 - 64 * j);
    m[1] = y + 1 < p.gy ? (s ^ sy) & in : 0ull;
    m[2] = z + 1 < p.gz ? (s ^ sz) & in : 0ull;
}

// Signs of every chunk: eight chunks a wavefront, one 4-byte load a lane and
// chunk, all in flight together.  It is the one pass over the whole field:
// 250 x 333 x 287 voxels in 18 us, 5.3 TB/s.  A count kernel that read the
// field itself took ten loads per four voxel rows (each row two and a half
// times) and was bound by their addresses: 41 us, against 32 for this kernel
// and the count of the signs.
__global__ __launch_bounds__(256) void weld_sign_kernel(const WeldParams w,
                                                        unsigned long long* __restrict__ signs,
                                                        uint32_t* __restrict__ nunits) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *nunits = 0;  // for the count kernel
    const McParams& p = w.mc;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t c0 = kSignChunks * (blockIdx.x * kWeldWaves + (uint32_t)wave);
    if (c0 >= (uint32_t)w.nchunks) return;
    // lane k (of every eight): chunk c0 + k (the last one past the end), its
    // first voxel and the voxels after that in its row
    const uint32_t cl = min(c0 + (uint32_t)(lane & 7), (uint32_t)w.nchunks - 1u);
    const uint32_t row = div31(cl, w.mul_cpr, w.sh_cpr), j = cl - row * (uint32_t)w.cpr;
    const unsigned long long start = (unsigned long long)row * (uint32_t)p.gx + 64ull * j;
    const int lo = (int)(uint32_t)start, hi = (int)(uint32_t)(start >> 32), last = p.gx - 1 - 64 * (int)j;
    float v[kSignChunks];
#pragma unroll
    for (int k = 0; k < kSignChunks; ++k) {
        const unsigned long long s = ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane(hi, k) << 32) |
                                     (uint32_t)__builtin_amdgcn_readlane(lo, k);
        const float* base = p.f + s;
        v[k] = base[(uint32_t)min(lane, __builtin_amdgcn_readlane(last, k))];
    }
    unsigned long long out = 0;
#pragma unroll
    for (int k = 0; k < kSignChunks; ++k) {
        const unsigned long long b = __ballot(v[k] < 0.0f);
        out = lane == k ? b : out;
    }
    if (lane < kSignChunks && c0 + lane < (uint32_t)w.nchunks) signs[c0 + lane] = out;
}

// Chunk c's place: chunk j of voxel row (y, z).
struct ChunkPlace {
    int j, y, z;
};
__device__ __forceinline__ ChunkPlace chunk_place(const WeldParams& w, uint32_t c) {
    const uint32_t row = div31(c, w.mul_cpr, w.sh_cpr), z = div31(row, w.mul_gy, w.sh_gy);
    return {(int)(c - row * (uint32_t)w.cpr), (int)(row - z * (uint32_t)w.mc.gy), (int)z};
}

// Triangle counts of 16 cubes of a chunk from voxel x on, 4 bits each, from
// the signs q of their rows (y,z), (y,z+1), (y+1,z), (y+1,z+1), 17 voxels
// each; `in`: the cubes' rows are in the grid.  A cube's byte holds the rows'
// bits in this order (corner order 0, 1, 3, 2, 4, 5, 7, 6).
struct CubeCounts {
    uint32_t w[2];
};
__device__ __forceinline__ uint32_t cube_byte(const uint32_t q[4], int j) {
    return ((q[0] >> j) & 3u) | (((q[1] >> j) & 3u) << 2) | (((q[2] >> j) & 3u) << 4) |
           (((q[3] >> j) & 3u) << 6);
}
__device__ __forceinline__ CubeCounts cube_counts(const McParams& p, const uint8_t* ntab,
                                                  const uint32_t q[4], bool in, int x) {
    CubeCounts n = {{0u, 0u}};
#pragma unroll
    for (int j = 0; j < 16; ++j) n.w[j >> 3] |= (uint32_t)ntab[cube_byte(q, j)] << (4 * (j & 7));
    const int left = in ? min(max(p.gx - 1 - x, 0), 16) : 0;
    const unsigned long long keep = low_bits(4 * left);
    n.w[0] &= (uint32_t)keep;
    n.w[1] &= (uint32_t)(keep >> 32);
    return n;
}
// Sum of the low 8, 4 or 2 of the 4-bit counts in w.
__device__ __forceinline__ int sum8(uint32_t w) {
    const uint32_t b = (w & 0x0F0F0F0Fu) + ((w >> 4) & 0x0F0F0F0Fu);
    return (int)((b * 0x01010101u) >> 24);
}

// Counts: one wavefront a group.  Lane 16 rr + i reads the signs of chunk i
// in row (y + (rr >> 1), z + (rr & 1)); the edges follow from the words, the
// triangles from the table, 16 cubes a lane, where any cube of the group has
// both signs.  A workgroup appends its groups' units of work to the write
// pass's list, in any order between workgroups (what a unit writes and where
// does not depend on it).  14 us for 24 000 groups, two thirds of them without
// a negative value: latency, of the loads and of the workgroup's two steps.
__global__ __launch_bounds__(64 * kBlockGroups) void weld_count_kernel(
    const WeldParams w, const unsigned long long* __restrict__ signs, int32_t* __restrict__ voff,
    int32_t* __restrict__ toff, int2* __restrict__ group, long long* __restrict__ vsums,
    long long* __restrict__ tsums, bool want_v, bool want_t, uint32_t* __restrict__ units,
    uint32_t* __restrict__ nunits) {
    __shared__ uint8_t ntab[256];
    __shared__ unsigned long long sl[kBlockGroups][64];
    __shared__ uint8_t nl[kBlockGroups][64];
    __shared__ int vc[kBlockChunks], tc[kBlockChunks];
    __shared__ int wv[kBlockChunks / 64], wt[kBlockChunks / 64], gu[kBlockGroups];
    const McParams& p = w.mc;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t nchunks = (uint32_t)w.nchunks;
    const uint32_t c0 = kGroupChunks * (blockIdx.x * kBlockGroups + (uint32_t)wave);
    const int rr = lane >> 4;
    const uint32_t c = c0 + (lane & 15);
    const ChunkPlace at = chunk_place(w, c < nchunks ? c : nchunks - 1u);
    const bool here = (c < nchunks) & (at.y + (rr >> 1) < p.gy) & (at.z + (rr & 1) < p.gz);
    const size_t cc = (size_t)c + (rr >> 1 ? (size_t)w.cpr : 0) + (rr & 1 ? (size_t)w.cpr * p.gy : 0);
    unsigned long long s = 0, sn = 0;
    if (here) {
        s = signs[cc];
        if (at.j + 1 < w.cpr) sn = signs[cc + 1];
    }
    if (threadIdx.x < 256) ntab[threadIdx.x] = mc_ntab_qbyte((int)threadIdx.x);
    __syncthreads();
    int nv = 0;
    bool mixed = false;
    if (__ballot((s | sn) != 0ull)) {  // any negative value in reach
        const unsigned long long sz = __shfl_down(s, 16, 64), sy = __shfl_down(s, 32, 64);
        if (rr == 0 && here) {
            unsigned long long m[3];
            weld_edges(p, at.j, at.y, at.z, s, sn, sy, sz, m);
            nv = __popcll(m[0]) + __popcll(m[1]) + __popcll(m[2]);
        }
        // a cube has both signs where the eight words' AND and OR differ
        const unsigned long long sx = (s >> 1) | (sn << 63);
        unsigned long long all = s & sx, any = s | sx;
        all &= __shfl_xor(all, 16, 64);
        any |= __shfl_xor(any, 16, 64);
        all &= __shfl_xor(all, 32, 64);
        any |= __shfl_xor(any, 32, 64);
        const bool cubes = (c < nchunks) & (at.y + 1 < p.gy) & (at.z + 1 < p.gz);
        mixed = cubes & (((any & ~all) & low_bits(p.gx - 1 - 64 * at.j)) != 0);
    }
    if (rr == 0) vc[kGroupChunks * wave + lane] = nv;
    const int nvg = __builtin_amdgcn_readlane(wave_inclusive_scan(nv, lane), 63);
    int ntg = 0;
    if (__ballot(mixed)) {
        sl[wave][lane] = s;
        nl[wave][lane] = (uint8_t)(sn & 1ull);
        __builtin_amdgcn_wave_barrier();
        const int i = lane >> 2, b = 16 * (lane & 3);
        const ChunkPlace mine = chunk_place(w, min(c0 + (uint32_t)i, nchunks - 1u));
        uint32_t q[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            q[k] = (uint32_t)(sl[wave][16 * k + i] >> b);
            if (b == 48) q[k] |= (uint32_t)nl[wave][16 * k + i] << 16;
        }
        const bool in = (c0 + (uint32_t)i < nchunks) & (mine.y + 1 < p.gy) & (mine.z + 1 < p.gz);
        const CubeCounts n = cube_counts(p, ntab, q, in, 64 * mine.j + b);
        const int incl = wave_inclusive_scan(sum8(n.w[0]) + sum8(n.w[1]), lane);
        ntg = __builtin_amdgcn_readlane(incl, 63);
        const int before = __shfl(incl, 4 * (lane & 15) - 1, 64);  // lanes 0..15: chunk lane's
        const int upto = __shfl(incl, 4 * (lane & 15) + 3, 64);
        if (lane < 16) tc[kGroupChunks * wave + lane] = upto - (lane ? before : 0);
    } else if (lane < 16) {
        tc[kGroupChunks * wave + lane] = 0;
    }
    if (lane == 0) {
        const int rounds = (want_v ? (nvg + 63) / 64 : 0) + (want_t ? (ntg + 63) / 64 : 0);
        gu[wave] = (rounds + kUnitRounds - 1) / kUnitRounds;
        if (c0 < nchunks) group[c0 / kGroupChunks] = make_int2(nvg, ntg);
    }
    __syncthreads();
    if (wave == kBlockGroups - 1) {
        const int mine = lane < kBlockGroups ? gu[lane] : 0;
        const int incl = wave_inclusive_scan(mine, lane);
        const int all_units = __builtin_amdgcn_readlane(incl, 63);
        if (all_units) {
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(nunits, (uint32_t)all_units);
            base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base) + (uint32_t)(incl - mine);
            const uint32_t g = kBlockGroups * blockIdx.x + (uint32_t)lane;
            for (int k = 0; k < mine; ++k) units[base + k] = (g << kUnitBits) | (uint32_t)k;
        }
    }
    const bool scan = wave < kBlockChunks / 64;
    int v = 0, t = 0, iv = 0, it = 0;
    if (scan) {
        v = vc[threadIdx.x];
        t = tc[threadIdx.x];
        iv = wave_inclusive_scan(v, lane);
        it = wave_inclusive_scan(t, lane);
        if (lane == 63) {
            wv[wave] = iv;
            wt[wave] = it;
        }
    }
    __syncthreads();
    if (scan) {
        int bv = 0, bt = 0, av = 0, at_ = 0;
#pragma unroll
        for (int k = 0; k < kBlockChunks / 64; ++k) {
            bv += k < wave ? wv[k] : 0;
            bt += k < wave ? wt[k] : 0;
            av += wv[k];
            at_ += wt[k];
        }
        const uint32_t ct = kBlockChunks * blockIdx.x + threadIdx.x;
        if (ct < nchunks) {
            voff[ct] = bv + iv - v;
            toff[ct] = bt + it - t;
        }
        if (threadIdx.x == 0) {
            vsums[blockIdx.x] = av;
            tsums[blockIdx.x] = at_;
        }
    }
}

// Block sums to first indices in place, the totals to total[0] (vertices) and
// total[1] (triangles): a workgroup an array.
__global__ __launch_bounds__(256) void weld_scan_kernel(long long* __restrict__ vsums,
                                                        long long* __restrict__ tsums, int nb,
                                                        long long* __restrict__ total) {
    constexpr int kItems = 8;
    __shared__ long long sh[4];
    long long* __restrict__ sums = blockIdx.x ? tsums : vsums;
    long long carry = 0;
    for (int base = 0; base < nb; base += 256 * kItems) {
        const int i0 = base + (int)threadIdx.x * kItems;
        long long v[kItems], s = 0;
#pragma unroll
        for (int k = 0; k < kItems; ++k) {
            v[k] = i0 + k < nb ? sums[i0 + k] : 0;
            s += v[k];
        }
        long long all;
        long long e = carry + block_exclusive_scan(s, sh, &all);
#pragma unroll
        for (int k = 0; k < kItems; ++k) {
            if (i0 + k < nb) sums[i0 + k] = e;
            e += v[k];
        }
        carry += all;
    }
    if (threadIdx.x == 0) total[blockIdx.x] = carry;
}

// Gradient component `a` of the field at voxel (x, y, z).
__device__ __forceinline__ float weld_grad(const McParams& p, int x, int y, int z, int a) {
    const int64_t st = a == 0 ? 1 : (a == 1 ? (int64_t)p.gx : (int64_t)p.gx * p.gy);
    const int c = a == 0 ? x : (a == 1 ? y : z);
    const int g = a == 0 ? p.gx : (a == 1 ? p.gy : p.gz);
    const int64_t i = (int64_t)x + (int64_t)p.gx * (y + (int64_t)p.gy * z);
    if (c > 0 && c < g - 1) return (p.f[i + st] - p.f[i - st]) / (p.vs[a] + p.vs[a]);
    if (c == 0) return (p.f[i + st] - p.f[i]) / p.vs[a];
    return (p.f[i] - p.f[i - st]) / p.vs[a];
}

// Vertex (and normal) `idx` on the edge from voxel (x, y, z) along axis a, by
// the divisions.
__device__ __forceinline__ void weld_vertex_exact(const WeldParams& w, int x, int y, int z, int a,
                                                  long long idx, float* __restrict__ verts,
                                                  float* __restrict__ normals) {
    const McParams& p = w.mc;
    const int row = y + p.gy * z;
    const int q[3] = {x + (a == 0), y + (a == 1), z + (a == 2)};
    const int64_t i = (int64_t)x + (int64_t)p.gx * row;
    const int64_t j = (int64_t)q[0] + (int64_t)p.gx * (q[1] + (int64_t)p.gy * q[2]);
    const bool neg_first = p.f[i] < 0.0f;
    const int pn[3] = {neg_first ? x : q[0], neg_first ? y : q[1], neg_first ? z : q[2]};
    const int pm[3] = {neg_first ? q[0] : x, neg_first ? q[1] : y, neg_first ? q[2] : z};
    const float dn = neg_first ? p.f[i] : p.f[j];
    const float dm = neg_first ? p.f[j] : p.f[i];
    const float r = (-dn) / (dm - dn);
    if (verts) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float sn = voxel_centre(pn[k], p.vs[k], p.off[k]);
            const float sm = voxel_centre(pm[k], p.vs[k], p.off[k]);
            const float e = sm - sn;
            const float o = r * e;
            verts[3 * idx + k] = sn + o;
        }
    }
    if (normals) {
        float g[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float gn = weld_grad(p, pn[0], pn[1], pn[2], k);
            const float gm = weld_grad(p, pm[0], pm[1], pm[2], k);
            const float e = gm - gn;
            const float o = r * e;
            g[k] = gn + o;
        }
        const float len2 = (g[0] * g[0] + g[1] * g[1]) + g[2] * g[2];
        if (len2 > 0.0f) {
            const float len = sqrtf(len2);
#pragma unroll
            for (int k = 0; k < 3; ++k) normals[3 * idx + k] = g[k] / len;
        } else {
#pragma unroll
            for (int k = 0; k < 3; ++k) normals[3 * idx + k] = 0.0f;
        }
    }
}

// num / den by y = RN(1/den) and div_by_rcp; `bad` is set where that might not
// be the division's bits (a quotient near the denormals or out of range, -0).
__device__ __forceinline__ float weld_quotient(float num, float den, float y, bool& bad) {
    const float an = fabsf(num);
    bad |= !((an >= 1e-30f) & (an <= 1e30f)) & (__float_as_uint(num) != 0u);
    return div_by_rcp(num, den, y);
}

// 1/vs and 1/(vs + vs) per axis, and whether weld_quotient covers them.
struct WeldSteps {
    float r1[3], r2[3];
    bool ok;
};

// Every lane with `on` writes vertex (and normal) `idx` of edge (x, y, z, a):
// weld_vertex_exact's bits.
__device__ __forceinline__ void weld_vertex(const WeldParams& w, const WeldSteps& st, bool on, int x, int y,
                                            int z, int a, long long idx, float* __restrict__ verts,
                                            float* __restrict__ normals) {
    const McParams& p = w.mc;
    bool bad = !st.ok;
    float pos[3] = {0.0f, 0.0f, 0.0f}, nrm[3] = {0.0f, 0.0f, 0.0f};
    if (on) {
        const int64_t sx[3] = {1, (int64_t)p.gx, (int64_t)p.gx * p.gy};
        const int c[3] = {x, y, z}, g[3] = {p.gx, p.gy, p.gz};
        const int64_t i = (int64_t)x + sx[1] * y + sx[2] * z;
        const int64_t sa = a == 0 ? sx[0] : (a == 1 ? sx[1] : sx[2]);
        const float fi = p.f[i], fj = p.f[i + sa];
        const bool first = fi < 0.0f;  // the negative end is (x, y, z)
        const float dn = first ? fi : fj, dm = first ? fj : fi;
        const float den = dm - dn;
        float res = 0.0f;
        const float y_den = recip_sum(den, res);
        bad |= !(res < kRecipBad) | !(fabsf(den) <= 1e7f);
        const float r = weld_quotient(-dn, den, y_den, bad);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float s0 = voxel_centre(c[k], p.vs[k], p.off[k]);
            const float s1 = voxel_centre(c[k] + (k == a ? 1 : 0), p.vs[k], p.off[k]);
            const float sn = first ? s0 : s1, sm = first ? s1 : s0;
            const float e = sm - sn;
            const float o = r * e;
            pos[k] = sn + o;
        }
        if (normals) {
            float gr[3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                float ge[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) {  // the lower end, then the upper
                    const int ck = c[k] + (q && k == a ? 1 : 0);
                    const int64_t iq = i + (q ? sa : 0);
                    // central differences inside, one-sided on the border
                    const bool lo = ck > 0, hi = ck < g[k] - 1;
                    const float num = p.f[hi ? iq + sx[k] : iq] - p.f[lo ? iq - sx[k] : iq];
                    const bool both = lo & hi;
                    ge[q] = weld_quotient(num, both ? p.vs[k] + p.vs[k] : p.vs[k],
                                          both ? st.r2[k] : st.r1[k], bad);
                }
                const float gn = first ? ge[0] : ge[1], gm = first ? ge[1] : ge[0];
                const float e = gm - gn;
                const float o = r * e;
                gr[k] = gn + o;
            }
            const float len2 = (gr[0] * gr[0] + gr[1] * gr[1]) + gr[2] * gr[2];
            if (len2 > 0.0f) {
                bad |= !((len2 >= 1e-30f) & (len2 <= 1e12f));
                const float len = sqrtf(len2);
                float rl = 0.0f;
                const float y_len = recip_sum(len, rl);
#pragma unroll
                for (int k = 0; k < 3; ++k) nrm[k] = weld_quotient(gr[k], len, y_len, bad);
            } else {
                bad |= !(len2 == 0.0f);
            }
        }
        if (__builtin_expect(bad, 0)) {
            weld_vertex_exact(w, x, y, z, a, idx, verts, normals);
        } else {
            if (verts) {
#pragma unroll
                for (int k = 0; k < 3; ++k) verts[3 * idx + k] = pos[k];
            }
            if (normals) {
#pragma unroll
                for (int k = 0; k < 3; ++k) normals[3 * idx + k] = nrm[k];
            }
        }
    }
}

// A group's neighbourhood in LDS, for the four rows (y + dy, z + dz) that its
// cubes reach: entry 17 (2 dy + dz) + i is chunk i's (16: the next one's) word
// of signs, edge masks and first vertex.
constexpr int kGroupEntries = kGroupChunks + 1;
struct WeldGroup {
    unsigned long long s[4 * kGroupEntries];
    unsigned long long m[4 * kGroupEntries][3];
    uint32_t base[4 * kGroupEntries];
    int x[kGroupChunks], y[kGroupChunks], z[kGroupChunks];
    int mark[64];
};

// The lane whose elements include element k0 + lane of the lanes' elements
// (first element excl, count n per lane; k0 below their total): marks at the
// first elements, a max-scan, and the lane that element k0 is in before the
// first mark.  Every lane calls.
__device__ __forceinline__ int weld_owner(int* mark, int excl, int n, int k0, int lane) {
    mark[lane] = 0;
    if (n > 0 && excl >= k0 && excl < k0 + 64) mark[excl - k0] = lane + 1;
    __builtin_amdgcn_wave_barrier();
    const int mx = wave_inclusive_max(mark[lane]);
    const int first = 63 - __builtin_clzll(__ballot(n > 0 && excl <= k0) | 1ull);
    __builtin_amdgcn_wave_barrier();
    return mx > 0 ? mx - 1 : first;
}

// Vertex index of the local edge of table word et (axis, lower end's dx, dy,
// dz) of the cube at voxel place xl of the group's chunks.
__device__ __forceinline__ int32_t weld_index(const WeldGroup& nb, int xl, unsigned et) {
    const int a = (int)(et & 3u), X = xl + (int)((et >> 2) & 1u), l = X & 63;
    const int n = kGroupEntries * (int)(et >> 3) + (X >> 6);
    const unsigned long long below = (1ull << l) - 1ull;
    const unsigned long long m0 = nb.m[n][0], m1 = nb.m[n][1], m2 = nb.m[n][2];
    int idx = (int)nb.base[n] + __popcll(m0 & below) + __popcll(m1 & below) + __popcll(m2 & below);
    idx += a > 0 ? (int)((m0 >> l) & 1ull) : 0;
    idx += a > 1 ? (int)((m1 >> l) & 1ull) : 0;
    return idx;
}

// Entry of chunk c (place at; of the grid) in row rr of the neighbourhood.
__device__ __forceinline__ void weld_entry_load(const WeldParams& w, uint32_t c, const ChunkPlace& at, int rr,
                                                const unsigned long long* __restrict__ signs,
                                                const int32_t* __restrict__ voff,
                                                const long long* __restrict__ vsums, bool in,
                                                WeldGroup& nb, int entry) {
    const McParams& p = w.mc;
    const int Y = at.y + (rr >> 1), Z = at.z + (rr & 1);
    unsigned long long s = 0, m[3] = {0, 0, 0};
    uint32_t base = 0;
    if (in & (Y < p.gy) & (Z < p.gz)) {
        const size_t cc = (size_t)c + (rr >> 1 ? (size_t)w.cpr : 0) + (rr & 1 ? (size_t)w.cpr * p.gy : 0);
        s = signs[cc];
        const unsigned long long sn = at.j + 1 < w.cpr ? signs[cc + 1] : 0ull;
        const unsigned long long sy = Y + 1 < p.gy ? signs[cc + w.cpr] : 0ull;
        const unsigned long long sz = Z + 1 < p.gz ? signs[cc + (size_t)w.cpr * p.gy] : 0ull;
        weld_edges(p, at.j, Y, Z, s, sn, sy, sz, m);
        base = (uint32_t)vsums[cc / kBlockChunks] + (uint32_t)voff[cc];
    }
    nb.s[entry] = s;
    nb.m[entry][0] = m[0];
    nb.m[entry][1] = m[1];
    nb.m[entry][2] = m[2];
    nb.base[entry] = base;
}

// Elements [first, first + 64 kUnitRounds) of the group of chunks from c0 on:
// its nv vertices rounded up to whole rounds, then its nt triangles.
__device__ __forceinline__ void weld_write_unit(
    const WeldParams& w, const WeldSteps& st, uint32_t c0, int lane, int first, int nv, int nt,
    const unsigned long long* __restrict__ signs, const int32_t* __restrict__ voff,
    const int32_t* __restrict__ toff, const long long* __restrict__ vsums,
    const long long* __restrict__ tsums, WeldGroup& nb, const uint64_t* tri, const uint8_t* ntab,
    const uint32_t* edges, float* __restrict__ verts, float* __restrict__ normals,
    int32_t* __restrict__ tris) {
    const McParams& p = w.mc;
    const uint32_t nchunks = (uint32_t)w.nchunks;
    {
        const uint32_t c = c0 + (lane & 15);
        const ChunkPlace at = chunk_place(w, min(c, nchunks - 1u));
        weld_entry_load(w, c, at, lane >> 4, signs, voff, vsums, c < nchunks, nb,
                        kGroupEntries * (lane >> 4) + (lane & 15));
        if (lane < kGroupChunks) {
            nb.x[lane] = 64 * at.j;
            nb.y[lane] = at.y;
            nb.z[lane] = at.z;
        }
    }
    const uint32_t cn = c0 + kGroupChunks;  // the next chunk, where it goes on with the row
    if (cn < nchunks && cn % (uint32_t)w.cpr) {
        const ChunkPlace at = chunk_place(w, cn);
        if (lane < 4)
            weld_entry_load(w, cn, at, lane, signs, voff, vsums, true, nb,
                            kGroupEntries * lane + kGroupChunks);
    }
    __builtin_amdgcn_wave_barrier();
    const int i = lane >> 2, b = 16 * (lane & 3);
    // rounds [first, first + kUnitRounds) of the vertices' and then the
    // triangles'
    const int nv64 = (nv + 63) & ~63, end = first + 64 * kUnitRounds;
    if (first < nv64) {
        const uint32_t own01 = (uint32_t)((nb.m[i][0] >> b) & 0xFFFFull) |
                               ((uint32_t)((nb.m[i][1] >> b) & 0xFFFFull) << 16);
        const uint32_t own2 = (uint32_t)((nb.m[i][2] >> b) & 0xFFFFull);
        const int mine = __popc(own01) + __popc(own2);
        const int excl = wave_inclusive_scan(mine, lane) - mine;
        const long long v0 = (long long)nb.base[0];
        for (int k0 = first; k0 < min(end, nv); k0 += 64) {
            const int owner = weld_owner(nb.mark, excl, mine, k0, lane);
            uint32_t o01 = (uint32_t)__shfl((int)own01, owner, 64), o2 = (uint32_t)__shfl((int)own2, owner, 64);
            int r = k0 + lane - __shfl(excl, owner, 64), v = 0;
            // edge r of the 16 voxels', in the order voxel, axis: halve the
            // voxels (bits shifted in from o01's upper half stay above the
            // bits that are left to look at)
#pragma unroll
            for (int h = 8; h >= 1; h >>= 1) {
                const uint32_t msk = (1u << h) - 1u;
                const int c = __popc(o01 & (msk | (msk << 16))) + __popc(o2 & msk);
                const bool up = r >= c;
                r -= up ? c : 0;
                v += up ? h : 0;
                o01 >>= up ? h : 0;
                o2 >>= up ? h : 0;
            }
            const bool ex = o01 & 1u, ey = (o01 >> 16) & 1u;
            const int a = r == 0 ? (ex ? 0 : (ey ? 1 : 2)) : (r == 1 && ex && ey ? 1 : 2);
            const int oi = owner >> 2;
            weld_vertex(w, st, k0 + lane < nv, nb.x[oi] + 16 * (owner & 3) + v, nb.y[oi], nb.z[oi], a,
                        v0 + k0 + lane, verts, normals);
        }
    }
    if (end <= nv64) return;
    uint32_t q[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        q[k] = (uint32_t)(nb.s[kGroupEntries * k + i] >> b) & 0x1FFFFu;
        // the next chunk's first voxel (of another row past the last: no cube)
        if (b == 48) q[k] |= ((uint32_t)nb.s[kGroupEntries * k + i + 1] & 1u) << 16;
    }
    const bool in = (c0 + (uint32_t)i < nchunks) & (nb.y[i] + 1 < p.gy) & (nb.z[i] + 1 < p.gz);
    const CubeCounts cn4 = cube_counts(p, ntab, q, in, nb.x[i] + b);
    const int mine = sum8(cn4.w[0]) + sum8(cn4.w[1]);
    const int excl = wave_inclusive_scan(mine, lane) - mine;
    const long long t0 = tsums[c0 / kBlockChunks] + toff[c0];
    for (int k0 = max(first - nv64, 0); k0 < min(end - nv64, nt); k0 += 64) {
        const int owner = weld_owner(nb.mark, excl, mine, k0, lane);
        const uint32_t w0 = (uint32_t)__shfl((int)cn4.w[0], owner, 64);
        const uint32_t w1 = (uint32_t)__shfl((int)cn4.w[1], owner, 64);
        uint32_t oq[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) oq[k] = (uint32_t)__shfl((int)q[k], owner, 64);
        int r = k0 + lane - __shfl(excl, owner, 64);
        // triangle r of the 16 cubes': halve the cubes
        int j = 0;
        const int c8 = sum8(w0);
        uint32_t left = r >= c8 ? w1 : w0;
        j += r >= c8 ? 8 : 0;
        r -= r >= c8 ? c8 : 0;
#pragma unroll
        for (int h = 4; h >= 1; h >>= 1) {
            const int c = sum8(left & ((1u << (4 * h)) - 1u));
            const bool up = r >= c;
            r -= up ? c : 0;
            j += up ? h : 0;
            left >>= up ? 4 * h : 0;
        }
        if (k0 + lane < nt) {
            const uint64_t word = tri[cube_byte(oq, j)] >> (4 + 12 * r);
            const long long t = t0 + k0 + lane;
#pragma unroll
            for (int e = 0; e < 3; ++e)
                tris[3 * t + e] = weld_index(nb, 64 * (owner >> 2) + 16 * (owner & 3) + j,
                                             edges[(word >> (4 * e)) & 0xFull]);
        }
    }
}

// The units of the list, strided over as many wavefronts as are resident: a
// unit's vertices, then its triangles, are spread over the lanes 64 at a time.
// The pass is bound by instruction issue and by its longest wavefront: lanes
// without work and groups that a surface runs along (48 rounds) are its cost.
// 250 x 333 x 287 voxels with 0.6 M vertices: chunk by chunk, with the field's
// corners read again for the classes, 106 us (ten vertices a round); in units
// of four chunks 59; a group a wavefront 52; units 34.
// Nothing is written when the totals (from the scan) exceed int32 indices or
// a requested output's capacity: the host reports that after the call.
constexpr int kWriteBlocks = 256 * 8;  // 8 workgroups a CU by registers
__global__ __launch_bounds__(64 * kWeldWaves) void weld_write_kernel(
    const WeldParams w, const unsigned long long* __restrict__ signs, const int32_t* __restrict__ voff,
    const int32_t* __restrict__ toff, const int2* __restrict__ group, const long long* __restrict__ vsums,
    const long long* __restrict__ tsums, const long long* __restrict__ total,
    const uint32_t* __restrict__ units, const uint32_t* __restrict__ nunits, long long vcap,
    long long tcap, float* __restrict__ verts, float* __restrict__ normals, int32_t* __restrict__ tris) {
    __shared__ WeldGroup groups[kWeldWaves];
    __shared__ uint64_t tri[256];    // triangle table by the signs' byte
    __shared__ uint8_t ntab[256];    // its triangle counts
    __shared__ uint32_t edges[16];   // axis | dx << 2 | (2 dy + dz) << 3 of an edge's lower end
    const McParams& p = w.mc;
    const bool want_v = verts || normals, want_t = tris != nullptr;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t nu = *nunits;
    const long long nvt = total[0], ntt = total[1];
    if (kWeldWaves * blockIdx.x >= nu || nvt > INT32_MAX || (want_v && nvt > vcap) || (want_t && ntt > tcap))
        return;
    tri[threadIdx.x] = c_tri[qbyte_class((int)threadIdx.x)];
    ntab[threadIdx.x] = mc_ntab_qbyte((int)threadIdx.x);
    if (threadIdx.x < 12) {
        // corner offsets packed as bits: dx = bit0, dy = bit1, dz = bit2
        // (0:000 1:001 2:101 3:100 4:010 5:011 6:111 7:110)
        constexpr unsigned k_off = (0u << 0) | (1u << 3) | (5u << 6) | (4u << 9) | (2u << 12) |
                                   (3u << 15) | (7u << 18) | (6u << 21);
        const int e = (int)threadIdx.x;
        const int ca = (int)((kEdgeA >> (4 * e)) & 0xFull), cb = (int)((kEdgeB >> (4 * e)) & 0xFull);
        const unsigned oa = (k_off >> (3 * ca)) & 7u, ob = (k_off >> (3 * cb)) & 7u;
        const unsigned lo = oa & ob;
        edges[e] = (unsigned)__builtin_ctz(oa ^ ob) | ((lo & 1u) << 2) | (((lo & 2u) | (lo >> 2)) << 3);
    }
    __syncthreads();
    WeldSteps st;
    st.ok = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float bad = 0.0f;
        st.r1[k] = recip_sum(p.vs[k], bad);
        st.r2[k] = recip_sum(p.vs[k] + p.vs[k], bad);
        st.ok = st.ok && bad < kRecipBad && p.vs[k] >= 1e-6f && p.vs[k] <= 1e6f;
    }
    for (uint32_t u = kWeldWaves * blockIdx.x + (uint32_t)wave; u < nu; u += kWeldWaves * gridDim.x) {
        const uint32_t unit = (uint32_t)__builtin_amdgcn_readfirstlane((int)units[u]);
        const uint32_t g = unit >> kUnitBits;
        const int2 n = group[g];
        weld_write_unit(w, st, g * kGroupChunks, lane,
                        64 * kUnitRounds * (int)(unit & ((1u << kUnitBits) - 1u)), want_v ? n.x : 0,
                        want_t ? n.y : 0, signs, voff, toff, vsums, tsums, groups[wave], tri, ntab, edges,
                        verts, normals, tris);
        __builtin_amdgcn_wave_barrier();
    }
}

static size_t align256(size_t b) { return (b + 255) / 256 * 256; }

// Counts (always), then writes what is asked for when it fits.
static int weld_run(const float* field, const int32_t grid[3], const float vs[3], const float off[3],
                    float* verts, float* normals, int64_t vcap, int32_t* tris, int64_t tcap,
                    int64_t* nv_out, int64_t* nt_out, void** scratch, size_t* scratch_bytes,
                    hipStream_t s, const char* fn) {
    *nv_out = 0;
    *nt_out = 0;
    if (grid[0] < 2 || grid[1] < 2 || grid[2] < 2) return RECON_OK;
    WeldParams w;
    McParams& p = w.mc;
    p.f = field;
    p.gx = grid[0];
    p.gy = grid[1];
    p.gz = grid[2];
    p.cx = grid[0] - 1;
    p.cyr = grid[1] - 1;
    p.rows = (grid[1] - 1) * (grid[2] - 1);
    for (int i = 0; i < 3; ++i) {
        p.vs[i] = vs[i];
        p.off[i] = off[i];
    }
    w.cpr = (grid[0] + 63) / 64;
    w.nchunks = w.cpr * grid[1] * grid[2];
    div31_make((uint32_t)w.cpr, w.mul_cpr, w.sh_cpr);
    div31_make((uint32_t)grid[1], w.mul_gy, w.sh_gy);
    const int nb = (w.nchunks + kBlockChunks - 1) / kBlockChunks;
    const size_t o_signs = 0;
    const size_t o_voff = o_signs + align256(8 * (size_t)w.nchunks);
    const size_t o_toff = o_voff + align256(4 * (size_t)w.nchunks);
    const size_t o_group = o_toff + align256(4 * (size_t)w.nchunks);
    const size_t o_vsums = o_group + align256(8 * (size_t)nb * kBlockGroups);
    const size_t o_tsums = o_vsums + align256(8 * (size_t)nb);
    const size_t o_total = o_tsums + align256(8 * (size_t)nb);
    const size_t o_nunits = o_total + 256;
    const size_t o_units = o_nunits + 256;
    const size_t need = o_units + align256((sizeof(uint32_t) << kUnitBits) * nb * kBlockGroups);
    if (*scratch_bytes < need) {
        if (*scratch) (void)hipFree(*scratch);
        *scratch = nullptr;
        *scratch_bytes = 0;
        RECON_HIP_TRY(hipMalloc(scratch, need), "welded marching cubes scratch");
        *scratch_bytes = need;
    }
    char* sb = static_cast<char*>(*scratch);
    auto* signs = reinterpret_cast<unsigned long long*>(sb + o_signs);
    auto* voff = reinterpret_cast<int32_t*>(sb + o_voff);
    auto* toff = reinterpret_cast<int32_t*>(sb + o_toff);
    auto* group = reinterpret_cast<int2*>(sb + o_group);
    auto* vsums = reinterpret_cast<long long*>(sb + o_vsums);
    auto* tsums = reinterpret_cast<long long*>(sb + o_tsums);
    auto* total = reinterpret_cast<long long*>(sb + o_total);
    auto* nunits = reinterpret_cast<uint32_t*>(sb + o_nunits);
    auto* units = reinterpret_cast<uint32_t*>(sb + o_units);
    const bool write = verts || normals || tris;
    constexpr int kSignBlock = kSignChunks * kWeldWaves;
    hipLaunchKernelGGL(weld_sign_kernel, dim3((w.nchunks + kSignBlock - 1) / kSignBlock),
                       dim3(64 * kWeldWaves), 0, s, w, signs, nunits);
    RECON_HIP_TRY(hipGetLastError(), "weld_sign_kernel launch");
    hipLaunchKernelGGL(weld_count_kernel, dim3(nb), dim3(64 * kBlockGroups), 0, s, w, signs, voff, toff,
                       group, vsums, tsums, verts || normals, tris != nullptr, units, nunits);
    RECON_HIP_TRY(hipGetLastError(), "weld_count_kernel launch");
    hipLaunchKernelGGL(weld_scan_kernel, dim3(2), dim3(256), 0, s, vsums, tsums, nb, total);
    RECON_HIP_TRY(hipGetLastError(), "weld_scan_kernel launch");
    // The write pass checks the totals on the device, so it is queued before
    // the host waits; the copy of the totals to pageable memory comes last,
    // since it returns only when the stream has reached it.
    if (write) {
        // most groups are empty and a busy one is one or two units
        const int blocks = std::min(kWriteBlocks, nb * kBlockGroups);
        hipLaunchKernelGGL(weld_write_kernel, dim3(blocks), dim3(64 * kWeldWaves), 0, s, w, signs, voff,
                           toff, group, vsums, tsums, total, units, nunits, (long long)vcap,
                           (long long)tcap, verts, normals, tris);
        RECON_HIP_TRY(hipGetLastError(), "weld_write_kernel launch");
    }
    long long totals[2] = {0, 0};
    RECON_HIP_TRY(hipMemcpyAsync(totals, total, 16, hipMemcpyDeviceToHost, s), "totals");
    RECON_HIP_TRY(hipStreamSynchronize(s), "welded marching cubes");
    *nv_out = totals[0];
    *nt_out = totals[1];
    if (!write) return RECON_OK;
    if (totals[0] > INT32_MAX)
        return fail(RECON_ERR_RANGE, "%s: %lld vertices exceed int32 indices", fn, totals[0]);
    if ((verts || normals) && totals[0] > vcap)
        return fail(RECON_ERR_CAPACITY, "%s: %lld vertices do not fit capacity %lld", fn, totals[0],
                    (long long)vcap);
    if (tris && totals[1] > tcap)
        return fail(RECON_ERR_CAPACITY, "%s: %lld triangles do not fit capacity %lld", fn, totals[1],
                    (long long)tcap);
    return RECON_OK;
}

static int weld_entry(const float* field, const int32_t grid[3], const float vs[3],
                      const float off[3], float* verts, float* normals, int64_t vcap,
                      int32_t* tris, int64_t tcap, int64_t* nv, int64_t* nt, void** scratch,
                      size_t* scratch_bytes, hipStream_t s, const char* fn) {
    if (!nv || !nt) return fail(RECON_ERR_NULL, "%s: count output is NULL", fn);
    *nv = 0;
    *nt = 0;
    if (!field || !grid || !vs || !off) return fail(RECON_ERR_NULL, "%s: null argument", fn);
    int64_t n = 1;
    for (int i = 0; i < 3; ++i) {
        if (grid[i] < 1) return fail(RECON_ERR_SIZE, "%s: grid[%d] = %d must be >= 1", fn, i, grid[i]);
        n *= grid[i];
    }
    if (n >= (int64_t(1) << 31)) return fail(RECON_ERR_RANGE, "%s: grid exceeds 2^31-1 voxels", fn);
    if (vcap < 0 || tcap < 0) return fail(RECON_ERR_SIZE, "%s: negative capacity", fn);
    const int rc = require_gfx950();
    if (rc) return rc;
    return weld_run(field, grid, vs, off, verts, normals, vcap, tris, tcap, nv, nt, scratch,
                    scratch_bytes, s, fn);
}

}  // namespace recon

using namespace recon;

extern "C" int recon_mc_extract_welded(const float* field, const int32_t grid[3],
                                       const float voxel_size[3], const float offset[3],
                                       float* vertices, float* normals, int64_t vertex_capacity,
                                       int32_t* triangles, int64_t triangle_capacity,
                                       int64_t* num_vertices, int64_t* num_triangles,
                                       recon_stream_t stream) {
    clear_error();
    void* scratch = nullptr;
    size_t bytes = 0;
    const int rc = weld_entry(field, grid, voxel_size, offset, vertices, normals, vertex_capacity,
                              triangles, triangle_capacity, num_vertices, num_triangles, &scratch,
                              &bytes, (hipStream_t)stream, "recon_mc_extract_welded");
    if (scratch) (void)hipFree(scratch);
    return rc;
}

extern "C" int recon_tsdf_extract_welded_mesh(recon_tsdf* h, float* vertices, float* normals,
                                              int64_t vertex_capacity, int32_t* triangles,
                                              int64_t triangle_capacity, int64_t* num_vertices,
                                              int64_t* num_triangles, recon_stream_t stream) {
    clear_error();
    const char* fn = "recon_tsdf_extract_welded_mesh";
    if (!h) {
        if (num_vertices) *num_vertices = 0;
        if (num_triangles) *num_triangles = 0;
        return fail(RECON_ERR_NULL, "%s: handle is NULL", fn);
    }
    return weld_entry(h->D, h->info.grid, h->info.voxel_size, h->info.global_offset, vertices,
                      normals, vertex_capacity, triangles, triangle_capacity, num_vertices,
                      num_triangles, &h->mc_scratch, &h->mc_scratch_bytes, (hipStream_t)stream, fn);
}
