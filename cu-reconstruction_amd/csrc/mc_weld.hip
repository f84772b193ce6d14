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
// which the vertex writer and the triangle writer both evaluate: 32 B of
// signs, counts and bases per 64 voxels.  The field is read whole once, by
// weld_count_kernel (signs, vertex and triangle counts); after two exclusive
// scans weld_write_kernel classifies cubes from the signs alone and reads the
// field at the vertices.
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

#include <cmath>

namespace recon {

constexpr int kWeldWaves = 4;  // one wavefront per voxel row, 256 threads

struct WeldParams {
    McParams mc;
    int32_t cpr;      // 64-voxel chunks per x-row
    int32_t nchunks;  // cpr * gy * gz
};

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

// Count pass: one wavefront per four voxel rows (y..y+3, z), streaming the
// ten voxel rows (y+i, z) and (y+i, z+1), i = 0..4, 64 voxels a step (the
// marching-cubes count's walk): each voxel's sign bit (v < 0) for the ten
// rows packs into one word, bit 2j the lane's voxel of row j and bit 2j+1
// the next lane's (a DPP wave shift; lane 63 takes the next step's lane 0).
// A row's sign word is a ballot of its bit; the cube byte of cube row i is
// bits 4i .. 4i+7 (corner order 0, 1, 3, 2, 4, 5, 7, 6, the count table
// mc_ntab_qbyte); lane i of the wave stores row i's signs and counts.
// Loads past a row's end read its last voxel, and rows past the grid (y+i
// >= gy, z+1 >= gz) read the last row (in bounds); their edges and cubes
// do not count.
constexpr int kWeldRows = 4;
constexpr int kWeldLoadRows = 2 * (kWeldRows + 1);

__global__ __launch_bounds__(256) void weld_count_kernel(const WeldParams w,
                                                         unsigned long long* __restrict__ signs,
                                                         int32_t* __restrict__ vcount,
                                                         int32_t* __restrict__ tcount) {
    __shared__ uint8_t ntab[256];
    ntab[threadIdx.x] = mc_ntab_qbyte((int)threadIdx.x);
    __syncthreads();
    const McParams& p = w.mc;
    const int lane = threadIdx.x & 63;
    const int gpl = (p.gy + kWeldRows - 1) / kWeldRows;
    const int q = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWeldWaves + (threadIdx.x >> 6)));
    const int z = q / gpl, y = kWeldRows * (q - z * gpl);
    if (z >= p.gz) return;
    const int k = min(kWeldRows, p.gy - y);         // voxel rows of the wave
    const int z1 = min(z + 1, p.gz - 1);
    const bool zin = z + 1 < p.gz;
    const char* rowp[kWeldLoadRows];
#pragma unroll
    for (int i = 0; i <= kWeldRows; ++i) {
        const int yy = min(y + i, p.gy - 1);
        rowp[2 * i] = reinterpret_cast<const char*>(p.f + (size_t)p.gx * ((size_t)yy + (size_t)p.gy * z));
        rowp[2 * i + 1] =
            reinterpret_cast<const char*>(p.f + (size_t)p.gx * ((size_t)yy + (size_t)p.gy * z1));
    }
    const uint32_t xlast = (uint32_t)(p.gx - 1);
    auto load = [&](int chunk, float v[kWeldLoadRows]) {
        const uint32_t off = min((uint32_t)(64 * chunk + lane), xlast) << 2;
#pragma unroll
        for (int j = 0; j < kWeldLoadRows; ++j) v[j] = *reinterpret_cast<const float*>(rowp[j] + off);
    };
    auto sign_bits = [&](const float v[kWeldLoadRows]) {
        uint32_t m = 0;
#pragma unroll
        for (int j = 0; j < kWeldLoadRows; ++j) m |= (v[j] < 0.0f ? 1u : 0u) << (2 * j);
        return m;
    };
    const int cpr = w.cpr;
    auto emit = [&](int c, uint32_t pc, uint32_t pn) {
        const uint32_t sh = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)pc, 0x130, 0xF, 0xF, false);
        const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)pn, 0);
        const uint32_t word = pc | ((lane == 63 ? first : sh) << 1);
        const int x = 64 * c + lane;
        const bool xin1 = x + 1 < p.gx;
        int n[kWeldRows];
        unsigned long long s[kWeldRows + 1];
        int nv[kWeldRows];
#pragma unroll
        for (int i = 0; i <= kWeldRows; ++i) s[i] = __ballot((pc >> (4 * i)) & 1u);
#pragma unroll
        for (int i = 0; i < kWeldRows; ++i) {
            unsigned long long m[3];
            weld_edges(p, c, y + i, z, s[i], (first >> (4 * i)) & 1u, s[i + 1],
                       __ballot((pc >> (4 * i + 2)) & 1u), m);
            nv[i] = __popcll(m[0]) + __popcll(m[1]) + __popcll(m[2]);
            const bool cube = xin1 && zin && y + i + 1 < p.gy;
            n[i] = cube ? (int)ntab[(word >> (4 * i)) & 0xFFu] : 0;
        }
        const int s01 = wave_inclusive_scan(n[0] | (n[1] << 16), lane);
        const int s23 = wave_inclusive_scan(n[2] | (n[3] << 16), lane);
        const int t01 = __builtin_amdgcn_readlane(s01, 63), t23 = __builtin_amdgcn_readlane(s23, 63);
        if (lane < k) {
            const int i = lane;
            const int tw = i < 2 ? t01 : t23;
            const int64_t cc = (int64_t)(y + i + p.gy * z) * cpr + c;
            signs[cc] = i == 0 ? s[0] : (i == 1 ? s[1] : (i == 2 ? s[2] : s[3]));
            vcount[cc] = i == 0 ? nv[0] : (i == 1 ? nv[1] : (i == 2 ? nv[2] : nv[3]));
            tcount[cc] = (i & 1) ? (tw >> 16) : (tw & 0xFFFF);
        }
    };
    float va[kWeldLoadRows], vb[kWeldLoadRows];
    load(0, va);
    load(1, vb);
    uint32_t pc = sign_bits(va);
    load(2, va);
    for (int c = 0; c < cpr; c += 2) {
        uint32_t pn = sign_bits(vb);  // chunk c+1
        load(c + 3, vb);
        emit(c, pc, pn);
        if (c + 1 >= cpr) break;
        pc = pn;
        pn = sign_bits(va);  // chunk c+2
        load(c + 4, va);
        emit(c + 1, pc, pn);
        pc = pn;
    }
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

// A window is up to four consecutive chunks of a voxel row; one wavefront
// writes it, lane l holding voxels and cubes 4l .. 4l+3 of its 256.  For the
// four rows (y + dy, z + dz) its cubes reach and its own chunks and the next,
// LDS holds the signs, edge masks and first vertex: entry 5 (2 dy + dz) + j.
constexpr int kWinChunks = 4, kWinEntries = 4 * (kWinChunks + 1);
struct WeldWindow {
    unsigned long long s[kWinEntries];
    unsigned long long m[kWinEntries][3];
    uint32_t base[kWinEntries];
    int mark[64];
};

// The lane whose elements include element k0 + lane of the lanes' elements
// (first element excl, count n per lane; carry: the round before's last
// owner): marks at the first elements and a max-scan.  Every lane calls.
__device__ __forceinline__ int weld_owner(int* mark, int excl, int n, int k0, int lane, int& carry) {
    mark[lane] = 0;
    if (n > 0 && excl >= k0 && excl < k0 + 64) mark[excl - k0] = lane + 1;
    __builtin_amdgcn_wave_barrier();
    const int mx = wave_inclusive_max(mark[lane]);
    const int owner = mx > 0 ? mx - 1 : carry;
    carry = __builtin_amdgcn_readlane(owner, 63);
    __builtin_amdgcn_wave_barrier();
    return owner;
}

// Vertex index of local edge e (table word et: axis, lower end's dx, dy, dz)
// of the window's cube at voxel place xl.
__device__ __forceinline__ int32_t weld_index(const WeldWindow& nb, int xl, unsigned et) {
    const int a = (int)(et & 3u), X = xl + (int)((et >> 2) & 1u), l = X & 63;
    const int n = 5 * (int)(et >> 3) + (X >> 6);
    const unsigned long long below = (1ull << l) - 1ull;
    const unsigned long long m0 = nb.m[n][0], m1 = nb.m[n][1], m2 = nb.m[n][2];
    int idx = (int)nb.base[n] + __popcll(m0 & below) + __popcll(m1 & below) + __popcll(m2 & below);
    idx += a > 0 ? (int)((m0 >> l) & 1ull) : 0;
    idx += a > 1 ? (int)((m1 >> l) & 1ull) : 0;
    return idx;
}

__device__ __forceinline__ void weld_write_window(const WeldParams& w, const WeldSteps& st, int row, int j0,
                                                  int lane, const unsigned long long* __restrict__ signs,
                                                  const long long* __restrict__ vbase, long long v0,
                                                  long long t0, bool want_v, bool want_t, WeldWindow& nb,
                                                  const uint64_t* tri, const uint8_t* ntab,
                                                  const uint32_t* edges, float* __restrict__ verts,
                                                  float* __restrict__ normals, int32_t* __restrict__ tris) {
    const McParams& p = w.mc;
    const int z = row / p.gy, y = row - z * p.gy;
    if (lane < kWinEntries) {
        const int rr = lane / 5, j = j0 + lane - 5 * rr;
        const int Y = y + (rr >> 1), Z = z + (rr & 1);
        unsigned long long s = 0, m[3] = {0, 0, 0};
        uint32_t base = 0;
        if (Y < p.gy && Z < p.gz && j < w.cpr) {
            const int64_t c = (int64_t)(Y + p.gy * Z) * w.cpr + j;
            s = signs[c];
            const unsigned long long sn = j + 1 < w.cpr ? signs[c + 1] : 0ull;
            const unsigned long long sy = Y + 1 < p.gy ? signs[c + w.cpr] : 0ull;
            const unsigned long long sz = Z + 1 < p.gz ? signs[c + (int64_t)w.cpr * p.gy] : 0ull;
            weld_edges(p, j, Y, Z, s, sn, sy, sz, m);
            base = (uint32_t)vbase[c];
        }
        nb.s[lane] = s;
        nb.m[lane][0] = m[0];
        nb.m[lane][1] = m[1];
        nb.m[lane][2] = m[2];
        nb.base[lane] = base;
    }
    __builtin_amdgcn_wave_barrier();
    const int slot = lane >> 4, b = 4 * (lane & 15);
    const int x0 = 64 * j0;
    if (want_v) {
        // the lane's edges, bit 3 v + axis of voxel 4 lane + v
        unsigned own = 0;
        if (j0 + slot < w.cpr) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const unsigned q = (unsigned)(nb.m[slot][a] >> b) & 0xFu;
                own |= ((q & 1u) | ((q & 2u) << 2) | ((q & 4u) << 4) | ((q & 8u) << 6)) << a;
            }
        }
        const int n = __popc(own);
        const int incl = wave_inclusive_scan(n, lane);
        const int excl = incl - n, total = __builtin_amdgcn_readlane(incl, 63);
        int carry = 0;
        for (int k0 = 0; k0 < total; k0 += 64) {
            const int owner = weld_owner(nb.mark, excl, n, k0, lane, carry);
            unsigned left = (unsigned)__shfl((int)own, owner, 64);
            const int r = k0 + lane - __shfl(excl, owner, 64);
            // the r-th set bit (r < 12), three at a time: a voxel's
            int v = 0, rr = r;
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const int c = __popc((left >> (3 * v)) & 7u);
                if (v == q && rr >= c) {
                    rr -= c;
                    ++v;
                }
            }
            left = (left >> (3 * v)) & 7u;
            const unsigned l1 = left & (left - 1u), l2 = l1 & (l1 - 1u);
            const unsigned bit = rr == 0 ? left : (rr == 1 ? l1 : l2);
            const int a = bit ? __builtin_ctz(bit) : 0;
            weld_vertex(w, st, k0 + lane < total, x0 + 4 * owner + v, y, z, a, v0 + k0 + lane, verts, normals);
        }
    }
    if (!want_t) return;
    // the lane's cubes from the signs of their rows (y,z), (y,z+1), (y+1,z),
    // (y+1,z+1), five voxels from bit b
    unsigned q[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        const unsigned long long s = nb.s[5 * rr + slot];
        q[rr] = (unsigned)(s >> b) & 0x1Fu;
        if (b == 60) q[rr] |= ((unsigned)nb.s[5 * rr + slot + 1] & 1u) << 4;
    }
    int nt[4], cls = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const unsigned byte = ((q[0] >> j) & 3u) | (((q[1] >> j) & 3u) << 2) | (((q[2] >> j) & 3u) << 4) |
                              (((q[3] >> j) & 3u) << 6);
        const bool cube = (x0 + 4 * lane + j + 1 < p.gx) & (y + 1 < p.gy) & (z + 1 < p.gz);
        nt[j] = cube ? (int)ntab[byte] : 0;
        cls |= (int)(byte << (8 * j));
    }
    const int c1 = nt[0], c2 = c1 + nt[1], c3 = c2 + nt[2], n = c3 + nt[3];
    const int cp = c1 | (c2 << 8) | (c3 << 16);  // each <= 15
    const int incl = wave_inclusive_scan(n, lane);
    const int excl = incl - n, total = __builtin_amdgcn_readlane(incl, 63);
    int carry = 0;
    for (int k0 = 0; k0 < total; k0 += 64) {
        const int owner = weld_owner(nb.mark, excl, n, k0, lane, carry);
        const int ocls = __shfl(cls, owner, 64), ocp = __shfl(cp, owner, 64);
        const int local = k0 + lane - __shfl(excl, owner, 64);
        const int o1 = ocp & 0xFF, o2 = (ocp >> 8) & 0xFF, o3 = (ocp >> 16) & 0xFF;
        const int j = (local >= o1 ? 1 : 0) + (local >= o2 ? 1 : 0) + (local >= o3 ? 1 : 0);
        const int slot3 = local - (j == 0 ? 0 : (j == 1 ? o1 : (j == 2 ? o2 : o3)));
        if (k0 + lane < total) {
            const uint64_t word = tri[(ocls >> (8 * j)) & 0xFF] >> (4 + 12 * slot3);
            const long long t = t0 + k0 + lane;
#pragma unroll
            for (int e = 0; e < 3; ++e)
                tris[3 * t + e] = weld_index(nb, 4 * owner + j, edges[(word >> (4 * e)) & 0xFull]);
        }
    }
}

// One wavefront per four windows: one load of their chunks' counts (most of a
// volume's windows hold neither vertices nor triangles), then each busy
// window.  A row's few vertices and triangles fill the lanes of one or two
// rounds; chunk by chunk, with the field's corners read again, the pass was
// bound by instruction issue (96 % VALU busy, ten vertices a round): 250 x
// 333 x 287 voxels and 0.6 M vertices took 106 us, 59 this way.  Nothing is
// written when the totals (*vtotal, *ttotal, from the scans) exceed int32
// indices or a requested output's capacity: the host reports that after the
// call.
__global__ __launch_bounds__(256) void weld_write_kernel(const WeldParams w,
                                                         const unsigned long long* __restrict__ signs,
                                                         const int32_t* __restrict__ vcount,
                                                         const long long* __restrict__ vbase,
                                                         const int32_t* __restrict__ tcount,
                                                         const long long* __restrict__ tbase,
                                                         const long long* __restrict__ vtotal,
                                                         const long long* __restrict__ ttotal,
                                                         long long vcap, long long tcap,
                                                         float* __restrict__ verts,
                                                         float* __restrict__ normals,
                                                         int32_t* __restrict__ tris) {
    __shared__ WeldWindow windows[kWeldWaves];
    __shared__ uint64_t tri[256];    // triangle table by the signs' byte
    __shared__ uint8_t ntab[256];    // its triangle counts
    __shared__ uint32_t edges[16];   // axis | dx << 2 | (2 dy + dz) << 3 of an edge's lower end
    const long long nvt = *vtotal, ntt = *ttotal;
    const bool want_v = verts || normals;
    if (nvt > INT32_MAX || (want_v && nvt > vcap) || (tris && ntt > tcap)) return;
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
    const McParams& p = w.mc;
    WeldSteps st;
    st.ok = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        float bad = 0.0f;
        st.r1[k] = recip_sum(p.vs[k], bad);
        st.r2[k] = recip_sum(p.vs[k] + p.vs[k], bad);
        st.ok = st.ok && bad < kRecipBad && p.vs[k] >= 1e-6f && p.vs[k] <= 1e6f;
    }
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int wpr = (w.cpr + kWinChunks - 1) / kWinChunks;  // windows per row
    const uint32_t nwin = (uint32_t)wpr * (uint32_t)(p.gy * p.gz);  // <= nchunks
    const uint32_t win0 = 4u * (blockIdx.x * kWeldWaves + (uint32_t)wave);
    int n = 0;
    if (lane < 16 && win0 + (lane >> 2) < nwin) {
        const uint32_t win = win0 + (lane >> 2);
        const int row = (int)(win / (uint32_t)wpr);
        const int j = kWinChunks * ((int)win - row * wpr) + (lane & 3);
        if (j < w.cpr) {
            const int64_t c = (int64_t)row * w.cpr + j;
            n = (want_v ? vcount[c] : 0) + (tris ? tcount[c] : 0);
        }
    }
    const unsigned long long busy = __ballot(n > 0);
    for (int k = 0; k < 4; ++k) {
        if (!((busy >> (4 * k)) & 15ull)) continue;
        const uint32_t win = win0 + k;
        const int row = (int)(win / (uint32_t)wpr), j0 = kWinChunks * ((int)win - row * wpr);
        const int64_t c = (int64_t)row * w.cpr + j0;
        weld_write_window(w, st, row, j0, lane, signs, vbase, vbase[c], tbase[c], want_v, tris != nullptr,
                          windows[wave], tri, ntab, edges, verts, normals, tris);
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
    const int nb = (w.nchunks + kScanBlock - 1) / kScanBlock;
    const size_t o_signs = 0;
    const size_t o_vcount = o_signs + align256(8 * (size_t)w.nchunks);
    const size_t o_tcount = o_vcount + align256(4 * (size_t)w.nchunks);
    const size_t o_vbase = o_tcount + align256(4 * (size_t)w.nchunks);
    const size_t o_tbase = o_vbase + align256(8 * (size_t)w.nchunks);
    const size_t o_vsums = o_tbase + align256(8 * (size_t)w.nchunks);
    const size_t o_tsums = o_vsums + align256(8 * (size_t)(nb + 1));
    const size_t need = o_tsums + align256(8 * (size_t)(nb + 1));
    if (*scratch_bytes < need) {
        if (*scratch) (void)hipFree(*scratch);
        *scratch = nullptr;
        *scratch_bytes = 0;
        RECON_HIP_TRY(hipMalloc(scratch, need), "welded marching cubes scratch");
        *scratch_bytes = need;
    }
    char* sb = static_cast<char*>(*scratch);
    auto* signs = reinterpret_cast<unsigned long long*>(sb + o_signs);
    auto* vcount = reinterpret_cast<int32_t*>(sb + o_vcount);
    auto* tcount = reinterpret_cast<int32_t*>(sb + o_tcount);
    auto* vbase = reinterpret_cast<long long*>(sb + o_vbase);
    auto* tbase = reinterpret_cast<long long*>(sb + o_tbase);
    auto* vsums = reinterpret_cast<long long*>(sb + o_vsums);
    auto* tsums = reinterpret_cast<long long*>(sb + o_tsums);
    const int count_blocks =
        (((grid[1] + kWeldRows - 1) / kWeldRows) * grid[2] + kWeldWaves - 1) / kWeldWaves;
    hipLaunchKernelGGL(weld_count_kernel, dim3(count_blocks), dim3(256), 0, s, w, signs, vcount,
                       tcount);
    RECON_HIP_TRY(hipGetLastError(), "weld_count_kernel launch");
    ScanJobs jobs;
    jobs.in[0] = vcount;
    jobs.in[1] = tcount;
    jobs.sums[0] = vsums;
    jobs.sums[1] = tsums;
    jobs.out[0] = vbase;
    jobs.out[1] = tbase;
    const int rc = launch_exclusive_scans(jobs, 2, w.nchunks, s);
    if (rc) return rc;
    // The write pass checks the totals on the device, so it is queued before
    // the host waits; the copies of the totals to pageable memory come last,
    // since each returns only when the stream has reached it.
    const bool write = verts || normals || tris;
    if (write) {
        const long long windows = (long long)((w.cpr + kWinChunks - 1) / kWinChunks) * grid[1] * grid[2];
        const unsigned blocks = (unsigned)((windows + 4 * kWeldWaves - 1) / (4 * kWeldWaves));
        hipLaunchKernelGGL(weld_write_kernel, dim3(blocks), dim3(256), 0, s, w, signs, vcount,
                           vbase, tcount, tbase, vsums + nb, tsums + nb, (long long)vcap,
                           (long long)tcap, verts, normals, tris);
        RECON_HIP_TRY(hipGetLastError(), "weld_write_kernel launch");
    }
    long long totals[2] = {0, 0};
    RECON_HIP_TRY(hipMemcpyAsync(&totals[0], vsums + nb, 8, hipMemcpyDeviceToHost, s), "vertex total");
    RECON_HIP_TRY(hipMemcpyAsync(&totals[1], tsums + nb, 8, hipMemcpyDeviceToHost, s), "triangle total");
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
