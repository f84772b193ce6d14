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
// signs and counts per 64 voxels.  The field is read whole once, by the sign
// pass (mc_signs.hip); after the counts and their scan weld_write_kernel
// classifies the cubes from the signs again and reads the field at the
// vertices.
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

#include "mc_signs.hpp"

#include <algorithm>
#include <cmath>

namespace recon {

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
__device__ __forceinline__ void weld_vertex_exact(const SignParams& w, int x, int y, int z, int a,
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

// 1/vs and 1/(vs + vs) per axis, and whether short_quotient covers them.
struct WeldSteps {
    float r1[3], r2[3];
    bool ok;
};

// Every lane with `on` writes vertex (and normal) `idx` of edge (x, y, z, a):
// weld_vertex_exact's bits.
__device__ __forceinline__ void weld_vertex(const SignParams& w, const WeldSteps& st, bool on, int x, int y,
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
        const float r = short_quotient(-dn, den, y_den, bad);
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
                    ge[q] = short_quotient(num, both ? p.vs[k] + p.vs[k] : p.vs[k],
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
                for (int k = 0; k < 3; ++k) nrm[k] = short_quotient(gr[k], len, y_len, bad);
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
__device__ __forceinline__ void weld_entry_load(const SignParams& w, uint32_t c, const ChunkPlace& at, int rr,
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
        sign_edges(p, at.j, Y, Z, s, sn, sy, sz, m);
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
    const SignParams& w, const WeldSteps& st, uint32_t c0, int lane, int first, int nv, int nt,
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
            const int owner = unit_owner(nb.mark, excl, mine, k0, lane);
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
        const int owner = unit_owner(nb.mark, excl, mine, k0, lane);
        int r = k0 + lane - __shfl(excl, owner, 64);
        const int j = cube_of((uint32_t)__shfl((int)cn4.w[0], owner, 64),
                              (uint32_t)__shfl((int)cn4.w[1], owner, 64), r);
        uint32_t oq[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) oq[k] = (uint32_t)__shfl((int)q[k], owner, 64);
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
constexpr int kWriteBlocks = 256 * 5;  // 5 workgroups a CU by registers (bound to 80 for 6: 4 % slower)
__global__ __launch_bounds__(64 * kUnitWaves) void weld_write_kernel(
    const SignParams w, const unsigned long long* __restrict__ signs, const int32_t* __restrict__ voff,
    const int32_t* __restrict__ toff, const int2* __restrict__ group, const long long* __restrict__ vsums,
    const long long* __restrict__ tsums, const long long* __restrict__ total,
    const uint32_t* __restrict__ units, const uint32_t* __restrict__ nunits, long long vcap,
    long long tcap, float* __restrict__ verts, float* __restrict__ normals, int32_t* __restrict__ tris) {
    __shared__ WeldGroup groups[kUnitWaves];
    __shared__ uint64_t tri[256];    // triangle table by the signs' byte
    __shared__ uint8_t ntab[256];    // its triangle counts
    __shared__ uint32_t edges[16];   // axis | dx << 2 | (2 dy + dz) << 3 of an edge's lower end
    const McParams& p = w.mc;
    const bool want_v = verts || normals, want_t = tris != nullptr;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t nu = *nunits;
    const long long nvt = total[0], ntt = total[1];
    if (kUnitWaves * blockIdx.x >= nu || nvt > INT32_MAX || (want_v && nvt > vcap) || (want_t && ntt > tcap))
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
    for (uint32_t u = kUnitWaves * blockIdx.x + (uint32_t)wave; u < nu; u += kUnitWaves * gridDim.x) {
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

// Counts (always), then writes what is asked for when it fits.
static int weld_run(const float* field, const int32_t grid[3], const float vs[3], const float off[3],
                    float* verts, float* normals, int64_t vcap, int32_t* tris, int64_t tcap,
                    int64_t* nv_out, int64_t* nt_out, void** scratch, size_t* scratch_bytes,
                    hipStream_t s, const char* fn) {
    *nv_out = 0;
    *nt_out = 0;
    if (grid[0] < 2 || grid[1] < 2 || grid[2] < 2) return RECON_OK;
    SignParams w;
    SignScratch sc;
    const size_t need = sign_layout(field, grid, vs, off, true, nullptr, w, sc);
    if (*scratch_bytes < need) {
        if (*scratch) (void)hipFree(*scratch);
        *scratch = nullptr;
        *scratch_bytes = 0;
        RECON_HIP_TRY(hipMalloc(scratch, need), "welded marching cubes scratch");
        *scratch_bytes = need;
    }
    sign_layout(field, grid, vs, off, true, static_cast<char*>(*scratch), w, sc);
    const bool write = verts || normals || tris;
    const int rc = launch_signs(w, sc, true, verts || normals, tris != nullptr, s);
    if (rc) return rc;
    // The write pass checks the totals on the device, so it is queued before
    // the host waits; the copy of the totals to pageable memory comes last,
    // since it returns only when the stream has reached it.
    if (write) {
        // most groups are empty and a busy one is one or two units
        const int blocks = std::min(kWriteBlocks, w.nchunks / kGroupChunks + 1);
        hipLaunchKernelGGL(weld_write_kernel, dim3(blocks), dim3(64 * kUnitWaves), 0, s, w, sc.signs, sc.voff,
                           sc.toff, sc.group, sc.vsums, sc.tsums, sc.total, static_cast<const uint32_t*>(sc.units), sc.nunits,
                           (long long)vcap, (long long)tcap, verts, normals, tris);
        RECON_HIP_TRY(hipGetLastError(), "weld_write_kernel launch");
    }
    long long totals[2] = {0, 0};
    RECON_HIP_TRY(hipMemcpyAsync(totals, sc.total, 16, hipMemcpyDeviceToHost, s), "totals");
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
