// marching_cubes.hip -- marching cubes over a dense TSDF for gfx950.
//
// Replaces generate_triangular_surface (cu-Reconstruction
// modules/src/cuda/marching_cubes.cu:102-236).  The reference launches one
// kernel per z layer, synchronises, and compacts each layer on the host from
// managed memory.  Here the whole volume is done on the device in four
// launches with a fixed, deterministic output order:
//   1-3. signs, counts, scan (mc_signs.hip): a word of signs per 64 voxels,
//        the triangles of every 64-cube chunk from the words, and a list of
//        units (runs of at most 64 chunks with up to 127 cubes that the surface
//        crosses, so up to 635 triangles), each with its first triangle;
//   4.   emit - the resident wavefronts stride over the units: a unit's crossed
//        cubes are spread over the lanes 64 at a time, one a lane, then their
//        triangles, a lane reading the six field values of its triangle's edges
//        (marching_cubes.cu:23-74).
// The allocation-free entry, whose static scratch has no room for the words
// and the list, keeps to a smaller one (2 B per 64 cubes):
//   1. chunk count - one wavefront per 4 cube rows (y..y+3, z), streaming
//                    their 10 voxel rows once, 256 cubes a step (16-byte
//                    loads; 64 with 4-byte loads where rows are not 16-byte
//                    aligned): every cube's class from the corners' sign
//                    bits, and per 64-cube chunk of each row its triangle
//                    count; per workgroup ("tile", 16 cube rows) the tile's
//                    total and its number of chunks with triangles;
//   2. tile scan   - one workgroup: exclusive scans of the tile totals and of
//                    the tiles' groups of four chunks with triangles;
//   3. emit        - each wavefront takes groups gi = wave, wave + waves, ...,
//                    finds the group's tile and chunks by a search and a walk,
//                    and spreads its triangles over its 64 lanes
//                    (mc_emit_group, also the batch's).
// Output order is cube z, y, x, table slot -- the order the reference's host
// loop produces (marching_cubes.cu:163-188 inside :213-225) -- as a triangle
// soup: triangle t owns vertices 3t, 3t+1, 3t+2 (marching_cubes.cu:171).
#pragma clang fp contract(off)

#include "mc_signs.hpp"

#include <algorithm>
#include <mutex>

namespace recon {

constexpr int kRowsPerBlock = 4;  // one wavefront per row, 256 threads

// ---- tile scan ------------------------------------------------------------------
// The scan takes kScanRows rows of kScanRow tiles a pass, thread t holding
// tiles 4t .. 4t+3 of each row, so every load and store instruction of a
// wavefront covers contiguous bytes (one workgroup's loads and stores all go
// through one CU).
constexpr int kScanRow = 4096, kScanRows = 2;

// One workgroup of 1024 threads: tile_off[i] = sum of tile_sum[0..i) and
// tile_off[n] = the total; when tile_nne is not null also group_off[i] = sum
// over tiles before i of ceil(tile_nne / 4) (the emit's four-chunk groups)
// and group_off[n] = their total.  All four arrays are 16-byte aligned.
__global__ __launch_bounds__(1024) void mc_tile_scan_kernel(const int32_t* __restrict__ tile_sum,
                                                            const int32_t* __restrict__ tile_nne,
                                                            int n, long long* __restrict__ tile_off,
                                                            int32_t* __restrict__ group_off) {
    __shared__ long long wtot[kScanRows][16];
    __shared__ int gtot[kScanRows][16];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    long long carry = 0;
    int gcarry = 0;
    for (int base = 0; base < n; base += kScanRow * kScanRows) {
        int v[kScanRows][4], g[kScanRows][4];
        long long sum[kScanRows], incl[kScanRows];
        int gsum[kScanRows], ginc[kScanRows];
#pragma unroll
        for (int q = 0; q < kScanRows; ++q) {
            const int i0 = base + kScanRow * q + 4 * t;
            if (i0 + 4 <= n) {
                const int4 a = *reinterpret_cast<const int4*>(tile_sum + i0);
                v[q][0] = a.x; v[q][1] = a.y; v[q][2] = a.z; v[q][3] = a.w;
                if (tile_nne) {
                    const int4 b = *reinterpret_cast<const int4*>(tile_nne + i0);
                    g[q][0] = (b.x + 3) >> 2; g[q][1] = (b.y + 3) >> 2;
                    g[q][2] = (b.z + 3) >> 2; g[q][3] = (b.w + 3) >> 2;
                } else {
                    g[q][0] = g[q][1] = g[q][2] = g[q][3] = 0;
                }
            } else {
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    v[q][k] = i0 + k < n ? tile_sum[i0 + k] : 0;
                    g[q][k] = (tile_nne && i0 + k < n) ? (tile_nne[i0 + k] + 3) >> 2 : 0;
                }
            }
            sum[q] = (long long)v[q][0] + v[q][1] + v[q][2] + v[q][3];
            gsum[q] = g[q][0] + g[q][1] + g[q][2] + g[q][3];
        }
#pragma unroll
        for (int q = 0; q < kScanRows; ++q) {
            incl[q] = wave_inclusive_scan64(sum[q]);
            ginc[q] = wave_inclusive_scan(gsum[q], lane);
        }
        if (lane == 63) {
#pragma unroll
            for (int q = 0; q < kScanRows; ++q) {
                wtot[q][wave] = incl[q];
                gtot[q][wave] = ginc[q];
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < kScanRows; ++q) {
            long long before = 0, all = 0;
            int gbefore = 0, gall = 0;
#pragma unroll
            for (int w = 0; w < 16; ++w) {
                before += w < wave ? wtot[q][w] : 0;
                all += wtot[q][w];
                gbefore += w < wave ? gtot[q][w] : 0;
                gall += gtot[q][w];
            }
            const long long e0 = carry + before + incl[q] - sum[q];
            const long long e1 = e0 + v[q][0], e2 = e1 + v[q][1], e3 = e2 + v[q][2];
            const int f0 = gcarry + gbefore + ginc[q] - gsum[q];
            const int f1 = f0 + g[q][0], f2 = f1 + g[q][1], f3 = f2 + g[q][2];
            const int i0 = base + kScanRow * q + 4 * t;
            if (i0 + 4 <= n) {
                longlong2* d2 = reinterpret_cast<longlong2*>(tile_off + i0);
                d2[0] = make_longlong2(e0, e1);
                d2[1] = make_longlong2(e2, e3);
                if (group_off) *reinterpret_cast<int4*>(group_off + i0) = make_int4(f0, f1, f2, f3);
            } else {
                const long long e[4] = {e0, e1, e2, e3};
                const int f[4] = {f0, f1, f2, f3};
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (i0 + k < n) {
                        tile_off[i0 + k] = e[k];
                        if (group_off) group_off[i0 + k] = f[k];
                    }
            }
            carry += all;
            gcarry += gall;
        }
        __syncthreads();  // wtot and gtot are rewritten by the next pass
    }
    if (t == 0) {
        tile_off[n] = carry;
        if (group_off) group_off[n] = gcarry;
    }
}

int launch_tile_scan(const int32_t* tile_sum, int n, long long* tile_off, hipStream_t s,
                     const int32_t* tile_nne, int32_t* group_off) {
    hipLaunchKernelGGL(mc_tile_scan_kernel, dim3(1), dim3(1024), 0, s, tile_sum, tile_nne, n,
                       tile_off, group_off);
    RECON_HIP_TRY(hipGetLastError(), "mc_tile_scan_kernel launch");
    return RECON_OK;
}

// ---- single-volume kernels ------------------------------------------------------
__global__ __launch_bounds__(256) void mc_chunk_count_kernel(const McParams p, const McTiling tl,
                                                             uint16_t* __restrict__ cc,
                                                             int32_t* __restrict__ tile_sum,
                                                             int32_t* __restrict__ tile_nne) {
    __shared__ uint8_t ntab[256];
    __shared__ int wtot[8];
    ntab[threadIdx.x] = mc_ntab_qbyte((int)threadIdx.x);
    __syncthreads();
    mc_count_tile(p, tl, blockIdx.x, cc, ntab, wtot, tile_sum + blockIdx.x, tile_nne + blockIdx.x);
}

// The same with 16-byte loads (mc_count_tile4): gx % 4 == 0 and a 16-byte
// aligned field.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(5))) void mc_chunk_count4_kernel(const McParams p, const McTiling tl,
                                                              uint16_t* __restrict__ cc,
                                                              int32_t* __restrict__ tile_sum,
                                                              int32_t* __restrict__ tile_nne) {
    __shared__ uint8_t ntab[256];
    __shared__ int wtot[8];
    ntab[threadIdx.x] = mc_ntab_qbyte((int)threadIdx.x);
    __syncthreads();
    mc_count_tile4(p, tl, blockIdx.x, cc, ntab, wtot, tile_sum + blockIdx.x, tile_nne + blockIdx.x);
}

// ---- emit from signs -------------------------------------------------------------
// LDS of a wavefront: the words of its unit's chunks (a lane each), of rows
// (y,z), (y,z+1), (y+1,z), (y+1,z+1).
struct UnitEmitLds {
    unsigned long long s[4][64];
    int mark[64];
    float stage[64 * 9];  // 64 triangles' vertices
};

// The place of set bit r of m.
__device__ __forceinline__ int set_bit(unsigned long long m, int r) {
    const uint32_t lo = (uint32_t)m;
    const int c32 = __popc(lo);
    uint32_t v = r >= c32 ? (uint32_t)(m >> 32) : lo;
    int k = r >= c32 ? 32 : 0;
    r -= r >= c32 ? c32 : 0;
#pragma unroll
    for (int h = 16; h >= 1; h >>= 1) {
        const int c = __popc(v & ((1u << h) - 1u));
        const bool up = r >= c;
        r -= up ? c : 0;
        k += up ? h : 0;
        v >>= up ? h : 0;
    }
    return k;
}

// One wavefront per unit, strided over as many as are resident: the cubes with
// both signs of its chunks, 64 at a time, and their triangles, 64 at a time;
// triangles below the capacity are written.  The lanes fill whether a surface
// crosses a row once (a wall) or runs along it (a floor): 512^3 voxels
// with 3.3 M triangles 70 us, 2.9 TB/s of field values and output, half of it
// instruction issue; by groups of four 64-cube chunks, their voxel values
// passed between the lanes, it took 116 and 5 for the groups' records.  Units
// of 64 cubes instead of 256 take 9 us off a mesh of 64^3 voxels (fewer
// rounds one after the other) and 1 us off this one.
constexpr int kEmitBlocks = 256 * 7;  // 7 workgroups a CU by LDS
__global__ __launch_bounds__(64 * kUnitWaves) void mc_unit_emit_kernel(
    const SignParams w, const unsigned long long* __restrict__ signs,
    const long long* __restrict__ tsums, const unsigned long long* __restrict__ units,
    const uint32_t* __restrict__ nunits, float* __restrict__ verts, int32_t* __restrict__ tris,
    long long capacity) {
    __shared__ UnitEmitLds lds[kUnitWaves];
    __shared__ uint64_t tri[256];   // triangle table by the signs' byte
    __shared__ uint8_t ntab[256];   // its triangle counts
    __shared__ int4 ends[12];       // an edge's ends: voxel offsets a, b; dx | dy << 1 | dz << 2 of a, b
    const McParams& p = w.mc;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t nu = *nunits;
    if (kUnitWaves * blockIdx.x >= nu) return;
    tri[threadIdx.x] = c_tri[qbyte_class((int)threadIdx.x)];
    ntab[threadIdx.x] = mc_ntab_qbyte((int)threadIdx.x);
    if (threadIdx.x < 12) {
        // corner offsets packed as bits: dx = bit0, dy = bit1, dz = bit2
        // (0:000 1:001 2:101 3:100 4:010 5:011 6:111 7:110)
        constexpr unsigned k_off = (0u << 0) | (1u << 3) | (5u << 6) | (4u << 9) | (2u << 12) |
                                   (3u << 15) | (7u << 18) | (6u << 21);
        const int e = (int)threadIdx.x;
        const int ca = (int)((kEdgeA >> (4 * e)) & 0xFull), cb = (int)((kEdgeB >> (4 * e)) & 0xFull);
        const int oa = (int)((k_off >> (3 * ca)) & 7u), ob = (int)((k_off >> (3 * cb)) & 7u);
        auto place = [&](int o) {
            return (o & 1) + ((o >> 1) & 1) * p.gx + (o >> 2) * p.gx * p.gy;
        };
        ends[e] = make_int4(place(oa), place(ob), oa, ob);
    }
    __syncthreads();
    UnitEmitLds& l = lds[wave];
    for (uint32_t u = kUnitWaves * blockIdx.x + (uint32_t)wave; u < nu; u += kUnitWaves * gridDim.x) {
        const unsigned long long unit = units[u];
        const uint32_t c0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(unit >> 6));
        const int len = 1 + __builtin_amdgcn_readfirstlane((int)(unit & 63ull));
        long long t0 = tsums[c0 / kBlockChunks] + (long long)(unit >> kSoupTriShift);
        const uint32_t c = c0 + (uint32_t)(lane < len ? lane : 0);
        const ChunkPlace at = chunk_place(w, c);
        const ChunkWords v = chunk_words(w, signs, c, at, lane < len);
        const unsigned long long mixed = mixed_cubes(p, v, at, lane < len);
        const uint32_t nb = next_bits(v);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) l.s[rr][lane] = v.s[rr];
        const int cubes = __popcll(mixed), incl = wave_inclusive_scan(cubes, lane);
        const int excl = incl - cubes, all = __builtin_amdgcn_readlane(incl, 63);
        for (int q0 = 0; q0 < all; q0 += 64) {
            // the lane's cube
            const int chunk = unit_owner(l.mark, excl, cubes, q0, lane);
            const unsigned long long om =
                ((unsigned long long)(uint32_t)__shfl((int)(mixed >> 32), chunk, 64) << 32) |
                (uint32_t)__shfl((int)mixed, chunk, 64);
            const int k = set_bit(om, q0 + lane - __shfl(excl, chunk, 64));
            const unsigned long long s[4] = {l.s[0][chunk], l.s[1][chunk], l.s[2][chunk], l.s[3][chunk]};
            const uint32_t byte = cube_byte64(s, (uint32_t)__shfl((int)nb, chunk, 64), k & 63) & 0xFFu;
            const ChunkPlace cat = chunk_place(w, c0 + (uint32_t)chunk);
            const int cx = 64 * cat.j + k;
            const int n = q0 + lane < all ? (int)ntab[byte] : 0;
            const int tincl = wave_inclusive_scan(n, lane), texcl = tincl - n;
            const int nt = __builtin_amdgcn_readlane(tincl, 63);
            const int pk = (int)byte | (texcl << 8);
            for (int k0 = 0; k0 < nt; k0 += 64) {
                const int owner = unit_owner(l.mark, texcl, n, k0, lane);
                const int opk = __shfl(pk, owner, 64);
                const int x = __shfl(cx, owner, 64), y = __shfl(cat.y, owner, 64), z = __shfl(cat.z, owner, 64);
                const int r = k0 + lane - (opk >> 8);
                if (k0 + lane < nt) {
                    const float* __restrict__ f = p.f + ((size_t)x + (size_t)p.gx * ((size_t)y + (size_t)p.gy * z));
                    const uint64_t word3 = tri[opk & 0xFF] >> (4 + 12 * r);
                    float wa[3], wb[3];
                    int da[3], db[3];
#pragma unroll
                    for (int e = 0; e < 3; ++e) {
                        const int4 d = ends[(word3 >> (4 * e)) & 0xFull];
                        wa[e] = f[d.x];
                        wb[e] = f[d.y];
                        da[e] = d.z;
                        db[e] = d.w;
                    }
                    const int cube[3] = {x, y, z};
                    float ctr[3][2];
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        ctr[k][0] = voxel_centre(cube[k], p.vs[k], p.off[k]);
                        ctr[k][1] = voxel_centre(cube[k] + 1, p.vs[k], p.off[k]);
                    }
                    float out[9];
#pragma unroll
                    for (int e = 0; e < 3; ++e) {
                        // from the negative end when the first is above zero and
                        // the second below (marching_cubes.cu:23-51)
                        const bool swap = (wa[e] > 0.0f) & (wb[e] < 0.0f);
                        const float s = swap ? wb[e] : wa[e], en = swap ? wa[e] : wb[e];
                        const int os = swap ? db[e] : da[e], oe = swap ? da[e] : db[e];
                        const float den = en - s;
                        float res = 0.0f;
                        const float y_den = recip_sum(den, res);
                        bool bad = !(res < kRecipBad) | !(fabsf(den) <= 1e7f);
                        float ratio = short_quotient(-s, den, y_den, bad);
                        if (__builtin_expect(bad, 0)) ratio = (-s) / den;
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            const float cs = (os >> k) & 1 ? ctr[k][1] : ctr[k][0];
                            const float ce = (oe >> k) & 1 ? ctr[k][1] : ctr[k][0];
                            const float edge = ce - cs;
                            const float o = ratio * edge;
                            out[3 * e + k] = cs + o;
                        }
                    }
#pragma unroll
                    for (int q = 0; q < 9; ++q) l.stage[9 * lane + q] = out[q];
                }
                __builtin_amdgcn_wave_barrier();
                const long long tb = t0 + k0;
                const int m = (int)min((long long)min(64, nt - k0), max(capacity - tb, 0ll));
                float* __restrict__ dst = verts + 9 * tb;
#pragma unroll
                for (int q = 0; q < 9; ++q)
                    if (64 * q + lane < 9 * m) dst[64 * q + lane] = l.stage[64 * q + lane];
                if (tris) {
#pragma unroll
                    for (int q = 0; q < 3; ++q)
                        if (64 * q + lane < 3 * m)
                            tris[3 * tb + 64 * q + lane] = (int32_t)(3 * tb + 64 * q + lane);
                }
                __builtin_amdgcn_wave_barrier();
            }
            t0 += nt;
        }
        __builtin_amdgcn_wave_barrier();
    }
}

// The emit of the allocation-free entry: a grid sized to the resident
// workgroups walks the volume's groups of four chunks with triangles,
// wavefront by wavefront; each finds its group's tile by a search over
// group_off and its chunks by a walk over the tile's chunk counts
// (mc_emit_group_at).
__global__ __launch_bounds__(256) void mc_chunk_emit_search_kernel(const McParams p, const McTiling tl,
                                                            const uint16_t* __restrict__ cc,
                                                            const long long* __restrict__ tile_off,
                                                            const int32_t* __restrict__ tile_nne,
                                                            const int32_t* __restrict__ group_off,
                                                            float* __restrict__ verts,
                                                            int32_t* __restrict__ tris,
                                                            long long capacity) {
    __shared__ McEmitLds lds;
    mc_emit_lds_init(lds);
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int ngroups = group_off[tl.tiles];
    const int waves = (int)gridDim.x * 4;
    for (int gi = (int)blockIdx.x * 4 + wave; gi < ngroups; gi += waves)
        mc_emit_group_at(p, tl, gi, cc, tile_off, tile_nne, group_off, lds, wave, lane, verts,
                         tris, capacity);
}

__global__ __launch_bounds__(256) void mc_class_hist_kernel(const McParams p,
                                                            unsigned long long* __restrict__ hist) {
    __shared__ unsigned int h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
    if (r < p.rows) {
        const int y = r % p.cyr, z = r / p.cyr;
        for (int x = lane; x < p.cx; x += 64) {
            float v[8];
            load_corners(p, x, y, z, v);
            atomicAdd(&h[cube_class(v)], 1u);
        }
    }
    __syncthreads();
    if (h[threadIdx.x]) atomicAdd(&hist[threadIdx.x], (unsigned long long)h[threadIdx.x]);
}

__global__ __launch_bounds__(256) void scan_block_sums_kernel(const int32_t* __restrict__ in, int n,
                                                              long long* __restrict__ sums) {
    __shared__ long long sh[256];
    const int b0 = blockIdx.x * kScanBlock + threadIdx.x * kScanItems;
    long long s = 0;
    if (b0 + kScanItems <= n && (reinterpret_cast<uintptr_t>(in) & 15) == 0) {
        const int4 a = *reinterpret_cast<const int4*>(in + b0);
        s = ((long long)a.x + a.y) + ((long long)a.z + a.w);
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
            if (b0 + k < n) s += in[b0 + k];
    }
    long long total;
    block_exclusive_scan(s, sh, &total);
    if (threadIdx.x == 0) sums[blockIdx.x] = total;
}

// One workgroup: exclusive scan of the block sums in place, total at [nb]; each thread takes kTopItems consecutive sums per pass, so up to
// 256 * kTopItems sums need one workgroup scan.
constexpr int kTopItems = 8;
__global__ __launch_bounds__(256) void scan_top_kernel(long long* __restrict__ sums, int nb) {
    __shared__ long long sh[256];
    long long carry = 0;
    for (int base = 0; base < nb; base += 256 * kTopItems) {
        const int i0 = base + threadIdx.x * kTopItems;
        long long v[kTopItems], s = 0;
#pragma unroll
        for (int k = 0; k < kTopItems; ++k) {
            v[k] = i0 + k < nb ? sums[i0 + k] : 0;
            s += v[k];
        }
        long long total;
        long long e = carry + block_exclusive_scan(s, sh, &total);
#pragma unroll
        for (int k = 0; k < kTopItems; ++k) {
            if (i0 + k < nb) sums[i0 + k] = e;
            e += v[k];
        }
        carry += total;
    }
    if (threadIdx.x == 0) sums[nb] = carry;
}

__global__ __launch_bounds__(256) void scan_apply_kernel(const int32_t* __restrict__ in, int n,
                                                         const long long* __restrict__ sums,
                                                         long long* __restrict__ out) {
    __shared__ long long sh[256];
    const int b0 = blockIdx.x * kScanBlock + threadIdx.x * kScanItems;
    const bool vec = b0 + kScanItems <= n && (reinterpret_cast<uintptr_t>(in) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    long long vals[kScanItems];
    if (vec) {
        const int4 a = *reinterpret_cast<const int4*>(in + b0);
        vals[0] = a.x; vals[1] = a.y; vals[2] = a.z; vals[3] = a.w;
    } else {
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) vals[k] = (b0 + k < n) ? in[b0 + k] : 0;
    }
    const long long s = (vals[0] + vals[1]) + (vals[2] + vals[3]);
    long long total;
    const long long e0 = block_exclusive_scan(s, sh, &total) + sums[blockIdx.x];
    const long long e1 = e0 + vals[0], e2 = e1 + vals[1], e3 = e2 + vals[2];
    if (vec) {
        longlong2* o2 = reinterpret_cast<longlong2*>(out + b0);
        o2[0] = make_longlong2(e0, e1);
        o2[1] = make_longlong2(e2, e3);
    } else {
        const long long e[kScanItems] = {e0, e1, e2, e3};
#pragma unroll
        for (int k = 0; k < kScanItems; ++k)
            if (b0 + k < n) out[b0 + k] = e[k];
    }
}

int launch_exclusive_scan(const int32_t* counts, int n, long long* offsets, long long* sums,
                          hipStream_t s) {
    const int nb = (n + kScanBlock - 1) / kScanBlock;
    hipLaunchKernelGGL(scan_block_sums_kernel, dim3(nb), dim3(256), 0, s, counts, n, sums);
    RECON_HIP_TRY(hipGetLastError(), "scan_block_sums_kernel launch");
    hipLaunchKernelGGL(scan_top_kernel, dim3(1), dim3(256), 0, s, sums, nb);
    RECON_HIP_TRY(hipGetLastError(), "scan_top_kernel launch");
    if (offsets) {
        hipLaunchKernelGGL(scan_apply_kernel, dim3(nb), dim3(256), 0, s, counts, n, sums, offsets);
        RECON_HIP_TRY(hipGetLastError(), "scan_apply_kernel launch");
    }
    return RECON_OK;
}

static McParams make_params(const float* field, const int32_t grid[3], const float vs[3],
                            const float off[3]) {
    McParams p;
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
    return p;
}

static int check_grid(const float* field, const int32_t grid[3], const float vs[3],
                      const float off[3], const char* fn) {
    if (!field || !grid || !vs || !off) return fail(RECON_ERR_NULL, "%s: null argument", fn);
    int64_t n = 1;
    for (int i = 0; i < 3; ++i) {
        if (grid[i] < 1) return fail(RECON_ERR_SIZE, "%s: grid[%d] = %d must be >= 1", fn, i, grid[i]);
        n *= grid[i];
    }
    if (n >= (int64_t(1) << 31)) return fail(RECON_ERR_RANGE, "%s: grid exceeds 2^31-1 voxels", fn);
    return RECON_OK;
}

// Tiling of a grid (host side) and the scratch layout of the allocation-free
// entry: chunk counts uint16[rows * nch] | tile sums int32[tiles] | tile chunks
// with triangles int32[tiles] | tile offsets int64[tiles+1] | tile first groups
// int32[tiles+1], each part 256-byte aligned.
struct McScratchLayout {
    McTiling t{0, 0, 0, 0};
    int gpl = 0, groups = 0, tiles = 0, nch = 0;
    size_t off_sum = 0, off_nne = 0, off_off = 0, off_goff = 0, need = 0;
    explicit McScratchLayout(const int32_t grid[3]) {
        if (grid[0] < 2 || grid[1] < 2 || grid[2] < 2) return;
        t = mc_tiling(grid[0], grid[1], grid[2]);
        gpl = t.gpl;
        groups = t.groups;
        tiles = t.tiles;
        nch = t.nch;
        const size_t rows = (size_t)(grid[1] - 1) * (size_t)(grid[2] - 1);
        auto a256 = [](size_t b) { return (b + 255) / 256 * 256; };
        off_sum = a256(2 * rows * (size_t)nch);
        off_nne = off_sum + a256(4 * (size_t)tiles);
        off_off = off_nne + a256(4 * (size_t)tiles);
        off_goff = off_off + a256(8 * ((size_t)tiles + 1));
        need = off_goff + 4 * ((size_t)tiles + 1);
    }
};

// Workgroups of the search emit: its resident slots on every CU of the current
// device (looked up once per device).
static int emit_grid() {
    static std::mutex mu;
    static int grid[64] = {0};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 1024;
    std::lock_guard<std::mutex> lk(mu);
    if (!grid[dev]) {
        int cus = 0, occ = 0;
        if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
            cus < 1)
            cus = 256;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, mc_chunk_emit_search_kernel, 256, 0) !=
                hipSuccess ||
            occ < 1)
            occ = 1;
        grid[dev] = cus * occ;
    }
    return grid[dev];
}

size_t mc_scratch_need(const int32_t grid[3]) { return McScratchLayout(grid).need; }

// The total of a run whose launches are all queued (the emit checks the
// capacity on the device): the copy to pageable memory comes last, since it
// returns only when the stream has reached it.
static int read_total(const long long* dev, int64_t* total, hipStream_t s) {
    long long host_total = 0;
    RECON_HIP_TRY(hipMemcpyAsync(&host_total, dev, sizeof(long long), hipMemcpyDeviceToHost, s),
                  "marching cubes total");
    RECON_HIP_TRY(hipStreamSynchronize(s), "marching cubes synchronize");
    *total = host_total;
    return RECON_OK;
}

// The allocation-free entry's passes.
static int mc_run_noalloc(const McParams& p, const int32_t grid[3], float* verts, int32_t* tris,
                          int64_t capacity, int64_t* total, bool count_only, void* scratch,
                          size_t scratch_bytes, hipStream_t s) {
    const McScratchLayout L(grid);
    if ((int64_t)(grid[1] - 1) * (grid[2] - 1) * L.nch >= (int64_t(1) << 31))
        return fail(RECON_ERR_RANGE, "marching cubes: more than 2^31 64-cube chunks");
    if (scratch_bytes < L.need)
        return fail(RECON_ERR_RANGE, "marching cubes needs %zu bytes of scratch, %zu available",
                    L.need, scratch_bytes);
    char* sb = static_cast<char*>(scratch);
    uint16_t* cc = reinterpret_cast<uint16_t*>(sb);
    int32_t* tile_sum = reinterpret_cast<int32_t*>(sb + L.off_sum);
    int32_t* tile_nne = reinterpret_cast<int32_t*>(sb + L.off_nne);
    long long* tile_off = reinterpret_cast<long long*>(sb + L.off_off);
    int32_t* group_off = reinterpret_cast<int32_t*>(sb + L.off_goff);
    if (grid[0] % 4 == 0 && reinterpret_cast<uintptr_t>(p.f) % 16 == 0)
        hipLaunchKernelGGL(mc_chunk_count4_kernel, dim3(L.tiles), dim3(256), 0, s, p, L.t, cc,
                           tile_sum, tile_nne);
    else
        hipLaunchKernelGGL(mc_chunk_count_kernel, dim3(L.tiles), dim3(256), 0, s, p, L.t, cc,
                           tile_sum, tile_nne);
    RECON_HIP_TRY(hipGetLastError(), "mc_chunk_count_kernel launch");
    const int rc = launch_tile_scan(tile_sum, L.tiles, tile_off, s, tile_nne, group_off);
    if (rc) return rc;
    if (!count_only && capacity > 0 && verts) {
        hipLaunchKernelGGL(mc_chunk_emit_search_kernel, dim3(emit_grid()), dim3(256), 0, s, p,
                           L.t, cc, tile_off, tile_nne, group_off, verts, tris,
                           (long long)capacity);
        RECON_HIP_TRY(hipGetLastError(), "mc_chunk_emit_search_kernel launch");
    }
    return read_total(tile_off + L.tiles, total, s);
}

int mc_run(const float* field, const int32_t grid[3], const float vs[3], const float off[3],
           float* verts, int32_t* tris, int64_t capacity, int64_t* total, bool count_only,
           void** scratch, size_t* scratch_bytes, hipStream_t s, bool may_allocate) {
    *total = 0;
    if (grid[0] < 2 || grid[1] < 2 || grid[2] < 2) return RECON_OK;
    if (!may_allocate)
        return mc_run_noalloc(make_params(field, grid, vs, off), grid, verts, tris, capacity, total,
                              count_only, *scratch, *scratch_bytes, s);
    SignParams w;
    SignScratch sc;
    const size_t need = sign_layout(field, grid, vs, off, false, nullptr, w, sc);
    if (*scratch_bytes < need) {
        if (*scratch) (void)hipFree(*scratch);
        *scratch = nullptr;
        *scratch_bytes = 0;
        RECON_HIP_TRY(hipMalloc(scratch, need), "marching cubes scratch");
        *scratch_bytes = need;
    }
    sign_layout(field, grid, vs, off, false, static_cast<char*>(*scratch), w, sc);
    const bool write = !count_only && capacity > 0 && verts;
    const int rc = launch_signs(w, sc, false, false, write, s);
    if (rc) return rc;
    if (write) {
        const int blocks = std::min(kEmitBlocks, w.nchunks / 16 + 1);
        hipLaunchKernelGGL(mc_unit_emit_kernel, dim3(blocks), dim3(64 * kUnitWaves), 0, s, w, sc.signs,
                           sc.tsums, static_cast<const unsigned long long*>(sc.units), sc.nunits, verts, tris,
                           (long long)capacity);
        RECON_HIP_TRY(hipGetLastError(), "mc_unit_emit_kernel launch");
    }
    return read_total(sc.total + 1, total, s);
}

}  // namespace recon

using namespace recon;

static int mc_entry(const float* field, const int32_t grid[3], const float vs[3], const float off[3],
                    float* verts, int32_t* tris, int64_t capacity, int64_t* n, bool count_only,
                    void** scratch, size_t* scratch_bytes, hipStream_t s, const char* fn,
                    bool may_allocate = true) {
    if (!n) return fail(RECON_ERR_NULL, "%s: num_triangles is NULL", fn);
    *n = 0;
    int rc = check_grid(field, grid, vs, off, fn);
    if (rc) return rc;
    if (!count_only) {
        if (capacity < 0) return fail(RECON_ERR_SIZE, "%s: negative capacity", fn);
        if (capacity > 0 && !verts) return fail(RECON_ERR_NULL, "%s: verts is NULL", fn);
        if (tris && capacity > (int64_t)715827882)
            return fail(RECON_ERR_RANGE, "%s: int32 vertex indices overflow above 715827882 triangles", fn);
    }
    rc = require_gfx950();
    if (rc) return rc;
    if (!may_allocate && mc_scratch_need(grid) > *scratch_bytes)
        return fail(RECON_ERR_RANGE,
                    "%s: a %d x %d x %d grid needs %zu bytes of scratch, above the static %zu",
                    fn, grid[0], grid[1], grid[2], mc_scratch_need(grid), *scratch_bytes);
    if (!may_allocate && !*scratch) return fail(RECON_ERR_HIP, "%s: no scratch address", fn);
    rc = mc_run(field, grid, vs, off, verts, tris, capacity, n, count_only, scratch, scratch_bytes,
                s, may_allocate);
    if (rc) return rc;
    if (!count_only && *n > capacity)
        return fail(RECON_ERR_CAPACITY, "%s: %lld triangles do not fit capacity %lld", fn,
                    (long long)*n, (long long)capacity);
    return RECON_OK;
}

extern "C" int recon_tsdf_count_triangles(recon_tsdf* h, int64_t* num_triangles,
                                          recon_stream_t stream) {
    clear_error();
    if (!h) return fail(RECON_ERR_NULL, "recon_tsdf_count_triangles: handle is NULL");
    return mc_entry(h->D, h->info.grid, h->info.voxel_size, h->info.global_offset, nullptr, nullptr,
                    0, num_triangles, true, &h->mc_scratch, &h->mc_scratch_bytes,
                    (hipStream_t)stream, "recon_tsdf_count_triangles");
}

extern "C" int recon_tsdf_extract_mesh(recon_tsdf* h, float* verts, int32_t* tris,
                                       int64_t capacity_triangles, int64_t* num_triangles,
                                       recon_stream_t stream) {
    clear_error();
    if (!h) return fail(RECON_ERR_NULL, "recon_tsdf_extract_mesh: handle is NULL");
    return mc_entry(h->D, h->info.grid, h->info.voxel_size, h->info.global_offset, verts, tris,
                    capacity_triangles, num_triangles, false, &h->mc_scratch, &h->mc_scratch_bytes,
                    (hipStream_t)stream, "recon_tsdf_extract_mesh");
}

extern "C" int recon_mc_count(const float* field, const int32_t grid[3], const float voxel_size[3],
                              const float offset[3], int64_t* num_triangles,
                              recon_stream_t stream) {
    clear_error();
    void* scratch = nullptr;
    size_t bytes = 0;
    const int rc = mc_entry(field, grid, voxel_size, offset, nullptr, nullptr, 0, num_triangles, true,
                            &scratch, &bytes, (hipStream_t)stream, "recon_mc_count");
    if (scratch) (void)hipFree(scratch);
    return rc;
}

extern "C" int recon_mc_extract(const float* field, const int32_t grid[3],
                                const float voxel_size[3], const float offset[3], float* verts,
                                int32_t* tris, int64_t capacity_triangles,
                                int64_t* num_triangles, recon_stream_t stream) {
    clear_error();
    void* scratch = nullptr;
    size_t bytes = 0;
    const int rc = mc_entry(field, grid, voxel_size, offset, verts, tris, capacity_triangles,
                            num_triangles, false, &scratch, &bytes, (hipStream_t)stream,
                            "recon_mc_extract");
    if (scratch) (void)hipFree(scratch);
    return rc;
}

// ---- marching cubes without allocation ---------------------------------------
// Scratch of recon_mc_extract_noalloc: the chunk counts (2 B per 64-cube
// chunk of every cube row) and the tile sums, chunk counts, triangle and
// group offsets (20 B per 16 cube rows) -- mc_scratch_need bytes -- in one
// static array that each GPU holds
// for the life of the process.  48 MiB covers a 1024^3 grid (1023^2 cube
// rows of 16 chunks: 34.6 MB).
constexpr size_t kMcNoAllocScratchBytes = size_t(48) << 20;
static __device__ __align__(256) unsigned char scratch[kMcNoAllocScratchBytes];

// The array's device address on the current device, looked up once per
// device (hipGetSymbolAddress; the host-side name is not a device address).
static int noalloc_scratch(void** out) {
    static std::mutex mu;
    static void* addr[64] = {nullptr};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
    if (dev < 0 || dev >= 64) return fail(RECON_ERR_DEVICE, "device index %d out of range", dev);
    std::lock_guard<std::mutex> lk(mu);
    if (!addr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) return hip_fail(e, "hipGetSymbolAddress(marching-cubes scratch)");
        addr[dev] = p;
    }
    *out = addr[dev];
    return RECON_OK;
}

extern "C" int recon_mc_extract_noalloc(const float* field, const int32_t grid[3],
                                        const float voxel_size[3], const float offset[3],
                                        float* verts, int32_t* tris, int64_t capacity_triangles,
                                        int64_t* num_triangles, recon_stream_t stream) {
    clear_error();
    const char* fn = "recon_mc_extract_noalloc";
    if (!num_triangles) return fail(RECON_ERR_NULL, "%s: num_triangles is NULL", fn);
    *num_triangles = 0;
    int rc = check_grid(field, grid, voxel_size, offset, fn);
    if (rc) return rc;
    if (mc_scratch_need(grid) > kMcNoAllocScratchBytes)
        return fail(RECON_ERR_RANGE,
                    "%s: a %d x %d x %d grid needs %zu bytes of scratch, above the static maximum "
                    "of %zu (2 B per 64-cube chunk of each of the (gy-1)*(gz-1) cube rows)",
                    fn, grid[0], grid[1], grid[2], mc_scratch_need(grid), kMcNoAllocScratchBytes);
    rc = require_gfx950();
    if (rc) return rc;
    void* sp = nullptr;
    rc = noalloc_scratch(&sp);
    if (rc) return rc;
    size_t bytes = kMcNoAllocScratchBytes;
    return mc_entry(field, grid, voxel_size, offset, verts, tris, capacity_triangles, num_triangles,
                    false, &sp, &bytes, (hipStream_t)stream, fn, false);
}

extern "C" int recon_mc_class_histogram(const float* field, const int32_t grid[3],
                                        unsigned long long* hist_device, recon_stream_t stream) {
    clear_error();
    const float one[3] = {1.f, 1.f, 1.f}, zero[3] = {0.f, 0.f, 0.f};
    int rc = check_grid(field, grid, one, zero, "recon_mc_class_histogram");
    if (rc) return rc;
    if (!hist_device) return fail(RECON_ERR_NULL, "recon_mc_class_histogram: hist is NULL");
    rc = require_gfx950();
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    RECON_HIP_TRY(hipMemsetAsync(hist_device, 0, 256 * sizeof(unsigned long long), s),
                  "histogram clear");
    if (grid[0] < 2 || grid[1] < 2 || grid[2] < 2) return RECON_OK;
    const McParams p = make_params(field, grid, one, zero);
    const int blocks = (p.rows + kRowsPerBlock - 1) / kRowsPerBlock;
    hipLaunchKernelGGL(mc_class_hist_kernel, dim3(blocks), dim3(256), 0, s, p, hist_device);
    RECON_HIP_TRY(hipGetLastError(), "mc_class_hist_kernel launch");
    return RECON_OK;
}
