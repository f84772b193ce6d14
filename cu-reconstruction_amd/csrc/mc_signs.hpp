// mc_signs.hpp -- marching cubes by sign words, for gfx950: what the soup's and
// the welded mesh's passes share.
//
// A voxel row is cut into chunks of 64 voxels; a 64-bit word holds a chunk's
// signs (v < 0, so -0 and NaN count as not negative, marching_cubes.cu:76-84).
// One pass reads the field and stores the words (8 B per 64 voxels); counts,
// cube classes and sign-changing edges follow from a chunk's word, the next
// one's and those of the three neighbouring rows, and the field is read again
// only at the vertices.
#pragma once

#include "mc_device.hpp"
#include "scan.hpp"

namespace recon {

// A group is 16 consecutive chunks (of one voxel row or several): what a
// wavefront of a write pass looks at, lane 4i + q holding voxels and cubes
// 16q .. 16q+15 of chunk i.  kBlockChunks chunks are a workgroup of the count
// pass; a chunk's first vertex or triangle is its block's plus its place in it.
constexpr int kGroupChunks = 16;
constexpr int kBlockChunks = 512, kBlockGroups = kBlockChunks / kGroupChunks;
// A unit of the soup's emit is a run of at most 64 consecutive chunks, within
// one of the count pass's wavefronts, whose cubes with both signs number at
// most kUnitCubes + 63; the list holds its first triangle in its count block
// (< 2^18) << kSoupTriShift | chunk << 6 | (chunks - 1).
constexpr int kUnitCubes = 64, kWaveUnits = 64 * 64 / kUnitCubes, kSoupTriShift = 38;
// A unit of the welded write pass is up to kUnitRounds rounds of 64 elements of a
// group: its vertices first, then its triangles (<= 48 + 80 rounds, so <= 32
// units).  The list holds group << kUnitBits | unit (group < 2^31 / 16).
constexpr int kUnitRounds = 4, kUnitBits = 5;
static_assert((16 * 64 * 3 + 16 * 64 * 5) / 64 <= kUnitRounds << kUnitBits, "a group's units fit the bits");
constexpr int kSignChunks = 8;  // chunks per wavefront of the sign pass
constexpr int kUnitWaves = 4;   // wavefronts per workgroup of the sign and write passes

struct SignParams {
    McParams mc;
    int32_t cpr;      // 64-voxel chunks per x-row
    int32_t nchunks;  // cpr * gy * gz
    uint32_t mul_cpr, mul_gy;  // div31's of cpr and gy
    int32_t sh_cpr, sh_gy;
};

// n / d for n < 2^31: ceil(2^(31 + l) / d), l = ceil(log2 d), errs by less
// than 2^-31 of n / d, too little to reach the next whole number.
inline void div31_make(uint32_t d, uint32_t& mul, int32_t& sh) {
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
__device__ __forceinline__ void sign_edges(const McParams& p, int j, int y, int z, unsigned long long s,
                                           unsigned long long sn, unsigned long long sy,
                                           unsigned long long sz, unsigned long long m[3]) {
    const unsigned long long in = low_bits(p.gx - 64 * j);
    m[0] = (s ^ ((s >> 1) | (sn << 63))) & low_bits(p.gx - 1 - 64 * j);
    m[1] = y + 1 < p.gy ? (s ^ sy) & in : 0ull;
    m[2] = z + 1 < p.gz ? (s ^ sz) & in : 0ull;
}

// Chunk c's place: chunk j of voxel row (y, z).
struct ChunkPlace {
    int j, y, z;
};
__device__ __forceinline__ ChunkPlace chunk_place(const SignParams& w, uint32_t c) {
    const uint32_t row = div31(c, w.mul_cpr, w.sh_cpr), z = div31(row, w.mul_gy, w.sh_gy);
    return {(int)(c - row * (uint32_t)w.cpr), (int)(row - z * (uint32_t)w.mc.gy), (int)z};
}

// The words a lane needs of chunk c (place at): its own and the next chunk's,
// of the rows (y,z), (y,z+1), (y+1,z), (y+1,z+1); 0 past the grid.
struct ChunkWords {
    unsigned long long s[4], sn[4];
};
__device__ __forceinline__ ChunkWords chunk_words(const SignParams& w,
                                                  const unsigned long long* __restrict__ signs, uint32_t c,
                                                  const ChunkPlace& at, bool in) {
    ChunkWords v;
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        v.s[rr] = v.sn[rr] = 0;
        if (in & (at.y + (rr >> 1) < w.mc.gy) & (at.z + (rr & 1) < w.mc.gz)) {
            const size_t cc = (size_t)c + (rr >> 1 ? (size_t)w.cpr : 0) + (rr & 1 ? (size_t)w.cpr * w.mc.gy : 0);
            v.s[rr] = signs[cc];
            if (at.j + 1 < w.cpr) v.sn[rr] = signs[cc + 1];
        }
    }
    return v;
}
__device__ __forceinline__ bool any_negative(const ChunkWords& v) {
    return (((v.s[0] | v.sn[0]) | (v.s[1] | v.sn[1])) | ((v.s[2] | v.sn[2]) | (v.s[3] | v.sn[3]))) != 0ull;
}
// The chunk's cubes whose corners have both signs.
__device__ __forceinline__ unsigned long long mixed_cubes(const McParams& p, const ChunkWords& v,
                                                          const ChunkPlace& at, bool in) {
    unsigned long long all = ~0ull, any = 0ull;
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
        const unsigned long long sx = (v.s[rr] >> 1) | (v.sn[rr] << 63);
        all &= v.s[rr] & sx;
        any |= v.s[rr] | sx;
    }
    return (in & (at.y + 1 < p.gy) & (at.z + 1 < p.gz)) ? (any & ~all) & low_bits(p.gx - 1 - 64 * at.j) : 0ull;
}
// The bits that the next chunk's first voxels have in the byte of cube 63.
__device__ __forceinline__ uint32_t next_bits(const ChunkWords& v) {
    return (((uint32_t)v.sn[0] & 1u) << 1) | (((uint32_t)v.sn[1] & 1u) << 3) |
           (((uint32_t)v.sn[2] & 1u) << 5) | (((uint32_t)v.sn[3] & 1u) << 7);
}
// Byte of cube k of a chunk with words s and next_bits nb.
__device__ __forceinline__ uint32_t cube_byte64(const unsigned long long s[4], uint32_t nb, int k) {
    return ((uint32_t)(s[0] >> k) & 3u) | (((uint32_t)(s[1] >> k) & 3u) << 2) |
           (((uint32_t)(s[2] >> k) & 3u) << 4) | (((uint32_t)(s[3] >> k) & 3u) << 6) | (k == 63 ? nb : 0u);
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

// The cube of triangle r among 16 cubes' counts w0 (the first 8), w1; r
// becomes the triangle's place in that cube.
__device__ __forceinline__ int cube_of(uint32_t w0, uint32_t w1, int& r) {
    const int c8 = sum8(w0);
    uint32_t left = r >= c8 ? w1 : w0;
    int j = r >= c8 ? 8 : 0;
    r -= r >= c8 ? c8 : 0;
#pragma unroll
    for (int h = 4; h >= 1; h >>= 1) {
        const int c = sum8(left & ((1u << (4 * h)) - 1u));
        const bool up = r >= c;
        r -= up ? c : 0;
        j += up ? h : 0;
        left >>= up ? 4 * h : 0;
    }
    return j;
}

// num / den by y = RN(1/den) and div_by_rcp; `bad` is set where that might not
// be the division's bits (a quotient near the denormals or out of range, -0).
__device__ __forceinline__ float short_quotient(float num, float den, float y, bool& bad) {
    const float an = fabsf(num);
    bad |= !((an >= 1e-30f) & (an <= 1e30f)) & (__float_as_uint(num) != 0u);
    return div_by_rcp(num, den, y);
}

// The lane whose elements include element k0 + lane of the lanes' elements
// (first element excl, count n per lane; k0 below their total): marks at the
// first elements, a max-scan, and the lane that element k0 is in before the
// first mark.  Every lane calls.
__device__ __forceinline__ int unit_owner(int* mark, int excl, int n, int k0, int lane) {
    mark[lane] = 0;
    if (n > 0 && excl >= k0 && excl < k0 + 64) mark[excl - k0] = lane + 1;
    __builtin_amdgcn_wave_barrier();
    const int mx = wave_inclusive_max(mark[lane]);
    const int first = 63 - __builtin_clzll(__ballot(n > 0 && excl <= k0) | 1ull);
    __builtin_amdgcn_wave_barrier();
    return mx > 0 ? mx - 1 : first;
}

// Scratch of the passes: the signs of every chunk; with `verts` its first
// vertex and triangle in its count block and every group's numbers of both;
// per count block its sums, the totals, and the list of units (uint32 with
// `verts`, else 64-bit words).
struct SignScratch {
    unsigned long long* signs;
    int32_t *voff, *toff;
    int2* group;
    long long *vsums, *tsums, *total;
    uint32_t* nunits;
    void* units;
};
// The parameters of a grid (each extent >= 2, fewer than 2^31 voxels) and the
// bytes of its scratch, laid out from base.
size_t sign_layout(const float* field, const int32_t grid[3], const float vs[3], const float off[3],
                   bool verts, char* base, SignParams& w, SignScratch& sc);
// Signs, counts and scan: vertices and total[0] only with `verts`; the list
// holds the units of the outputs that are wanted.
int launch_signs(const SignParams& w, const SignScratch& sc, bool verts, bool want_v, bool want_t,
                 hipStream_t s);

}  // namespace recon
