// mc_signs.hip -- the sign, count and scan passes of marching cubes
// (mc_signs.hpp), for the soup (marching_cubes.hip) and the welded mesh
// (mc_weld.hip).  They replace the reference's per-layer classification and
// host compaction (marching_cubes.cu:76-84,118-130,163-188).
#pragma clang fp contract(off)

#include "mc_signs.hpp"

namespace recon {

// Signs of every chunk: eight chunks a wavefront, one 4-byte load a lane and
// chunk, all in flight together.  It is the one pass over the whole field:
// 250 x 333 x 287 voxels in 18 us, 5.3 TB/s.  A count kernel that read the
// field itself took ten loads per four voxel rows (each row two and a half
// times) and was bound by their addresses: 41 us there, against 29 for this
// kernel and the count of the signs.  512^3 voxels in 110 us, 4.9 TB/s, where
// the soup's count of the field took 129.  16 chunks a wavefront are no faster.
__global__ __launch_bounds__(64 * kUnitWaves) void sign_kernel(const SignParams w,
                                                              unsigned long long* __restrict__ signs,
                                                              uint32_t* __restrict__ nunits) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *nunits = 0;  // for the count kernel
    const McParams& p = w.mc;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t c0 = kSignChunks * (blockIdx.x * kUnitWaves + (uint32_t)wave);
    if (c0 >= (uint32_t)w.nchunks) return;
    // lane k (of every eight): chunk c0 + k (the last one past the end), its
    // first voxel and the voxels after that in its row
    const uint32_t cl = min(c0 + (uint32_t)(lane & (kSignChunks - 1)), (uint32_t)w.nchunks - 1u);
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

// Counts: a lane a chunk.  The lane's eight words (its own and the next
// chunk's, of four rows) give its vertices and its cubes with both signs, whose
// triangles come from the table: cube by cube in every lane at once, or, where
// a few chunks hold many, chunk by chunk with a cube a lane.  A workgroup
// stores its chunks' places and appends the units of work to the write pass's
// list, in any order between workgroups (what a unit writes and where does not
// depend on it).  250 x 333 x 287 voxels 12 us, 512^3 29; with the chunks one
// by one throughout 23 and 45, 16 lanes a chunk 14 (the first).
template <bool VERTS>
__global__ __launch_bounds__(kBlockChunks) void sign_count_kernel(
    const SignParams w, const unsigned long long* __restrict__ signs, int32_t* __restrict__ voff,
    int32_t* __restrict__ toff, int2* __restrict__ group, long long* __restrict__ vsums,
    long long* __restrict__ tsums, bool want_v, bool want_t, void* __restrict__ units,
    uint32_t* __restrict__ nunits) {
    constexpr int kWaves = kBlockChunks / 64;
    __shared__ uint8_t ntab[256];
    __shared__ int wv[kWaves], wt[kWaves], wu[kWaves];
    __shared__ uint32_t ubase;
    const McParams& p = w.mc;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t nchunks = (uint32_t)w.nchunks;
    const uint32_t c = kBlockChunks * blockIdx.x + threadIdx.x;
    const bool in = c < nchunks;
    const ChunkPlace at = chunk_place(w, min(c, nchunks - 1u));
    const ChunkWords v = chunk_words(w, signs, c, at, in);
    if (threadIdx.x < 256) ntab[threadIdx.x] = mc_ntab_qbyte((int)threadIdx.x);
    __syncthreads();
    int nv = 0, nt = 0;
    unsigned long long mixed = 0;
    if (__ballot(any_negative(v))) {
        if (VERTS && in) {
            unsigned long long m[3];
            sign_edges(p, at.j, at.y, at.z, v.s[0], v.sn[0], v.s[2], v.s[1], m);
            nv = __popcll(m[0]) + __popcll(m[1]) + __popcll(m[2]);
        }
        mixed = mixed_cubes(p, v, at, in);
    }
    const int cubes = __popcll(mixed);
    const uint32_t nb = next_bits(v);
    unsigned long long todo = __ballot(mixed != 0ull);
    const int most = __builtin_amdgcn_readlane(wave_inclusive_max(cubes), 63);
    if (most <= 4 * __popcll(todo)) {
        for (unsigned long long left = mixed; left;) {  // the lowest and the highest at once
            const int lo = __builtin_ctzll(left), hi = 63 - __builtin_clzll(left);
            const int nlo = (int)ntab[cube_byte64(v.s, nb, lo)], nhi = (int)ntab[cube_byte64(v.s, nb, hi)];
            nt += nlo + (hi != lo ? nhi : 0);
            left &= ~((1ull << lo) | (1ull << hi));
        }
    } else {
        auto lane64 = [](unsigned long long x, int k) {
            return ((unsigned long long)(uint32_t)__builtin_amdgcn_readlane((int)(x >> 32), k) << 32) |
                   (uint32_t)__builtin_amdgcn_readlane((int)x, k);
        };
        while (todo) {
            const int k = __builtin_ctzll(todo);
            todo &= todo - 1ull;
            const unsigned long long s[4] = {lane64(v.s[0], k), lane64(v.s[1], k), lane64(v.s[2], k),
                                             lane64(v.s[3], k)};
            const uint32_t byte = cube_byte64(s, (uint32_t)__builtin_amdgcn_readlane((int)nb, k), lane);
            const int n = (int)(lane64(mixed, k) >> lane) & 1 ? (int)ntab[byte] : 0;  // <= 5
            const int sum =
                __popcll(__ballot(n & 1)) + 2 * __popcll(__ballot(n & 2)) + 4 * __popcll(__ballot(n & 4));
            nt = lane == k ? sum : nt;
        }
    }
    const int iv = VERTS ? wave_inclusive_scan(nv, lane) : 0, it = wave_inclusive_scan(nt, lane);
    int mine = 0;                    // units that the lane appends
    unsigned long long starts = 0;   // soup: lanes whose chunk begins a unit
    if (VERTS) {
        // per group (16 lanes) its counts and units
        const int last = lane | 15, prev = (lane - 16) | 15;
        const int lv = __shfl(iv, last, 64), pv = __shfl(iv, prev, 64);
        const int lt = __shfl(it, last, 64), pt = __shfl(it, prev, 64);
        const int gv = lv - (lane > 15 ? pv : 0), gt = lt - (lane > 15 ? pt : 0);
        if ((lane & 15) == 0 && in) {
            group[c / kGroupChunks] = make_int2(gv, gt);
            const int rounds = (want_v ? (gv + 63) / 64 : 0) + (want_t ? (gt + 63) / 64 : 0);
            mine = (rounds + kUnitRounds - 1) / kUnitRounds;
        }
    } else if (want_t) {
        // units by the cubes before the chunk, in steps of kUnitCubes
        const int step = (wave_inclusive_scan(cubes, lane) - cubes) / kUnitCubes;
        const unsigned long long act = __ballot(cubes > 0), below = act & ((1ull << lane) - 1ull);
        const int before = __shfl(step, below ? 63 - __builtin_clzll(below) : 0, 64);
        mine = cubes > 0 && (!below || before != step) ? 1 : 0;
        starts = __ballot(mine);
    }
    const int iu = wave_inclusive_scan(mine, lane);
    if (lane == 63) {
        wv[wave] = iv;
        wt[wave] = it;
        wu[wave] = iu;
    }
    __syncthreads();
    int bv = 0, bt = 0, bu = 0, av = 0, at_all = 0, au = 0;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) {
        bv += k < wave ? wv[k] : 0;
        bt += k < wave ? wt[k] : 0;
        bu += k < wave ? wu[k] : 0;
        av += wv[k];
        at_all += wt[k];
        au += wu[k];
    }
    if (in) {
        if (VERTS) voff[c] = bv + iv - nv;
        if (VERTS) toff[c] = bt + it - nt;
    }
    if (threadIdx.x == 0) {
        if (VERTS) vsums[blockIdx.x] = av;
        tsums[blockIdx.x] = at_all;
        if (au) ubase = atomicAdd(nunits, (uint32_t)au);
    }
    if (!au) return;
    __syncthreads();
    const uint32_t base = ubase + (uint32_t)(bu + iu - mine);
    if (VERTS) {
        for (int k = 0; k < mine; ++k)
            static_cast<uint32_t*>(units)[base + k] = (c / kGroupChunks << kUnitBits) | (uint32_t)k;
    } else if (mine) {
        const unsigned long long after = lane < 63 ? starts >> (lane + 1) : 0ull;
        const int len = after ? 1 + __builtin_ctzll(after) : 64 - lane;
        static_cast<unsigned long long*>(units)[base] = ((unsigned long long)(unsigned)(bt + it - nt) << kSoupTriShift) |
                                                        ((unsigned long long)c << 6) | (unsigned)(len - 1);
    }
}

// Block sums to first indices in place, the totals to total[0] (vertices) and
// total[1] (triangles): a workgroup an array, the first the triangles'.
__global__ __launch_bounds__(256) void sign_scan_kernel(long long* __restrict__ tsums,
                                                        long long* __restrict__ vsums, int nb,
                                                        long long* __restrict__ total) {
    constexpr int kItems = 8;
    __shared__ long long sh[4];
    long long* __restrict__ sums = blockIdx.x ? vsums : tsums;
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
    if (threadIdx.x == 0) total[1 - (int)blockIdx.x] = carry;
}

static size_t align256(size_t b) { return (b + 255) / 256 * 256; }

size_t sign_layout(const float* field, const int32_t grid[3], const float vs[3], const float off[3],
                   bool verts, char* base, SignParams& w, SignScratch& sc) {
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
    const size_t n = (size_t)w.nchunks, nb = (n + kBlockChunks - 1) / kBlockChunks;
    const size_t ng = verts ? nb * kBlockGroups : 0;
    size_t at = 0;
    auto take = [&](size_t bytes) {
        char* q = base + at;
        at += align256(bytes);
        return q;
    };
    sc.signs = reinterpret_cast<unsigned long long*>(take(8 * n));
    sc.voff = reinterpret_cast<int32_t*>(take(verts ? 4 * n : 0));
    sc.toff = reinterpret_cast<int32_t*>(take(verts ? 4 * n : 0));
    sc.group = reinterpret_cast<int2*>(take(8 * ng));
    sc.vsums = reinterpret_cast<long long*>(take(verts ? 8 * nb : 0));
    sc.tsums = reinterpret_cast<long long*>(take(8 * nb));
    sc.total = reinterpret_cast<long long*>(take(16));
    sc.nunits = reinterpret_cast<uint32_t*>(take(4));
    sc.units = take(verts ? (sizeof(uint32_t) << kUnitBits) * ng
                          : sizeof(unsigned long long) * kWaveUnits * nb * (kBlockChunks / 64));
    return at;
}

int launch_signs(const SignParams& w, const SignScratch& sc, bool verts, bool want_v, bool want_t,
                 hipStream_t s) {
    const unsigned n = (unsigned)w.nchunks, nb = (n + kBlockChunks - 1) / kBlockChunks;
    constexpr unsigned kSignBlock = kSignChunks * kUnitWaves;
    hipLaunchKernelGGL(sign_kernel, dim3((n + kSignBlock - 1) / kSignBlock), dim3(64 * kUnitWaves), 0, s, w,
                       sc.signs, sc.nunits);
    RECON_HIP_TRY(hipGetLastError(), "sign_kernel launch");
    if (verts)
        hipLaunchKernelGGL(sign_count_kernel<true>, dim3(nb), dim3(kBlockChunks), 0, s, w, sc.signs, sc.voff,
                           sc.toff, sc.group, sc.vsums, sc.tsums, want_v, want_t, sc.units, sc.nunits);
    else
        hipLaunchKernelGGL(sign_count_kernel<false>, dim3(nb), dim3(kBlockChunks), 0, s, w, sc.signs, sc.voff,
                           sc.toff, sc.group, sc.vsums, sc.tsums, want_v, want_t, sc.units, sc.nunits);
    RECON_HIP_TRY(hipGetLastError(), "sign_count_kernel launch");
    hipLaunchKernelGGL(sign_scan_kernel, dim3(verts ? 2 : 1), dim3(256), 0, s, sc.tsums, sc.vsums, (int)nb,
                       sc.total);
    RECON_HIP_TRY(hipGetLastError(), "sign_scan_kernel launch");
    return RECON_OK;
}

}  // namespace recon
