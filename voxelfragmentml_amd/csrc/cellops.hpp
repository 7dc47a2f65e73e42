// Device helpers for cell-parallel stages: each thread owns 8 consecutive
// cells of one job's linear index range (x*ny*nz + y*nz + z), loaded and
// stored as one 16-byte access when the run is complete, element-wise at the
// tail; or 8 cells of a column, a byte of its occupancy words, in bricks (CellGroup).
#pragma once

#include <algorithm>

#include "jobs.hpp"
#include "tune.hpp"

namespace vf {

// Bits of the correctly rounded float square root of an integer n < 2^24, exactly: the estimate
// moves to a float neighbour while sqrt(n) lies beyond the midpoint towards it.  Midpoints of
// adjacent floats have at most 25 significant bits, so their sums and squares are exact in double,
// and no midpoint squares to an integer below 2^48, so there are no ties.
__device__ inline uint32_t sqrt_rn_bits(uint32_t n)
{
    uint32_t b = __float_as_uint(__builtin_sqrtf((float)n));
    const double dn = (double)n;
    for (int it = 0; it < 4; ++it) {
        const double f = (double)__uint_as_float(b);
        if (b > 0u) {
            const double lo = 0.5 * ((double)__uint_as_float(b - 1u) + f);
            if (lo * lo > dn) {
                --b;
                continue;
            }
        }
        const double hi = 0.5 * (f + (double)__uint_as_float(b + 1u));
        if (hi * hi < dn) {
            ++b;
            continue;
        }
        break;
    }
    return b;
}


// x / d for x below 2^24, d below 2^16 and inv = 1 / d: a float estimate off by at most one, corrected.
__device__ inline uint32_t small_div(uint32_t x, uint32_t d, float inv)
{
    uint32_t q = (uint32_t)((float)x * inv);
    const int r = (int)x - (int)(q * d);
    if (r < 0) --q;
    else if (r >= (int)d) ++q;
    return q;
}

constexpr uint32_t kCellThreads = 256;
constexpr uint32_t kCellsPerThread = 8;
static_assert(kCellThreads * kCellsPerThread == kTileCells, "tile shape");

__device__ inline void load8(const uint16_t* p, uint64_t c0, uint64_t V, uint16_t v[8])
{
    if (c0 + 8 <= V) {
        const uint4 q = gload4(p + c0);
        v[0] = (uint16_t)q.x; v[1] = (uint16_t)(q.x >> 16);
        v[2] = (uint16_t)q.y; v[3] = (uint16_t)(q.y >> 16);
        v[4] = (uint16_t)q.z; v[5] = (uint16_t)(q.z >> 16);
        v[6] = (uint16_t)q.w; v[7] = (uint16_t)(q.w >> 16);
    } else {
        for (int k = 0; k < 8; ++k) v[k] = c0 + k < V ? gcast<const uint16_t>(p)[c0 + k] : (uint16_t)0;
    }
}

__device__ inline void store8(uint16_t* p, uint64_t c0, uint64_t V, const uint16_t v[8])
{
    if (c0 + 8 <= V) {
        uint4 q;
        q.x = (uint32_t)v[0] | ((uint32_t)v[1] << 16);
        q.y = (uint32_t)v[2] | ((uint32_t)v[3] << 16);
        q.z = (uint32_t)v[4] | ((uint32_t)v[5] << 16);
        q.w = (uint32_t)v[6] | ((uint32_t)v[7] << 16);
        gstore4(p + c0, q);
    } else {
        for (int k = 0; k < 8; ++k)
            if (c0 + k < V) gcast<uint16_t>(p)[c0 + k] = v[k];
    }
}

// Brick `id` of job J: its first cell.
struct BrickAt {
    uint32_t x, y, z;
};
__device__ inline BrickAt brick_at(const JobDev& J, uint32_t id)
{
    const uint32_t tz = (J.nz + kBrickZ - 1u) / kBrickZ, ty = (J.ny + kBrickY - 1u) / kBrickY, t = id / tz;
    return BrickAt{ t / ty * kBrickX, t % ty * kBrickY, id % tz * kBrickZ };
}

// The cells of one thread in a brick: byte tid % 4 of the occupancy word of row tid / 4, i.e. cells z0 .. z0 + n - 1 of
// column col (n = 8, less at the column's end, 0 outside the grid), linear index c0.
static_assert(kBrickX * kBrickY * 4 == kCellThreads && kBrickZ == 32, "a thread owns a byte of occupancy");
struct CellGroup {
    uint64_t c0;
    uint32_t col, z0, n;
};
__device__ inline CellGroup cell_group(const JobDev& J, const BrickAt& b)
{
    CellGroup g;
    const uint32_t row = threadIdx.x >> 2, x = b.x + row / kBrickY, y = b.y + row % kBrickY;
    g.col = x * J.ny + y;
    g.z0 = b.z + (threadIdx.x & 3u) * 8u;
    g.n = x < J.nx && y < J.ny && g.z0 < J.nz ? min(8u, J.nz - g.z0) : 0u;
    g.c0 = (uint64_t)g.col * J.nz + g.z0;
    return g;
}
__device__ inline CellGroup cell_group(const JobDev& J, uint32_t brick) { return cell_group(J, brick_at(J, brick)); }
// Which of the n <= N bricks from brick `first` of job J on hold an occupied cell, as bits, the same for the whole workgroup
// (of kCellThreads threads, all of which call this): a brick's rows are one occupancy word each, and lane l looks at rows of
// brick first + l % N, so a run costs about as much as one brick by itself (which divides its index in every lane).
template <uint32_t N>
__device__ inline uint32_t live_bricks(const JobDev& J, uint32_t first, uint32_t n)
{
    static_assert((N & (N - 1)) == 0 && N <= 32, "lanes of a wave repeat the run");
    constexpr uint32_t kRows = N < 4 ? 1 : N / 4, kColumns = kBrickX * kBrickY;
    const uint32_t r = threadIdx.x % N, row0 = threadIdx.x / N * kRows;
    uint32_t occ = 0;
    if (r < n && row0 < kColumns) {
        const BrickAt b = brick_at(J, first + r);
#pragma unroll
        for (uint32_t k = 0; k < kRows; ++k) {
            const uint32_t x = b.x + (row0 + k) / kBrickY, y = b.y + (row0 + k) % kBrickY;
            if (x < J.nx && y < J.ny) occ |= gcast<const uint32_t>(J.occ)[((size_t)x * J.ny + y) * J.wp + b.z / 32u];
        }
    }
    uint64_t m = __ballot(occ != 0u);
#pragma unroll
    for (uint32_t o = 32; o >= N; o >>= 1) m |= m >> o;
    const uint32_t mine = N < 32 ? (uint32_t)m & ((1u << (N & 31u)) - 1u) : (uint32_t)m;
    return (uint32_t)__ockl_wgred_or_i32((int)mine);
}
// the group's byte of an array of occupancy words
__device__ inline size_t group_byte(const JobDev& J, const CellGroup& g) { return (size_t)g.col * J.wp * 4u + (g.z0 >> 3); }
// the group's occupancy bits (0 for a group without cells)
__device__ inline uint32_t group_occ(const JobDev& J, const CellGroup& g)
{
    return g.n ? gcast<const uint8_t>(J.occ)[group_byte(J, g)] : 0u;
}
__device__ inline void store_group(uint16_t* p, const CellGroup& g, uint4 q)
{
    if (g.n == 8u) {
        gstore4_cells(p + g.c0, q);
    } else {
        const uint32_t w[4] = { q.x, q.y, q.z, q.w };
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k)
            if (k < g.n) gcast<uint16_t>(p)[g.c0 + k] = (uint16_t)(w[k >> 1] >> (16u * (k & 1u)));
    }
}
__device__ inline uint4 load_group(const uint16_t* p, const CellGroup& g)
{
    if (g.n == 8u) return gload4_cells(p + g.c0);
    uint32_t w[4] = { 0u, 0u, 0u, 0u };
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k)
        if (k < g.n) w[k >> 1] |= (uint32_t)gcast<const uint16_t>(p)[g.c0 + k] << (16u * (k & 1u));
    return make_uint4(w[0], w[1], w[2], w[3]);
}
__device__ inline uint4 pack_cells(const uint16_t v[8])
{
    return make_uint4((uint32_t)v[0] | ((uint32_t)v[1] << 16), (uint32_t)v[2] | ((uint32_t)v[3] << 16),
                      (uint32_t)v[4] | ((uint32_t)v[5] << 16), (uint32_t)v[6] | ((uint32_t)v[7] << 16));
}
__device__ inline bool occ_bit(const JobDev& J, uint32_t x, uint32_t y, uint32_t z)
{
    return (gcast<const uint32_t>(J.occ)[((size_t)x * J.ny + y) * J.wp + (z >> 5)] >> (z & 31u)) & 1u;
}

// Contiguous tile range of this block (keeps a block on one job for long
// stretches so per-job reductions flush rarely).
__device__ inline void block_tile_range(uint32_t total, uint32_t& b, uint32_t& e)
{
    uint32_t per = (total + gridDim.x - 1) / gridDim.x;
    b = blockIdx.x * per;
    if (b > total) b = total;
    e = b + per;
    if (e > total) e = total;
}

// Copy a job descriptor into LDS (block-wide; every thread must call it).
__device__ inline void stage_job(JobDev* sJ, const JobDev* src)
{
    static_assert(sizeof(JobDev) % 4 == 0, "JobDev is copied as words");
    __syncthreads();
    const uint32_t* s = reinterpret_cast<const uint32_t*>(src);
    uint32_t* d = reinterpret_cast<uint32_t*>(sJ);
    for (uint32_t i = threadIdx.x; i < sizeof(JobDev) / 4; i += blockDim.x) d[i] = s[i];
    __syncthreads();
}

// Walk this block's contiguous range of the global tiles (prefix: njobs + 1
// tile prefix over the jobs).  The job is tracked incrementally and its
// descriptor staged in LDS on every change, so a tile costs no lookup and no
// dependent descriptor loads.  f(J, j, local_tile) runs block-uniformly;
// leave(j) runs before the block moves off job j and at the end.
template <class F, class G>
__device__ inline void walk_tiles(const Launch& L, const uint32_t* prefix, uint32_t total, JobDev* sJ, F&& f, G&& leave)
{
    uint32_t tb, te;
    block_tile_range(total, tb, te);
    if (tb >= te) return;
    uint32_t j = find_job(prefix, L.njobs, tb);
    uint32_t jb = prefix[j], je = prefix[j + 1];
    stage_job(sJ, L.jobs + j);
    for (uint32_t t = tb; t < te; ++t) {
        if (t >= je) {
            leave(j);
            do {
                ++j;
                jb = je;
                je = prefix[j + 1];
            } while (t >= je);
            stage_job(sJ, L.jobs + j);
        }
        f(*sJ, j, t - jb, t);
    }
    leave(j);
}

template <class F>
__device__ inline void walk_tiles(const Launch& L, const uint32_t* prefix, uint32_t total, JobDev* sJ, F&& f)
{
    walk_tiles(L, prefix, total, sJ, f, [](uint32_t) {});
}

// The same walk in runs of up to N consecutive tiles of one job:
// f(J, j, first_local_tile, n) handles tiles first .. first + n - 1 (n <= N),
// so a streaming stage can issue all its loads before using any of them.
// leave(j) runs when the block is done with job j (as in walk_tiles).
template <uint32_t N, class F, class G>
__device__ inline void walk_tile_runs(const Launch& L, const uint32_t* prefix, uint32_t total, JobDev* sJ, F&& f, G&& leave)
{
    uint32_t tb, te;
    block_tile_range(total, tb, te);
    if (tb >= te) return;
    uint32_t j = find_job(prefix, L.njobs, tb);
    uint32_t jb = prefix[j], je = prefix[j + 1];
    stage_job(sJ, L.jobs + j);
    for (uint32_t t = tb; t < te;) {
        if (t >= je) {
            leave(j);
            do {
                ++j;
                jb = je;
                je = prefix[j + 1];
            } while (t >= je);
            stage_job(sJ, L.jobs + j);
        }
        const uint32_t n = min(N, min(te, je) - t);
        f(*sJ, j, t - jb, n);
        t += n;
    }
    leave(j);
}

template <uint32_t N, class F>
__device__ inline void walk_tile_runs(const Launch& L, const uint32_t* prefix, uint32_t total, JobDev* sJ, F&& f)
{
    walk_tile_runs<N>(L, prefix, total, sJ, f, [](uint32_t) {});
}

// Runs of N consecutive tiles by workgroups that keep to one job (their per-job sums are flushed once, by leave(j)):
// job j has prefix[j + 1] / per - prefix[j] / per + 1 workgroups (total / per + njobs in all), which take its runs in
// turn, so each sees the job's full and empty regions alike.
template <uint32_t N, class F, class G>
__device__ inline void walk_job_runs(const Launch& L, const uint32_t* prefix, uint32_t total, uint32_t per, JobDev* sJ, F&& f,
                                     G&& leave)
{
    uint32_t lo = 0, hi = L.njobs;  // largest j whose first workgroup, prefix[j] / per + j, is not after this one
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (prefix[mid] / per + mid <= blockIdx.x) lo = mid; else hi = mid;
    }
    const uint32_t jb = prefix[lo], n = prefix[lo + 1] - jb, b0 = jb / per + lo, nb = (jb + n) / per + lo + 1 - b0;
    if ((uint64_t)(blockIdx.x - b0) * N >= n) return;
    stage_job(sJ, L.jobs + lo);
    for (uint64_t t = (uint64_t)(blockIdx.x - b0) * N; t < n; t += (uint64_t)nb * N) f(*sJ, (uint32_t)t, min(N, n - (uint32_t)t));
    leave(lo);
}

// Job prefixes kept in LDS by the stages that search them per tile (njobs <= 1024).
constexpr uint32_t kWalkMaxJobs = 1024;

// Grid-stride over runs of N consecutive tiles: run r (tiles r*N .. r*N + N - 1, split where a job
// ends) goes to block r % gridDim.x, and f(J, j, first_local_tile, n) handles n <= N tiles of job j,
// so a stage whose tiles differ in cost keeps the round-robin balance and can still issue the
// loads of a whole run before using any of them.
template <uint32_t N, class F>
__device__ inline void walk_tile_runs_strided(const Launch& L, const uint32_t* prefix, uint32_t total, JobDev* sJ,
                                              uint32_t* sp, F&& f)
{
    for (uint32_t i = threadIdx.x; i <= L.njobs && i <= kWalkMaxJobs; i += blockDim.x) sp[i] = prefix[i];
    __syncthreads();
    uint32_t cur = 0xFFFFFFFFu;
    const uint32_t runs = (total + N - 1) / N;
    for (uint32_t r = blockIdx.x; r < runs; r += gridDim.x) {
        uint32_t t = r * N;
        const uint32_t t1 = min(t + N, total);
        while (t < t1) {
            uint32_t lo = 0, hi = L.njobs;  // largest j with sp[j] <= t
            while (hi - lo > 1) {
                const uint32_t mid = (lo + hi) >> 1;
                if (sp[mid] <= t) lo = mid; else hi = mid;
            }
            if (lo != cur) {
                stage_job(sJ, L.jobs + lo);
                cur = lo;
            }
            const uint32_t n = min(t1, sp[lo + 1]) - t;
            f(*sJ, lo, t - sp[lo], n);
            t += n;
        }
    }
}

__device__ inline void decompose(uint64_t c, const JobDev* J, uint32_t& x, uint32_t& y, uint32_t& z)
{
    uint32_t yz = J->ny * J->nz;
    uint32_t cc = (uint32_t)c;
    x = cc / yz;
    uint32_t r = cc - x * yz;
    y = r / J->nz;
    z = r - y * J->nz;
}

__device__ inline void advance(uint32_t& x, uint32_t& y, uint32_t& z, const JobDev* J)
{
    if (++z == J->nz) {
        z = 0;
        if (++y == J->ny) {
            y = 0;
            ++x;
        }
    }
}

__device__ inline unsigned long long wave_sum_u64(unsigned long long v)
{
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

}  // namespace vf
