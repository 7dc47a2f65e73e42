// Cell-parallel grid stages: occupancy <-> labels, homogenize, mask removal,
// boundary detection (optionally fused with the per-fragment histogram),
// histogram, occupied count and the order-independent grid checksum.
// All are HBM-bound streaming passes; each thread owns 8 cells.
#include <type_traits>

#include "cellops.hpp"

namespace vf {

namespace {

template <class F>
__device__ inline void for_each_tile(const Launch& L, F&& f)
{
    __shared__ JobDev sJ;
    walk_tiles(L, L.tile_prefix, L.total_tiles, &sJ, [&](const JobDev& J, uint32_t, uint32_t local, uint32_t) {
        if (!J.active) return;
        const uint64_t c0 = (uint64_t)local * kTileCells + threadIdx.x * kCellsPerThread;
        if (c0 < J.V) f(J, c0);
    });
}

// f(J, group) for every group of cells of a single grid, in the order of its columns' bytes of occupancy: lanes read and write
// one after another whatever the edges are (by bricks of 8 x 8 x 32 cells, a 2048 x 2048 x 1 grid took 50 us from labels and 42 to
// labels, now 24 and 16; 301 x 430 x 223 30 and 24, now 24 and 19).
template <class F>
__device__ inline void for_each_group(const Launch& L, F&& f)
{
    const JobDev& J = *L.jobs;
    const uint32_t nz = J.nz, per = (nz + 7u) / 8u, total = J.nx * J.ny * per;
    for (uint32_t id = blockIdx.x * kCellThreads + threadIdx.x; id < total; id += gridDim.x * kCellThreads) {
        CellGroup g;
        g.col = id / per;
        g.z0 = (id - g.col * per) * 8u;
        g.n = min(8u, nz - g.z0);
        g.c0 = (uint64_t)g.col * nz + g.z0;
        f(J, g);
    }
}
inline uint32_t group_blocks(const Launch& L)
{
    return std::max(1u, std::min(L.total_bricks, 2u * active_shape().cell_blocks));  // a brick has 256 groups at most
}

// The last group of a column of at least 8 cells takes the column's last 8 in its place (first: the cell they begin at), so
// that every group is one access: its own are the upper ones, and the others' values are what their own group has.
__device__ inline uint32_t whole_group(const JobDev& J, const CellGroup& g) { return g.n < 8u && J.nz >= 8u ? J.nz - 8u : g.z0; }

__global__ __launch_bounds__(kCellThreads) void k_occ_to_labels(Launch L)
{
    for_each_group(L, [&](const JobDev& J, CellGroup g) {
        const auto* byte = gcast<const uint8_t>(J.occ) + group_byte(J, g);
        const uint32_t z = whole_group(J, g), back = g.z0 - z;  // cells of the group before
        uint32_t o = byte[0];
        if (back) {
            o = (o << 8 | byte[-1]) >> (8u - back);
            g.n = 8u;
            g.c0 -= back;
        }
        uint16_t v[8];
        for (int k = 0; k < 8; ++k) v[k] = (uint16_t)((o >> k) & 1u);
        store_group(J.labels, g, pack_cells(v));
    });
}

__global__ __launch_bounds__(kCellThreads) void k_labels_to_occ(Launch L)
{
    for_each_group(L, [&](const JobDev& J, CellGroup g) {
        const uint32_t back = g.z0 - whole_group(J, g);
        if (back) {
            g.n = 8u;
            g.c0 -= back;
        }
        const uint4 q = load_group(J.labels, g);
        const uint32_t w[4] = { q.x, q.y, q.z, q.w };
        uint32_t o = 0;
        for (int k = 0; k < 8; ++k) o |= ((w[k >> 1] >> (16 * (k & 1))) & 0xFFFFu ? 1u : 0u) << k;
        o >>= back;
        auto* byte = gcast<uint8_t>(J.occ) + group_byte(J, g);
        const uint32_t in_word = (g.z0 >> 3) & 3u;
        if (g.z0 + 8u < J.nz) byte[0] = (uint8_t)o;
        else if (in_word == 0) *(VF_AS_GLOBAL uint32_t*)byte = o;  // with the rest of the column's last word
        else
            for (uint32_t k = in_word; k < 4u; ++k, o = 0) byte[k - in_word] = (uint8_t)o;
    });
}

__global__ __launch_bounds__(kCellThreads) void k_occ_free(Launch L, const uint32_t* bits)
{
    for_each_group(L, [&](const JobDev& J, const CellGroup& g) {
        const uint32_t o = gcast<const uint8_t>(bits)[group_byte(J, g)];
        for (uint32_t k = 0; k < 8u; ++k)
            if ((o >> k) & 1u) gcast<uint16_t>(J.labels)[g.c0 + k] = kFree;
    });
}

__global__ __launch_bounds__(kCellThreads) void k_occ_bytes(Launch L, uint8_t* out)
{
    for_each_group(L, [&](const JobDev& J, const CellGroup& g) {
        const uint32_t o = group_occ(J, g);
        uint32_t w[2];  // four bits to four bytes
        for (uint32_t q = 0; q < 2u; ++q) w[q] = (((o >> (4u * q)) & 15u) * 0x00204081u) & 0x01010101u;
        if (g.n == 8u) gstore2_bytes(out + g.c0, make_uint2(w[0], w[1]));
        else
            for (uint32_t k = 0; k < g.n; ++k) gcast<uint8_t>(out)[g.c0 + k] = (uint8_t)(w[k >> 2] >> (8u * (k & 3u)));
    });
}

// All cells EMPTY, in the cells' linear order: whole lines written one after another run at the rate of a fill (512^3:
// 268 MB in 35 us), where the fractures' bricks write rows of 64 bytes (the same bytes in 87 to 115 us).
__global__ __launch_bounds__(kCellThreads) void k_clear_labels(Launch L)
{
    __shared__ JobDev sJ;
    walk_tile_runs<8>(L, L.tile_prefix, L.total_tiles, &sJ, [&](const JobDev& J, uint32_t, uint32_t tile, uint32_t n) {
        if (!J.active) return;
        const uint16_t zero[8] = {};
        for (uint32_t r = 0; r < n; ++r) {
            const uint64_t c0 = (uint64_t)(tile + r) * kTileCells + threadIdx.x * kCellsPerThread;
            if (c0 < J.V) store8(J.labels, c0, J.V, zero);
        }
    });
}

__global__ __launch_bounds__(kCellThreads) void k_homogenize(Launch L)
{
    for_each_tile(L, [&](const JobDev& J, uint64_t c0) {
        uint16_t v[8];
        load8(J.labels, c0, J.V, v);
        for (int k = 0; k < 8; ++k) v[k] = v[k] != kEmpty ? kFree : kEmpty;
        store8(J.labels, c0, J.V, v);
    });
}

__global__ __launch_bounds__(kCellThreads) void k_undo_mask(Launch L, uint16_t keep)
{
    for_each_tile(L, [&](const JobDev& J, uint64_t c0) {
        uint16_t v[8];
        load8(J.labels, c0, J.V, v);
        for (int k = 0; k < 8; ++k) v[k] = (uint16_t)(v[k] & keep);
        store8(J.labels, c0, J.V, v);
    });
}

__global__ void k_put_head(GridHead* dst, GridHead h)
{
    static_assert(sizeof(GridHead) % 4 == 0, "copied as words");
    const uint32_t* s = reinterpret_cast<const uint32_t*>(&h);
    for (uint32_t i = threadIdx.x; i < sizeof(GridHead) / 4; i += blockDim.x) reinterpret_cast<uint32_t*>(dst)[i] = s[i];
}

constexpr uint32_t kPutSeeds = 128;  // seeds per launch: 2 KiB of arguments
struct SeedArgs {
    uint4 s[kPutSeeds];
};
__global__ void k_put_seeds(uint4* dst, SeedArgs a, uint32_t n)
{
    if (threadIdx.x < n) dst[threadIdx.x] = a.s[threadIdx.x];
}

__global__ void k_report(const unsigned long long* stats, const uint4* seeds, uint32_t n, uint32_t* host)
{
    if (threadIdx.x < kStatCount) reinterpret_cast<unsigned long long*>(host + kPinStats)[threadIdx.x] = stats[threadIdx.x];
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) reinterpret_cast<uint4*>(host + kPinSeeds)[i] = seeds[i];
}

// The histogram of a single grid.  Labels below kHistLds are counted in LDS by kHistBlocks workgroups of 16 waves,
// which then store the counts of those below kHistBins (1 MiB) for k_hist_sum and add the others, where there are any, to
// the counts in HBM; still larger labels go there cell by cell.  Bound by HBM: 2 bytes
// per cell.  A lane adds the cells of one label among its 8 with one LDS atomic; lanes of a wave that hold the same label
// follow each other at one a cycle, which costs less than counting them over the wave first (110 us for a 512^3 grid).
// 8192 workgroups that added their counts to the same few addresses in HBM took 98 us for a 512^3 grid and 57 us for a
// 256^3 one; now 75 and 20 us, of which clearing and summing take 10.  The word after the partial counts receives the largest
// label of kHistBins or more.  With those counted in HBM alone, 1500 labels in 8^3 blocks of a 256^3 grid took 400 us.
// 4096 bins: 12288 cost a grid of few labels 1.5 us of clearing and looking through them.
constexpr uint32_t kHistThreads = 1024, kHistLds = 4096;
__global__ __launch_bounds__(kHistThreads) void k_histogram(Launch L, uint32_t* part)
{
    __shared__ __attribute__((aligned(16))) uint32_t bins[kHistLds];
    __shared__ uint32_t largest;  // label, 0 where all are below kHistBins
    const JobDev& J = L.jobs[0];
    const uint16_t* labels = J.labels;
    const uint64_t V = J.V;
    for (uint32_t i = threadIdx.x; i < kHistLds / 4; i += kHistThreads) reinterpret_cast<uint4*>(bins)[i] = make_uint4(0u, 0u, 0u, 0u);
    if (threadIdx.x == 0) largest = 0;
    uint32_t top = 0;
    __syncthreads();
    constexpr uint64_t kStep = (uint64_t)kHistThreads * kCellsPerThread;
    constexpr uint32_t kRun = 4;  // steps whose loads are issued together
    const uint64_t steps = (V + kStep - 1) / kStep;
    // steps are dealt round-robin: a vessel's cells lie in some slabs of the box and not in others
    for (uint64_t s = blockIdx.x; s < steps; s += (uint64_t)kRun * gridDim.x) {
        uint4 q[kRun];
#pragma unroll
        for (uint32_t r = 0; r < kRun; ++r) {
            const uint64_t c0 = (s + (uint64_t)r * gridDim.x) * kStep + threadIdx.x * kCellsPerThread;
            q[r] = make_uint4(0u, 0u, 0u, 0u);
            if (c0 < V) {
                uint16_t v[8];
                load8(labels, c0, V, v);
                q[r] = pack_cells(v);
            }
        }
#pragma unroll
        for (uint32_t r = 0; r < kRun; ++r) {
            const uint32_t w[4] = { q[r].x, q[r].y, q[r].z, q[r].w };
            if ((w[0] | w[1] | w[2] | w[3]) == 0u) continue;
            uint32_t m[8], rest = 0;  // masked labels; the cells still to count
#pragma unroll
            for (uint32_t k = 0; k < 8u; ++k) {
                const uint32_t raw = (w[k >> 1] >> (16u * (k & 1u))) & 0xFFFFu;
                m[k] = raw & kMask15;
                rest |= raw > kFree ? 1u << k : 0u;
            }
            while (rest) {
                uint32_t l = 0, eq = 0;  // the first cell still to count; the cells of its label
#pragma unroll
                for (int k = 7; k >= 0; --k) l = (rest >> k) & 1u ? m[k] : l;
#pragma unroll
                for (uint32_t k = 0; k < 8u; ++k) eq |= m[k] == l ? 1u << k : 0u;
                eq &= rest;
                rest &= ~eq;
                if (l < kHistLds) {
                    atomicAdd(&bins[l], (uint32_t)__popc(eq));
                } else {
                    atomicAdd(J.hist + l, (uint32_t)__popc(eq));
                    top = max(top, l);
                }
            }
        }
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < kHistBins; i += kHistThreads) part[blockIdx.x * kHistBins + i] = bins[i];
#pragma unroll
    for (uint32_t i = kHistBins + threadIdx.x; i < kHistLds; i += kHistThreads) {
        const uint32_t c = bins[i];
        if (c) {
            atomicAdd(J.hist + i, c);
            top = max(top, i);
        }
    }
    if (top) atomicMax(&largest, top);
    __syncthreads();
    if (threadIdx.x == 0 && largest) atomicMax(part + kHistBlocks * kHistBins, largest);
}

// Sums nparts partial counts of 64 bins per workgroup into hist and, where given, host memory; the workgroups after those
// store the counts of larger labels there, where they occur.
constexpr uint32_t kLargeBlocks = 8;
__global__ __launch_bounds__(256) void k_hist_sum(const uint32_t* part, uint32_t nparts, uint32_t* hist, uint32_t* host)
{
    __shared__ uint32_t sum[4][64];
    if (blockIdx.x >= kHistBins / 64) {
        const uint32_t top = part[kHistBlocks * kHistBins];  // 0: no larger label
        for (uint32_t i = (blockIdx.x - kHistBins / 64) * 256u + threadIdx.x; i < kHistLargeHost && kHistBins + i <= top; i += kLargeBlocks * 256u)
            host[kPinLarge + i] = hist[kHistBins + i];
        return;
    }
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, bin = blockIdx.x * 64u + lane;
    uint32_t n = 0;
#pragma unroll 8
    for (uint32_t p = wave; p < nparts; p += 4u) n += part[p * kHistBins + bin];
    sum[wave][lane] = n;
    __syncthreads();
    if (wave == 0) {
        n = sum[0][lane] + sum[1][lane] + sum[2][lane] + sum[3][lane];
        hist[bin] = n;
        if (host) host[bin] = n;
    }
    if (host && blockIdx.x == 0 && threadIdx.x == 0) host[kHistBins] = part[kHistBlocks * kHistBins];
}

// The first kHistBins counts of every job to host memory.
__global__ __launch_bounds__(kHistBins / 4) void k_hist_heads(const JobDev* jobs, uint32_t* host)
{
    reinterpret_cast<uint4*>(host)[blockIdx.x * (kHistBins / 4) + threadIdx.x] = reinterpret_cast<const uint4*>(jobs[blockIdx.x].hist)[threadIdx.x];
}

__global__ void k_hist_clear(uint32_t* hist, uint32_t* flag)
{
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < 65536 / 4; i += gridDim.x * blockDim.x)
        gstore4(hist + 4 * i, make_uint4(0u, 0u, 0u, 0u));
    if (blockIdx.x == 0 && threadIdx.x == 0) *flag = 0u;
}

constexpr uint32_t kLdsBins = 4096;
constexpr uint32_t kTiledBins = 1024;  // LDS histogram bins of the tiled boundary kernel (larger labels go to HBM)

// Per-job sum of a per-thread value: wave sums, then one device atomic per block and job.
struct BlockSum {
    unsigned long long part[kCellThreads / 64];
    // stat of job J, in the block's line of its sums where it has any
    __device__ void flush(unsigned long long& acc, const JobDev& J, int stat)
    {
        unsigned long long* dst = J.sums ? J.sums + (blockIdx.x % kSumSlots) * kStatCount + stat : J.stats + stat;
        const unsigned long long s = wave_sum_u64(acc);
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned long long tot = 0;
            for (int w = 0; w < (int)(kCellThreads / 64); ++w) tot += part[w];
            if (tot) atomicAdd(dst, tot);
        }
        __syncthreads();
        acc = 0;
    }
};

// Checksum term of one cell c (linear index) holding v: a = fmix32(c ^ v * 0x9E3779B1),
// term = (a << 32) | fmix32(a ^ c ^ 0x7F4A7C15); EMPTY adds nothing.
__device__ inline unsigned long long checksum_term(uint16_t v, uint32_t c)
{
    if (!v) return 0ull;
    const uint32_t a = fmix32(c ^ ((uint32_t)v * 0x9E3779B1u));
    return ((unsigned long long)a << 32) | fmix32(a ^ c ^ 0x7F4A7C15u);
}


__device__ inline uint32_t ceil_div_d(uint32_t a, uint32_t b) { return (a + b - 1) / b; }

// Boundary bit of one labelled cell (detectBoundaries-comp.glsl:18-43).
__device__ inline bool is_boundary_cell(const JobDev* J, uint32_t x, uint32_t y, uint32_t z, uint16_t c, int b)
{
    const int nx = (int)J->nx, ny = (int)J->ny, nz = (int)J->nz;
    int x0 = max((int)x - b, 0), x1 = min((int)x + b, nx - 1);
    int y0 = max((int)y - b, 0), y1 = min((int)y + b, ny - 1);
    int z0 = max((int)z - b, 0), z1 = min((int)z + b, nz - 1);
    const uint16_t* g = J->labels;
    for (int xx = x0; xx <= x1; ++xx)
        for (int yy = y0; yy <= y1; ++yy) {
            const uint16_t* row = g + ((size_t)xx * ny + yy) * nz;
            for (int zz = z0; zz <= z1; ++zz) {
                uint16_t v = (uint16_t)(row[zz] & kMask15);
                if (v > kFree && v != c) return true;
            }
        }
    return false;
}

// Sets the boundary bits; HIST: and accumulates the per-fragment histogram.
// Generic path (any window size; used for jobs with size > 1).  In a table (HIST)
// it is restricted to those jobs, the tiled kernel handles the rest.
template <bool HIST>
__global__ __launch_bounds__(kCellThreads) void k_cells_post(Launch L, int bsize)
{
    __shared__ uint32_t bins[HIST ? kLdsBins : 1];
    uint32_t tb, te;
    block_tile_range(L.total_tiles, tb, te);
    if (tb >= te) return;
    uint32_t cur_job = find_job(L.tile_prefix, L.njobs, tb);
    if (HIST) {
        for (uint32_t i = threadIdx.x; i < kLdsBins; i += blockDim.x) bins[i] = 0;
        __syncthreads();
    }
    auto flush = [&](uint32_t j) {
        if (!HIST) return;
        __syncthreads();
        uint32_t* h = L.jobs[j].hist;
        for (uint32_t i = threadIdx.x; i < kLdsBins; i += blockDim.x) {
            uint32_t c = bins[i];
            if (c) {
                atomicAdd(h + i, c);
                bins[i] = 0;
            }
        }
        __syncthreads();
    };
    for (uint32_t t = tb; t < te; ++t) {
        uint32_t j = find_job(L.tile_prefix, L.njobs, t);
        if (j != cur_job) {
            flush(cur_job);
            cur_job = j;
        }
        const JobDev* J = L.jobs + j;
        if (!J->active || (HIST && J->bsize <= 1)) continue;
        uint64_t c0 = (uint64_t)(t - L.tile_prefix[j]) * kTileCells + threadIdx.x * kCellsPerThread;
        if (c0 >= J->V) continue;
        uint16_t v[8];
        load8(J->labels, c0, J->V, v);
        bool any = false;
        for (int k = 0; k < 8; ++k) any |= v[k] > kFree;
        if (!any) continue;
        bool changed = false;
        {
            const int bs = bsize >= 0 ? bsize : J->bsize;
            uint32_t x, y, z;
            decompose(c0, J, x, y, z);
            for (int k = 0; k < 8; ++k) {
                if (c0 + k < J->V && v[k] > kFree && is_boundary_cell(J, x, y, z, v[k], bs)) {
                    v[k] = (uint16_t)(v[k] | 0x8000u);
                    changed = true;
                }
                advance(x, y, z, J);
            }
        }
        if (HIST) {
            for (int k = 0; k < 8; ++k) {
                if (c0 + k < J->V && v[k] > kFree) {
                    uint32_t m = v[k] & kMask15;
                    if (m < kLdsBins) atomicAdd(&bins[m], 1u);
                    else atomicAdd(J->hist + m, 1u);
                }
            }
        }
        if (changed) store8(J->labels, c0, J->V, v);
    }
    flush(cur_job);
}

// Tiled detectBoundaries(1) + histogram.  A labelled cell c (2 <= raw < 0x8000)
// is a boundary cell iff its clamped 3x3x3 window holds a label > FREE other than
// its own, i.e. iff the window max of A = (m > 1 ? m : 0) or the window min of
// B = (m > 1 ? m : 0xFFFF) differs from raw(c) (m = value & 0x7FFF; c itself is in
// the window).  Cells whose bit 15 is already set never change.  Clamping the
// window equals replicate padding for max/min, so the halo is loaded with
// clamped coordinates.  8x8x32 bricks: the interior is loaded first with one
// 16-byte load per thread and bricks without a label stop there; live bricks
// load the halo and run separable max/min passes z, y, x in LDS.
constexpr int kBTX = 8, kBTY = 8, kBTZ = 32;
constexpr int kBHX = kBTX + 2, kBHY = kBTY + 2;
// z-pass row stride (words): a multiple of 4, so a thread's 8-value segment is two 16-byte LDS accesses;
// 36 = 9 groups of 4 banks per row, so the 16-byte accesses of 8 consecutive lanes (2 rows x 4 segments)
// fall on distinct bank groups
constexpr int kAZ = kBTZ + 4;

// TABLE: the jobs of a table, whose labels follow their occupancy; also accumulate
// the histogram and the grid checksum of the final cells (jobs with a window size <= 1; the others
// get theirs from k_checksum).
//
// Each thread owns an 8-cell z segment of one of the brick's 64 rows and loads
// it with its two z neighbours (clamped coordinates = replicate padding), so
// the z window is done in registers; 144 of the threads also do one segment
// of the 36 halo rows.  Only the z-window max/min of the 100 rows goes
// through LDS, for the 3x3 x/y window of each labelled cell.
//
// Bound by instructions: 20 to 30 % of the cells of the bricks with labels are labelled, in 30 to 40 % of the
// segments, but those lie in most of the waves.  The windows, counts and checksum are therefore worked for the
// segments that are not EMPTY, listed in LDS, by the first waves: 64 mixed grids 1.36 -> 0.94 ms, of which
// the runs dealt over a whole job (full and empty regions of a grid made some workgroups several times slower than
// others) and the look at a run's bricks by 4-byte occupancy words together made 1.28 -> 0.94.
// lane-wise max of two packed u16 pairs
__device__ inline uint32_t pk_max_u16(uint32_t a, uint32_t b)
{
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}
// a label as the packed pair (label | 0xFFFF - label)
__device__ inline uint32_t packed_self(uint32_t m) { return m | ((0xFFFFu - m) << 16); }

template <bool TABLE, uint32_t RUN>
__global__ __launch_bounds__(256) void k_boundaries_tiled(Launch L, uint32_t per)
{
    // z-window max (low 16 bits) | 0xFFFF - min (high 16) over labelled cells (EMPTY / FREE contribute 0),
    // so one packed u16 max combines both halves; row = hx * kBHY + hy
    __shared__ __attribute__((aligned(16))) uint32_t zmm[kBHX * kBHY * kAZ];
    __shared__ uint32_t bins[TABLE ? kTiledBins : 1];
    __shared__ JobDev sJ;
    __shared__ BlockSum csum_part;
    __shared__ uint4 cells[256];  // a brick's segments that are not EMPTY, by wave
    __shared__ uint8_t listed[256];
    __shared__ uint32_t count[4];
    unsigned long long csum = 0;
    if (TABLE) {
        for (uint32_t i = threadIdx.x; i < kTiledBins; i += blockDim.x) bins[i] = 0;
    }
    auto flush = [&](uint32_t j) {
        if (TABLE) csum_part.flush(csum, L.jobs[j], kStatChecksum);
        if (!TABLE) return;
        __syncthreads();
        uint32_t* h = L.jobs[j].hist;
        for (uint32_t i = threadIdx.x; i < kTiledBins; i += blockDim.x) {
            const uint32_t c = bins[i];
            if (c) {
                atomicAdd(h + i, c);
                bins[i] = 0;
            }
        }
        __syncthreads();
    };
    // this thread's interior segment: row (tx, ty) = tid / 4, z segment (tid % 4) * 8
    const int row = threadIdx.x >> 2, seg = (threadIdx.x & 3) * 8;
    const int tx = row / kBTY, ty = row % kBTY;
    // halo task (threads < 144): ring row r = tid / 4 of the 36 rows with hx in {0, 9} or hy in {0, 9}
    const bool halo_task = threadIdx.x < (2 * kBHY + 2 * kBTX) * 4;
    int hhx = 0, hhy = 0;
    {
        const int r = threadIdx.x >> 2;
        if (r < kBHY) { hhx = 0; hhy = r; }
        else if (r < 2 * kBHY) { hhx = kBHX - 1; hhy = r - kBHY; }
        else if (r < 2 * kBHY + kBTX) { hhx = r - 2 * kBHY + 1; hhy = 0; }
        else { hhx = r - 2 * kBHY - kBTX + 1; hhy = kBHY - 1; }
    }
    // packed z-window (max | 0xFFFF - min) of 8 cells from their 10 raw values w[0..9] (w[k+1] is cell k)
    auto zwin = [](const uint16_t w[10], uint32_t out[8]) {
        uint32_t p[10];
#pragma unroll
        for (int k = 0; k < 10; ++k) {
            const uint32_t m = w[k] & kMask15;
            p[k] = m > kFree ? packed_self(m) : 0u;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) out[k] = pk_max_u16(pk_max_u16(p[k], p[k + 1]), p[k + 2]);
    };
    constexpr uint32_t kRun = RUN;  // bricks per step: their interior loads are issued together
    walk_job_runs<kRun>(L, L.bt_prefix, L.total_bricks, per, &sJ, [&](const JobDev& J, uint32_t first, uint32_t nrun) {
        if (!J.active || J.bsize > 1) return;
        const int nx = (int)J.nx, ny = (int)J.ny, nz = (int)J.nz;
        const uint32_t tz = ceil_div_d(J.nz, kBTZ), tyn = ceil_div_d(J.ny, kBTY);
        const bool bound = J.bsize == 1;
        const uint16_t* lab = J.labels;
        // ten raw values of row (gx, gy) at z = zs - 1 .. zs + 8, clamped to the grid
        auto load_row = [&](int gx, int gy, int zs, uint16_t w[10]) {
            const int cx = min(max(gx, 0), nx - 1), cy = min(max(gy, 0), ny - 1);
            const uint16_t* r = lab + ((size_t)cx * ny + cy) * nz;
            if (zs + 8 <= nz) {
                const uint4 q = gload4_cells(r + zs);
                w[1] = (uint16_t)q.x; w[2] = (uint16_t)(q.x >> 16); w[3] = (uint16_t)q.y; w[4] = (uint16_t)(q.y >> 16);
                w[5] = (uint16_t)q.z; w[6] = (uint16_t)(q.z >> 16); w[7] = (uint16_t)q.w; w[8] = (uint16_t)(q.w >> 16);
                w[0] = gcast<const uint16_t>(r)[max(zs - 1, 0)];  // clamped window: z = -1 reads z = 0
                w[9] = gcast<const uint16_t>(r)[min(zs + 8, nz - 1)];
            } else {
#pragma unroll
                for (int k = 0; k < 10; ++k) w[k] = r[min(max(zs - 1 + k, 0), nz - 1)];
            }
        };
        // brick `local`: its origin, this thread's row segment (gx, gy, gz) and how many of its 8 cells lie in the grid
        auto segment = [&](uint32_t local, int& x0, int& y0, int& z0, int& gx, int& gy, int& gz, int& nval) {
            x0 = (int)(local / (tz * tyn)) * kBTX;
            y0 = (int)((local / tz) % tyn) * kBTY;
            z0 = (int)(local % tz) * kBTZ;
            gx = x0 + tx;
            gy = y0 + ty;
            gz = z0 + seg;
            nval = gx < nx && gy < ny ? max(0, min(8, nz - gz)) : 0;
        };
        // the 8 in-grid cells of a segment as packed pairs (cells beyond the grid read 0)
        auto load_seg = [&](int gx, int gy, int gz, int nval, uint32_t p[4]) {
            p[0] = p[1] = p[2] = p[3] = 0u;
            const uint16_t* r = lab + ((size_t)(nval ? gx : 0) * ny + (nval ? gy : 0)) * nz + gz;
            if (nval == 8) {
                const uint4 q = gload4_cells(r);
                p[0] = q.x; p[1] = q.y; p[2] = q.z; p[3] = q.w;
            } else {
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (k < nval) p[k >> 1] |= (uint32_t)r[k] << (16 * (k & 1));
            }
        };

        // phase 1: whether each brick of the run holds a label, all loads issued together; the others end here
        uint32_t live = 0;
        if constexpr (TABLE) {
            // a table's labels are not EMPTY only where the occupancy is set, and a brick's rows are one occupancy
            // word each: 4 bytes a row instead of its 64 bytes of labels; bricks without a bit add nothing
            live = live_bricks<kRun>(J, first, nrun);
        } else {
            uint32_t pr[kRun][4];
#pragma unroll
            for (uint32_t r = 0; r < kRun; ++r) {
                int x0, y0, z0, gx, gy, gz, nval;
                segment(first + r, x0, y0, z0, gx, gy, gz, nval);
                load_seg(gx, gy, gz, r < nrun ? nval : 0, pr[r]);
            }
#pragma unroll
            for (uint32_t r = 0; r < kRun; ++r) {
                bool mine = false;
#pragma unroll
                for (int k = 0; k < 4; ++k) mine |= (pr[r][k] & 0xFFFFu) > kFree || (pr[r][k] >> 16) > kFree;
                live |= mine ? 1u << r : 0u;
            }
            live = (uint32_t)__ockl_wgred_or_i32((int)live);  // block-uniform: bit r = brick r holds a label
        }

        // phase 2: bricks with a label
        for (uint32_t r = 0; r < nrun; ++r) {
            if (!((live >> r) & 1u)) continue;
            int x0, y0, z0, gx, gy, gz, nval;
            segment(first + r, x0, y0, z0, gx, gy, gz, nval);
            uint16_t w[10];
            load_row(gx, gy, gz, w);  // the segment again (a cache hit) with its z neighbours
            uint32_t own[4];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                own[k] = (2 * k < nval ? (uint32_t)w[2 * k + 1] : 0u) | (2 * k + 1 < nval ? (uint32_t)w[2 * k + 2] << 16 : 0u);
            // list the segments with cells that are not EMPTY, a wave's after one another
            const bool some = (own[0] | own[1] | own[2] | own[3]) != 0u;
            const uint64_t mask = __ballot(some);
            if (some) {
                const uint32_t at = (threadIdx.x & ~63u) + (uint32_t)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
                listed[at] = (uint8_t)threadIdx.x;
                cells[at] = make_uint4(own[0], own[1], own[2], own[3]);
            }
            if ((threadIdx.x & 63u) == 0) count[threadIdx.x >> 6] = (uint32_t)__builtin_popcountll(mask);
            if (bound) {
                uint32_t zw[8];
                zwin(w, zw);
                uint4* dst = reinterpret_cast<uint4*>(zmm + ((tx + 1) * kBHY + ty + 1) * kAZ + seg);
                dst[0] = make_uint4(zw[0], zw[1], zw[2], zw[3]);
                dst[1] = make_uint4(zw[4], zw[5], zw[6], zw[7]);
                if (halo_task) {
                    uint16_t hw[10];
                    load_row(x0 + hhx - 1, y0 + hhy - 1, z0 + seg, hw);
                    zwin(hw, zw);
                    dst = reinterpret_cast<uint4*>(zmm + (hhx * kBHY + hhy) * kAZ + seg);
                    dst[0] = make_uint4(zw[0], zw[1], zw[2], zw[3]);
                    dst[1] = make_uint4(zw[4], zw[5], zw[6], zw[7]);
                }
            }
            __syncthreads();
            uint32_t at = threadIdx.x, wv = 0;  // the at-th listed segment: place `at` of wave wv's
            while (wv < 4u && at >= count[wv]) at -= count[wv++];
            if (wv < 4u) {
                const uint32_t id = listed[64u * wv + at];
                const uint4 q = cells[64u * wv + at];
                const int r2 = (int)(id >> 2), zs = (int)(id & 3u) * 8, sx = r2 / kBTY, sy = r2 % kBTY;
                const uint32_t qw[4] = { q.x, q.y, q.z, q.w };
                uint16_t v[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) v[k] = (uint16_t)(qw[k >> 1] >> (16 * (k & 1)));
                if (TABLE) {
                    // one LDS atomic per label of the segment
                    uint32_t rest = 0;
#pragma unroll
                    for (int k = 0; k < 8; ++k) rest |= v[k] > kFree ? 1u << k : 0u;
                    while (rest) {
                        uint32_t l = 0, eq = 0;  // the first cell still to count; the cells of its label
#pragma unroll
                        for (int k = 7; k >= 0; --k) l = (rest >> k) & 1u ? (uint32_t)(v[k] & kMask15) : l;
#pragma unroll
                        for (int k = 0; k < 8; ++k) eq |= (v[k] & kMask15) == l ? 1u << k : 0u;
                        eq &= rest;
                        rest &= ~eq;
                        if (l < kTiledBins) atomicAdd(&bins[l], (uint32_t)__popc(eq));
                        else atomicAdd(J.hist + l, (uint32_t)__popc(eq));
                    }
                }
                const int ax = x0 + sx, ay = y0 + sy, az = z0 + zs, n = min(8, nz - az);
                bool changed = false;
                if (bound) {
                    // x and y windows together: a labelled cell without the bit is interior iff the packed
                    // window (max | 0xFFFF - min) equals its own packed value; cells beyond the grid are 0
                    uint32_t accs[8] = { 0, 0, 0, 0, 0, 0, 0, 0 };
#pragma unroll
                    for (int dx = 0; dx < 3; ++dx)
#pragma unroll
                        for (int dy = 0; dy < 3; ++dy) {
                            const uint4* row = reinterpret_cast<const uint4*>(zmm + ((sx + dx) * kBHY + sy + dy) * kAZ + zs);
                            const uint4 a = row[0], b = row[1];
                            accs[0] = pk_max_u16(accs[0], a.x); accs[1] = pk_max_u16(accs[1], a.y);
                            accs[2] = pk_max_u16(accs[2], a.z); accs[3] = pk_max_u16(accs[3], a.w);
                            accs[4] = pk_max_u16(accs[4], b.x); accs[5] = pk_max_u16(accs[5], b.y);
                            accs[6] = pk_max_u16(accs[6], b.z); accs[7] = pk_max_u16(accs[7], b.w);
                        }
#pragma unroll
                    for (int k = 0; k < 8; ++k) {
                        const uint32_t c = v[k];
                        const bool bnd = c > kFree && (c & 0x8000u) == 0 && accs[k] != packed_self(c);
                        v[k] = bnd ? (uint16_t)(c | 0x8000u) : (uint16_t)c;
                        changed |= bnd;
                    }
                }
                if (TABLE) {
                    const uint32_t c0 = (uint32_t)(((size_t)ax * ny + ay) * nz + az);
#pragma unroll
                    for (int k = 0; k < 8; ++k) csum += checksum_term(v[k], c0 + k);  // EMPTY cells add nothing
                }
                if (changed) {
                    uint16_t* dst = J.labels + ((size_t)ax * ny + ay) * nz + az;
                    if (n == 8) {
                        gstore4_cells(dst, pack_cells(v));
                    } else {
                        for (int k = 0; k < n; ++k) dst[k] = v[k];
                    }
                }
            }
            __syncthreads();
        }
    }, flush);
}

// Order-independent grid checksum, the sum over the non-EMPTY cells of checksum_term, of the jobs whose boundary
// window is wider than 1 (the tiled boundary kernel sums the others).
__global__ __launch_bounds__(kCellThreads) void k_checksum(Launch L)
{
    __shared__ BlockSum bs;
    __shared__ JobDev sJ;
    unsigned long long acc = 0;
    walk_tiles(L, L.tile_prefix, L.total_tiles, &sJ, [&](const JobDev& J, uint32_t, uint32_t local, uint32_t) {
        if (!J.active || J.bsize <= 1) return;
        const uint64_t c0 = (uint64_t)local * kTileCells + threadIdx.x * kCellsPerThread;
        if (c0 >= J.V) return;
        uint16_t v[8];
        load8(J.labels, c0, J.V, v);
        for (int k = 0; k < 8; ++k) acc += checksum_term(v[k], (uint32_t)(c0 + k));  // cells beyond V load as 0
    }, [&](uint32_t j) { bs.flush(acc, L.jobs[j], kStatChecksum); });
}

__global__ __launch_bounds__(kCellThreads) void k_count_occupied(Launch L)
{
    __shared__ BlockSum bs;
    __shared__ JobDev sJ;
    unsigned long long acc = 0;
    walk_tiles(L, L.bt_prefix, L.total_bricks, &sJ, [&](const JobDev& J, uint32_t, uint32_t brick, uint32_t) {
        if (J.active) acc += __popc(group_occ(J, cell_group(J, brick)));
    }, [&](uint32_t j) { bs.flush(acc, L.jobs[j], kStatOccupied); });
}

// One block per job: number of labels >= 2 with a nonzero count.
// kStatLabels: labels >= 2 with a nonzero count.  kSummaryParts blocks per job, each over 65536 /
// kSummaryParts bins with 16-byte loads issued together, add their counts (the slot is zeroed by job_init).
constexpr uint32_t kSummaryParts = 8;
__global__ __launch_bounds__(256) void k_hist_summary(Launch L)
{
    constexpr uint32_t kBins = 65536 / kSummaryParts, kIters = kBins / 4 / 256;
    __shared__ uint32_t wsum[4];
    const JobDev* J = L.jobs + blockIdx.x / kSummaryParts;
    if (!J->active) return;
    const uint32_t part = blockIdx.x % kSummaryParts;
    const uint4* h = reinterpret_cast<const uint4*>(J->hist + part * kBins);
    uint4 q[kIters];
#pragma unroll
    for (uint32_t i = 0; i < kIters; ++i) q[i] = gload4(h + i * 256 + threadIdx.x);
    uint32_t n = 0;
#pragma unroll
    for (uint32_t i = 0; i < kIters; ++i) {
        const bool first = part == 0 && i == 0 && threadIdx.x == 0;  // bins 0 (EMPTY) and 1 (FREE) are not labels
        n += (q[i].x != 0 && !first) + (q[i].y != 0 && !first) + (q[i].z != 0) + (q[i].w != 0);
    }
    for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
    if ((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = n;
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t t = wsum[0] + wsum[1] + wsum[2] + wsum[3];
        if (t) atomicAdd(J->stats + kStatLabels, (unsigned long long)t);
    }
}

// Block per job: zero the per-job statistics, histogram and flood control.
__global__ __launch_bounds__(256) void k_job_init(Launch L)
{
    const JobDev* J = L.jobs + blockIdx.x;
    if (!J->active) return;
    for (uint32_t i = threadIdx.x; i < 65536 / 4; i += blockDim.x) gstore4(J->hist + 4 * i, make_uint4(0u, 0u, 0u, 0u));
    if (threadIdx.x < kStatCount) J->stats[threadIdx.x] = 0;
    if (J->fctl && threadIdx.x < 64) J->fctl[threadIdx.x] = 0;
    if (J->sums)
        for (uint32_t i = threadIdx.x; i < kSumSlots * kStatCount; i += blockDim.x) J->sums[i] = 0ull;
}

// Block per job: stats and flood state into a compact table for one readback.
__global__ void k_gather(Launch L, uint32_t* out)
{
    const JobDev* J = L.jobs + blockIdx.x;
    uint32_t* o = out + 16 * (size_t)blockIdx.x;
    const uint32_t t = threadIdx.x;
    static_assert(kSumSlots == 64 && kStatCount == 8, "8 lines a step, a sum per lane");
    unsigned long long v = 0;
    if (J->active && J->sums)
        for (uint32_t i = t; i < kSumSlots * kStatCount; i += 64u) v += J->sums[i];
    for (int o = 8; o < 64; o <<= 1) v += __shfl_xor(v, o, 64);  // lanes with the same statistic
    if (t < kStatCount) {
        if (J->active) v += J->stats[t];
        o[2 * t] = (uint32_t)v;
        o[2 * t + 1] = (uint32_t)(v >> 32);
    }
}

inline uint32_t bgrid_for(const Launch& L) { return std::max(1u, std::min(L.total_bricks, active_shape().cell_blocks)); }
inline uint32_t grid_for(const Launch& L) { return std::max(1u, std::min(L.total_tiles, active_shape().cell_blocks)); }

}  // namespace

void launch_put_head(GridHead* dst, const GridHead& h, hipStream_t s)
{
    TimedLaunch tl("put_head", s);
    k_put_head<<<1, 128, 0, s>>>(dst, h);
    VF_CHECK_LAUNCH();
}

void launch_put_seeds(uint4* dst, const vf_seed* seeds, uint32_t n, hipStream_t s)
{
    static_assert(sizeof(vf_seed) == sizeof(uint4), "copied as they are");
    for (uint32_t i = 0; i < n; i += kPutSeeds) {
        SeedArgs a;
        const uint32_t m = std::min(kPutSeeds, n - i);
        __builtin_memcpy(a.s, seeds + i, (size_t)m * sizeof(uint4));
        TimedLaunch tl("put_seeds", s);
        k_put_seeds<<<1, kPutSeeds, 0, s>>>(dst + i, a, m);
        VF_CHECK_LAUNCH();
    }
}

void launch_report(const unsigned long long* stats, const uint4* seeds, uint32_t n, uint32_t* host, hipStream_t s)
{
    if (n > kMaxDeviceSeeds) fail(VF_ERR_INVALID_ARG, "report of %u seeds", n);
    TimedLaunch tl("report", s);
    k_report<<<1, 256, 0, s>>>(stats, seeds, n, host);
    VF_CHECK_LAUNCH();
}

void launch_occ_to_labels(const Launch& L)
{
    TimedLaunch tl("occ_to_labels", L.s);
    k_occ_to_labels<<<group_blocks(L), kCellThreads, 0, L.s>>>(L);
    VF_CHECK_LAUNCH();
}

void launch_labels_to_occ(const Launch& L)
{
    TimedLaunch tl("labels_to_occ", L.s);
    k_labels_to_occ<<<group_blocks(L), kCellThreads, 0, L.s>>>(L);
    VF_CHECK_LAUNCH();
}

void launch_occ_free(const Launch& L, const uint32_t* bits)
{
    TimedLaunch tl("occ_free", L.s);
    k_occ_free<<<group_blocks(L), kCellThreads, 0, L.s>>>(L, bits);
    VF_CHECK_LAUNCH();
}

void launch_occ_bytes(const Launch& L, uint8_t* out)
{
    TimedLaunch tl("occ_bytes", L.s);
    k_occ_bytes<<<group_blocks(L), kCellThreads, 0, L.s>>>(L, out);
    VF_CHECK_LAUNCH();
}

void launch_clear_labels(const Launch& L)
{
    TimedLaunch tl("clear_labels", L.s);
    k_clear_labels<<<grid_for(L), kCellThreads, 0, L.s>>>(L);
    VF_CHECK_LAUNCH();
}

void launch_homogenize(const Launch& L)
{
    TimedLaunch tl("homogenize", L.s);
    k_homogenize<<<grid_for(L), kCellThreads, 0, L.s>>>(L);
    VF_CHECK_LAUNCH();
}

void launch_undo_mask(const Launch& L, uint16_t keep)
{
    TimedLaunch tl("undo_mask", L.s);
    k_undo_mask<<<grid_for(L), kCellThreads, 0, L.s>>>(L, keep);
    VF_CHECK_LAUNCH();
}

void launch_hist_heads(const Launch& L, uint32_t* host)
{
    TimedLaunch tl("hist_heads", L.s);
    k_hist_heads<<<L.njobs, kHistBins / 4, 0, L.s>>>(L.jobs, host);
    VF_CHECK_LAUNCH();
}

void launch_histogram(const Launch& L, uint32_t* hist, uint32_t* part, uint32_t* host)
{
    TimedLaunch tl("histogram", L.s);
    const uint32_t blocks = std::max(1u, std::min(kHistBlocks, ceil_div((uint64_t)L.total_tiles * kTileCells, kHistThreads * kCellsPerThread)));
    k_hist_clear<<<16, 256, 0, L.s>>>(hist, part + kHistBlocks * kHistBins);
    VF_CHECK_LAUNCH();
    k_histogram<<<blocks, kHistThreads, 0, L.s>>>(L, part);
    VF_CHECK_LAUNCH();
    k_hist_sum<<<kHistBins / 64 + (host ? kLargeBlocks : 0u), 256, 0, L.s>>>(part, blocks, hist, host);
    VF_CHECK_LAUNCH();
}

void launch_boundaries(const Launch& L, int size)
{
    TimedLaunch tl("boundaries", L.s);
    k_cells_post<false><<<grid_for(L), kCellThreads, 0, L.s>>>(L, size);
    VF_CHECK_LAUNCH();
}

void launch_boundaries_tiled(const Launch& L, bool any_wide, bool table)
{
    {
        TimedLaunch tl("boundaries_hist", L.s);
        const LaunchShape sh = active_shape();
        const uint32_t per = std::max(1u, L.total_bricks / std::max(1u, sh.brick_blocks));
        const uint32_t blocks = L.total_bricks / per + L.njobs;
        auto go = [&](auto run) {
            constexpr uint32_t R = decltype(run)::value;
            if (table) k_boundaries_tiled<true, R><<<blocks, 256, 0, L.s>>>(L, per);
            else k_boundaries_tiled<false, R><<<blocks, 256, 0, L.s>>>(L, per);
        };
        // long runs look at many bricks at once, but leave workgroups idle where there are few bricks: a 256^3 grid (8192)
        // takes 26 us with runs of 4 and 30 with 8, a 512^3 grid (65536) 99 and 81, 64 mixed grids 1010 and 945; a 64^3 grid
        // (128) 15 with runs of 4 and 7.5 brick by brick, a 160^3 one (2000) 16 and 11.  Without a table, which reads every
        // label: 512^3 102 with runs of 4 and 95 with 8, 256^3 18.7 with 4 and 22 brick by brick, 128^3 12.3 and 7.7
        const uint32_t run = L.total_bricks < 4096u ? 1u : L.total_bricks < 32768u ? std::min(sh.brick_run, 4u) : sh.brick_run;
        if (run == 1) go(std::integral_constant<uint32_t, 1>{});
        else if (run == 2) go(std::integral_constant<uint32_t, 2>{});
        else if (run == 8) go(std::integral_constant<uint32_t, 8>{});
        else go(std::integral_constant<uint32_t, 4>{});
        VF_CHECK_LAUNCH();
    }
    if (any_wide) {
        TimedLaunch tl("boundaries_wide", L.s);
        k_cells_post<true><<<grid_for(L), kCellThreads, 0, L.s>>>(L, -1);
        VF_CHECK_LAUNCH();
        if (table) {
            TimedLaunch tc("checksum", L.s);
            k_checksum<<<grid_for(L), kCellThreads, 0, L.s>>>(L);
            VF_CHECK_LAUNCH();
        }
    }
}

void launch_job_init(const Launch& L)
{
    TimedLaunch tl("job_init", L.s);
    k_job_init<<<L.njobs, 256, 0, L.s>>>(L);
    VF_CHECK_LAUNCH();
}

void launch_gather(const Launch& L, uint32_t* out)
{
    k_gather<<<L.njobs, 64, 0, L.s>>>(L, out);
    VF_CHECK_LAUNCH();
}

void launch_hist_summary(const Launch& L)
{
    TimedLaunch tl("hist_summary", L.s);
    k_hist_summary<<<L.njobs * kSummaryParts, 256, 0, L.s>>>(L);
    VF_CHECK_LAUNCH();
}

void launch_count_occupied(const Launch& L)
{
    TimedLaunch tl("count_occupied", L.s);
    k_count_occupied<<<bgrid_for(L), kCellThreads, 0, L.s>>>(L);
    VF_CHECK_LAUNCH();
}

}  // namespace vf
