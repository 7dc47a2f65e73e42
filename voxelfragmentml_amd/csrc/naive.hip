// Naive Voronoi fracture (NaiveFracturer::buildCPU, NaiveFracturer.cpp:26-68;
// naiveFracturer-comp.glsl:19-42) and the optional isolated-region removal
// (removeIsolatedRegionsCPU, NaiveFracturer.cpp:111-150).
//
// Every non-EMPTY cell takes the label of argmin over seeds of (distance,
// seed index).  Distances are exact integers: squared Euclidean, L1, L-inf
// (the reference's float distances on integer offsets order identically),
// except Euclidean on grids large enough for float roots to collide, which
// ranks by the float root itself.
// The argmin is a single unsigned min over packed keys (distance << b | i),
// so ties go to the lowest index exactly as the reference's strict '<' does.
// Work goes by bricks of 8 x 8 x 32 cells: a brick's occupied cells are
// compacted, the seeds that cannot be nearest to any of its cells are dropped,
// and a thread applies the rest to its few cells in registers.  Flat grids of
// many bricks go by tiles of cells in linear order instead.
#include <type_traits>

#include "cellops.hpp"

namespace vf {

namespace {

constexpr uint32_t kSeedChunk = 1024;
constexpr uint32_t kNaiveSmall = 8192;  // bricks of a launch below which runs are of one

// (d << b) | i.  32-bit keys: d < 2^24 (at most 3 * 2047^2) and b <= 17, so it is one 24-bit
// multiply-add, d * 2^b + i.
template <typename K>
__device__ inline K pack_key(uint32_t d, uint32_t i, uint32_t b)
{
    if constexpr (sizeof(K) == 4) return (K)(__umul24(d, 1u << b) + i);
    else return ((K)d << b) | (K)i;
}

// |a.lo - b.lo| + |a.hi - b.hi| + acc over the 16-bit halves (v_sad_u16, one instruction); cell and seed
// coordinates are below 2^11 (grid edges of at most 2048 cells), so the halves never wrap.
__device__ inline uint32_t sad16(uint32_t a, uint32_t b, uint32_t acc) { return __builtin_amdgcn_sad_u16(a, b, acc); }

// The distance of offsets (ax, ay, az), each below 2^11.  kDistEuclidF32 (64-bit keys only) ranks by the bits of the
// correctly rounded float root of the squared distance, which is below 2^24 and so converts exactly: the
// reference's float sqrt (NaiveFracturer.cpp:12-15).
template <int DIST>
__device__ inline uint32_t offset_dist(uint32_t ax, uint32_t ay, uint32_t az)
{
    if (DIST == VF_MANHATTAN) return ax + ay + az;
    if (DIST == VF_CHEBYSHEV) return max(ax, max(ay, az));
    // offsets < 2^11: 16-bit operands select the full-rate 24-bit multiply
    const uint32_t d = (ax & 0xFFFFu) * (ax & 0xFFFFu) + (ay & 0xFFFFu) * (ay & 0xFFFFu) + (az & 0xFFFFu) * (az & 0xFFFFu);
    return DIST == kDistEuclidF32 ? sqrt_rn_bits(d) : d;
}

// Distance key of one cell (xy = x | y << 16, z) to one seed (sxy, sz).
template <int DIST, typename K>
__device__ inline K seed_key(uint32_t xy, uint32_t z, uint32_t sxy, uint32_t sz, uint32_t id, uint32_t b)
{
    uint32_t d;
    if (DIST == VF_MANHATTAN) {
        d = sad16(xy, sxy, sad16(z, sz, 0u));
    } else {
        const uint32_t ax = sad16(xy & 0xFFFFu, sxy & 0xFFFFu, 0u), ay = sad16(xy >> 16, sxy >> 16, 0u), az = sad16(z, sz, 0u);
        d = offset_dist<DIST>(ax, ay, az);
    }
    return pack_key<K>(d, id, b);
}

// Seeds in LDS: x | y << 16, then z | (index in the chunk) << 16.
static_assert(kSeedChunk <= 65536, "16-bit seed index");

// argmin over the n seeds of `list` for Q compacted cells of a thread: each seed is read once (an LDS broadcast, its
// parts split on the scalar unit) and applied to all Q cells held in registers.
template <int DIST, typename K, int Q>
__device__ inline void naive_cells_q(K best[4], const uint32_t cxy[4], const uint32_t cz[4], const uint2* list, uint32_t base,
                                     uint32_t n, uint32_t b)
{
    K m[Q];
    uint32_t xy[Q], z[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        m[q] = best[q];
        xy[q] = cxy[q];
        z[q] = cz[q];
    }
    auto apply = [&](uint32_t vxy, uint32_t vzi) {
        const uint32_t sxy = (uint32_t)__builtin_amdgcn_readfirstlane((int)vxy), szi = (uint32_t)__builtin_amdgcn_readfirstlane((int)vzi);
        const uint32_t sz = szi & 0xFFFFu, id = base + (szi >> 16);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const K key = seed_key<DIST, K>(xy[q], z[q], sxy, sz, id, b);
            m[q] = key < m[q] ? key : m[q];
        }
    };
    // four seeds per step, two 16-byte LDS reads (the list is 16-byte aligned)
    uint32_t i = 0;
    for (; i + 4 <= n; i += 4) {
        const uint4 a = *reinterpret_cast<const uint4*>(list + i), c = *reinterpret_cast<const uint4*>(list + i + 2);
        apply(a.x, a.y);
        apply(a.z, a.w);
        apply(c.x, c.y);
        apply(c.z, c.w);
    }
    for (; i < n; ++i) {
        const uint2 a = list[i];
        apply(a.x, a.y);
    }
#pragma unroll
    for (int q = 0; q < Q; ++q) best[q] = m[q];
}

// qmax (1..4): cells per thread, the same for the whole wave (lanes past the
// brick's last occupied cell compute on a dummy cell)
template <int DIST, typename K>
__device__ inline void naive_cells(K best[4], const uint32_t cxy[4], const uint32_t cz[4], uint32_t qmax, const uint2* list,
                                   uint32_t base, uint32_t n, uint32_t b)
{
    if (qmax <= 1) naive_cells_q<DIST, K, 1>(best, cxy, cz, list, base, n, b);
    else if (qmax == 2) naive_cells_q<DIST, K, 2>(best, cxy, cz, list, base, n, b);
    else if (qmax == 3) naive_cells_q<DIST, K, 3>(best, cxy, cz, list, base, n, b);
    else naive_cells_q<DIST, K, 4>(best, cxy, cz, list, base, n, b);
}

// The least and the greatest distance of a seed from the cells of a box.
template <int DIST>
__device__ inline void box_dist(uint32_t xy, uint32_t z, const uint32_t lo[3], const uint32_t hi[3], uint32_t& dmin, uint32_t& dmax)
{
    const uint32_t s[3] = { xy & 0xFFFFu, xy >> 16, z };
    uint32_t a[3], f[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        const int below = (int)lo[q] - (int)s[q], above = (int)s[q] - (int)hi[q];  // > 0 outside the box
        a[q] = (uint32_t)max(max(below, above), 0);
        f[q] = (uint32_t)max(-below, -above);
    }
    dmin = offset_dist<DIST>(a[0], a[1], a[2]);
    dmax = offset_dist<DIST>(f[0], f[1], f[2]);
}

// Seeds below which a brick applies all of them: dropping the far ones (a box distance per seed, a block minimum, a
// compaction) costs about as much as applying this many.
constexpr uint32_t kPruneSeeds = 16;

// One brick per step.  Its occupied cells are compacted in LDS, so the seed loop runs over occupied cells only (shells
// occupy a few percent of their box); of more than kPruneSeeds seeds, those farther from the whole brick than some
// other seed's farthest cell are dropped first (strictly farther: ties stay, and a dropped seed is never nearest or
// tied), which leaves a few of 128; labels return through LDS and leave as one 16-byte store per
// occupied group (launch_clear_labels has written the rest).  Bound by the latency of the block's barriers, so the
// register budget is set for more waves in flight: 5 per SIMD with 32-bit keys, 4 with 64-bit keys.  RUN bricks form a walker run
// whose occupancy loads are issued together (a launch shape the tuner picks).
// 512^3, 128 seeds, Chebyshev: 442 us applying every seed in linear tiles, 84 us by bricks and 34 us of clearing, 68 us
// since a run's bricks are looked at by occupancy words together (live_bricks) instead of a byte a thread.
// LINEAR: tiles of 2048 cells in linear order in place of bricks, for grids that fill little of their bricks (launch_naive).
template <typename K, uint32_t RUN, bool LINEAR>
__global__ __launch_bounds__(kCellThreads) __attribute__((amdgpu_waves_per_eu(sizeof(K) == 4 ? 5 : 4))) void k_naive(Launch L)
{
    __shared__ __attribute__((aligned(16))) uint2 seeds[kSeedChunk];
    __shared__ __attribute__((aligned(16))) uint2 near[kSeedChunk];
    __shared__ uint16_t sw[kSeedChunk];
    __shared__ uint16_t cells[kTileCells];  // compacted offsets of the occupied cells
    __shared__ uint4 lab4[kTileCells / 8];  // the brick's output labels, 8 per thread
    typedef uint16_t __attribute__((may_alias)) label_alias;  // single labels of lab4
    label_alias* lab = reinterpret_cast<label_alias*>(lab4);
    __shared__ uint32_t wsum[kCellThreads / 64], wmin[kCellThreads / 64];
    __shared__ JobDev sJ;
    __shared__ uint32_t sp[kWalkMaxJobs + 1];
    constexpr int kWant = sizeof(K) == 8 ? 1 : 0;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    uint32_t staged = 0xFFFFFFFFu;  // job whose seeds (one chunk) sit in LDS
    auto stage = [&](const JobDev& J, uint32_t base, uint32_t n) {
        __syncthreads();
        for (uint32_t i = tid; i < n; i += blockDim.x) {
            const uint4 q = J.seeds[base + i];
            seeds[i] = make_uint2(q.x | q.y << 16, q.z | i << 16);
            sw[i] = (uint16_t)q.w;
        }
        __syncthreads();
    };
    // the seeds of the n staged ones that may be nearest to a cell of the box, into near; bound: the least of the seeds'
    // greatest distances so far.  Block-wide.
    auto prune = [&](auto dist, uint32_t n, const uint32_t lo[3], const uint32_t hi[3], uint32_t& bound) {
        constexpr int DIST = decltype(dist)::value;
        constexpr uint32_t kPer = kSeedChunk / kCellThreads;
        uint32_t dmin[kPer], far = 0xFFFFFFFFu;
#pragma unroll
        for (uint32_t c = 0; c < kPer; ++c) {
            dmin[c] = 0xFFFFFFFFu;
            const uint32_t i = c * kCellThreads + tid;
            if (c * kCellThreads < n && i < n) {
                uint32_t dmax;
                box_dist<DIST>(seeds[i].x, seeds[i].y & 0xFFFFu, lo, hi, dmin[c], dmax);
                far = min(far, dmax);
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) far = min(far, (uint32_t)__shfl_xor((int)far, o, 64));
        if (lane == 0) wmin[wave] = far;
        __syncthreads();
        for (uint32_t w = 0; w < kCellThreads / 64; ++w) bound = min(bound, wmin[w]);
        uint32_t m = 0;
#pragma unroll
        for (uint32_t c = 0; c < kPer; ++c) {
            if (c * kCellThreads >= n) break;
            const uint64_t keep = __ballot(dmin[c] <= bound);
            if (lane == 0) wsum[wave] = (uint32_t)__popcll(keep);
            __syncthreads();
            uint32_t pos = m;
            for (uint32_t w = 0; w < kCellThreads / 64; ++w) {
                if (w < wave) pos += wsum[w];
                m += wsum[w];
            }
            if ((keep >> lane) & 1u) near[pos + (uint32_t)__popcll(keep & ((1ull << lane) - 1ull))] = seeds[c * kCellThreads + tid];
            __syncthreads();
        }
        return m;
    };
    constexpr uint32_t kRun = RUN;
    walk_tile_runs_strided<kRun>(L, LINEAR ? L.tile_prefix : L.bt_prefix, LINEAR ? L.total_tiles : L.total_bricks, &sJ, sp,
                                 [&](const JobDev& J, uint32_t j, uint32_t first, uint32_t nrun) {
        if (!J.active || J.algo != VF_NAIVE || J.naive_key64 != kWant || J.S == 0) return;
        const uint32_t S = J.S;
        const bool one_chunk = S <= kSeedChunk;
        if (one_chunk && staged != j) {  // block-uniform
            stage(J, 0, S);
            staged = j;
        }
        auto brick = [&](uint32_t id) {
        BrickAt at;
        CellGroup grp;
        uint32_t occ = 0;
        const uint32_t c0 = id * kTileCells + tid * kCellsPerThread;  // LINEAR: the thread's first cell
        if constexpr (LINEAR) {
            if (c0 < J.V) {
                uint32_t x, y, z;
                decompose(c0, &J, x, y, z);
                for (uint32_t k = 0; k < kCellsPerThread && c0 + k < J.V; ++k) {
                    occ |= occ_bit(J, x, y, z) ? 1u << k : 0u;
                    advance(x, y, z, &J);
                }
            }
        } else {
            at = brick_at(J, id);
            grp = cell_group(J, at);
            occ = group_occ(J, grp);
        }
        // block-wide exclusive scan of the occupied counts -> compacted positions
        const uint32_t n = (uint32_t)__popc(occ);
        uint32_t inc = n;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t t = __shfl_up(inc, o, 64);
            if (lane >= (uint32_t)o) inc += t;
        }
        if (lane == 63u) wsum[wave] = inc;
        lab4[tid] = make_uint4(0u, 0u, 0u, 0u);  // EMPTY unless written below
        __syncthreads();
        uint32_t pos = inc - n, total = 0;
        for (uint32_t w = 0; w < kCellThreads / 64; ++w) {
            if (w < wave) pos += wsum[w];
            total += wsum[w];
        }
        for (int k = 0; k < 8; ++k)
            if ((occ >> k) & 1u) cells[pos++] = (uint16_t)(tid * 8 + k);  // row of the brick * 32 + z; place in the tile
        __syncthreads();
        if (LINEAR && total == 0) return;  // block-uniform
        uint32_t lo[3], hi[3];  // the box of the brick or tile
        if constexpr (LINEAR) {
            decompose((uint64_t)id * kTileCells, &J, lo[0], lo[1], lo[2]);
            decompose(min((uint64_t)(id + 1u) * kTileCells, J.V) - 1u, &J, hi[0], hi[1], hi[2]);
            if (lo[0] != hi[0]) {
                lo[1] = 0;
                hi[1] = J.ny - 1u;
            }
            if (lo[0] != hi[0] || lo[1] != hi[1]) {
                lo[2] = 0;
                hi[2] = J.nz - 1u;
            }
        } else {
            lo[0] = at.x;
            lo[1] = at.y;
            lo[2] = at.z;
            hi[0] = min(at.x + kBrickX, J.nx) - 1u;
            hi[1] = min(at.y + kBrickY, J.ny) - 1u;
            hi[2] = min(at.z + kBrickZ, J.nz) - 1u;
        }
        const int dist = J.dist;
        const bool drop = S > kPruneSeeds;
        uint32_t bound = 0xFFFFFFFFu;
        auto prune_any = [&](uint32_t m) {
            if (dist == VF_MANHATTAN) return prune(std::integral_constant<int, VF_MANHATTAN>{}, m, lo, hi, bound);
            if (dist == VF_CHEBYSHEV) return prune(std::integral_constant<int, VF_CHEBYSHEV>{}, m, lo, hi, bound);
            if constexpr (sizeof(K) == 8)
                if (dist == kDistEuclidF32) return prune(std::integral_constant<int, kDistEuclidF32>{}, m, lo, hi, bound);
            return prune(std::integral_constant<int, VF_EUCLIDEAN>{}, m, lo, hi, bound);
        };
        uint32_t nnear = S;
        if (one_chunk && drop) nnear = prune_any(S);
        const uint2* list = drop ? near : seeds;
        // thread t holds compacted cells t, t + 256, ...: a wave's first lane holds the most, so
        // waves past the last cell skip the seed loop.  Cells are taken four per thread at a time
        // (the second group only in bricks with more than 1024 occupied cells), so the registers
        // hold four cells' coordinates and keys, not eight.
        const uint32_t nq = tid < total ? (total - tid + kCellThreads - 1) / kCellThreads : 0u;
        const uint32_t tid0 = wave * 64u;
        const uint32_t qmax = tid0 < total ? (total - tid0 + kCellThreads - 1) / kCellThreads : 0u;  // wave-uniform
        const uint32_t b = J.key_bits;
        const K mask = ((K)1 << b) - 1;
        const uint32_t groups = total > 4u * kCellThreads ? 2u : 1u;  // block-uniform
        for (uint32_t g = 0; g < groups; ++g) {
            const uint32_t q0 = 4u * g;
            const uint32_t gq = nq > q0 ? min(nq - q0, 4u) : 0u;
            const uint32_t gqmax = qmax > q0 ? min(qmax - q0, 4u) : 0u;  // wave-uniform
            uint32_t cxy[4], cz[4];
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                const uint32_t c = q < gq ? cells[tid + (q0 + q) * kCellThreads] : 0u, row = c >> 5;
                if constexpr (LINEAR) {
                    uint32_t x, y;
                    decompose((uint64_t)id * kTileCells + c, &J, x, y, cz[q]);
                    cxy[q] = x | y << 16;
                } else {
                    cxy[q] = (at.x + row / kBrickY) | (at.y + row % kBrickY) << 16;
                    cz[q] = at.z + (c & 31u);
                }
            }
            K best[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) best[q] = ~(K)0;
            for (uint32_t base = 0; base < S; base += kSeedChunk) {
                uint32_t m = one_chunk ? nnear : min(kSeedChunk, S - base);
                if (!one_chunk) {
                    stage(J, base, m);
                    staged = 0xFFFFFFFFu;
                    m = prune_any(m);
                }
                if (gqmax == 0) continue;  // staging above stays block-wide
                if (dist == VF_MANHATTAN) naive_cells<VF_MANHATTAN, K>(best, cxy, cz, gqmax, list, base, m, b);
                else if (dist == VF_CHEBYSHEV) naive_cells<VF_CHEBYSHEV, K>(best, cxy, cz, gqmax, list, base, m, b);
                else if (dist == VF_EUCLIDEAN) naive_cells<VF_EUCLIDEAN, K>(best, cxy, cz, gqmax, list, base, m, b);
                else if constexpr (sizeof(K) == 8) naive_cells<kDistEuclidF32, K>(best, cxy, cz, gqmax, list, base, m, b);
            }
#pragma unroll
            for (uint32_t q = 0; q < 4; ++q) {
                if (q >= gq) break;
                const uint32_t id = (uint32_t)(best[q] & mask);
                lab[cells[tid + (q0 + q) * kCellThreads]] = one_chunk ? sw[id] : (uint16_t)J.seeds[id].w;
            }
        }
        __syncthreads();
        if (occ) {
            const uint4 out = lab4[tid];
            if constexpr (LINEAR) {
                const uint32_t w[4] = { out.x, out.y, out.z, out.w };
                uint16_t v[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) v[k] = (uint16_t)(w[k >> 1] >> (16 * (k & 1)));
                store8(J.labels, c0, J.V, v);
            } else {
                store_group(J.labels, grp, out);
            }
        }
        __syncthreads();  // lab and cells are reused by the next brick
        };
        // the bricks of the run with an occupied cell; the others (most of a vessel's box) stay EMPTY
        if constexpr (LINEAR) {
#pragma unroll 1
            for (uint32_t r = 0; r < nrun; ++r) brick(first + r);
        } else {
#pragma unroll 1
            for (uint32_t any = live_bricks<kRun>(J, first, nrun); any; any &= any - 1u) brick(first + (uint32_t)__builtin_ctz(any));
        }
    });
}

// ---------------------------------------------------------------------------
// Isolated-region removal: label-propagation BFS from the seeds through cells
// holding the seed's label.  Each cell can be claimed by one label only (its
// own), so the reached set, and thus the result, is independent of order.
__global__ void k_ri_init(const uint16_t* labels, uint16_t* out, uint32_t* visited, uint64_t V, uint64_t words)
{
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < V; i += (uint64_t)gridDim.x * blockDim.x)
        out[i] = 0;
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < words; i += (uint64_t)gridDim.x * blockDim.x)
        visited[i] = 0;
}

__global__ void k_ri_seed(uint16_t* out, uint32_t* visited, uint32_t* frontier, uint32_t* fl, uint32_t* counters,
                          uint32_t ny, uint32_t nz, const uint4* seeds, uint32_t S)
{
    // seeds stamped in list order: the last seed on a cell keeps it
    if (threadIdx.x == 0 && blockIdx.x == 0) {
        for (uint32_t s = 0; s < S; ++s) {
            uint32_t c = (seeds[s].x * ny + seeds[s].y) * nz + seeds[s].z;
            out[c] = (uint16_t)seeds[s].w;
            visited[c >> 5] |= 1u << (c & 31);
            frontier[s] = c;
            fl[s] = seeds[s].w;
        }
        counters[0] = S;
        counters[1] = 0;
    }
}

__global__ void k_ri_step(const uint16_t* labels, uint16_t* out, uint32_t* visited, const uint32_t* fa, const uint32_t* la,
                          uint32_t* fb, uint32_t* lb, uint32_t* counters, uint32_t cur, uint32_t nx, uint32_t ny, uint32_t nz)
{
    const uint32_t n = counters[cur];
    for (uint32_t e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
        const uint32_t v = fa[e], w = la[e];
        const uint32_t yz = ny * nz;
        const uint32_t x = v / yz, r = v - x * yz, y = r / nz, z = r - y * nz;
        const int dx[6] = { 1, -1, 0, 0, 0, 0 }, dy[6] = { 0, 0, 1, -1, 0, 0 }, dz[6] = { 0, 0, 0, 0, 1, -1 };
        for (int k = 0; k < 6; ++k) {
            const int xx = (int)x + dx[k], yy = (int)y + dy[k], zz = (int)z + dz[k];
            if (xx < 0 || yy < 0 || zz < 0 || xx >= (int)nx || yy >= (int)ny || zz >= (int)nz) continue;
            const uint32_t u = ((uint32_t)xx * ny + (uint32_t)yy) * nz + (uint32_t)zz;
            if ((uint32_t)labels[u] != w) continue;
            const uint32_t bit = 1u << (u & 31);
            if (visited[u >> 5] & bit) continue;
            const uint32_t old = atomicOr(visited + (u >> 5), bit);
            if (old & bit) continue;
            out[u] = (uint16_t)w;
            const uint32_t slot = atomicAdd(counters + (cur ^ 1), 1u);
            fb[slot] = u;
            lb[slot] = w;
        }
    }
}

__global__ void k_ri_reset(uint32_t* counters, uint32_t idx) { counters[idx] = 0; }

}  // namespace

void launch_naive(const Launch& L, bool key64)
{
    if (L.njobs > kWalkMaxJobs) fail(VF_ERR_INVALID_ARG, "naive launch with %u jobs (max %u)", L.njobs, kWalkMaxJobs);
    TimedLaunch tl(key64 ? "naive64" : "naive", L.s);
    // grids of few bricks: one brick per run, so that they spread over the device (in runs of 8 a 64^3 grid's 128
    // bricks kept 16 workgroups busy)
    // Many bricks with few cells each (2048 x 2048 x 1: 64 of 2048): tiles of cells in linear order, 2.0 to 5.0 times as fast
    // as bricks there with 4 to 128 seeds (272 -> 54 us for 32 seeds and every 20th cell occupied), 1.2 to 2.4 at
    // 2048 x 1500 x 4; at a quarter of the cells it depends on the seeds (2 x 2048 x 2048: 0.5 to 1.3), and with few bricks
    // they are even (300 x 300 x 2, 1444 bricks: 0.8 to 1.1)
    const bool thin = L.total_bricks >= kNaiveSmall && (uint64_t)L.total_tiles * 6u < L.total_bricks;
    const uint32_t run = thin || L.total_bricks < kNaiveSmall ? 1u : active_shape().naive_run;
    const uint32_t blocks = std::max(1u, std::min(thin ? L.total_tiles : L.total_bricks, active_shape().cell_blocks));
    auto go = [&](auto r, auto linear) {
        constexpr uint32_t R = decltype(r)::value;
        constexpr bool LINEAR = decltype(linear)::value;
        if (key64) k_naive<unsigned long long, R, LINEAR><<<blocks, kCellThreads, 0, L.s>>>(L);
        else k_naive<uint32_t, R, LINEAR><<<blocks, kCellThreads, 0, L.s>>>(L);
    };
    if (thin) go(std::integral_constant<uint32_t, 1>{}, std::true_type{});
    else if (run == 1) go(std::integral_constant<uint32_t, 1>{}, std::false_type{});
    else if (run == 4) go(std::integral_constant<uint32_t, 4>{}, std::false_type{});
    else if (run == 16) go(std::integral_constant<uint32_t, 16>{}, std::false_type{});
    else go(std::integral_constant<uint32_t, 8>{}, std::false_type{});
    VF_CHECK_LAUNCH();
}

void launch_remove_isolated(hipStream_t s, uint16_t* labels, uint16_t* out, uint32_t* fa, uint32_t* fb, uint32_t* counters,
                            uint32_t* visited, const uint32_t dims[3], const uint4* seeds, uint32_t S, uint32_t* host_counter)
{
    // fa/fb each hold 2*V uint32 (cell, label) halves; host_counter is pinned memory
    const uint64_t V = (uint64_t)dims[0] * dims[1] * dims[2];
    uint32_t* la = fa + V;
    uint32_t* lb = fb + V;
    TimedLaunch tl("remove_isolated", s);
    k_ri_init<<<1024, 256, 0, s>>>(labels, out, visited, V, (V + 31) / 32);
    k_ri_seed<<<1, 64, 0, s>>>(out, visited, fa, la, counters, dims[1], dims[2], seeds, S);
    VF_CHECK_LAUNCH();
    uint32_t cur = 0;
    for (;;) {
        k_ri_step<<<1024, 256, 0, s>>>(labels, out, visited, cur ? fb : fa, cur ? lb : la, cur ? fa : fb, cur ? la : lb,
                                       counters, cur, dims[0], dims[1], dims[2]);
        VF_CHECK_LAUNCH();
        k_ri_reset<<<1, 1, 0, s>>>(counters, cur);
        VF_HIP(hipMemcpyAsync(host_counter, counters + (cur ^ 1), sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        VF_HIP(hipStreamSynchronize(s));
        cur ^= 1;
        if (*host_counter == 0) break;
    }
}

}  // namespace vf
