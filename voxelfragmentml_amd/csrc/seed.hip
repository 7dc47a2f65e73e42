// Device-side uniform seeding: Seeder::uniform (MF/Source/Fracturer/Seeder.cpp:154-208)
// with a counter-based draw so results are reproducible across platforms.
// Candidates are occupied cells (optionally only surface / only interior
// cells by RegularGrid::isBoundary, RegularGrid.cpp:543-558).  The j-th draw
// is rank floor(hash32(key, j) * O / 2^32) among the O candidates in linear
// order; repeated ranks are skipped until S distinct ranks are accepted (at
// most 10^6 draws, Seeder.cpp MAX_TRIES), then seeds are emitted in (x,y,z)
// order with labels 2..S+1.
#include "cellops.hpp"

namespace vf {

namespace {

constexpr uint32_t kSeedThreads = 256;
constexpr uint32_t kMaxDraws = 1000000u;

// Occupancy words of a 32-cell run and its two z neighbours: the word itself, and the words whose bit k is the
// cell below (above) cell k, cells beyond the grid counting as occupied.
struct ColumnRun {
    uint32_t own, dn, up;
};
__device__ inline ColumnRun column_run(const JobDev& J, uint32_t x, uint32_t y, uint32_t wz)
{
    const auto* p = gcast<const uint32_t>(J.occ) + ((size_t)x * J.ny + y) * J.wp;
    const uint32_t z0 = wz * 32u;
    const uint32_t w = p[wz];
    const uint32_t below = wz ? p[wz - 1u] >> 31 : 1u;
    const uint32_t above = z0 + 32u < J.nz ? p[wz + 1u] & 1u : 1u;
    ColumnRun r{ w, (w << 1) | below, (w >> 1) | (above << 31) };
    if (J.nz - z0 < 32u) r.up |= 1u << (J.nz - z0 - 1u);  // the last cell has no upper neighbour
    return r;
}

// Seed candidates among the cells of word wz of column (x, y): occupied cells, of jobs that seed on the surface or
// inside only those whose clamped 3x3x3 window holds an EMPTY cell (RegularGrid::isBoundary) or none.
__device__ inline uint32_t candidates(const JobDev& J, uint32_t x, uint32_t y, uint32_t wz)
{
    if (wz * 32u >= J.nz) return 0u;
    const uint32_t own = gcast<const uint32_t>(J.occ)[((size_t)x * J.ny + y) * J.wp + wz];
    if (J.seed_location == VF_SEED_BOTH || own == 0u) return own;
    uint32_t inner = ~0u;
    for (uint32_t a = x ? x - 1u : 0u; a <= min(x + 1u, J.nx - 1u); ++a)
        for (uint32_t b = y ? y - 1u : 0u; b <= min(y + 1u, J.ny - 1u); ++b) {
            const ColumnRun r = column_run(J, a, b, wz);
            inner &= r.own & r.dn & r.up;
        }
    return J.seed_location == VF_SEED_OUTER ? own & ~inner : own & inner;
}

__device__ inline bool surface_cell(const JobDev& J, uint32_t x, uint32_t y, uint32_t z)
{
    for (uint32_t a = x ? x - 1u : 0u; a <= min(x + 1u, J.nx - 1u); ++a)
        for (uint32_t b = y ? y - 1u : 0u; b <= min(y + 1u, J.ny - 1u); ++b) {
            const ColumnRun r = column_run(J, a, b, z >> 5);
            if (!(((r.own & r.dn & r.up) >> (z & 31u)) & 1u)) return true;
        }
    return false;
}

// the candidates of word w of job J (0 past its last word)
__device__ inline uint32_t word_candidates(const JobDev& J, uint32_t w)
{
    const uint32_t lg = (uint32_t)__builtin_ctz(J.wp), col = w >> lg;
    if (col >= J.nx * J.ny) return 0u;
    const uint32_t x = col / J.ny;
    return candidates(J, x, col - x * J.ny, w & (J.wp - 1u));
}

// Candidates per word tile, one wave per tile and one lane per word: surface and interior cells are found 32 at a
// time from the words of nine columns (cell by cell, 27 byte loads each, eight grids of 64^3 to 160^3 took
// 310 us).  skip_both: jobs that seed anywhere were counted by the voxelizer's fill.
__global__ __launch_bounds__(kCellThreads) void k_seed_count(Launch L, uint32_t* tile_cnt, bool skip_both)
{
    const uint32_t lane = threadIdx.x & 63u, waves = gridDim.x * (kCellThreads / 64u);
    const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * (kCellThreads / 64u) + (threadIdx.x >> 6)));
    for (uint32_t t = first; t < L.total_wtiles; t += waves) {
        const uint32_t j = find_job(L.wtile_prefix, L.njobs, t);
        const JobDev& J = L.jobs[j];
        if (skip_both && J.seed_location == VF_SEED_BOTH) continue;  // wave-uniform
        uint32_t n = J.active ? (uint32_t)__popc(word_candidates(J, (t - L.wtile_prefix[j]) * kTileWords + lane)) : 0u;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) n += __shfl_xor(n, o, 64);
        if (lane == 0) tile_cnt[t] = n;
    }
}

// The largest t in [lo, hi) with off[t] <= want, off ascending and off[lo] <= want, searched by a wave with 64
// probes a step.
__device__ inline uint32_t wave_last_below(const unsigned long long* off, uint32_t lo, uint32_t hi, unsigned long long want)
{
    const uint32_t lane = threadIdx.x & 63u;
    while (hi - lo > 1u) {
        const uint32_t step = (hi - lo + 63u) / 64u, idx = lo + lane * step;
        const uint64_t m = __ballot(idx < hi && off[idx] <= want);
        lo += (63u - (uint32_t)__clzll((long long)m)) * step;
        hi = min(lo + step, hi);
    }
    return lo;
}

// The index of the n-th set bit of v (n below its bit count).
__device__ inline uint32_t nth_bit(uint32_t v, uint32_t n)
{
    uint32_t pos = 0;
#pragma unroll
    for (uint32_t half = 16u; half; half >>= 1) {
        const uint32_t c = (uint32_t)__popc(v & ((1u << half) - 1u));
        if (n >= c) {
            n -= c;
            v >>= half;
            pos += half;
        }
    }
    return pos;
}

// kPickParts blocks per job: each draws and sorts the job's ranks by itself (in LDS, a few microseconds) and then
// finds the cells of its share of them, a wave per seed.  Bound by latency: three dependent probes of the tile
// offsets, the tile's words, a bit select.  One block per job, a binary search per seed and a walk over the tile's
// cells took 180 us for the 128 seeds of a 512^3 grid.
constexpr uint32_t kPickParts = 8;
__global__ __launch_bounds__(kSeedThreads) void k_seed_pick(Launch L, const unsigned long long* tile_off)
{
    __shared__ __attribute__((aligned(16))) uint32_t chosen[kMaxDeviceSeeds];
    __shared__ uint32_t sorted[kMaxDeviceSeeds];
    __shared__ __attribute__((aligned(16))) uint32_t cand[kSeedThreads];
    __shared__ uint32_t wsum[kSeedThreads / 64];
    __shared__ uint32_t s_got;
    const uint32_t j = blockIdx.x / kPickParts, part = blockIdx.x % kPickParts;
    const JobDev* J = L.jobs + j;
    if (!J->active) return;
    const uint32_t S = J->S_draw;
    constexpr uint32_t kWaves = kSeedThreads / 64u;
    if (part * kWaves >= S) return;  // no seed of this part
    const uint32_t t0 = L.wtile_prefix[j], t1 = L.wtile_prefix[j + 1];
    const unsigned long long base = tile_off[t0];
    const unsigned long long O = tile_off[t1] - base;
    // on failure every seed is parked on cell (0,0,0) so later stages stay in bounds
    auto park = [&]() {
        if (part) return;
        if (threadIdx.x == 0) atomicOr(reinterpret_cast<unsigned int*>(J->stats + kStatError), (unsigned int)kDevErrSeeding);
        for (uint32_t i = threadIdx.x; i < S; i += blockDim.x) J->seeds[i] = make_uint4(0u, 0u, 0u, 2u + (i & 0xFFu));
    };
    if (O < S || O > 0xFFFFFFFFull || S > kMaxDeviceSeeds) {
        park();
        return;
    }
    if (threadIdx.x == 0) s_got = 0;
    __syncthreads();
    // how many of the first n entries of a list equal r (n may differ by lane): 16-byte reads, no early way out, so that
    // the reads of a wave's lanes stream
    auto count_if = [](const uint32_t* list, uint32_t n, auto&& test) {
        uint32_t c = 0;
        for (uint32_t k = 0; k < n; k += 4u) {
            const uint4 q = *reinterpret_cast<const uint4*>(list + k);
            c += (test(q.x) ? 1u : 0u) + (k + 1u < n && test(q.y) ? 1u : 0u) + (k + 2u < n && test(q.z) ? 1u : 0u) +
                 (k + 3u < n && test(q.w) ? 1u : 0u);
        }
        return c;
    };
    // as many draws a step as the missing seeds are expected to take (a draw is accepted or not by those before it
    // alone): no more than are missing where few cells are taken, but a whole step for the last cells of a full draw,
    // which take about O draws each (4096 of 4096 cells: 15.8 ms, 1370 with as many draws as seeds were missing)
    for (uint32_t j0 = 0; j0 < kMaxDraws;) {
        const uint32_t got = s_got;
        if (got >= S) break;
        const uint32_t step = (uint32_t)min((float)kSeedThreads, ceilf((float)(S - got) * ((float)O / (float)(O - got))));
        const uint32_t draw = j0 + threadIdx.x;
        j0 += step;
        const uint32_t r = (uint32_t)(((unsigned long long)hash32(J->seed_key, draw) * O) >> 32);
        cand[threadIdx.x] = r;
        __syncthreads();
        bool dup = draw >= kMaxDraws || threadIdx.x >= step;
        if (!dup) {
            auto same = [&](uint32_t v) { return v == r; };
            dup = count_if(chosen, got, same) + count_if(cand, threadIdx.x, same) != 0u;
        }
        // block exclusive scan of the accept flags
        uint32_t a = dup ? 0u : 1u, x = a;
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        for (int o = 1; o < 64; o <<= 1) {
            uint32_t y = __shfl_up(x, o, 64);
            if (lane >= (uint32_t)o) x += y;
        }
        if (lane == 63) wsum[wave] = x;
        __syncthreads();
        uint32_t wofs = 0, tot = 0;
        for (uint32_t w = 0; w < kSeedThreads / 64; ++w) {
            if (w < wave) wofs += wsum[w];
            tot += wsum[w];
        }
        const uint32_t pos = got + wofs + x - a;
        if (a && pos < S) chosen[pos] = r;
        __syncthreads();
        if (threadIdx.x == 0) s_got = min(S, got + tot);
        __syncthreads();
    }
    if (s_got < S) {
        park();
        return;
    }
    // sort the distinct ranks: position = number of smaller ranks
    for (uint32_t i = threadIdx.x; i < S; i += blockDim.x) {
        const uint32_t r = chosen[i];
        sorted[count_if(chosen, S, [&](uint32_t v) { return v < r; })] = r;
    }
    __syncthreads();
    // rank -> tile -> cell: lane l holds the candidates of the tile's word l, a wave scan finds the lane with the
    // wanted one
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    for (uint32_t i = part * kWaves + wave; i < S; i += kPickParts * kWaves) {
        const unsigned long long want = base + sorted[i];
        const uint32_t t = wave_last_below(tile_off, t0, t1, want);
        const uint32_t need = (uint32_t)(want - tile_off[t]);
        const uint32_t w = (t - t0) * kTileWords + lane;
        const uint32_t bits = word_candidates(*J, w);
        const uint32_t cnt = (uint32_t)__popc(bits);
        uint32_t inc = cnt;  // wave inclusive scan
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t v = __shfl_up(inc, o, 64);
            if (lane >= (uint32_t)o) inc += v;
        }
        const bool holder = inc > need && inc - cnt <= need;
        if (holder) {
            const uint32_t col = w >> (uint32_t)__builtin_ctz(J->wp), x = col / J->ny;
            J->seeds[i] = make_uint4(x, col - x * J->ny, (w & (J->wp - 1u)) * 32u + nth_bit(bits, need - (inc - cnt)), 2u + i);
        }
        if (__ballot(holder) == 0ull && lane == 0) {  // the counts disagree with the tile prefix
            J->seeds[i] = make_uint4(0u, 0u, 0u, 2u + i);
            atomicOr(reinterpret_cast<unsigned int*>(J->stats + kStatError), (unsigned int)kDevErrSeeding);
        }
    }
}

// Seeder::mergeSeeds (Seeder.cpp:115-152) in CADScene::fractureModel's order (CADScene.cpp:647-655): the
// merged list is the fragment seeds followed by the extra draw (at seeds[xoff..]); each entry takes the label of its nearest
// fragment seed (the reference's float distances on the coordinates, strict '<': the first fragment wins
// ties) with that fragment's running sub-seed id (1, 2, ... in list order) in bits 8..15.  The fragments
// stay first, the merged list follows them.  One block per job; entries staged in LDS.
constexpr uint32_t kMaxMerge = 2048;  // fragments + extra seeds of one job
__global__ __launch_bounds__(kSeedThreads) void k_seed_merge(Launch L)
{
    __shared__ uint32_t px[kMaxMerge], py[kMaxMerge], pz[kMaxMerge];
    __shared__ uint16_t near[kMaxMerge];
    const JobDev* J = L.jobs + blockIdx.x;
    if (!J->active || J->extra == 0) return;
    const uint32_t F = J->S0, M = J->S0 + J->extra;
    uint4* seeds = J->seeds;
    for (uint32_t i = threadIdx.x; i < M; i += blockDim.x) {
        const uint4 q = i < F ? seeds[i] : seeds[J->xoff + (i - F)];
        px[i] = q.x;
        py[i] = q.y;
        pz[i] = q.z;
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < M; i += blockDim.x) {
        uint32_t best = 0xFFFFFFFFu, arg = 0;
        for (uint32_t f = 0; f < F; ++f) {
            const uint32_t dx = px[i] > px[f] ? px[i] - px[f] : px[f] - px[i];
            const uint32_t dy = py[i] > py[f] ? py[i] - py[f] : py[f] - py[i];
            const uint32_t dz = pz[i] > pz[f] ? pz[i] - pz[f] : pz[f] - pz[i];
            // integer forms of the float distances (coordinates below 2^11): Manhattan and Chebyshev
            // exact, Euclidean as the correctly rounded float root of the squared distance
            const uint32_t d = J->merge_dist == VF_MANHATTAN ? dx + dy + dz
                               : J->merge_dist == VF_CHEBYSHEV ? max(dx, max(dy, dz))
                                                               : sqrt_rn_bits(dx * dx + dy * dy + dz * dz);
            if (d < best) {
                best = d;
                arg = f;
            }
        }
        near[i] = (uint16_t)arg;
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < M; i += blockDim.x) {
        const uint32_t f = near[i];
        uint32_t id = 1;
        for (uint32_t k = 0; k < i; ++k) id += near[k] == f ? 1u : 0u;
        if (id > 255u) atomicOr(reinterpret_cast<unsigned int*>(J->stats + kStatError), (unsigned int)kDevErrMerge);
        seeds[F + i] = make_uint4(px[i], py[i], pz[i], (seeds[f].w & 0xFFu) | ((id & 0xFFu) << 8));
    }
}

// floor(mn + (mx - mn) * h / 2^32): static_cast<int>(min + (max - min) * u) of
// RandomUtilities::getUniformRandomInt (RandomUtilities.h:141-144) for
// u = h / 2^32 wherever that is not negative.
__device__ inline int64_t uniform_int(int64_t mn, int64_t mx, uint32_t h)
{
    const int64_t t = (mx - mn) * (int64_t)h;
    return mn + (t >= 0 ? (t >> 32) : -((-t + 0xFFFFFFFFll) >> 32));
}

// Seeder::nearSeeds (Seeder.cpp:49-113) for one grid, one block.  Impact i
// draws with key k_i = key + (i + 1) * 0x9E3779B97F4A7C15: the fragment seed
// uniform_int(0, F - 1, h(k_i, 0)), the seed count min(uniform_int(1,
// pending, h(k_i, 1)), pending), and candidate t's axis a as
// n_a / 2 - sum_{j < spreading} h(k_i, 2 + (3t + a) spreading + j) mod
// (n_a / spreading) (getBiasedRandomInt) wrapped around the fragment seed.  A
// candidate is accepted, in draw order, when it lies within min(n) / 2 of the
// fragment seed, is occupied, on the surface (isBoundary) and new.  Batches of
// kSeedThreads candidates are tested in parallel; one lane accepts them in
// order.  out receives the fragments (unless out == frags) and then the new
// seeds; returns the number of new seeds, err = 1 if an impact hit the draw cap.
__device__ __forceinline__ uint32_t near_draw(const JobDev* J, const uint4* frags, uint32_t F, uint32_t impacts,
                                              uint32_t num_seeds, uint32_t spreading, uint64_t key, uint4* out,
                                              uint32_t& err)
{
    __shared__ uint32_t chosen[kMaxDeviceSeeds];
    __shared__ uint32_t sorted[kMaxDeviceSeeds];
    __shared__ uint32_t cand[kSeedThreads];
    __shared__ uint32_t s_n, s_got, s_err;
    const uint32_t n[3] = { J->nx, J->ny, J->nz };
    const uint32_t m[3] = { n[0] / spreading, n[1] / spreading, n[2] / spreading };
    const uint32_t mind = min(n[0], min(n[1], n[2])) / 2;
    if (threadIdx.x == 0) {
        s_n = 0;
        s_err = 0;
    }
    __syncthreads();
    uint32_t pending = num_seeds;
    for (uint32_t i = 0; i < impacts && !s_err; ++i) {
        const uint64_t k = key + (uint64_t)(i + 1u) * 0x9E3779B97F4A7C15ull;
        const uint4 fr = frags[uniform_int(0, (int64_t)F - 1, hash32(k, 0))];
        const int64_t w = uniform_int(1, pending, hash32(k, 1));
        const uint32_t want = (uint32_t)max<int64_t>(0, min<int64_t>(w, pending));
        if (threadIdx.x == 0) s_got = 0;
        __syncthreads();
        for (uint32_t t0 = 0; s_got < want; t0 += kSeedThreads) {
            if (t0 >= kMaxDraws) {
                if (threadIdx.x == 0) s_err = 1;
                break;
            }
            const uint32_t t = t0 + threadIdx.x;
            const uint32_t f[3] = { fr.x, fr.y, fr.z };
            uint32_t c[3];
            int64_t d2 = 0;
            for (int a = 0; a < 3; ++a) {
                uint32_t b = 0;
                for (uint32_t j = 0; j < spreading; ++j) b += hash32(k, 2u + (3u * t + (uint32_t)a) * spreading + j) % m[a];
                const int64_t o = (int64_t)(n[a] / 2) - (int64_t)b;
                c[a] = (uint32_t)(((int64_t)f[a] + o + n[a]) % n[a]);
                d2 += ((int64_t)c[a] - f[a]) * ((int64_t)c[a] - f[a]);
            }
            uint32_t id = 0xFFFFFFFFu;
            if (t < kMaxDraws && d2 <= (int64_t)mind * mind) {
                const size_t cell = ((size_t)c[0] * n[1] + c[1]) * n[2] + c[2];
                if (occ_bit(*J, c[0], c[1], c[2]) && surface_cell(*J, c[0], c[1], c[2])) {
                    id = (uint32_t)cell;
                    for (uint32_t q = 0; q < s_n && id != 0xFFFFFFFFu; ++q)
                        if (chosen[q] == id) id = 0xFFFFFFFFu;
                }
            }
            cand[threadIdx.x] = id;
            __syncthreads();
            if (threadIdx.x == 0) {
                const uint32_t first = s_n;
                for (uint32_t q = 0; q < kSeedThreads && s_got < want; ++q) {
                    const uint32_t v = cand[q];
                    if (v == 0xFFFFFFFFu) continue;
                    bool dup = false;
                    for (uint32_t r = first; r < s_n && !dup; ++r) dup = chosen[r] == v;
                    if (dup) continue;
                    chosen[s_n++] = v;
                    ++s_got;
                }
            }
            __syncthreads();
        }
        pending -= want;
        __syncthreads();
    }
    const uint32_t N = s_n;
    for (uint32_t i = threadIdx.x; i < N; i += blockDim.x) {
        const uint32_t v = chosen[i];
        uint32_t p = 0;
        for (uint32_t q = 0; q < N; ++q) p += chosen[q] < v ? 1u : 0u;
        sorted[p] = v;
    }
    __syncthreads();
    if (out != frags)
        for (uint32_t i = threadIdx.x; i < F; i += blockDim.x) out[i] = frags[i];
    const uint32_t label0 = frags[F - 1].w;
    for (uint32_t i = threadIdx.x; i < N; i += blockDim.x) {
        const uint32_t v = sorted[i];
        out[F + i] = make_uint4(v / (n[1] * n[2]), (v / n[2]) % n[1], v % n[2], label0 + 1u + i);
    }
    err = s_err;
    return N;
}

// One grid's nearSeeds.  result: [0] seeds written (fragments first), [1] 1 if an impact hit the draw cap.
__global__ __launch_bounds__(kSeedThreads) void k_seed_near(const JobDev* J, const uint4* frags, uint32_t F,
                                                             uint32_t impacts, uint32_t num_seeds, uint32_t spreading,
                                                             uint64_t key, uint4* out, uint32_t* result)
{
    uint32_t err = 0;
    const uint32_t N = near_draw(J, frags, F, impacts, num_seeds, spreading, key, out, err);
    if (threadIdx.x == 0) {
        result[0] = F + N;
        result[1] = err;
    }
}

// nearSeeds of every job with impacts (CADScene::fractureModel, CADScene.cpp:636-646), one block per job, in
// place: the new seeds follow the F_in fragment seeds, and the job's fragment count S0 and seed count S
// (fragments, then their merged copies and the extra draw when mergeSeeds follows) are set in the table.
__global__ __launch_bounds__(kSeedThreads) void k_seed_near_jobs(Launch L)
{
    JobDev* J = const_cast<JobDev*>(L.jobs + blockIdx.x);
    if (!J->active || J->impacts == 0) return;
    const uint32_t F = J->F_in;
    uint32_t err = 0;
    const uint32_t N = near_draw(J, J->seeds, F, J->impacts, J->near_seeds, J->spreading, J->near_key, J->seeds, err);
    if (threadIdx.x == 0) {
        const uint32_t S0 = F + N;
        J->S0 = S0;
        J->S = S0 + (J->extra ? S0 + J->extra : 0u);
        J->fctl[kCtlSeedCounts] = J->S;  // for tables made later
        J->fctl[kCtlSeedCounts + 1] = S0;
        if (err) atomicOr(reinterpret_cast<unsigned int*>(J->stats + kStatError), (unsigned int)kDevErrSeeding);
    }
}

__global__ void k_seed_counts(Launch L)
{
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= L.njobs) return;
    JobDev* J = const_cast<JobDev*>(L.jobs + j);
    if (!J->impacts) return;
    J->S = J->fctl[kCtlSeedCounts];
    J->S0 = J->fctl[kCtlSeedCounts + 1];
}

}  // namespace

void launch_seed_merge(const Launch& L)
{
    TimedLaunch tl("seed_merge", L.s);
    k_seed_merge<<<L.njobs, kSeedThreads, 0, L.s>>>(L);
    VF_CHECK_LAUNCH();
}

void launch_seed_near(const Launch& L, const uint4* frags, uint32_t F, uint32_t impacts, uint32_t num_seeds,
                      uint32_t spreading, uint64_t key, uint4* out, uint32_t* result)
{
    if (!F || !spreading || spreading > 64 || num_seeds > kMaxDeviceSeeds)
        fail(VF_ERR_INVALID_ARG, "near seeding needs fragment seeds, spreading 1..64 and at most %u seeds",
             kMaxDeviceSeeds);
    TimedLaunch tl("seed_near", L.s);
    k_seed_near<<<1, kSeedThreads, 0, L.s>>>(L.jobs, frags, F, impacts, num_seeds, spreading, key, out, result);
    VF_CHECK_LAUNCH();
}

void launch_seed_near_jobs(const Launch& L)
{
    TimedLaunch tl("seed_near", L.s);
    k_seed_near_jobs<<<L.njobs, kSeedThreads, 0, L.s>>>(L);
    VF_CHECK_LAUNCH();
}

void launch_seed_counts(const Launch& L)
{
    TimedLaunch tl("seed_counts", L.s);
    k_seed_counts<<<ceil_div(L.njobs, 64u), 64, 0, L.s>>>(L);
    VF_CHECK_LAUNCH();
}

void launch_seed_count(const Launch& L, uint32_t* tile_cnt, bool skip_both)
{
    TimedLaunch tl("seed_count", L.s);
    const uint32_t blocks = std::max(1u, std::min(ceil_div(L.total_wtiles, kCellThreads / 64u), active_shape().cell_blocks));
    k_seed_count<<<blocks, kCellThreads, 0, L.s>>>(L, tile_cnt, skip_both);
    VF_CHECK_LAUNCH();
}

void launch_seed_pick(const Launch& L, const unsigned long long* tile_off)
{
    TimedLaunch tl("seed_pick", L.s);
    k_seed_pick<<<L.njobs * kPickParts, kSeedThreads, 0, L.s>>>(L, tile_off);
    VF_CHECK_LAUNCH();
}

}  // namespace vf
