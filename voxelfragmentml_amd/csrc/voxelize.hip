// Conservative voxelization: FP32 triangle/box SAT shell plus a z-parity
// interior fill, replacing the reference's raster Tetravoxelizer
// (RegularGrid::fill, RegularGrid.cpp:173-212; Tetravoxelizer.cpp:264-315).
//
// Pipeline (all jobs of a launch together, no host synchronisation):
//   1. k_vox_setup   per triangle: SAT candidate cell box, snapped fixed-point
//                    vertices, parity column range, pair counts
//   2. scans         exclusive prefix of the pair counts (load balancing)
//   3. k_vox_pairs   shell: one thread per (triangle, column, 32-cell z word): SAT
//                    (Intersections3D.h:204-420 arithmetic) per cell with the
//                    z-free terms once per column, one atomicOr per word;
//                    parity: one thread per (triangle, column) pair: top-left covered
//                    column centres toggle the first cell centre above the
//                    crossing (exact int64 edge functions), atomicXor
//   4. k_vox_fill    one lane per 32-cell column word: prefix-XOR in the word,
//                    carry across the column by wave ballot, occupancy bits
//                    = shell | parity, occupied count
// Compiled with -ffp-contract=off: FP32 results equal the CPU oracle's.
#include "cellops.hpp"

namespace vf {

namespace {

constexpr int kSub = 256;
constexpr float kSnapLim = 524288.0f;
constexpr uint32_t kVoxThreads = 256;
constexpr float kRangeMargin = 0.015625f;   // 1/64 cell
constexpr uint32_t kInlineShell = 8;        // SAT candidates a setup thread tests itself
constexpr uint32_t kInlineCols = 8;         // parity columns a setup thread toggles itself
constexpr uint32_t kWildTriangle = 1u << 31;  // TriSetup::job flag: coordinates of kTameLimit or more
constexpr uint32_t kColBits = 4;            // column index bits in the setup kernel's owner tables
static_assert(kInlineShell <= (1u << kColBits) && kInlineCols <= (1u << kColBits), "owner table encoding");

// A separating-axis test in two forms with the same outcome.  Exact: comparisons as the reference makes them.  Tame (no
// operand is infinite or NaN): each axis yields a value above 0 where it separates, and a cell's values are combined by
// one running maximum, which takes fewer instructions than a comparison each: x > y exactly where x - y > 0.
template <bool TAME>
struct Separation {
    float most = -1.0f;
    bool sep = false;
    // projections pa, pb both beyond rad on one side: min(pa, pb) > rad || max(pa, pb) < -rad (the median of pa, pb and
    // 0 is the one nearer to 0 when both lie on one side of it, else 0)
    __device__ inline void axis(float pa, float pb, float rad)
    {
        if (TAME) {
            most = __builtin_fmaxf(most, fabsf(__builtin_amdgcn_fmed3f(pa, pb, 0.0f)) - rad);
        } else {
            float mn = pa < pb ? pa : pb;
            float mx = pa < pb ? pb : pa;
            sep |= mn > rad || mx < -rad;
        }
    }
    // a box face: all three of a, b, c beyond h on one side
    __device__ inline void face(float a, float b, float c, float h)
    {
        if (TAME) {
            const float mn = __builtin_fminf(__builtin_fminf(a, b), c), mx = __builtin_fmaxf(__builtin_fmaxf(a, b), c);
            most = __builtin_fmaxf(most, __builtin_fmaxf(mn, -mx) - h);
        } else {
            float mn = a, mx = a;
            if (b < mn) mn = b;
            if (b > mx) mx = b;
            if (c < mn) mn = c;
            if (c > mx) mx = c;
            sep |= mn > h || mx < -h;
        }
    }
    // the triangle's plane: the box's least and greatest distance along the normal
    __device__ inline void plane(float dmin, float dmax)
    {
        if (TAME) most = __builtin_fmaxf(__builtin_fmaxf(most, dmin), -dmax);
        else sep |= dmin > 0.0f || !(dmax >= 0.0f);
    }
    __device__ inline bool any() const { return TAME ? most > 0.0f : sep; }
};

// n times the end of [lo, hi] that makes it least, and greatest.
template <bool TAME>
__device__ inline void span(float n, float lo, float hi, float& least, float& greatest)
{
    if (TAME) {
        const float a = n * lo, b = n * hi;
        least = __builtin_fminf(a, b);
        greatest = __builtin_fmaxf(a, b);
    } else {
        least = n * (n > 0.0f ? lo : hi);
        greatest = n * (n > 0.0f ? hi : lo);
    }
}

// Coordinates below this keep every product and sum of the SAT finite (three factors of at most 4e12 and sums of
// three of them stay below 3e38), so no operand of a comparison is NaN.
constexpr float kTameLimit = 1e12f;

__device__ inline void cell_box(int i, float mn, float cs, float* center, float* half)
{
    float lo = mn + (float)i * cs;
    float hi = mn + (float)(i + 1) * cs;
    *center = (hi + lo) / 2.0f;
    *half = hi - *center;
}

// The triangle/box SAT of Intersections3D::intersect(Triangle3D&, AABB&) (Intersections3D.h:204-420:
// nine edge-cross axes, the three box faces, the triangle plane) for the cells of one grid column.  For
// each cell every FP32 operation is the reference's (same operands, same order, no contraction), so
// a cell passes exactly when the per-cell test passes; which axis separates first does not change the outcome.
// Column: what a column of cells shares, the vertices' x and y offsets from its centre, its half extents and the
// vertices' z.
struct Column {
    float v0x, v1x, v2x, v0y, v1y, v2y, hx, hy, az, bz, cz;
};
__device__ inline Column make_column(const float* a, const float* b, const float* c, float cx, float hx, float cy, float hy)
{
    return Column{ a[0] - cx, b[0] - cx, c[0] - cx, a[1] - cy, b[1] - cy, c[1] - cy, hx, hy, a[2], b[2], c[2] };
}

// The tests that do not depend on z (the third axis of each edge, the x and y faces): false when no cell passes.
template <bool TAME>
__device__ __forceinline__ bool column_open(const Column& q)
{
    const float e0x = q.v1x - q.v0x, e1x = q.v2x - q.v1x, e2x = q.v0x - q.v2x;
    const float e0y = q.v1y - q.v0y, e1y = q.v2y - q.v1y, e2y = q.v0y - q.v2y;
    Separation<TAME> s;
    s.axis(e0y * q.v1x - e0x * q.v1y, e0y * q.v2x - e0x * q.v2y, fabsf(e0y) * q.hx + fabsf(e0x) * q.hy);
    s.axis(e1y * q.v0x - e1x * q.v0y, e1y * q.v1x - e1x * q.v1y, fabsf(e1y) * q.hx + fabsf(e1x) * q.hy);
    s.axis(e2y * q.v1x - e2x * q.v1y, e2y * q.v2x - e2x * q.v2y, fabsf(e2y) * q.hx + fabsf(e2x) * q.hy);
    s.face(q.v0x, q.v1x, q.v2x, q.hx);
    s.face(q.v0y, q.v1y, q.v2y, q.hy);
    return !s.any();
}

// The tests that do, for the cell between z planes lo and hi of an open column.
template <bool TAME>
__device__ __forceinline__ bool cell_passes(const Column& q, float lo, float hi)
{
    const float e0x = q.v1x - q.v0x, e1x = q.v2x - q.v1x, e2x = q.v0x - q.v2x;
    const float e0y = q.v1y - q.v0y, e1y = q.v2y - q.v1y, e2y = q.v0y - q.v2y;
    const float f0x = fabsf(e0x), f0y = fabsf(e0y), f1x = fabsf(e1x), f1y = fabsf(e1y), f2x = fabsf(e2x), f2y = fabsf(e2y);
    const float cz = (hi + lo) / 2.0f, hz = hi - cz;
    const float v0z = q.az - cz, v1z = q.bz - cz, v2z = q.cz - cz;
    const float e0z = v1z - v0z, e1z = v2z - v1z, e2z = v0z - v2z;
    const float f0z = fabsf(e0z), f1z = fabsf(e1z), f2z = fabsf(e2z);
    Separation<TAME> s;
    s.axis(e0z * q.v0y - e0y * v0z, e0z * q.v2y - e0y * v2z, f0z * q.hy + f0y * hz);
    s.axis(-e0z * q.v0x + e0x * v0z, -e0z * q.v2x + e0x * v2z, f0z * q.hx + f0x * hz);
    s.axis(e1z * q.v0y - e1y * v0z, e1z * q.v2y - e1y * v2z, f1z * q.hy + f1y * hz);
    s.axis(-e1z * q.v0x + e1x * v0z, -e1z * q.v2x + e1x * v2z, f1z * q.hx + f1x * hz);
    s.axis(e2z * q.v0y - e2y * v0z, e2z * q.v1y - e2y * v1z, f2z * q.hy + f2y * hz);
    s.axis(-e2z * q.v0x + e2x * v0z, -e2z * q.v1x + e2x * v1z, f2z * q.hx + f2x * hz);
    s.face(v0z, v1z, v2z, hz);
    const float n0 = e0y * e1z - e1y * e0z;
    const float n1 = e0z * e1x - e1z * e0x;
    const float n2 = e0x * e1y - e1x * e0y;
    float min0, max0, min1, max1, min2, max2;
    span<TAME>(n0, -q.hx - q.v0x, q.hx - q.v0x, min0, max0);
    span<TAME>(n1, -q.hy - q.v0y, q.hy - q.v0y, min1, max1);
    span<TAME>(n2, -hz - v0z, hz - v0z, min2, max2);
    s.plane(min0 + min1 + min2, max0 + max1 + max2);
    return !s.any();
}

// The cells z0..z1 (inside one 32-cell word) of an open column of finite coordinates, from the z intervals in which the
// tests that depend on z pass: `sure` are cells that pass every test, `maybe` those too near an interval's end to tell.
// Along a column every such test is linear in the cell's number: with v_z = a - k cs an edge's projections are
// c + k e cs, so the axis separates outside [(-rad - max c) / (e cs), (rad - min c) / (e cs)]; the plane's distance and
// the z face likewise.  An interval is widened (to what may pass) and narrowed (to what surely does) by the rounding of
// the FP32 tests and of this function.  With E the largest edge component, V a bound on the vertices' offsets, and S one on
// the coordinates (|mn| + |a| + V), a cell's centre is off by less than 2^-21 S, an offset along z by 3 times that, an edge's
// z component by 2^-22 V, so that
//   an axis' projections and radius, here and there:  2^-20 V (V + E) + 2^-17.7 |e| S  <  2^-18 V (V + E) + 2^-15 |e| S,
//   the plane's:  2^-18.4 E V^2 + 2^-18.8 E^2 V + 2^-17.7 |n_z| S  <  2^-17 E V (V + E) + 2^-15 |n_z| S,
//   the z face's:  6 * 2^-21 S  <  2^-18 S.
// A slope below 1/64 of the error is taken as that much: over a word's 32 cells it moves the projection by less than
// half the error.
struct ZCells {
    uint32_t sure, maybe;
};
__device__ __forceinline__ ZCells z_cells(const Column& q, int z0, int z1, float mnz, float csz)
{
    const float e0x = q.v1x - q.v0x, e1x = q.v2x - q.v1x, e2x = q.v0x - q.v2x;
    const float e0y = q.v1y - q.v0y, e1y = q.v2y - q.v1y, e2y = q.v0y - q.v2y;
    const float e0z = q.bz - q.az, e1z = q.cz - q.bz, e2z = q.az - q.cz;
    const float base = mnz + ((float)z0 + 0.5f) * csz, hz = 0.5f * csz;
    const float a = q.az - base, b = q.bz - base, c = q.cz - base;
    auto max3 = [](float x, float y, float z) { return __builtin_fmaxf(__builtin_fmaxf(fabsf(x), fabsf(y)), fabsf(z)); };
    const float E = max3(max3(e0x, e1x, e2x), max3(e0y, e1y, e2y), max3(e0z, e1z, e2z));
    const float V = max3(max3(q.v0x, q.v1x, q.v2x), max3(q.v0y, q.v1y, q.v2y), E) + 2.0f * (csz + q.hx + q.hy);
    const float S = fabsf(mnz) + fabsf(q.az) + V;
    const float err = 0x1p-18f * V * (V + E), far = 0x1p-15f * S;
    const float last = (float)(z1 - z0);
    float olo = 0.0f, ohi = last, ilo = 0.0f, ihi = last;  // k of cells that may pass, that surely do
    auto interval = [&](float lo, float hi, float e) {
        olo = __builtin_fmaxf(olo, lo - e);
        ohi = __builtin_fminf(ohi, hi + e);
        ilo = __builtin_fmaxf(ilo, lo + e);
        ihi = __builtin_fminf(ihi, hi - e);
    };
    // lower <= s k <= upper, both off by less than er
    auto linear = [&](float s, float lower, float upper, float er) {
        const float inv = __builtin_amdgcn_rcpf(__builtin_fmaxf(fabsf(s), er * 0x1p-6f));
        const float lo = s < 0.0f ? -upper : lower, hi = s < 0.0f ? -lower : upper;
        interval(lo * inv, hi * inv, er * inv + 0x1p-12f);
    };
    auto axis = [&](float ez, float ey, float py, float pz, float qy, float qz, float h) {
        const float cp = __builtin_fmaf(ez, py, -(ey * pz)), cq = __builtin_fmaf(ez, qy, -(ey * qz));
        const float er = __builtin_fmaf(far, fabsf(ey), err);
        // an edge along the other coordinate separates nothing: all its products are 0
        const float rad = ez == 0.0f && ey == 0.0f ? 4.0f * er : __builtin_fmaf(fabsf(ez), h, fabsf(ey) * hz);
        linear(ey * csz, -rad - __builtin_fmaxf(cp, cq), rad - __builtin_fminf(cp, cq), er);
    };
    axis(e0z, e0y, q.v0y, a, q.v2y, c, q.hy);
    axis(e0z, e0x, q.v0x, a, q.v2x, c, q.hx);
    axis(e1z, e1y, q.v0y, a, q.v2y, c, q.hy);
    axis(e1z, e1x, q.v0x, a, q.v2x, c, q.hx);
    axis(e2z, e2y, q.v0y, a, q.v1y, b, q.hy);
    axis(e2z, e2x, q.v0x, a, q.v1x, b, q.hx);
    const float ic = __builtin_amdgcn_rcpf(csz);
    interval((__builtin_fminf(__builtin_fminf(a, b), c) - hz) * ic, (__builtin_fmaxf(__builtin_fmaxf(a, b), c) + hz) * ic,
             0x1p-18f * S * ic + 0x1p-12f);
    const float n0 = e0y * e1z - e1y * e0z, n1 = e0z * e1x - e1z * e0x, n2 = e0x * e1y - e1x * e0y;
    const float g = n0 * q.v0x + n1 * q.v0y + n2 * a;  // |g - n2 cs k| <= r
    const float r = fabsf(n0) * q.hx + fabsf(n1) * q.hy + fabsf(n2) * hz;
    const float errn = __builtin_fmaf(far, fabsf(n2), 0x1p-17f * E * V * (V + E));
    linear(n2 * csz, g - r, g + r, errn);
    // a triangle or cells so small or large that these lose their meaning: every cell by its tests
    const bool good = err > 1e-30f && errn > 1e-30f && errn < 1e30f && csz > 1e-30f;
    auto bits = [&](float lo, float hi) {
        const int l = (int)__builtin_ceilf(lo), h = (int)__builtin_floorf(hi);  // both in -1 .. 32 where it matters
        return l > h ? 0u : ((2u << (h & 31)) - 1u) & ~((1u << (l & 31)) - 1u);
    };
    const uint32_t all = bits(0.0f, last), may = good ? bits(__builtin_fminf(olo, 32.0f), __builtin_fmaxf(ohi, -1.0f)) : all;
    const uint32_t sure = good ? bits(__builtin_fminf(ilo, 32.0f), __builtin_fmaxf(ihi, -1.0f)) : 0u;
    return ZCells{ sure << (z0 & 31), (may & ~sure) << (z0 & 31) };
}

// z plane k of a grid (the lower face of cell k, the upper of cell k - 1), as cell_box has it
__device__ inline float z_plane(int k, float mnz, float csz) { return mnz + (float)k * csz; }

// The cells z0..z1 (inside one 32-cell word) of a column: bit (z & 31) is set when cell z passes.
template <bool TAME>
__device__ __forceinline__ uint32_t sat_column(const Column& q, int z0, int z1, float mnz, float csz)
{
    if (!column_open<TAME>(q)) return 0u;
    uint32_t bits = 0;
    float lo = z_plane(z0, mnz, csz);
    for (int z = z0; z <= z1; ++z) {
        const float hi = z_plane(z + 1, mnz, csz);
        bits |= cell_passes<TAME>(q, lo, hi) ? 1u << (z & 31) : 0u;
        lo = hi;
    }
    return bits;
}

// (x - mn) / cs in grid cells, the quotient both the candidate range and the snap start from
__device__ inline float grid_coord(float x, float mn, float cs) { return (x - mn) / cs; }

__device__ inline int32_t snap_coord(float q)
{
    q = q * (float)kSub;
    if (!(q >= -kSnapLim)) q = -kSnapLim;
    if (q > kSnapLim) q = kSnapLim;
    return (int32_t)rintf(q);
}

__device__ inline int clampi(int v, int lo, int hi) { return v < lo ? lo : (v > hi ? hi : v); }

// TriSetup records are stored as 8 planes of 16-byte pieces: piece k of record g at plane k, index g.
// A wave's stores of 64 consecutive records are then 8 contiguous 1 KiB runs instead of 16-byte pieces
// 128 bytes apart; readers fetch the pieces they use.
static_assert(sizeof(TriSetup) == 8 * sizeof(uint4), "TriSetup is eight 16-byte pieces");
__device__ inline void store_setup(TriSetup* base, uint32_t total, uint32_t g, const TriSetup& S)
{
    uint4 piece[8];
    __builtin_memcpy(piece, &S, sizeof(TriSetup));
    uint4* dst = reinterpret_cast<uint4*>(base);
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) gstore4(dst + (size_t)k * total + g, piece[k]);
}
__device__ inline TriSetup load_setup(const TriSetup* base, uint32_t total, uint32_t g)
{
    uint4 piece[8];
    const uint4* src = reinterpret_cast<const uint4*>(base);
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) piece[k] = src[(size_t)k * total + g];
    TriSetup S;
    __builtin_memcpy(&S, piece, sizeof(TriSetup));
    return S;
}

__device__ inline bool edge_incl(int64_t e, int64_t dx, int64_t dy)
{
    return e > 0 || (e == 0 && (dy < 0 || (dy == 0 && dx < 0)));
}

// floor(a / b) for b > 0: an FP32 estimate, then exact int64 remainder corrections (the estimate is
// within one of the quotient wherever |a / b| < 2^20; the loops make it exact everywhere)
__device__ inline int64_t floordiv64(int64_t a, int64_t b)
{
    int64_t q = (int64_t)floorf((float)a * __builtin_amdgcn_rcpf((float)b));
    int64_t r = a - q * b;
    while (r < 0) {
        --q;
        r += b;
    }
    while (r >= b) {
        ++q;
        r -= b;
    }
    return q;
}

// Column (i, j): if its centre is covered by the triangle's xy projection
// (top-left rule on exact int64 edge functions), the parity bit of the
// first cell whose centre lies above the crossing, to be toggled.
__device__ inline void parity_column(const JobDev* J, const TriSetup& S, int i, int jj, uint32_t& word, uint32_t& bit)
{
    const int64_t X0 = S.X[0], X1 = S.X[1], X2 = S.X[2];
    const int64_t Y0 = S.Y[0], Y1 = S.Y[1], Y2 = S.Y[2];
    const int64_t px = (int64_t)i * kSub + kSub / 2, py = (int64_t)jj * kSub + kSub / 2;
    const int64_t d0x = X2 - X1, d0y = Y2 - Y1, d1x = X0 - X2, d1y = Y0 - Y2, d2x = X1 - X0, d2y = Y1 - Y0;
    const int64_t E0 = d0x * (py - Y1) - d0y * (px - X1);
    const int64_t E1 = d1x * (py - Y2) - d1y * (px - X2);
    const int64_t E2 = d2x * (py - Y0) - d2y * (px - X0);
    if (!edge_incl(E0, d0x, d0y) || !edge_incl(E1, d1x, d1y) || !edge_incl(E2, d2x, d2y)) return;
    const int64_t num = E0 * (int64_t)S.Z[0] + E1 * (int64_t)S.Z[1] + E2 * (int64_t)S.Z[2];
    int64_t k = floordiv64(num - (int64_t)(kSub / 2) * S.area, (int64_t)kSub * S.area) + 1;
    if (k < 0) k = 0;
    if (k >= (int64_t)J->nz) return;
    word = (uint32_t)(((size_t)i * J->ny + (size_t)jj) * J->wp + (size_t)(k >> 5));
    bit = 1u << (k & 31);
}

__global__ __launch_bounds__(kVoxThreads) void k_vox_setup(const JobDev* jobs, uint32_t njobs, const uint32_t* tri_prefix,
                                                           uint32_t total, TriSetup* setup, uint32_t* cnt_shell, uint32_t* cnt_col)
{
    // Small triangles' candidate columns (shell) and covered columns (parity) are tested in this kernel,
    // shared by the lanes of a wave: each lane stashes its triangle in the wave's slots and lists its
    // columns as (lane << kColBits | column) in an owner table; the wave then takes the listed columns 64 at a
    // time, instead of every lane looping over its own (as many steps as its largest triangle).
    // Bound by the memory side's atomics first: 0.93 ms for the 9.2 M triangles of 64 mixed grids, with 13 M atomics.
    // Timed with one part left out each: 0.51 ms without the atomics, 0.62 without the parity columns, 0.74 without the
    // shell's cells, 0.76 without the record stores, 0.26 with neither columns, cells nor stores.  Combining the
    // words in LDS before their atomics, as the pairs do, was 0.91 ms here and at 64^3 15.7 us instead of 13.4.
    constexpr uint32_t kWaves = kVoxThreads / 64;
    // 16-bit pairs hold cell indices (< 2048) and extents: lo0 | lo1 << 16, lo2 | hi2 << 16, ey | nj << 16, i0 | j0 << 16
    enum { kLo01, kLo2Hi2, kEyNj, kI0J0, kJob, kX, kY = kX + 3, kZ = kY + 3, kAreaLo = kZ + 3, kAreaHi, kFields };
    __shared__ uint32_t sp[kWalkMaxJobs + 1];
    __shared__ float sP[kWaves][9][64];
    __shared__ int32_t sF[kWaves][kFields][64];
    __shared__ uint16_t sOwnS[kWaves][64 * kInlineShell], sOwnP[kWaves][64 * kInlineCols];
    for (uint32_t i = threadIdx.x; i <= njobs; i += blockDim.x) sp[i] = tri_prefix[i];
    __syncthreads();
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    for (uint32_t g0 = blockIdx.x * blockDim.x; g0 < total; g0 += gridDim.x * blockDim.x) {  // block-uniform
        const uint32_t g = g0 + threadIdx.x;
        const bool valid = g < total;
        const uint32_t j = valid ? find_job(sp, njobs, g) : 0u;
        const JobDev* J = jobs + j;
        TriSetup S;
        S.job = j;
        S.area = 0;
        S.i0 = S.j0 = 0;
        S.i1 = S.j1 = -1;
        for (int q = 0; q < 3; ++q) S.lo[q] = S.hi[q] = S.X[q] = S.Y[q] = S.Z[q] = 0;
        uint32_t nshell = 0, ncol = 0;
        const uint32_t t = g - sp[j];
        uint32_t vi[3] = { 0, 0, 0 };
        bool in_range = true, wild = false;
        if (valid && J->active) {
            for (int k = 0; k < 3; ++k) {
                vi[k] = J->tri[3 * (size_t)t + k];
                in_range &= vi[k] < J->nv;
            }
            if (!in_range)  // a device mesh with a bad index: flag the job and skip the triangle
                atomicOr(reinterpret_cast<unsigned int*>(J->stats + kStatError), (unsigned int)kDevErrMesh);
        }
        if (valid && J->active && in_range) {
            const float* p[3] = { J->xyz + 3 * (size_t)vi[0], J->xyz + 3 * (size_t)vi[1], J->xyz + 3 * (size_t)vi[2] };
            float P[3][3];
            bool finite = true;
            for (int k = 0; k < 3; ++k)
                for (int q = 0; q < 3; ++q) {
                    P[k][q] = p[k][q];
                    S.P[k][q] = P[k][q];
                    finite &= __builtin_isfinite(P[k][q]);
                    wild |= !(fabsf(P[k][q]) < kTameLimit);
                }
            for (int q = 0; q < 3; ++q) wild |= !(fabsf(J->mn[q]) < kTameLimit) || !(fabsf(J->mx[q]) < kTameLimit);
            const uint32_t dims[3] = { J->nx, J->ny, J->nz };
            if (finite) {
                // vertex coordinates in cells; (v - mn) / cs is monotone in v, so the extremes
                // of these are the quotients of the extreme coordinates
                float G[3][3];
                for (int k = 0; k < 3; ++k)
                    for (int q = 0; q < 3; ++q) G[k][q] = grid_coord(P[k][q], J->mn[q], J->cs[q]);
                bool empty = false;
                for (int q = 0; q < 3; ++q) {
                    float mn = G[0][q], mx = G[0][q];
                    if (G[1][q] < mn) mn = G[1][q];
                    if (G[1][q] > mx) mx = G[1][q];
                    if (G[2][q] < mn) mn = G[2][q];
                    if (G[2][q] > mx) mx = G[2][q];
                    // candidate cells: those within 1/64 cell of the triangle's extent (the
                    // SAT's FP32 box test can only accept touching cells, and its rounding
                    // is far below the margin)
                    float fl = floorf(mn - kRangeMargin);
                    float fh = floorf(mx + kRangeMargin);
                    const float lim = (float)dims[q] + 1.0f;
                    fl = fl < -2.0f ? -2.0f : (fl > lim ? lim : fl);
                    fh = fh < -2.0f ? -2.0f : (fh > lim ? lim : fh);
                    if ((int)fh < 0 || (int)fl > (int)dims[q] - 1) empty = true;
                    S.lo[q] = clampi((int)fl, 0, (int)dims[q] - 1);
                    S.hi[q] = clampi((int)fh, 0, (int)dims[q] - 1);
                }
                if (!empty)
                    nshell = (uint32_t)(S.hi[0] - S.lo[0] + 1) * (uint32_t)(S.hi[1] - S.lo[1] + 1) *
                             (uint32_t)(S.hi[2] - S.lo[2] + 1);
                int64_t X[3], Y[3], Z[3];
                for (int k = 0; k < 3; ++k) {
                    X[k] = snap_coord(G[k][0]);
                    Y[k] = snap_coord(G[k][1]);
                    Z[k] = snap_coord(G[k][2]);
                }
                int64_t area = (X[1] - X[0]) * (Y[2] - Y[0]) - (Y[1] - Y[0]) * (X[2] - X[0]);
                if (area != 0) {
                    if (area < 0) {
                        int64_t tx = X[1], ty = Y[1], tz = Z[1];
                        X[1] = X[2]; Y[1] = Y[2]; Z[1] = Z[2];
                        X[2] = tx; Y[2] = ty; Z[2] = tz;
                        area = -area;
                    }
                    int32_t mnx = (int32_t)X[0], mxx = (int32_t)X[0], mny = (int32_t)Y[0], mxy = (int32_t)Y[0];
                    for (int k = 1; k < 3; ++k) {
                        mnx = min(mnx, (int32_t)X[k]); mxx = max(mxx, (int32_t)X[k]);
                        mny = min(mny, (int32_t)Y[k]); mxy = max(mxy, (int32_t)Y[k]);
                    }
                    int i0 = (mnx - kSub / 2 + kSub - 1) >> 8, i1 = (mxx - kSub / 2) >> 8;
                    int j0 = (mny - kSub / 2 + kSub - 1) >> 8, j1 = (mxy - kSub / 2) >> 8;
                    i0 = max(i0, 0); j0 = max(j0, 0);
                    i1 = min(i1, (int)dims[0] - 1); j1 = min(j1, (int)dims[1] - 1);
                    for (int k = 0; k < 3; ++k) {
                        S.X[k] = (int32_t)X[k]; S.Y[k] = (int32_t)Y[k]; S.Z[k] = (int32_t)Z[k];
                    }
                    S.area = area;
                    S.i0 = i0; S.i1 = i1; S.j0 = j0; S.j1 = j1;
                    if (i1 >= i0 && j1 >= j0) ncol = (uint32_t)(i1 - i0 + 1) * (uint32_t)(j1 - j0 + 1);
                }
            }
        }
        // small triangles are tested here; the others go to the pair kernels, the shell as segments of
        // a column (x, y) that lie in one 32-cell word of z
        uint32_t nis = 0, nip = 0;  // this lane's inline shell columns and parity columns
        S.job |= wild ? kWildTriangle : 0u;
        if (nshell && nshell <= kInlineShell && !wild) {
            nis = (uint32_t)(S.hi[0] - S.lo[0] + 1) * (uint32_t)(S.hi[1] - S.lo[1] + 1);
            nshell = 0;
        } else if (nshell) {
            nshell = (uint32_t)(S.hi[0] - S.lo[0] + 1) * (uint32_t)(S.hi[1] - S.lo[1] + 1) *
                     (uint32_t)((S.hi[2] >> 5) - (S.lo[2] >> 5) + 1);
        }
        if (ncol && ncol <= kInlineCols) {
            nip = ncol;
            ncol = 0;
        }
        if (valid) {
            // only the pair kernels read a record, and only a triangle with pairs left
            if (nshell | ncol) store_setup(setup, total, g, S);
            cnt_shell[g] = nshell;
            cnt_col[g] = ncol;
        }
        // stash the triangle and list its columns
        if (nis | nip) {
#pragma unroll
            for (int k = 0; k < 3; ++k)
#pragma unroll
                for (int q = 0; q < 3; ++q) sP[wave][3 * k + q][lane] = S.P[k][q];
            sF[wave][kLo01][lane] = S.lo[0] | S.lo[1] << 16;
            sF[wave][kLo2Hi2][lane] = S.lo[2] | S.hi[2] << 16;
            sF[wave][kEyNj][lane] = (S.hi[1] - S.lo[1] + 1) | (S.j1 - S.j0 + 1) << 16;
            sF[wave][kI0J0][lane] = S.i0 | S.j0 << 16;
            sF[wave][kJob][lane] = (int32_t)j;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                sF[wave][kX + k][lane] = S.X[k];
                sF[wave][kY + k][lane] = S.Y[k];
                sF[wave][kZ + k][lane] = S.Z[k];
            }
            sF[wave][kAreaLo][lane] = (int32_t)(uint32_t)S.area;
            sF[wave][kAreaHi][lane] = (int32_t)(uint32_t)((uint64_t)S.area >> 32);
        }
        uint32_t es = nis, ep = nip;  // wave inclusive scans
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const uint32_t us = __shfl_up(es, o, 64), up = __shfl_up(ep, o, 64);
            if (lane >= (uint32_t)o) {
                es += us;
                ep += up;
            }
        }
        for (uint32_t k = 0; k < nis; ++k) sOwnS[wave][es - nis + k] = (uint16_t)(lane << kColBits | k);
        for (uint32_t k = 0; k < nip; ++k) sOwnP[wave][ep - nip + k] = (uint16_t)(lane << kColBits | k);
        const uint32_t ts = __shfl(es, 63, 64), tp = __shfl(ep, 63, 64);
        __syncthreads();
        for (uint32_t it = lane; it < ts; it += 64) {
            const uint32_t e = sOwnS[wave][it], o = e >> kColBits, c = e & ((1u << kColBits) - 1u);
            const int ey = sF[wave][kEyNj][o] & 0xFFFF, lo01 = sF[wave][kLo01][o], z2 = sF[wave][kLo2Hi2][o];
            const int x = (lo01 & 0xFFFF) + (int)c / ey, y = (lo01 >> 16) + (int)c % ey;
            const int lo2 = z2 & 0xFFFF, hi2 = z2 >> 16;
            const JobDev* Jo = jobs + sF[wave][kJob][o];
            float pa[3], pb[3], pc[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                pa[q] = sP[wave][q][o];
                pb[q] = sP[wave][3 + q][o];
                pc[q] = sP[wave][6 + q][o];
            }
            float cx, hx, cy, hy;
            cell_box(x, Jo->mn[0], Jo->cs[0], &cx, &hx);
            cell_box(y, Jo->mn[1], Jo->cs[1], &cy, &hy);
            for (int w = lo2 >> 5; w <= hi2 >> 5; ++w) {
                const uint32_t bits = sat_column<true>(make_column(pa, pb, pc, cx, hx, cy, hy), max(lo2, 32 * w),
                                                       min(hi2, 32 * w + 31), Jo->mn[2], Jo->cs[2]);
                if (bits) atomicOr(Jo->shell_bits + ((size_t)x * Jo->ny + (size_t)y) * Jo->wp + (size_t)w, bits);
            }
        }
        for (uint32_t it = lane; it < tp; it += 64) {
            const uint32_t e = sOwnP[wave][it], o = e >> kColBits, c = e & ((1u << kColBits) - 1u);
            TriSetup Q;
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                Q.X[k] = sF[wave][kX + k][o];
                Q.Y[k] = sF[wave][kY + k][o];
                Q.Z[k] = sF[wave][kZ + k][o];
            }
            Q.area = (int64_t)(((uint64_t)(uint32_t)sF[wave][kAreaHi][o] << 32) | (uint32_t)sF[wave][kAreaLo][o]);
            const int nj = sF[wave][kEyNj][o] >> 16, ij = sF[wave][kI0J0][o];
            const JobDev* Jo = jobs + sF[wave][kJob][o];
            uint32_t word = 0, bit = 0;
            parity_column(Jo, Q, (ij & 0xFFFF) + (int)c / nj, (ij >> 16) + (int)c % nj, word, bit);
            if (bit) atomicXor(Jo->toggle_bits + word, bit);
        }
        __syncthreads();  // the slots and owner tables are reused by the next 256 triangles
    }
}

// Largest g in [0, n) with off[g] <= p (off[0] == 0 <= p), searched by the
// whole wave with 64 probes per step: four dependent loads cover 16M entries.
__device__ inline uint32_t wave_search(const unsigned long long* off, uint32_t n, unsigned long long p)
{
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t lo = 0, hi = n;
    while (hi - lo > 64u) {
        const uint32_t step = (hi - lo + 63u) / 64u;
        const uint32_t idx = lo + lane * step;
        const bool ok = idx < hi && off[idx] <= p;
        const uint64_t m = __ballot(ok);
        const uint32_t last = 63u - (uint32_t)__clzll((long long)m);
        lo = lo + last * step;
        hi = min(lo + step, hi);
    }
    const uint32_t idx = lo + lane;
    const bool ok = idx < hi && off[idx] <= p;
    const uint64_t m = __ballot(ok);
    return lo + (63u - (uint32_t)__clzll((long long)m));
}

// A block takes chunks of up to kPairChunk consecutive pairs.  Two waves locate the chunk's first and last triangle, the
// block caches their offsets in LDS and each thread finds its triangle there.
constexpr uint32_t kPairChunk = 4 * kVoxThreads;
constexpr uint32_t kOffCache = 1024;

// The pairs p0 .. p1 - 1 (at most kPairChunk) of the ntris triangles whose offsets are off: f(g, local, valid) for pair
// `local` of triangle g, called by whole waves (valid: the lane has a pair).
template <class F>
__device__ inline void pair_chunk(const unsigned long long* off, uint32_t ntris, unsigned long long p0, unsigned long long p1,
                                  uint32_t* soff, uint32_t* sg, F&& f)
{
    const uint32_t wave = threadIdx.x >> 6;
    if (wave < 2) {
        const uint32_t g = wave_search(off, ntris + 1, wave == 0 ? p0 : p1 - 1);
        if ((threadIdx.x & 63u) == 0) sg[wave] = g;
    }
    __syncthreads();
    const uint32_t g0 = sg[0], n = sg[1] - g0 + 1;  // triangles g0 .. g0 + n - 1 hold the chunk
    const unsigned long long base = off[g0];
    const bool cached = n <= kOffCache;
    if (cached)  // from the first triangle's offset on: below it by less than 2^32 pairs of a triangle
        for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) soff[i] = (uint32_t)(off[g0 + i] - base);
    __syncthreads();
    for (unsigned long long pw = p0 + wave * 64u; pw < p1; pw += blockDim.x) {  // wave-uniform
        const unsigned long long p = min(pw + (threadIdx.x & 63u), p1 - 1);
        const uint32_t at = (uint32_t)(p - base);
        uint32_t lo = 0, hi = n;  // largest i with off[g0 + i] <= p
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if ((cached ? soff[mid] : (uint32_t)(off[g0 + mid] - base)) <= at) lo = mid; else hi = mid;
        }
        const uint32_t g = g0 + lo;
        f(g, at - (cached ? soff[lo] : (uint32_t)(off[g] - base)), pw + (threadIdx.x & 63u) < p1);
    }
    __syncthreads();
}

// The words that a wave's lanes are to change, combined in LDS first: neighbouring triangles meet the same words, and
// each change is an atomic at the memory side, of which the chip executes about 24 a nanosecond.
struct WordTable {
    uint32_t key[128], bits[128];  // open addressing; a key is 0xFFFFFFFF and its bits 0 while free
};
__device__ inline void wave_lds_fence()
{
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
__device__ inline void clear_table(WordTable& T)
{
    for (uint32_t e = threadIdx.x & 63u; e < 128u; e += 64u) {
        T.key[e] = 0xFFFFFFFFu;
        T.bits[e] = 0u;
    }
    wave_lds_fence();
}
// OR of bits into words[word], by all lanes of a wave; words: the lane's job's array (bits 0: nothing)
__device__ inline void combine_words(WordTable& T, uint32_t* words, uint32_t word, uint32_t bits)
{
    const uint64_t with = __ballot(bits != 0u);
    if (with == 0ull) return;
    // lanes of one job share the table; a wave across two jobs changes its words one by one
    const uint32_t first = (uint32_t)__builtin_ctzll(with);
    const uint64_t w0 = (uint64_t)words;
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)w0, (int)first),
                   hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(w0 >> 32), (int)first);
    uint32_t* const base = (uint32_t*)(((uint64_t)hi << 32) | lo);
    if (__ballot(bits != 0u && words != base)) {
        if (bits) atomicOr(words + word, bits);
        return;
    }
    bool pending = bits != 0u;
    uint32_t h = (word * 0x9E3779B1u) >> 25;
    while (__ballot(pending)) {  // at most 64 distinct words in 128 entries: every lane finds its own or a free one
        if (pending) {
            const uint32_t old = atomicCAS(&T.key[h], 0xFFFFFFFFu, word);
            if (old == 0xFFFFFFFFu || old == word) {
                atomicOr(&T.bits[h], bits);
                pending = false;
            } else {
                h = (h + 1u) & 127u;
            }
        }
    }
    wave_lds_fence();
#pragma unroll
    for (uint32_t e = threadIdx.x & 63u; e < 128u; e += 64u) {
        const uint32_t k = T.key[e], b = T.bits[e];
        if (k != 0xFFFFFFFFu) {
            if (b) atomicOr(base + k, b);
            T.key[e] = 0xFFFFFFFFu;
            T.bits[e] = 0u;
        }
    }
    wave_lds_fence();
}

// The pairs left by the setup kernel, shell and parity in one launch (one after the other, each paid a launch of
// thousands of workgroups and a tail).
// Shell: one lane per column segment of a triangle's candidate box, the cells (x, y, z) with z in one 32-cell word: the
// tests that do not depend on z, then the cells between the ends of the others' intervals (z_cells) at once and those
// near an end one by one (all of them where no lane of the wave has more than two).  The words of a wave are combined and
// then merged by atomicOr, where it has many triangles; those of one triangle are all different, and of two or three hardly the same
// (600 x 600 x 16 with 50 k triangles: 123 us combining all, 91; 2048 x 2048 x 1 with 20 k: 550 and 434).
// Bound by FP32 instruction issue (91 % of the rate).  Testing cell after cell, about 140 instructions each, a lane ran as
// long as the wave's longest column and merged every segment's word by itself: 2.14 ms for 64 mixed grids, 181 us
// at 512^3 with a million triangles; with the cells listed over the wave and the words combined (50.3 -> 33.7 M
// atomics) 1.82 ms and 135 us; by intervals 1.61 ms and 124 us, 256^3 with 200 k triangles 52 -> 39 us.
// Parity: one lane per column of a triangle's column range, one atomicXor each (combining them too gained nothing at any size,
// 512^3 with a million triangles 141 us either way, and cost up to 8 % on flat grids).
__global__ __launch_bounds__(kVoxThreads) __attribute__((amdgpu_waves_per_eu(5))) void k_vox_pairs(const JobDev* jobs, const TriSetup* setup,
                                                           const unsigned long long* off, uint32_t ntris, uint32_t chunk)
{
    __shared__ uint32_t soff[kOffCache];
    __shared__ uint32_t sg[2];
    __shared__ WordTable tables[kVoxThreads / 64];
    WordTable& table = tables[threadIdx.x >> 6];
    clear_table(table);
    // pairs [0, off[ntris]) are the shell's, [off[ntris], off[2 ntris]) the parity's
    const unsigned long long shell = off[ntris], total = off[2 * (size_t)ntris];
    const unsigned long long ns = (shell + chunk - 1) / chunk, np = (total - shell + chunk - 1) / chunk;
    for (unsigned long long c = blockIdx.x; c < ns + np; c += gridDim.x) {
        if (c < ns) {
            const unsigned long long p0 = c * chunk;
            pair_chunk(off, ntris, p0, min(p0 + chunk, shell), soff, sg, [&](uint32_t g, uint32_t col, bool valid) {
                const TriSetup Sg = load_setup(setup, ntris, g);
                const TriSetup* S = &Sg;
                const JobDev* J = jobs + (S->job & ~kWildTriangle);
                const int lo2 = S->lo[2], hi2 = S->hi[2];
                const uint32_t w0 = (uint32_t)lo2 >> 5, nseg = ((uint32_t)hi2 >> 5) - w0 + 1;
                const uint32_t ey = (uint32_t)(S->hi[1] - S->lo[1] + 1);
                uint32_t seg = 0;
                if (nseg > 1) {
                    seg = col % nseg;
                    col /= nseg;
                }
                const int y = S->lo[1] + (int)(col % ey), x = S->lo[0] + (int)(col / ey);
                const uint32_t w = w0 + seg;
                const float mnz = J->mn[2], csz = J->cs[2];
                float cx, hx, cy, hy;
                cell_box(x, J->mn[0], J->cs[0], &cx, &hx);
                cell_box(y, J->mn[1], J->cs[1], &cy, &hy);
                const int z0 = max(lo2, (int)(32 * w)), z1 = min(hi2, (int)(32 * w + 31));
                const Column q = make_column(S->P[0], S->P[1], S->P[2], cx, hx, cy, hy);
                uint32_t bits = 0;
                const bool few = __ballot(valid && z1 - z0 >= 2) == 0ull;
                if (valid) {
                    if (S->job & kWildTriangle) {
                        bits = sat_column<false>(q, z0, z1, mnz, csz);
                    } else if (column_open<true>(q)) {
                        ZCells z{ 0u, ((2u << (z1 - z0)) - 1u) << (z0 & 31) };
                        if (!few) z = z_cells(q, z0, z1, mnz, csz);
                        bits = z.sure;
                        for (uint32_t m = z.maybe; m; m &= m - 1u) {
                            const int k = (int)(32 * w) + (int)__builtin_ctz(m);
                            if (cell_passes<true>(q, z_plane(k, mnz, csz), z_plane(k + 1, mnz, csz))) bits |= m & -m;
                        }
                    }
                }
                const uint32_t word = (uint32_t)(((size_t)x * J->ny + (size_t)y) * J->wp + w);
                // lanes of a wave have ascending triangles
                const uint32_t triangles = (uint32_t)__builtin_amdgcn_readlane((int)g, 63) - (uint32_t)__builtin_amdgcn_readfirstlane((int)g) + 1u;
                if (triangles > 3u) combine_words(table, J->shell_bits, word, bits);
                else if (bits) atomicOr(J->shell_bits + word, bits);
            });
        } else {
            const unsigned long long p0 = shell + (c - ns) * chunk;
            pair_chunk(off + ntris, ntris, p0, min(p0 + chunk, total), soff, sg, [&](uint32_t g, uint32_t local, bool valid) {
                const TriSetup Sg = load_setup(setup, ntris, g);
                const uint32_t nj = (uint32_t)(Sg.j1 - Sg.j0 + 1);
                const JobDev* J = jobs + (Sg.job & ~kWildTriangle);
                uint32_t word = 0, bit = 0;
                if (valid) parity_column(J, Sg, Sg.i0 + (int)(local / nj), Sg.j0 + (int)(local % nj), word, bit);
                if (bit) atomicXor(J->toggle_bits + word, bit);
            });
        }
    }
}

// Occupancy bits = shell | parity interior, left in place of the shell bits.  Bound by HBM: 8 bytes read and 4
// written per 32 cells (as one byte per cell, 32 written, the 512^3 fill took 80 us, and every later stage
// read those bytes).  tile_cnt (or null): a wave's 64 words are one word tile, whose occupied cells it counts
// for jobs that seed anywhere.
__global__ __launch_bounds__(kVoxThreads) void k_vox_fill(Launch L, const uint32_t* col_prefix, uint32_t total_groups,
                                                          uint32_t* tile_cnt)
{
    __shared__ JobDev sJ;
    __shared__ unsigned long long part[kVoxThreads / 64];
    static_assert(kTileWords == 64, "a wave's words are one tile");
    unsigned long long acc = 0;
    constexpr uint32_t kRun = 4;  // column groups per step: all their bit loads are issued first
    walk_tile_runs<kRun>(L, col_prefix, total_groups, &sJ, [&](const JobDev& J, uint32_t jidx, uint32_t first, uint32_t nrun) {
        if (!J.active) return;
        const uint64_t nwords = (uint64_t)J.nx * J.ny * J.wp;
        uint32_t tgs[kRun], shs[kRun];
#pragma unroll
        for (uint32_t r = 0; r < kRun; ++r) {
            const uint64_t w = (uint64_t)(first + r) * kVoxThreads + threadIdx.x;
            const bool valid = r < nrun && w < nwords;
            tgs[r] = valid ? gcast<const uint32_t>(J.toggle_bits)[w] : 0u;
            shs[r] = valid ? gcast<const uint32_t>(J.shell_bits)[w] : 0u;
        }
        const uint32_t lane = threadIdx.x & 63u;
        const uint32_t seg = lane & ~(J.wp - 1u);
        const uint64_t below = (lane ? (~0ull >> (64u - lane)) : 0ull) & ~(seg ? (~0ull >> (64u - seg)) : 0ull);
#pragma unroll
        for (uint32_t r = 0; r < kRun; ++r) {
            if (r >= nrun) break;
            const uint64_t w = (uint64_t)(first + r) * kVoxThreads + threadIdx.x;
            const uint32_t tg = tgs[r];
            uint32_t p = tg;
            p ^= p << 1; p ^= p << 2; p ^= p << 4; p ^= p << 8; p ^= p << 16;
            const uint64_t par = __ballot(__popc(tg) & 1);
            if (__popcll(par & below) & 1) p = ~p;
            uint32_t bits = 0;
            if (w < nwords) {
                const uint32_t z0 = (uint32_t)(w & (J.wp - 1u)) * 32u;
                if (z0 < J.nz) {
                    const uint32_t nb = min(32u, J.nz - z0);
                    bits = (shs[r] | p) & (nb == 32 ? 0xFFFFFFFFu : ((1u << nb) - 1u));
                }
                gcast<uint32_t>(J.shell_bits)[w] = bits;
            }
            uint32_t cnt = (uint32_t)__popc(bits);
            acc += cnt;
            if (tile_cnt && J.seed_location == VF_SEED_BOTH) {  // block-uniform
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) cnt += __shfl_xor(cnt, o, 64);
                if (lane == 0 && w < nwords) tile_cnt[L.wtile_prefix[jidx] + (uint32_t)(w / kTileWords)] = cnt;
            }
        }
    }, [&](uint32_t j) {
        const unsigned long long s = wave_sum_u64(acc);
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
        __syncthreads();
        if (threadIdx.x == 0) {
            unsigned long long tot = 0;
            for (uint32_t w = 0; w < kVoxThreads / 64; ++w) tot += part[w];
            const JobDev& J = L.jobs[j];
            if (tot && J.sums) atomicAdd(J.sums + (blockIdx.x % kSumSlots) * kStatCount + kStatOccupied, tot);
        }
        __syncthreads();
        acc = 0;
    });
}

__global__ __launch_bounds__(kVoxThreads) void k_vox_clear(Launch L, const uint32_t* col_prefix, uint32_t total_groups)
{
    __shared__ JobDev sJ;
    walk_tiles(L, col_prefix, total_groups, &sJ, [&](const JobDev& J, uint32_t, uint32_t group, uint32_t) {
        if (!J.active) return;
        const uint64_t nwords = (uint64_t)J.nx * J.ny * J.wp;
        const uint64_t w = (uint64_t)group * kVoxThreads + threadIdx.x;
        if (w < nwords) {
            gcast<uint32_t>(J.toggle_bits)[w] = 0u;
            gcast<uint32_t>(J.shell_bits)[w] = 0u;
        }
    });
}

}  // namespace


void launch_clear_bits(const Launch& L, const uint32_t* col_prefix, uint32_t total_groups)
{
    TimedLaunch tl("vox_clear", L.s);
    const uint32_t blocks = std::max(1u, std::min(total_groups, active_shape().cell_blocks));
    k_vox_clear<<<blocks, kVoxThreads, 0, L.s>>>(L, col_prefix, total_groups);
    VF_CHECK_LAUNCH();
}

// X.setup / X.counts / X.shell_off / X.scan_tmp sized for X.total_tris (shell_off and the scan for twice that).
void launch_voxelize(const Launch& L, const VoxScratch& X, const uint32_t* col_prefix, uint32_t total_groups,
                     uint32_t* tile_cnt)
{
    if (L.njobs > kWalkMaxJobs) fail(VF_ERR_INVALID_ARG, "voxelize launch with %u jobs (max %u)", L.njobs, kWalkMaxJobs);
    launch_clear_bits(L, col_prefix, total_groups);
    if (X.total_tris) {
        uint32_t* cnt_shell = X.counts;
        uint32_t* cnt_col = cnt_shell + X.total_tris;
        {
            TimedLaunch tl("vox_setup", L.s);
            k_vox_setup<<<stride_blocks(X.total_tris, kVoxThreads), kVoxThreads, 0, L.s>>>(
                L.jobs, L.njobs, X.tri_prefix, X.total_tris, X.setup, cnt_shell, cnt_col);
            VF_CHECK_LAUNCH();
        }
        // one scan over both count arrays (contiguous): the parity offsets continue from the shell total
        scan_exclusive_u32_to_u64(cnt_shell, X.shell_off, 2ull * X.total_tris, X.scan_tmp, L.s);
        // workgroups for as many pairs as a mesh of this size commonly leaves (a few surfaces across every column, a few
        // columns per triangle); more pairs take more steps
        const uint64_t likely = (uint64_t)total_groups * 256u * 4u + 8ull * X.total_tris;
        // few pairs: shorter chunks, so that no wave takes several steps while others have none (64^3 with 5 k triangles
        // 22.6 -> 10.7 us, 128^3 with 20 k 30.8 -> 15.5; from 1024 chunks on the longer ones' one search for four steps pays)
        const uint32_t chunk = (uint32_t)std::min<uint64_t>(kPairChunk, std::max<uint64_t>(1, likely / (1024u * kVoxThreads)) * kVoxThreads);
        TimedLaunch tl("vox_pairs", L.s);
        k_vox_pairs<<<std::min(active_shape().pair_blocks, std::max(256u, ceil_div(likely, chunk))), kVoxThreads, 0, L.s>>>(
            L.jobs, X.setup, X.shell_off, X.total_tris, chunk);
        VF_CHECK_LAUNCH();
    }
    TimedLaunch tl("vox_fill", L.s);
    const uint32_t blocks = std::max(1u, std::min(total_groups, active_shape().cell_blocks));
    k_vox_fill<<<blocks, kVoxThreads, 0, L.s>>>(L, col_prefix, total_groups, tile_cnt);
    VF_CHECK_LAUNCH();
}

}  // namespace vf
