// Grid erosion: RegularGrid::erode (MF/Source/DataStructures/RegularGrid.cpp:82-159),
// erodeGrid-comp.glsl:26-59, copyGrid-comp.glsl, and the final
// removeIsolatedRegions (RegularGrid.cpp:1006-1015,
// removeIsolatedRegionsGrid-comp.glsl:16-38).
//
// One erosion iteration is detectBoundaries(1) (in place, launch_boundaries_tiled)
// followed by one stencil step that reads one state of the grid, as the
// reference's erode / copyGrid pair does.
// The step's noise gate is the reference's uniform float noise buffer as a
// counter-based draw per cell: (hash32(seed, cell) >> 8) / 2^24.
//
// Both stencils find the cells that become EMPTY first (a bit per cell) and empty them in the grid in a second
// pass over those bits: the grid is read and written where there is something, never copied.
#include "cellops.hpp"

#include <cmath>
#include <limits>
#include <vector>

namespace vf {

namespace {

// Pairs of cells in a 32-bit register.
typedef uint16_t cells2 __attribute__((ext_vector_type(2)));
__device__ inline cells2 as_cells(uint32_t w) { return __builtin_bit_cast(cells2, w); }

// Cells to empty, by bricks, bits of thread t's cells at kill[256 * brick + t].
// kErode (erodeGrid-comp.glsl): the shader's isBoundary is unmaskedBit(value, 15) != 0, which holds for every non-EMPTY
// cell, so every cell above FREE that passes the noise gate is tested.  Neighbours count when their raw value (boundary
// bit included) equals the cell's and the mask is set; the cell empties when count / (in-bounds window cells) <
// limit, all in FP32.
// Otherwise (removeIsolatedRegionsGrid-comp.glsl): a cell with fewer than 6 other cells of its raw value in the clamped
// 3x3x3 window empties.  The shader updates in place (thread-order dependent); this reads one state of the grid.
// A brick with cells to test is staged in LDS with its surroundings, 0 (which equals no tested cell) outside the grid;
// a thread compares its 8 cells with a row of the window at a time, two cells to an instruction.  SIDE 3 has the
// row's cells in registers; 0 is any side, read from LDS once for each step along the row.
// Bound by the latency of the staging loads and then LDS: a thread per cell that read its window from memory took
// 79 us a step (side 3) and 100 us (isolated cells) for a 189 x 211 x 175 grid, and 7 to copy the grid back; now 31 and
// 35, and 5 to empty the cells.
template <uint32_t SIDE, bool kErode>
__global__ __launch_bounds__(kCellThreads) void k_stencil(const JobDev* Jg, uint8_t* kill, const uint8_t* mask, uint32_t dyn_side,
                                                          float limit, float probability, uint64_t noise_seed)
{
    extern __shared__ uint32_t lds[];
    const uint32_t side = SIDE ? SIDE : dyn_side, h = side / 2, len = kBrickZ + 2 * h, ry = kBrickY + 2 * h;
    const JobDev& J = *Jg;
    const BrickAt b = brick_at(J, blockIdx.x);
    const CellGroup g = cell_group(J, b);
    uint8_t* bits = kill + (size_t)blockIdx.x * kCellThreads + threadIdx.x;
    const uint4 own = g.n ? load_group(J.labels, g) : make_uint4(0u, 0u, 0u, 0u);
    const uint32_t v2[4] = { own.x, own.y, own.z, own.w };
    uint32_t test = 0;
    if (own.x | own.y | own.z | own.w) {
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const uint32_t v = (v2[k >> 1] >> (16u * (k & 1u))) & 0xFFFFu;
            const bool yes = kErode ? v > kFree && (v & 0x7FFFu) != 0 &&
                                          (float)(hash32(noise_seed, (uint32_t)(g.c0 + k)) >> 8) * (1.0f / 16777216.0f) < probability
                                    : v != 0;
            test |= yes ? 1u << k : 0u;
        }
    }
    if (!__syncthreads_or((int)test)) {
        *bits = 0;
        return;
    }
    uint16_t* tile = reinterpret_cast<uint16_t*>(lds);
    uint32_t* rows = lds + (kBrickX + 2 * h) * ry * len / 2;  // the mask's rows as bits
    const uint32_t cells = (kBrickX + 2 * h) * ry * len;
    const int bx = (int)b.x - (int)h, by = (int)b.y - (int)h, bz = (int)b.z - (int)h;
#pragma unroll 7
    for (uint32_t i = threadIdx.x; i < cells; i += kCellThreads) {
        const uint32_t r = i / len, z = i - r * len, rx = r / ry;
        const int cx = bx + (int)rx, cy = by + (int)(r - rx * ry), cz = bz + (int)z;
        const bool in = (uint32_t)cx < J.nx && (uint32_t)cy < J.ny && (uint32_t)cz < J.nz;
        tile[i] = in ? J.labels[((uint64_t)(uint32_t)cx * J.ny + (uint32_t)cy) * J.nz + (uint32_t)cz] : (uint16_t)0;
    }
    uint32_t ones = side * side * side;
    if (kErode) {
        for (uint32_t r = threadIdx.x; r < side * side; r += kCellThreads) {
            uint32_t m = 0;
            for (uint32_t z = 0; z < side; ++z) m |= mask[r * side + z] ? 1u << z : 0u;
            rows[r] = m;
        }
    }
    __syncthreads();
    uint32_t emptied = 0;
    if (test) {
        if (kErode) ones = 0;
        const uint32_t row = threadIdx.x >> 2, tx = row / kBrickY, ty = row % kBrickY;
        cells2 off[4] = {};  // window cells that differ, of the four pairs
        const cells2 one = { 1, 1 };
        auto compare = [&](const uint32_t (&q)[4]) {
#pragma unroll
            for (uint32_t k = 0; k < 4u; ++k) off[k] += __builtin_elementwise_min(as_cells(q[k] ^ v2[k]), one);
        };
        for (uint32_t dx = 0; dx < side; ++dx)
            for (uint32_t dy = 0; dy < side; ++dy) {
                const uint32_t m = kErode ? (uint32_t)__builtin_amdgcn_readfirstlane((int)rows[dx * side + dy]) : 7u;
                if (kErode) ones += (uint32_t)__builtin_popcount(m);
                // the row of the window from the first cell's corner on; even cells begin a word
                const uint32_t* w = lds + (((tx + dx) * ry + ty + dy) * len + (threadIdx.x & 3u) * 8u) / 2u;
                if (SIDE == 3u) {
                    uint32_t q[5];
#pragma unroll
                    for (uint32_t k = 0; k < 5u; ++k) q[k] = w[k];
                    if (m & 1u) compare({ q[0], q[1], q[2], q[3] });
                    if (m & 2u)
                        compare({ __builtin_amdgcn_alignbit(q[1], q[0], 16), __builtin_amdgcn_alignbit(q[2], q[1], 16),
                                  __builtin_amdgcn_alignbit(q[3], q[2], 16), __builtin_amdgcn_alignbit(q[4], q[3], 16) });
                    if (m & 4u) compare({ q[1], q[2], q[3], q[4] });
                } else {
                    for (uint32_t dz = 0; dz < side; ++dz) {
                        if (!((m >> dz) & 1u)) continue;
                        const uint32_t* p = w + dz / 2u;
                        if (dz & 1u)
                            compare({ __builtin_amdgcn_alignbit(p[1], p[0], 16), __builtin_amdgcn_alignbit(p[2], p[1], 16),
                                      __builtin_amdgcn_alignbit(p[3], p[2], 16), __builtin_amdgcn_alignbit(p[4], p[3], 16) });
                        else
                            compare({ p[0], p[1], p[2], p[3] });
                    }
                }
            }
        auto span = [&](uint32_t c, uint32_t n) { return min(c + h, n - 1u) - (c > h ? c - h : 0u) + 1u; };
        const uint32_t xy = kErode ? span(b.x + tx, J.nx) * span(b.y + ty, J.ny) : 0u;
#pragma unroll
        for (uint32_t k = 0; k < 8u; ++k) {
            const uint32_t count = ones - (uint32_t)off[k >> 1][k & 1u];
            const bool gone = kErode ? (float)count / (float)(xy * span(g.z0 + k, J.nz)) < limit : count < 7u;
            emptied |= gone ? 1u << k : 0u;
        }
        emptied &= test;
    }
    *bits = (uint8_t)emptied;
}

__global__ __launch_bounds__(kCellThreads) void k_empty_cells(const JobDev* Jg, const uint8_t* kill)
{
    const uint32_t bits = kill[(size_t)blockIdx.x * kCellThreads + threadIdx.x];
    if (!bits) return;
    const CellGroup g = cell_group(*Jg, blockIdx.x);
    const uint4 q = load_group(Jg->labels, g);
    uint32_t w[4] = { q.x, q.y, q.z, q.w };
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k)
        if ((bits >> k) & 1u) w[k >> 1] &= k & 1u ? 0x0000FFFFu : 0xFFFF0000u;
    store_group(Jg->labels, g, make_uint4(w[0], w[1], w[2], w[3]));
}

// The same by a thread per cell in linear order that reads its window from memory: cell c's bit is bit c % 64 of word
// c / 64.  For grids where bricks do not pay (by_cells).
template <bool kErode>
__global__ __launch_bounds__(kCellThreads) void k_stencil_cells(const JobDev* Jg, unsigned long long* kill, const uint8_t* mask,
                                                                uint32_t side, float limit, float probability, uint64_t noise_seed)
{
    __shared__ uint8_t smask[kErode ? kMaxErosionSide * kMaxErosionSide * kMaxErosionSide : 1];
    if (kErode) {
        for (uint32_t i = threadIdx.x; i < side * side * side; i += kCellThreads) smask[i] = mask[i];
        __syncthreads();
    }
    const JobDev& J = *Jg;
    const auto* in = gcast<const uint16_t>(J.labels);
    const int nx = (int)J.nx, ny = (int)J.ny, nz = (int)J.nz, h = (int)side / 2;
    const uint64_t c = (uint64_t)blockIdx.x * kCellThreads + threadIdx.x;
    const uint32_t v = c < J.V ? in[c] : 0u;
    const bool test = kErode ? v > kFree && (v & 0x7FFFu) != 0 &&
                                   (float)(hash32(noise_seed, (uint32_t)c) >> 8) * (1.0f / 16777216.0f) < probability
                             : v != 0;
    bool gone = false;
    if (test) {
        uint32_t cx, cy, cz;
        decompose(c, &J, cx, cy, cz);
        const int x = (int)cx, y = (int)cy, z = (int)cz;
        const int x0 = max(x - h, 0), x1 = min(x + h, nx - 1), y0 = max(y - h, 0), y1 = min(y + h, ny - 1),
                  z0 = max(z - h, 0), z1 = min(z + h, nz - 1);
        uint32_t count = 0;
        for (int xx = x0; xx <= x1; ++xx)
            for (int yy = y0; yy <= y1; ++yy) {
                const auto* row = in + ((size_t)xx * ny + yy) * nz;
                const int m0 = kErode ? ((xx - x + h) * (int)side + (yy - y + h)) * (int)side - z + h : 0;
                for (int zz = z0; zz <= z1; ++zz) count += row[zz] == v && (!kErode || smask[m0 + zz]) ? 1u : 0u;
            }
        gone = kErode ? (float)count / (float)((x1 - x0 + 1) * (y1 - y0 + 1) * (z1 - z0 + 1)) < limit : count < 7u;
    }
    const uint64_t m = __ballot(gone);
    if ((threadIdx.x & 63u) == 0 && c < J.V) kill[c / 64u] = m;
}

__global__ __launch_bounds__(kCellThreads) void k_empty_linear(const JobDev* Jg, const uint8_t* kill)
{
    const uint64_t g = (uint64_t)blockIdx.x * kCellThreads + threadIdx.x;
    if (8u * g >= Jg->V) return;
    const uint32_t bits = kill[g];
    if (!bits) return;
    uint16_t v[8];
    load8(Jg->labels, 8u * g, Jg->V, v);
#pragma unroll
    for (uint32_t k = 0; k < 8u; ++k)
        if ((bits >> k) & 1u) v[k] = kEmpty;
    store8(Jg->labels, 8u * g, Jg->V, v);
}

// Thin grids, whose cells are less than a third of their bricks' (2048 x 2048 x 1, window 3: 824 us a step by bricks, 159 by
// cells; 600 x 600 x 9, where they are 0.28: 98 and 80; x 12, 0.38: 102 and 96; x 16, 0.5: 106 and 119), and grids of too
// few bricks for the chip, which a brick's steps one after another take longer: isolated cells 27.1 us by bricks and 21.5 by
// cells at 64^3 (128 bricks), 34.7 and 30.7 at 96^3 (432), 38.8 and 40.6 at 128^3 (1024; six jobs of 120^3 with 900 bricks
// each take 739 us by bricks, 756 by cells); window 3 17.2 and 15.2 at 64^3, 19.3 and 18.2 at 80^3 (300), 20.6 and 23.1 at
// 96^3; larger windows are even up to 50 bricks (40^3: 32 and 30 for 5, 221 and 191 for 15) and then better by bricks (64^3:
// 52 and 60 for 7).
bool by_cells(uint64_t V, uint32_t bricks, uint32_t side, bool erode)
{
    return V * 3u < (uint64_t)bricks * kTileCells || bricks < (!erode ? 640u : side <= 3u ? 320u : 64u);
}

template <uint32_t SIDE, bool kErode>
void launch_stencil(const Launch& L, uint64_t V, uint8_t* kill, const uint8_t* mask, uint32_t side, float limit, float probability,
                    uint64_t noise_seed)
{
    if (by_cells(V, L.total_bricks, side, kErode)) {
        k_stencil_cells<kErode><<<ceil_div(V, kCellThreads), kCellThreads, 0, L.s>>>(L.jobs, reinterpret_cast<unsigned long long*>(kill), mask, side,
                                                                                     limit, probability, noise_seed);
        VF_CHECK_LAUNCH();
        k_empty_linear<<<ceil_div(V, 8u * kCellThreads), kCellThreads, 0, L.s>>>(L.jobs, kill);
        VF_CHECK_LAUNCH();
        return;
    }
    const size_t wide = kBrickX + 2 * (side / 2), lds = wide * wide * (kBrickZ + 2 * (side / 2)) * 2 + side * side * 4;
    k_stencil<SIDE, kErode><<<L.total_bricks, kCellThreads, lds, L.s>>>(L.jobs, kill, mask, side, limit, probability, noise_seed);
    VF_CHECK_LAUNCH();
    k_empty_cells<<<L.total_bricks, kCellThreads, 0, L.s>>>(L.jobs, kill);
    VF_CHECK_LAUNCH();
}

}  // namespace

int erosion_mask(int type, uint32_t size, std::vector<uint8_t>& mask, float& activations)
{
    if (size % 2 == 0) ++size;
    const uint32_t n = size * size * size, c = size / 2;
    mask.assign(n, 0);
    float act = 0.0f;
    if (type == VF_EROSION_SQUARE) {
        std::fill(mask.begin(), mask.end(), 1);
        act = (float)n;
    } else if (type == VF_EROSION_CROSS) {
        for (uint32_t i = 0; i < size; ++i) {
            mask[i * size * size + c * size + c] = 1;
            mask[c * size * size + i * size + c] = 1;
            mask[c * size * size + c * size + i] = 1;
        }
        act = 1.0f / 3.0f * (float)n;  // as RegularGrid.cpp:104 sets it, not the cell count
    } else if (type == VF_EROSION_ELLIPSE) {
        for (uint32_t x = 0; x < size; ++x)
            for (uint32_t y = 0; y < size; ++y)
                for (uint32_t z = 0; z < size; ++z) {
                    const float dx = (float)x - (float)c, dy = (float)y - (float)c, dz = (float)z - (float)c;
                    if (std::sqrt(dx * dx + dy * dy + dz * dz) < (float)c + std::numeric_limits<float>::epsilon()) {
                        mask[x * size * size + y * size + z] = 1;
                        act += 1.0f;
                    }
                }
    } else {
        return -1;
    }
    activations = act / (float)n;
    return (int)size;
}

size_t erode_bytes(const uint32_t dims[3])
{
    return (size_t)brick_count(dims[0], dims[1], dims[2]) * kCellThreads;
}

void launch_erode_step(const Launch& L, uint64_t V, uint8_t* kill, const uint8_t* mask, uint32_t side, float limit,
                       float probability, uint64_t noise_seed)
{
    if (side > kMaxErosionSide || side % 2 == 0) fail(VF_ERR_INVALID_ARG, "erosion window side %u", side);
    TimedLaunch tl("erode_step", L.s);
    if (side == 3) launch_stencil<3, true>(L, V, kill, mask, side, limit, probability, noise_seed);
    else launch_stencil<0, true>(L, V, kill, mask, side, limit, probability, noise_seed);
}

void launch_isolated_cells(const Launch& L, uint64_t V, uint8_t* kill)
{
    TimedLaunch tl("isolated_cells", L.s);
    launch_stencil<3, false>(L, V, kill, nullptr, 3, 0.0f, 0.0f, 0);
}

}  // namespace vf
