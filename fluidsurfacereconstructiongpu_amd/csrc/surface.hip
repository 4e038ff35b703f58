// Surface-particle detection and band seeding.
//
//   k_cell_surface      extractionOfSurfaceParticles (ReconstructionCUDA.cu:70-120)
//                       and the surface half of extractionOfSurfaceAndInvolveParticles
//                       (ReconstructionCUDA.cu:466-551): an occupied cell that is
//                       not on the last layer of the grid and has an empty cell in
//                       its clamped 3^3 block is a surface cell.
//   k_involve_window    the involve half of the latter: every cell of the clamped
//                       5^3 block of a surface cell gets its particle count.
//   k_flags_from_cells  marks the particles of surface cells (the reference's
//                       per-cell loop over the cell's range, written per particle).
//   k_colorfield        extractionOfSurfaceParticlesUsingColorField
//                       (ReconstructionCUDA.cu:909-971): surface iff fewer than 25
//                       particles with |r|^2 > 0 in the clamped 3^3 cell block, or
//                       |sum m/rho_j gradW_spiky(r) r_hat| > 3.  With the radius-count
//                       surface mode (either method): surface iff fewer than 25
//                       particles at 0 < |r|^2 < h^2 (FP32 squared distances).
// Every surface particle then seeds the band: its scalar cell is set in a byte
// mask of "surface scalar cells" that band.hip dilates, or, when it lies outside
// the scalar grid, it is appended to an exception list that band.hip treats with
// the reference's per-particle box loop.  On a grid where the dilation is exact
// for no particle there is neither: band.hip walks the surface flags.
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace fsr {

namespace {

__device__ __forceinline__ int clampi(int v, int lo, int hi) {
    return v < lo ? lo : (v > hi ? hi : v);
}

// Truncating conversion of a cell coordinate that may lie outside the grid;
// NaN maps to 0 (what v_cvt_i32_f32 returns) and the value is clamped so the
// conversion stays defined.
__device__ __forceinline__ int trunc_cell(float q, int res) {
    if (!(q == q)) return 0;
    const float lo = -4.0f, hi = (float)res + 4.0f;
    q = q < lo ? lo : (q > hi ? hi : q);
    return (int)q;
}

// Surface cells, and the frame's surface particle count (the particles of those
// cells; st may be null): counted here, once per cell, because the per-particle
// pass would end in an atomic per workgroup on one address, and about a
// thousand of those took most of its time.
__global__ __launch_bounds__(256) void k_cell_surface(const float* __restrict__ occupancy,
                                                      const fsr_index_range* __restrict__ ranges,
                                                      GridDev sp, uint8_t* __restrict__ surf_cell,
                                                      fsr_frame_stats* __restrict__ st,
                                                      int all_exceptions) {
    __shared__ uint32_t part[4];
    const uint32_t C = sp.rx * sp.ry * sp.rz;
    uint32_t n_surf = 0;
    for (uint64_t c0 = (uint64_t)blockIdx.x * 256u; c0 < C; c0 += (uint64_t)gridDim.x * 256u) {
        const uint64_t cc = c0 + threadIdx.x;
        if (cc >= C) break;
        const uint32_t c = (uint32_t)cc;
        const uint32_t x = c % sp.rx, y = (c / sp.rx) % sp.ry, z = c / (sp.rx * sp.ry);
        uint8_t surf = 0;
        if (x < sp.rx - 1 && y < sp.ry - 1 && z < sp.rz - 1 && occupancy[c] >= 1.0f) {
            // the clamped 3^3 block as 27 clamped offsets (a clamped offset repeats
            // a cell of the block, which leaves the test unchanged), all read with
            // no early exit, so that their loads issue together
            const fsr_index_range own = ranges[c];
#pragma unroll
            for (int dz = -1; dz <= 1; ++dz) {
                const uint32_t zz = (uint32_t)clampi((int)z + dz, 0, sp.rz - 1);
#pragma unroll
                for (int dy = -1; dy <= 1; ++dy) {
                    const uint32_t yy = (uint32_t)clampi((int)y + dy, 0, sp.ry - 1);
#pragma unroll
                    for (int dx = -1; dx <= 1; ++dx) {
                        const uint32_t xx = (uint32_t)clampi((int)x + dx, 0, sp.rx - 1);
                        surf |= occupancy[(zz * sp.ry + yy) * sp.rx + xx] < 1.0f ? 1 : 0;
                    }
                }
            }
            if (surf) n_surf += own.end - own.start;
        }
        surf_cell[c] = surf;
    }
    if (!st) return;
    const uint32_t sum = wave_sum(n_surf);
    if (__lane_id() == 0) part[threadIdx.x >> 6] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        const uint32_t total = part[0] + part[1] + part[2] + part[3];
        if (total) {
            atomicAdd(&st->num_surface_particles, total);
            if (all_exceptions) atomicAdd(&st->band_exceptions, total);
        }
    }
}

// Involve counts (K4, the Yu13 half): an occupied cell within the clamped 5^3
// block of some surface cell gets its particle count, every other cell 0.  The
// block test is separable: a workgroup owns a tile of 28 x 4 x 4 cells and makes a
// 32-bit word of each row of the tile with its halo of 2 (cells outside the grid
// are 0, as the block is clamped to it); the words of the 5 x 5 rows around a row
// are ORed, and shifted copies of the sum ORed along x.  Every cell is written, so
// no clearing pass is needed.  (A launch for each axis took 3 x 4.6 us of a
// 1M-particle frame and 1.5 to 2 each of a 9,216-particle one; this one 5.6 and 4.2.)
constexpr int kInvX = 28, kInvY = 4, kInvZ = 4;
__global__ __launch_bounds__(256) void k_involve_window(const uint8_t* __restrict__ surf_cell,
                                                       GridDev sp,
                                                       const fsr_index_range* __restrict__ ranges,
                                                       uint32_t* __restrict__ involve) {
    constexpr int kHy = kInvY + 4, kRows = kHy * (kInvZ + 4);
    __shared__ uint32_t rows[kRows];
    __shared__ uint32_t any[kInvY * kInvZ];
    const uint32_t tx = (sp.rx + kInvX - 1) / kInvX, ty = (sp.ry + kInvY - 1) / kInvY,
                   tz = (sp.rz + kInvZ - 1) / kInvZ;
    const int64_t rx = sp.rx, ry = sp.ry, rz = sp.rz;
    const uint64_t tiles = (uint64_t)tx * ty * tz;
    for (uint64_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int64_t x0 = (int64_t)(tile % tx) * kInvX, y0 = (int64_t)(tile / tx % ty) * kInvY,
                      z0 = (int64_t)(tile / ((uint64_t)tx * ty)) * kInvZ;
        // 8 rows at a time, 32 lanes a row, and the ranges of the cells to write: all
        // loads of a thread together
        constexpr int kTurns = kRows / 8, kOut = 32 * kInvY * kInvZ / 256;
        uint8_t v[kTurns];
        fsr_index_range r[kOut];
        uint64_t cell[kOut];
        const int b = (int)(threadIdx.x & 31u), sub = (int)(threadIdx.x >> 5);
#pragma unroll
        for (int k = 0; k < kTurns; ++k) {
            const int row = 8 * k + sub;
            const int64_t x = x0 - 2 + b, y = y0 - 2 + row % kHy, z = z0 - 2 + row / kHy;
            const bool in = x >= 0 && x < rx && y >= 0 && y < ry && z >= 0 && z < rz;
            v[k] = in ? surf_cell[((uint32_t)z * sp.ry + (uint32_t)y) * sp.rx + (uint32_t)x] : 0;
        }
#pragma unroll
        for (int k = 0; k < kOut; ++k) {
            const int yz = 8 * k + sub;
            const int64_t x = x0 + b, y = y0 + yz % kInvY, z = z0 + yz / kInvY;
            const bool in = b < kInvX && x < rx && y < ry && z < rz;
            cell[k] = in ? ((uint32_t)z * sp.ry + (uint32_t)y) * sp.rx + (uint32_t)x : ~0ull;
            if (in) r[k] = ranges[cell[k]];
        }
#pragma unroll
        for (int k = 0; k < kTurns; ++k) {
            const uint64_t m = __ballot(v[k] != 0);
            if (b == 0) rows[8 * k + sub] = (uint32_t)(m >> (threadIdx.x & 32u));
        }
        __syncthreads();
        if (threadIdx.x < (uint32_t)(kInvY * kInvZ)) {
            const int y = (int)threadIdx.x % kInvY, z = (int)threadIdx.x / kInvY;
            uint32_t m = 0;
#pragma unroll
            for (int dz = 0; dz < 5; ++dz)
#pragma unroll
                for (int dy = 0; dy < 5; ++dy) m |= rows[(z + dz) * kHy + y + dy];
            any[threadIdx.x] = m | (m >> 1) | (m >> 2) | (m >> 3) | (m >> 4);
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kOut; ++k) {
            if (cell[k] == ~0ull) continue;
            const bool take = ((any[8 * k + sub] >> b) & 1u) && r[k].start != 0xFFFFFFFFu;
            involve[cell[k]] = take ? r[k].end - r[k].start : 0u;
        }
        __syncthreads();  // the next tile rewrites the rows
    }
}

// Band seeding of one particle: its scalar cell is set in the surface-cell
// byte mask, or the particle is appended to the exception list (exact path).
// When every surface particle takes the exact path that pass walks the surface
// flags, so no list is made (its counter was one address for every wave: the
// flag pass of a 1M-particle frame took 51.6 us with it, 17.1 us without).
// Called with all 64 lanes of the wave active (lanes without a particle pass
// surf = false); returns whether the particle became an exception.
__device__ __forceinline__ bool seed_particle(const SurfaceArgs& a, uint32_t i, float px,
                                              float py, float pz, bool surf) {
    if (a.all_exceptions) return surf;
    const float qx = cell_coord(px, a.sc.minx, a.sc.cell);
    const float qy = cell_coord(py, a.sc.miny, a.sc.cell);
    const float qz = cell_coord(pz, a.sc.minz, a.sc.cell);
    const bool in_grid = qx > -1.0f && qx < (float)a.sc.rx && qy > -1.0f &&
                         qy < (float)a.sc.ry && qz > -1.0f && qz < (float)a.sc.rz;
    const bool exc = surf && !in_grid;
    if (surf && !exc) {
        // one byte per scalar cell, rows padded to whole mask words: a plain
        // byte store (every writer stores 1), no read-modify-write
        const uint32_t ix = (uint32_t)(int)qx, iy = (uint32_t)(int)qy, iz = (uint32_t)(int)qz;
        const uint32_t wx = row_words(a.sc.rx);
        uint8_t* seeds = reinterpret_cast<uint8_t*>(a.sbits);
        seeds[(((uint64_t)iz * a.sc.ry + iy) * wx << 5) + ix] = 1u;
        // and in the map, the words that its x dilation [ix - 3, ix + 2] meets
        uint8_t* map = seeds + seed_map_offset(a.sc) + seed_map_index(a.sc, 0, iy, iz);
        const uint32_t w0 = (ix < 3u ? 0u : ix - 3u) >> 5, w1 = min((ix + 2u) >> 5, wx - 1u);
        map[w0] = 1u;
        if (w1 != w0) map[w1] = 1u;
    }
    const uint64_t m = __ballot(exc);
    if (m) {
        uint32_t base = 0;
        if (__lane_id() == (uint32_t)(__ffsll((unsigned long long)m) - 1))
            base = atomicAdd(&a.counters->num_exceptions, (uint32_t)__popcll(m));
        base = __shfl(base, __ffsll((unsigned long long)m) - 1, 64);
        if (exc) a.exceptions[base + mask_rank(m)] = i;
    }
    return exc;
}

// Elements per thread and grid-stride step of the per-particle kernels below:
// their loads are issued together, so one step waits for memory once per
// dependent load rather than once per element.
constexpr uint32_t kPerThread = 4;

// Surface flags from the surface hash cells (ZB05 occupancy method) and band
// seeding.  HBM-bound in the large: 4N read, 4N written, 16 bytes and a byte
// store per surface particle.
__global__ __launch_bounds__(256) void k_flags_from_cells(SurfaceArgs a,
                                                          const uint8_t* __restrict__ surf_cell) {
    const uint32_t C = a.sp.rx * a.sp.ry * a.sp.rz;
    const uint32_t span = blockDim.x * kPerThread;
    const bool seeds = a.sbits && !a.all_exceptions;
    uint32_t n_exc = 0;
    for (uint32_t base = blockIdx.x * span; base < a.n; base += gridDim.x * span) {
        uint32_t key[kPerThread];
#pragma unroll
        for (uint32_t k = 0; k < kPerThread; ++k) {
            const uint32_t i = base + k * blockDim.x + threadIdx.x;
            key[k] = i < a.n ? a.keys[i] : C;
        }
        bool surf[kPerThread];
#pragma unroll
        for (uint32_t k = 0; k < kPerThread; ++k) {
            const uint32_t i = base + k * blockDim.x + threadIdx.x;
            surf[k] = key[k] < C && surf_cell[key[k]] != 0;
            if (i < a.n) a.flags[i] = surf[k] ? 1u : 0u;
        }
        if (!seeds) continue;
        // positions only of the surface particles (the band seeds)
        float4 p[kPerThread];
#pragma unroll
        for (uint32_t k = 0; k < kPerThread; ++k) {
            const uint32_t i = base + k * blockDim.x + threadIdx.x;
            p[k] = surf[k] ? a.sorted[i] : make_float4(0.f, 0.f, 0.f, 0.f);
        }
#pragma unroll
        for (uint32_t k = 0; k < kPerThread; ++k) {
            const uint32_t i = base + k * blockDim.x + threadIdx.x;
            n_exc += seed_particle(a, i, p[k].x, p[k].y, p[k].z, surf[k]) ? 1u : 0u;
        }
    }
    // particles outside the scalar grid: few, if any
    if (seeds && a.st) wave_count_add(&a.st->band_exceptions, n_exc);
}

// Particles outside the hash grid (sorted last, in no cell): one thread each,
// over the clamped block around their own clamped cell.  Grid-stride over the
// device-side count; the surface / exception counts are added once per block.
__global__ __launch_bounds__(256) void k_colorfield_tail(SurfaceArgs a, float mass) {
    const uint32_t first = a.n - a.st->num_out_of_grid;
    const float h = a.h;
    const float inv_h = 1.0f / h;
    const float gcoef = -45.0f / (3.14159265358979f * (h * h) * (h * h));
    uint32_t n_surf = 0, n_exc = 0;
    // block-uniform trip count: seed_particle needs whole waves
    for (uint32_t base = first + blockIdx.x * blockDim.x; base < a.n;
         base += gridDim.x * blockDim.x) {
        const uint32_t i = base + threadIdx.x;
        bool surf = false;
        float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i < a.n) {
            p = a.sorted[i];
            const int cx = trunc_cell(cell_coord(p.x, a.sp.minx, a.sp.cell), a.sp.rx);
            const int cy = trunc_cell(cell_coord(p.y, a.sp.miny, a.sp.cell), a.sp.ry);
            const int cz = trunc_cell(cell_coord(p.z, a.sp.minz, a.sp.cell), a.sp.rz);
            const int x0 = clampi(cx - 1, 0, a.sp.rx - 1), x1 = clampi(cx + 1, 0, a.sp.rx - 1);
            const int y0 = clampi(cy - 1, 0, a.sp.ry - 1), y1 = clampi(cy + 1, 0, a.sp.ry - 1);
            const int z0 = clampi(cz - 1, 0, a.sp.rz - 1), z1 = clampi(cz + 1, 0, a.sp.rz - 1);
            uint32_t count = 0, count_r = 0;
            const float h2 = h * h;
            float gx = 0.f, gy = 0.f, gz = 0.f;
            for (int zz = z0; zz <= z1; ++zz)
                for (int yy = y0; yy <= y1; ++yy) {
                    const uint32_t row = ((uint32_t)zz * a.sp.ry + yy) * a.sp.rx;
                    uint32_t s = 0xFFFFFFFFu, e = 0;
                    for (int xx = x0; xx <= x1; ++xx) {
                        const fsr_index_range r = a.ranges[row + xx];
                        if (r.start != 0xFFFFFFFFu) {
                            if (s == 0xFFFFFFFFu) s = r.start;
                            e = r.end;
                        }
                    }
                    if (s == 0xFFFFFFFFu) continue;
                    for (uint32_t j = s; j < e; ++j) {
                        const float4 q = a.sorted[j];
                        const float rx = p.x - q.x, ry = p.y - q.y, rz = p.z - q.z;
                        const float d2 = __builtin_fmaf(rz, rz, __builtin_fmaf(ry, ry, rx * rx));
                        if (d2 > 0.0f) {
                            ++count;
                            if (d2 < h2) {
                                ++count_r;
                                const float ri = __builtin_amdgcn_rsqf(d2);
                                const float x = 1.0f - d2 * ri * inv_h;
                                const float c = mass / q.w * gcoef * x * x * ri;
                                gx = __builtin_fmaf(c, rx, gx);
                                gy = __builtin_fmaf(c, ry, gy);
                                gz = __builtin_fmaf(c, rz, gz);
                            }
                        }
                    }
                }
            const float g2 = __builtin_fmaf(gz, gz, __builtin_fmaf(gy, gy, gx * gx));
            surf = a.radius_count ? count_r < 25u : (count < 25u || __builtin_sqrtf(g2) > 3.0f);
            a.flags[i] = surf ? 1u : 0u;
        }
        const bool exc = a.sbits ? seed_particle(a, i, p.x, p.y, p.z, surf) : false;
        n_surf += surf ? 1u : 0u;
        n_exc += exc ? 1u : 0u;
    }
    block_count_add2(&a.st->num_surface_particles, n_surf, &a.st->band_exceptions, n_exc);
}

struct ColorChunks {
    const uint32_t* chunk_cell;
    const uint32_t* chunk_off;
    const uint32_t* num_chunks;
    uint32_t* next;  // per-XCD fetch counters
    uint32_t* work;  // per wave: candidates staged, kept by the box test, pairs within h
};

// The colour-field test of the particles of the hash cells, a wave per chunk of
// up to 64 particles of one cell, a lane per particle; each lane sums its
// candidates in their order (x-runs of the cell's 3^3 block), with the arithmetic
// of the kernel above.  Both take the reference's test |r| < h as |r|^2 < h^2 and
// the distance as |r|^2 rsqrt(|r|^2), one reciprocal square root per pair within
// h and no square root: the distance enters the gradient through (1 - |r|/h)^2,
// which vanishes where the two forms of the test could differ.
//
// VALU-bound: a candidate costs the wave some 20 operations, whichever lanes it
// is within h of (about one in five).  So
//   * the chunk's lanes form two groups, the halves of its box along x, each with a
//     queue of its own in LDS.  A candidate enters the queues of the groups whose
//     box it is within h * (1 + 5e-5) of, and a lane reads its group's: the wave
//     makes as many steps as the longer queue needs, four fifths of those for one
//     box around a full cell.  Along x, the order within a run, the queues fill
//     most evenly.  (Quarters, in x and y, need two thirds of the steps, but twice
//     the tests, and rings that fill less evenly: 441 us against 398 for the 1M
//     frame below);
//   * the count of neighbours (d^2 > 0), which decides for particles with fewer
//     than 25, is that of the block less those at distance 0, which lie in the
//     particle's own cell: it is not looked at when the other cells hold 25.  And
//     only queue parts that can hold own-cell candidates test for distance 0 (the
//     particle itself): particles of different cells differ in a coordinate (the
//     host checks that the square of the least difference does not underflow);
//   * four candidates are loaded together; in smaller frames (kSmall), where a SIMD
//     has few waves to change to, their terms are formed side by side with no
//     branch between them, a pair that is not within h weighing 0.
// Akinci12 frames, before (one group, counting every pair) and now: 1M-particle
// dam break 472 -> 383 us, 150k particles 179 -> 141, 16k 126 -> 66.
//
// A queue is a ring of kColorRing entries.  When a ring holds more than kColorRing
// - 64, steps are made for both groups at once, as many as the shorter queue holds,
// or as many more as the next staging round needs; a lane whose ring has fewer
// idles.  Heads stay multiples of 4 (the last step's 4 are padded with entries out
// of reach).
constexpr uint32_t kColorRing = 128;
constexpr uint32_t kOgt = 2, kOlt = 4;  // ordered > and <, as the compare builtin numbers them

template <bool kSmall, bool kRadius>
__global__ __launch_bounds__(256, kSmall ? 6 : 8) void k_colorfield(SurfaceArgs a, float mass,
                                                                    ColorChunks cl,
                                                                    int own_zero_only) {
    constexpr int G = 2;
    // a group's ring starts 4 banks after the one before
    __shared__ float4 queue[4][G][kColorRing + 1];
    __shared__ FetchState fetch;
    fetch_init(&fetch);
    const uint32_t lane = __lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t nch = *cl.num_chunks;
    if (kSmall) {
        // entries that no group's candidate was put in are multiplied by 0 there
        for (uint32_t t = lane; t < (uint32_t)G * (kColorRing + 1u); t += 64u)
            (&queue[wave][0][0])[t] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    const float h = a.h;
    const float inv_h = 1.0f / h;
    const float gcoef = -45.0f / (3.14159265358979f * (h * h) * (h * h));
    const float cull2 = (h * h) * 1.0001f;
    const float h2 = h * h;
    constexpr float kFar = 3.0e38f;  // a coordinate out of reach: its distance is infinite
    uint32_t n_surf = 0, n_exc = 0;
    // work of this wave: candidates staged, kept for a group, and pairs within h
    uint32_t n_staged = 0, n_kept = 0, n_inh = 0;
    ItemFetch<4, kSmall> items(cl.next, nch, &fetch);
    for (;;) {
        const uint32_t ch = items.next(wave);
        if (ch >= nch) break;
        const uint32_t c = cl.chunk_cell[ch];
        const uint32_t k = ch - cl.chunk_off[c];
        const fsr_index_range own = a.ranges[c];
        const uint32_t i = own.start + 64u * k + lane;
        const bool live = i < own.end;
        const int cx = (int)(c % a.sp.rx), cy = (int)((c / a.sp.rx) % a.sp.ry);
        const int cz = (int)(c / (a.sp.rx * a.sp.ry));
        const int x0 = clampi(cx - 1, 0, a.sp.rx - 1), x1 = clampi(cx + 1, 0, a.sp.rx - 1);
        const int y0 = clampi(cy - 1, 0, a.sp.ry - 1), y1 = clampi(cy + 1, 0, a.sp.ry - 1);
        const int z0 = clampi(cz - 1, 0, a.sp.rz - 1), z1 = clampi(cz + 1, 0, a.sp.rz - 1);
        const int ny = y1 - y0 + 1;
        const int nrows = ny * (z1 - z0 + 1);
        uint32_t len = 0, rs = 0;
        if ((int)lane < nrows) {
            const int yy = y0 + (int)lane % ny, zz = z0 + (int)lane / ny;
            const uint32_t rowc = ((uint32_t)zz * a.sp.ry + yy) * a.sp.rx;
            // the row's 3 cells as clamped offsets (a repeated edge cell leaves
            // the run unchanged), loaded together
            fsr_index_range rg[3];
#pragma unroll
            for (int d = 0; d < 3; ++d) rg[d] = a.ranges[rowc + clampi(cx - 1 + d, x0, x1)];
            uint32_t s0 = 0xFFFFFFFFu, e0 = 0;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                if (rg[d].start != 0xFFFFFFFFu) {
                    if (s0 == 0xFFFFFFFFu) s0 = rg[d].start;
                    e0 = rg[d].end;
                }
            }
            if (s0 != 0xFFFFFFFFu) { rs = s0; len = e0 - s0; }
        }
        // lane j < nrows holds row j's first candidate index (rp) and the
        // offset from candidate index to sorted index in that row (ro)
        const uint32_t incl = wave_inclusive_sum(len);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        const uint32_t rp = incl - len;
        const uint32_t ro = rs - rp;
        // Row of candidate index gg of the staging round that starts at nb:
        // jc, a row whose first index is at most nb, only grows; the rows
        // that start inside the round are visited with wave-uniform reads, and
        // a lane takes the last one that starts at or before gg (an empty row
        // shares its first index with the next row, visited after it).
        uint32_t jc = 0;
        auto row_offset = [&](uint32_t nb, uint32_t gg) {
            uint32_t off = (uint32_t)__builtin_amdgcn_readlane((int)ro, (int)jc);
            for (uint32_t jj = jc + 1u; jj < (uint32_t)nrows; ++jj) {
                const uint32_t pj = (uint32_t)__builtin_amdgcn_readlane((int)rp, (int)jj);
                if (pj >= nb + 64u) break;
                if (gg >= pj) off = (uint32_t)__builtin_amdgcn_readlane((int)ro, (int)jj);
                jc = jj;
            }
            return off;
        };
        // the candidate indices of the own cell's particles
        const uint32_t oj = (uint32_t)((cz - z0) * ny + (cy - y0));
        const uint32_t own_first = own.start - (uint32_t)__builtin_amdgcn_readlane((int)ro, (int)oj);
        const uint32_t own_n = own.end - own.start;
        const bool need_count = kRadius || !own_zero_only || total - own_n < 25u;

        float4 p = make_float4(-kFar, -kFar, -kFar, 0.f);
        if (live) p = a.sorted[i];
        float bx0, bx1;
        wave_range(live, p.x, &bx0, &bx1);
        const uint32_t grp = p.x > 0.5f * (bx0 + bx1) ? 1u : 0u;
        // the groups' boxes; an empty one is out of reach
        float lo[G][3], hi[G][3];
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const bool in = live && grp == (uint32_t)g;
            wave_range(in, p.x, &lo[g][0], &hi[g][0]);
            wave_range(in, p.y, &lo[g][1], &hi[g][1]);
            wave_range(in, p.z, &lo[g][2], &hi[g][2]);
            if (!__ballot(in)) lo[g][0] = hi[g][0] = kFar;
        }
        // rings: entries [head, head + fill) of each wait for evaluation
        uint32_t head[G], fill[G], done[G], put[G], mark[G];
#pragma unroll
        for (int g = 0; g < G; ++g) head[g] = fill[g] = done[g] = put[g] = mark[g] = 0;
        uint32_t zeros = 0, count_r = 0;
        float gx = 0.f, gy = 0.f, gz = 0.f;
        const char* ring = reinterpret_cast<const char*>(&queue[wave][grp][0]);
        auto by_group = [&](const uint32_t (&v)[G]) { return grp ? v[1] : v[0]; };
        // the next mine candidates of the lane's ring (a multiple of 4, at most n)
        auto steps = [&](auto zt, uint32_t n, uint32_t mine, uint32_t at) {
            constexpr bool kZero = decltype(zt)::value;
            for (uint32_t t = 0; t < n; t += 4u) {
                const uint64_t act = __ballot(t < mine);
                const float4* e =
                    reinterpret_cast<const float4*>(ring + ((16u * (at + t)) & (16u * kColorRing - 1u)));
                float rx[4], ry[4], rz[4], d2[4];
                float4 qq[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) qq[u] = e[u];
                // whole entries, all four before the first is used
                asm volatile("" : "+v"(qq[0].w), "+v"(qq[1].w), "+v"(qq[2].w), "+v"(qq[3].w));
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    rx[u] = p.x - qq[u].x;
                    ry[u] = p.y - qq[u].y;
                    rz[u] = p.z - qq[u].z;
                    d2[u] = __builtin_fmaf(rz[u], rz[u], __builtin_fmaf(ry[u], ry[u], rx[u] * rx[u]));
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    // lane masks straight from the compares (a ballot of the
                    // conditions took two more operations per candidate)
                    uint64_t in = act & __builtin_amdgcn_fcmpf(d2[u], h2, kOlt);
                    if (kZero) {
                        const uint64_t apart = __builtin_amdgcn_fcmpf(d2[u], 0.0f, kOgt);
                        in &= apart;
                        zeros += __builtin_amdgcn_inverse_ballot_w64(act & ~apart) ? 1u : 0u;
                    }
                    n_inh += (uint32_t)__popcll(in);
                    const bool take = __builtin_amdgcn_inverse_ballot_w64(in);
                    if (kRadius) count_r += take ? 1u : 0u;
                    if (kSmall || take) {
                        const float ri = __builtin_amdgcn_rsqf(d2[u]);
                        const float x = 1.0f - d2[u] * ri * inv_h;
                        float cc = qq[u].w * x * x * ri;
                        if (kSmall) cc = take ? cc : 0.0f;
                        gx = __builtin_fmaf(cc, rx[u], gx);
                        gy = __builtin_fmaf(cc, ry[u], gy);
                        gz = __builtin_fmaf(cc, rz[u], gz);
                    }
                }
            }
        };
        auto run = [&](uint32_t n) {
            uint32_t take[G];
            bool zero = need_count;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                take[g] = min(n, fill[g] & ~3u);
                zero |= done[g] < mark[g];
            }
            const uint32_t mine = by_group(take), at = by_group(head);
            wave_lds_sync();
            if (zero) steps(std::true_type{}, n, mine, at);
            else steps(std::false_type{}, n, mine, at);
            wave_lds_sync();
#pragma unroll
            for (int g = 0; g < G; ++g) {
                fill[g] -= take[g];
                done[g] += take[g];
                head[g] = (head[g] + take[g]) & (kColorRing - 1u);
            }
        };
        // each lane's candidate is loaded one staging round ahead
        float4 next = make_float4(0.f, 0.f, 0.f, 0.f);
        {
            const uint32_t off = row_offset(0u, lane);
            if (lane < total) next = a.sorted[off + lane];
        }
        for (uint32_t base = 0; base < total; base += 64u) {
            const uint32_t g0 = base + lane;
            const float4 cand = next;
            if (base + 64u < total) {
                const uint32_t off = row_offset(base + 64u, g0 + 64u);
                if (g0 + 64u < total) next = a.sorted[off + g0 + 64u];
            }
            // (m / rho_j) * gcoef, in the per-thread kernel's operation order
            const float4 st = make_float4(cand.x, cand.y, cand.z, mass / cand.w * gcoef);
            const bool has_own = base < own_first + own_n && base + 64u > own_first;
            uint32_t most = 0, least = kColorRing;
            uint64_t any = 0;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                // c - clamp(c, lo, hi): its square equals that of max(lo - c, c - hi, 0)
                const float dx = cand.x - __builtin_amdgcn_fmed3f(cand.x, lo[g][0], hi[g][0]);
                const float dy = cand.y - __builtin_amdgcn_fmed3f(cand.y, lo[g][1], hi[g][1]);
                const float dz = cand.z - __builtin_amdgcn_fmed3f(cand.z, lo[g][2], hi[g][2]);
                const bool keep =
                    g0 < total && __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx)) < cull2;
                const uint64_t m = __ballot(keep);
                if (keep) queue[wave][g][(head[g] + fill[g] + mask_rank(m)) & (kColorRing - 1u)] = st;
                const uint32_t added = (uint32_t)__popcll(m);
                any |= m;
                fill[g] += added;
                put[g] += added;
                if (has_own) mark[g] = put[g];
                most = max(most, fill[g]);
                least = min(least, fill[g]);
            }
            n_kept += (uint32_t)__popcll(any);
            if (most > kColorRing - 64u)
                run(max(least & ~3u, (most - (kColorRing - 64u) + 3u) & ~3u));
        }
        // the rest, each ring padded to a multiple of 4 with entries out of reach
        uint32_t most = 0;
#pragma unroll
        for (int g = 0; g < G; ++g) {
            const uint32_t n = (fill[g] + 3u) & ~3u;
            if (lane < n - fill[g])
                queue[wave][g][(head[g] + fill[g] + lane) & (kColorRing - 1u)] =
                    make_float4(kFar, kFar, kFar, 0.f);
            fill[g] = n;
            most = max(most, n);
        }
        if (most) run(most);
        n_staged += total;
        bool surf = false;
        if (live) {
            const float g2 = __builtin_fmaf(gz, gz, __builtin_fmaf(gy, gy, gx * gx));
            // candidates that the lane did not see lie beyond h: they count as
            // neighbours, and never in count_r
            surf = kRadius ? count_r < 25u
                           : ((need_count && total - zeros < 25u) || __builtin_sqrtf(g2) > 3.0f);
            a.flags[i] = surf ? 1u : 0u;
        }
        bool exc = false;
        if (a.sbits) exc = seed_particle(a, i, p.x, p.y, p.z, surf);
        n_surf += surf ? 1u : 0u;
        n_exc += exc ? 1u : 0u;
    }
    if (lane == 0) {
        uint32_t* w = cl.work + 3u * (blockIdx.x * (blockDim.x >> 6) + wave);
        w[0] = n_staged;
        w[1] = n_kept;
        w[2] = n_inh;
    }
    block_count_add2(&a.st->num_surface_particles, n_surf, &a.st->band_exceptions, n_exc);
}

// band seeding from given flags (stage entry point of the band)
__global__ __launch_bounds__(256) void k_seed_flags(SurfaceArgs a) {
    const uint32_t span = blockDim.x * kPerThread;
    uint32_t n_surf = 0, n_exc = 0;
    for (uint32_t base = blockIdx.x * span; base < a.n; base += gridDim.x * span) {
        bool surf[kPerThread];
        float4 p[kPerThread];
#pragma unroll
        for (uint32_t k = 0; k < kPerThread; ++k) {
            const uint32_t i = base + k * blockDim.x + threadIdx.x;
            surf[k] = false;
            p[k] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (i < a.n) {
                surf[k] = a.flags[i] != 0;
                p[k] = a.sorted[i];
            }
        }
#pragma unroll
        for (uint32_t k = 0; k < kPerThread; ++k) {
            const uint32_t i = base + k * blockDim.x + threadIdx.x;
            const bool exc = a.sbits ? seed_particle(a, i, p[k].x, p[k].y, p[k].z, surf[k]) : false;
            n_surf += surf[k] ? 1u : 0u;
            n_exc += exc ? 1u : 0u;
        }
    }
    if (a.st) block_count_add2(&a.st->num_surface_particles, n_surf, &a.st->band_exceptions, n_exc);
}

}  // namespace

// Grid of the per-particle kernels that end in block counter atomics.
static uint32_t count_blocks(fsr_context* ctx, uint32_t n) {
    const uint32_t cap = (uint32_t)persistent_blocks(ctx, 256, 4, TUNE_BAND);
    return std::max(1u, std::min((n + 256u * kPerThread - 1u) / (256u * kPerThread), cap));
}

fsr_status surface_seed_from_flags(fsr_context* ctx, const SurfaceArgs& a, hipStream_t s) {
    if (a.n) {
        hipLaunchKernelGGL(k_seed_flags, dim3(count_blocks(ctx, a.n)), dim3(256), 0, s, a);
        FSR_LAUNCH_CHECK("k_seed_flags");
    }
    return FSR_OK;
}

fsr_status surface_occupancy(fsr_context* ctx, const SurfaceArgs& a, uint8_t* surf_cell,
                             uint32_t* involve, hipStream_t s) {
    const uint32_t C = a.sp.rx * a.sp.ry * a.sp.rz;
    hipLaunchKernelGGL(k_cell_surface, dim3(std::min((C + 255) / 256, 1024u)), dim3(256), 0, s,
                       a.occupancy, a.ranges, a.sp, surf_cell, a.st, a.all_exceptions);
    FSR_LAUNCH_CHECK("k_cell_surface");
    if (involve) {
        const uint64_t tiles = (uint64_t)((a.sp.rx + kInvX - 1) / kInvX) *
                               ((a.sp.ry + kInvY - 1) / kInvY) * ((a.sp.rz + kInvZ - 1) / kInvZ);
        hipLaunchKernelGGL(k_involve_window, dim3((uint32_t)std::min<uint64_t>(tiles, 65536)),
                           dim3(256), 0, s, (const uint8_t*)surf_cell, a.sp, a.ranges, involve);
        FSR_LAUNCH_CHECK("k_involve_window");
    }
    if (a.n) {
        hipLaunchKernelGGL(k_flags_from_cells, dim3(count_blocks(ctx, a.n)), dim3(256), 0, s, a,
                           (const uint8_t*)surf_cell);
        FSR_LAUNCH_CHECK("k_flags_from_cells");
    }
    return FSR_OK;
}

fsr_status surface_colorfield(fsr_context* ctx, const SurfaceArgs& a, float mass,
                              hipStream_t s) {
    if (!a.n) return FSR_OK;
    const uint32_t C = a.sp.rx * a.sp.ry * a.sp.rz;
    const uint64_t max_chunks = (uint64_t)a.n / 64 + C + 1;
    uint32_t* scratch;
    FSR_TRY(arena_typed(ctx, A_SURF_CHUNKS, C + max_chunks, &scratch));
    uint32_t* total = &a.counters->aux[4];
    FSR_TRY(cell_chunk_list(ctx, a.ranges, nullptr, C, scratch, scratch + C, max_chunks, total, s));
    const int blocks = persistent_blocks(ctx, 256, 8, TUNE_FIELD);
    uint32_t* work;
    FSR_TRY(arena_typed(ctx, A_COLOR_WORK, 3ull * blocks * 4, &work));
    ColorChunks cl{scratch + C, scratch, total, a.counters->xcd_next, work};
    // n / 64 chunks and up to as many remainders: a list that may be shorter than
    // the waves is dealt out (see ItemFetch)
    const bool small = a.n / 64u <= 4u * (uint32_t)(blocks / ctx->in_flight);
    auto kernel = a.radius_count ? (small ? k_colorfield<true, true> : k_colorfield<false, true>)
                                 : (small ? k_colorfield<true, false> : k_colorfield<false, false>);
    // Two floats x whose x - min round to either side of a cell boundary B >= cell
    // have |x| >= ulp(B) / 4 (min is a float), so they are at least cell * 2^-49
    // apart; the square of that must not underflow.
    const int own_zero_only = a.sp.cell > 1.0e-5f ? 1 : 0;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, s, a, mass, cl, own_zero_only);
    FSR_LAUNCH_CHECK("k_colorfield");
    // particles outside the grid (a device-side count)
    hipLaunchKernelGGL(k_colorfield_tail, dim3(64), dim3(256), 0, s, a, mass);
    FSR_LAUNCH_CHECK("k_colorfield_tail");
    return FSR_OK;
}

}  // namespace fsr
