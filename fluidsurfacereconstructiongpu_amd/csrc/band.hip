// Surface band of scalar vertices, its compaction, and the cell-major work
// list of the field kernels.
//
// The reference (estimationOfSurfaceVertices, ReconstructionCUDA.cu:554-595)
// loops, for every surface particle in scalar cell (i, j, k), over the vertices
//   x in [clamp(i-3), clamp(i+3))   (upper bound exclusive)
//   y in [clamp(j-3), clamp(j+3)],  z in [clamp(k-3), clamp(k+3)]
// (clamp to [0, res-1]) and marks those with FP32 |v - p| < 1.5 h (compared in
// double) in a dense u32[V] grid, which is then scanned (thrust) and compacted
// (compactSurfaceVertex, ReconstructionCUDA.cu:293-304).
//
// Here the band is a bit mask (V/8 bytes instead of 4V).  When every vertex of
// such a box lies within 1.5 h of any point of the particle's scalar cell
// (4*sqrt(3) scalar cells < 1.5 h, checked on the host with a rounding margin),
// the distance test never rejects and the band of in-grid particles is exactly
// the dilation of the set S of their scalar cells by the box
//   x - s_x in [-3, 2] (and x <= resx-2),  |y - s_y| <= 3,  |z - s_z| <= 3,
// done as three separable passes over the mask.  Particles outside the scalar
// grid, and every particle when the condition fails, go through the exact
// per-particle loop of the reference (k_band_exceptions).
//
// Compaction: set bits counted per 256 words -> each block of 256 words offsets
// and scans its words' counts -> 16 lanes a word write its set bits in ascending
// order (the reference's surfaceVerticesIndexArray; see band_emit).
//
// Cell-major work list: the field kernels process the band grouped by the hash cell
// each vertex falls in (getIndex3D of the vertex position, exactly as the
// reference's field kernels compute it), so that all 64 lanes of a wave share
// one neighbour-cell block.  Cells outside the hash grid are folded into a ring
// of `radius` virtual cells on each side (their clamped neighbour blocks
// coincide).  The list holds 64-vertex chunks, not vertices: a chunk's are read
// from the mask (chunk_vertex).  The order of vertices inside a cell does not
// affect any value: every vertex sums its candidates in the cell's fixed order.
#include <algorithm>
#include <cmath>
#include <limits>

#include "common.hpp"

namespace fsr {

namespace {

// Bits of four 0/1 bytes (byte k -> bit k).
__device__ __forceinline__ uint32_t pack4(uint32_t x) {
    return (x & 1u) | ((x >> 7) & 2u) | ((x >> 14) & 4u) | ((x >> 21) & 8u);
}

// The x pass reads the seed mask as bytes (one per scalar cell, rows padded to
// whole words: word w covers bytes 32w .. 32w + 31) and writes bits.
__global__ __launch_bounds__(256) void k_dilate_x(const uint8_t* __restrict__ in,
                                                  uint32_t* __restrict__ out, uint32_t wx,
                                                  uint64_t nwords, uint32_t rx) {
    const uint64_t w = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= nwords) return;
    const uint32_t xw = (uint32_t)(w % wx);
    const uint4* chunk = reinterpret_cast<const uint4*>(in + (w << 5));
    const uint4 lo = chunk[0], hi = chunk[1];
    const uint32_t cur = pack4(lo.x) | (pack4(lo.y) << 4) | (pack4(lo.z) << 8) |
                         (pack4(lo.w) << 12) | (pack4(hi.x) << 16) | (pack4(hi.y) << 20) |
                         (pack4(hi.z) << 24) | (pack4(hi.w) << 28);
    // the two top bits of the previous word and the three low bits of the next
    const uint32_t prev =
        xw > 0 ? pack4(reinterpret_cast<const uint32_t*>(in + (w << 5))[-1]) << 28 : 0u;
    const uint32_t next = xw + 1 < wx ? pack4(reinterpret_cast<const uint32_t*>(in + (w << 5))[8]) : 0u;
    uint32_t o = cur;
    o |= (cur >> 1) | (next << 31);
    o |= (cur >> 2) | (next << 30);
    o |= (cur >> 3) | (next << 29);
    o |= (cur << 1) | (prev >> 31);
    o |= (cur << 2) | (prev >> 30);
    // the reference's exclusive x bound after clamping: x <= rx - 2
    const uint32_t lim = rx >= 1 ? rx - 1 : 0;
    const uint32_t x0 = xw * 32u;
    if (x0 >= lim) o = 0;
    else if (lim - x0 < 32u) o &= (1u << (lim - x0)) - 1u;
    out[w] = o;
}

// out(w, row) = OR of in over rows row + d*stride, |d| <= 3, inside [0, extent)
__global__ __launch_bounds__(256) void k_dilate_rows(const uint32_t* __restrict__ in,
                                                     uint32_t* __restrict__ out,
                                                     uint64_t nwords, uint64_t stride,
                                                     uint32_t extent, uint64_t period) {
    const uint64_t w = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w >= nwords) return;
    const uint32_t c = (uint32_t)((w / stride) % period);
    uint32_t o = 0;
#pragma unroll
    for (int d = -3; d <= 3; ++d) {
        const int cc = (int)c + d;
        if (cc >= 0 && cc < (int)extent) o |= in[(uint64_t)((int64_t)w + (int64_t)d * (int64_t)stride)];
    }
    out[w] = o;
}

// x dilation of one band-mask word from the byte seed mask (the body of
// k_dilate_x): w = word index in the row, rowbase = first byte of the row.
__device__ __forceinline__ uint32_t dilate_x_word(const uint8_t* __restrict__ in, uint64_t rowbase,
                                                  uint32_t xw, uint32_t wx, uint32_t rx) {
    const uint8_t* src = in + rowbase + ((uint64_t)xw << 5);
    const uint4* chunk = reinterpret_cast<const uint4*>(src);
    const uint4 lo = chunk[0], hi = chunk[1];
    const uint32_t cur = pack4(lo.x) | (pack4(lo.y) << 4) | (pack4(lo.z) << 8) |
                         (pack4(lo.w) << 12) | (pack4(hi.x) << 16) | (pack4(hi.y) << 20) |
                         (pack4(hi.z) << 24) | (pack4(hi.w) << 28);
    const uint32_t prev = xw > 0 ? pack4(reinterpret_cast<const uint32_t*>(src)[-1]) << 28 : 0u;
    const uint32_t next = xw + 1 < wx ? pack4(reinterpret_cast<const uint32_t*>(src)[8]) : 0u;
    uint32_t o = cur;
    o |= (cur >> 1) | (next << 31);
    o |= (cur >> 2) | (next << 30);
    o |= (cur >> 3) | (next << 29);
    o |= (cur << 1) | (prev >> 31);
    o |= (cur << 2) | (prev >> 30);
    const uint32_t lim = rx >= 1 ? rx - 1 : 0;
    const uint32_t x0 = xw * 32u;
    if (x0 >= lim) o = 0;
    else if (lim - x0 < 32u) o &= (1u << (lim - x0)) - 1u;
    return o;
}

// The three dilation passes in one launch: a workgroup owns a tile of kTW
// words x kTYZ rows x kTYZ layers of the output; it x-dilates the tile's input
// with a halo of 3 rows and 3 layers on each side into LDS (from the byte
// mask), ORs the 7 rows (y), then the 7 layers (z), and writes the tile.
// Rows and layers outside the grid contribute nothing, as in the separate
// passes.  The forms, by the number of 8-word x 16 x 16 tiles:
//   * at least one per CU: that tile, 1024 threads, kMap.  Reading the seeds
//     bounds it (the halo nearly doubles their V bytes), and most of a grid has
//     no seed near: only words that the seeds' map marks are read, and a tile
//     without one is just cleared.  27 -> 14 us at 320^3, 42 -> 19 at 384^3, 9.2
//     -> 8.3 at 256^3 (dam breaks).
//   * fewer: the same tile without the map, whose load would be one more in the
//     chain that a tile takes: at 192^3 7.8 us, 8.7 with the map.
//   * fewer than half a tile per CU: 4 words x 8 x 8, 512 threads, which leaves
//     fewer CUs idle and takes 2 rounds of loads for 4: 7.9 -> 4.4 us at 128^3,
//     7.5 -> 6.1 at 161^3 (at 192^3 9.2, hence the line).
constexpr int kH = 3;
template <int kTW, int kTYZ, int kThreads, bool kMap>
__global__ __launch_bounds__(kThreads) void k_dilate_box(const uint8_t* __restrict__ in,
                                                         uint32_t* __restrict__ out, uint32_t wx,
                                                         GridDev sc) {
    constexpr int kIn = kTYZ + 2 * kH;
    __shared__ uint32_t xs[kIn][kIn][kTW];
    __shared__ uint32_t ys[kIn][kTYZ][kTW];
    const uint32_t w0 = blockIdx.x * kTW;
    const int y0 = (int)(blockIdx.y * kTYZ), z0 = (int)(blockIdx.z * kTYZ);
    constexpr int nxs = kIn * kIn * kTW;
    constexpr int kRounds = (nxs + kThreads - 1) / kThreads;
    const uint8_t* map = in + seed_map_offset(sc);
    // the map entries of the thread's words, loaded together
    bool seeded[kRounds];
#pragma unroll
    for (int k = 0; k < kRounds; ++k) {
        const int t = (int)threadIdx.x + k * kThreads;
        const int w = t % kTW, r = t / kTW;
        const int yy = y0 - kH + r % kIn, zz = z0 - kH + r / kIn;
        seeded[k] = t < nxs && w0 + w < wx && yy >= 0 && yy < (int)sc.ry && zz >= 0 &&
                    zz < (int)sc.rz &&
                    (!kMap || map[seed_map_index(sc, w0 + w, yy, zz)] != 0);
    }
    bool any = false;
#pragma unroll
    for (int k = 0; k < kRounds; ++k) {
        const int t = (int)threadIdx.x + k * kThreads;
        const int w = t % kTW, r = t / kTW;
        const int yy = y0 - kH + r % kIn, zz = z0 - kH + r / kIn;
        uint32_t v = 0;
        if (seeded[k])
            v = dilate_x_word(in, (((uint64_t)zz * sc.ry + yy) * wx) << 5, w0 + w, wx, sc.rx);
        if (t < nxs) xs[r / kIn][r % kIn][w] = v;
        any |= seeded[k];
    }
    constexpr int nout = kTYZ * kTYZ * kTW;
    if (kMap) {
        if (!__syncthreads_or(any)) {
            // no seed near the tile
            for (int t = threadIdx.x; t < nout; t += kThreads) {
                const int w = t % kTW, yy = y0 + (t / kTW) % kTYZ, zz = z0 + t / (kTW * kTYZ);
                if (w0 + w < wx && yy < (int)sc.ry && zz < (int)sc.rz)
                    out[((uint64_t)zz * sc.ry + yy) * wx + w0 + w] = 0u;
            }
            return;
        }
    } else {
        __syncthreads();
    }
    constexpr int nys = kIn * kTYZ * kTW;
    for (int t = threadIdx.x; t < nys; t += kThreads) {
        const int w = t % kTW, y = (t / kTW) % kTYZ, zr = t / (kTW * kTYZ);
        uint32_t v = 0;
#pragma unroll
        for (int d = 0; d <= 2 * kH; ++d) v |= xs[zr][y + d][w];
        ys[zr][y][w] = v;
    }
    __syncthreads();
    for (int t = threadIdx.x; t < nout; t += kThreads) {
        const int w = t % kTW, y = (t / kTW) % kTYZ, z = t / (kTW * kTYZ);
        const int yy = y0 + y, zz = z0 + z;
        if (w0 + w >= wx || yy >= (int)sc.ry || zz >= (int)sc.rz) continue;
        uint32_t v = 0;
#pragma unroll
        for (int d = 0; d <= 2 * kH; ++d) v |= ys[z + d][y][w];
        out[((uint64_t)zz * sc.ry + yy) * wx + w0 + w] = v;
    }
}

__device__ __forceinline__ int clampi(int v, int lo, int hi) {
    return v < lo ? lo : (v > hi ? hi : v);
}

__device__ __forceinline__ int trunc_clamped(float q, int res) {
    if (!(q == q)) return 0;
    const float lo = -4.0f, hi = (float)res + 4.0f;
    q = q < lo ? lo : (q > hi ? hi : q);
    return (int)q;
}

// The reference's per-particle band loop (the exact path), for the exception
// list or, when every surface particle takes it, for the surface flags in
// particle order.  A wave takes `group` consecutive list entries (particles),
// one per lane for the box and its cell, and compacts the live ones into LDS;
// then it treats 8 particles at a time, 8 lanes each: lane k of a particle's 8
// walks layer z0 + k of its box (at most 7 layers of 7 rows of 6 vertices).
// `group` shrinks with the particle count (32 down to 8), so that a small
// frame still has a wave for every 8 particles.  One particle per lane, its 294
// tests in a row, took 28.9 us for a 960-particle block and 128.9 us for
// 1,000,000 dam-break particles on the half-hash-cell grid; this form takes 6.3
// and 41.2 us (groups of 16 and 64: 50 and 52 us).
//
// The reference tests the FP32 distance sqrt(d2) < 1.5 h.  The square root is
// monotonic and correctly rounded, so this is d2 < a.d2_limit exactly, the
// smallest float whose root fails (found on the host).  d2 = fma(dz, dz,
// fma(dy, dy, dx dx)) as the reference forms it, its dx dx once per particle.
// A particle with a NaN coordinate has no vertex in the band.
//
// It is bound by the tests' VALU work and then by the ORs: device-scope atomics
// are slow here, and a word takes bits from every particle within 3 cells of its
// 32 vertices.  So the bits are gathered in an LDS window first: the waves of a
// workgroup (up to 128 consecutive sorted particles, whose boxes share their
// words) use one window when the box of their boxes has at most kExcWindow
// words; else each wave its own part of it, and a wave whose box does not fit
// there ORs straight into the mask.  Each nonzero window word then costs one
// atomic.  (Windows of one wave took 61 us, of 16 waves 71 us: too few, too
// uneven workgroups.)
constexpr int kExcWaves = 4;
constexpr int kExcWindow = 2048;                      // words of the workgroup's window
constexpr int kExcWaveWindow = kExcWindow / kExcWaves;
constexpr uint32_t kExcLanes = 8;                     // lanes per particle
constexpr uint32_t kExcPart = 64 / kExcLanes;         // particles per step of a wave

// Words [w0, w0 + nw) of rows [y0, y0 + ny) of layers [z0, z0 + nz) of the mask
// that the clamped boxes about the cells [lo, hi] touch.
struct MaskBox {
    int w0, y0, z0, nw, ny, nz;
    __device__ __forceinline__ MaskBox(const GridDev& sc, const int* lo, const int* hi) {
        w0 = clampi(lo[0] - 3, 0, sc.rx - 1) >> 5;
        y0 = clampi(lo[1] - 3, 0, sc.ry - 1);
        z0 = clampi(lo[2] - 3, 0, sc.rz - 1);
        nw = (clampi(hi[0] + 3, 0, sc.rx - 1) >> 5) - w0 + 1;
        ny = clampi(hi[1] + 3, 0, sc.ry - 1) - y0 + 1;
        nz = clampi(hi[2] + 3, 0, sc.rz - 1) - z0 + 1;
    }
    __device__ __forceinline__ bool fits(int words) const {
        return (int64_t)nw * ny * nz <= (int64_t)words;
    }
    // ORs the window's words into the mask: thread t of n
    __device__ __forceinline__ void flush(const uint32_t* win, uint32_t* bits, const GridDev& sc,
                                          uint32_t wx, int t, int n) const {
        for (int r = t; r < ny * nz; r += n) {
            const int zi = r / ny, yi = r - zi * ny;
            uint32_t* row = bits + ((uint64_t)(z0 + zi) * sc.ry + (uint32_t)(y0 + yi)) * wx + w0;
            for (int k = 0; k < nw; ++k) {
                const uint32_t m = win[r * nw + k];
                if (m) atomicOr(row + k, m);
            }
        }
    }
};

__global__ __launch_bounds__(64 * kExcWaves) void k_band_exceptions(BandArgs a, uint32_t group) {
    __shared__ float4 pos[kExcWaves][64];  // a wave's live particles, compacted
    __shared__ int3 cell[kExcWaves][64];   // their scalar cells
    __shared__ uint32_t window[kExcWindow];
    __shared__ int box[6];                 // cell box of the workgroup's particles
    const bool by_flags = a.all_exceptions != 0 && a.flags != nullptr;
    const uint32_t count = by_flags ? a.num_particles : a.counters->num_exceptions;
    const uint32_t wx = row_words(a.sc.rx);
    const uint32_t lane = __lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    const uint64_t per_block = (uint64_t)kExcWaves * group;
    const int big = 0x3fffffff;
    // workgroup-uniform loop
    for (uint64_t b0 = blockIdx.x * per_block; b0 < count; b0 += gridDim.x * per_block) {
        if (threadIdx.x < 6) box[threadIdx.x] = threadIdx.x < 3 ? big : -big;
        const uint64_t e = b0 + (uint64_t)wave * group + lane;
        bool live = lane < group && e < count;
        uint32_t pi = 0;
        if (live) {
            if (by_flags) {
                live = a.flags[e] != 0u;
                pi = (uint32_t)e;
            } else {
                pi = a.exceptions[e];
            }
        }
        float4 p = make_float4(0.f, 0.f, 0.f, 0.f);
        if (live) {
            p = a.sorted[pi];
            live = p.x == p.x && p.y == p.y && p.z == p.z;
        }
        const uint64_t m = __ballot(live);
        const uint32_t n = (uint32_t)__popcll(m);
        int lo[3] = {big, big, big}, hi[3] = {-big, -big, -big};
        if (n) {
            if (live) {
                lo[0] = hi[0] = trunc_clamped(cell_coord(p.x, a.sc.minx, a.sc.cell), a.sc.rx);
                lo[1] = hi[1] = trunc_clamped(cell_coord(p.y, a.sc.miny, a.sc.cell), a.sc.ry);
                lo[2] = hi[2] = trunc_clamped(cell_coord(p.z, a.sc.minz, a.sc.cell), a.sc.rz);
                pos[wave][mask_rank(m)] = p;
                cell[wave][mask_rank(m)] = make_int3(lo[0], lo[1], lo[2]);
            }
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                lo[d] = wave_min_i(lo[d]);
                hi[d] = wave_max_i(hi[d]);
            }
        }
        __syncthreads();
        if (n && lane == 0) {
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                atomicMin(&box[d], lo[d]);
                atomicMax(&box[3 + d], hi[d]);
            }
        }
        __syncthreads();
        int blo[3], bhi[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            blo[d] = box[d];
            bhi[d] = box[3 + d];
        }
        __syncthreads();  // box is rewritten by the next round
        // no surface particle in the workgroup's entries (uniform)
        if (blo[0] > bhi[0]) continue;
        MaskBox mb(a.sc, blo, bhi);
        const bool shared = mb.fits(kExcWindow);
        uint32_t* win = window;
        bool windowed = shared;
        if (!shared && n) {
            mb = MaskBox(a.sc, lo, hi);
            windowed = mb.fits(kExcWaveWindow);
            win = window + wave * kExcWaveWindow;
        }
        const int nwin = mb.nw * mb.ny * mb.nz;
        if (shared) {
            for (int t = (int)threadIdx.x; t < nwin; t += 64 * kExcWaves) win[t] = 0u;
            __syncthreads();
        } else {
            if (windowed)
                for (int t = (int)lane; t < nwin; t += 64) win[t] = 0u;
            wave_lds_sync();
        }
        for (uint32_t it = 0; it < n; it += kExcPart) {
            const uint32_t slot = it + lane / kExcLanes;
            if (slot >= n) continue;
            const float4 p = pos[wave][slot];
            const int3 pc = cell[wave][slot];
            const int x0 = clampi(pc.x - 3, 0, a.sc.rx - 1), x1 = clampi(pc.x + 3, 0, a.sc.rx - 1);
            const int y0 = clampi(pc.y - 3, 0, a.sc.ry - 1), y1 = clampi(pc.y + 3, 0, a.sc.ry - 1);
            const int z0 = clampi(pc.z - 3, 0, a.sc.rz - 1), z1 = clampi(pc.z + 3, 0, a.sc.rz - 1);
            const int z = z0 + (int)(lane % kExcLanes);
            if (z > z1) continue;
            const float dz = vertex_coord((uint32_t)z, a.sc.minz, a.sc.cell) - p.z;
            // a row has vertices x in [x0, x1), at most 6, in one or two words
            const uint32_t w0 = (uint32_t)x0 >> 5, sh = (uint32_t)x0 & 31u;
            const uint32_t valid = (1u << (x1 - x0)) - 1u;
            float xx[6];
#pragma unroll
            for (int k = 0; k < 6; ++k) {
                const float dx = vertex_coord((uint32_t)(x0 + k), a.sc.minx, a.sc.cell) - p.x;
                xx[k] = dx * dx;
            }
            const int at = ((z - mb.z0) * mb.ny + (y0 - mb.y0)) * mb.nw + ((int)w0 - mb.w0);
            uint32_t* row = a.bits + ((uint64_t)z * a.sc.ry + (uint32_t)y0) * wx + w0;
#pragma unroll
            for (int ky = 0; ky < 7; ++ky) {
                const float dy = vertex_coord((uint32_t)(y0 + ky), a.sc.miny, a.sc.cell) - p.y;
                // bit k: d2 < a.d2_limit, as the sign of the difference (exact:
                // a float difference is negative exactly when it should be)
                uint32_t in = 0;
#pragma unroll
                for (int k = 5; k >= 0; --k) {
                    const float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, xx[k]));
                    in = __builtin_amdgcn_alignbit(in, (uint32_t)__float_as_int(d2 - a.d2_limit),
                                                   31);
                }
                const uint64_t bits = (uint64_t)(in & valid) << sh;
                const uint32_t m0 = (uint32_t)bits, m1 = (uint32_t)(bits >> 32);
                if (y0 + ky > y1) continue;
                if (windowed) {
                    if (m0) atomicOr(&win[at + ky * mb.nw], m0);
                    if (m1) atomicOr(&win[at + ky * mb.nw + 1], m1);
                } else {
                    if (m0) atomicOr(row + (uint64_t)ky * wx, m0);
                    if (m1) atomicOr(row + (uint64_t)ky * wx + 1, m1);
                }
            }
        }
        if (shared) {
            __syncthreads();
            mb.flush(win, a.bits, a.sc, wx, (int)threadIdx.x, 64 * kExcWaves);
            __syncthreads();
        } else {
            wave_lds_sync();
            if (windowed && n) mb.flush(win, a.bits, a.sc, wx, (int)lane, 64);
            wave_lds_sync();
        }
    }
}

// Compaction of the band mask into the ascending band index (the reference's
// scan + compactSurfaceVertex): k_axis_maps counts the set bits of every 256-word
// block; then band_emit gives each block its offset
// (the sum of the counts of the blocks before it, at most 8 words per thread
// from L2), scans its words' counts, writes each word's offset (word_off, the
// band rank of the word's first vertex) and the block's vertices, 16 lanes for a
// word: its lanes store to consecutive entries.  (A lane for each word, writing
// its ids into LDS for the block to copy out, met bank conflicts, and stored
// directly when the block had more than 4096.)  12.4 -> 8.0 us for a 1M dam break
// at 256^3, 39 -> 10.5 with the wider band of Akinci12, 25 -> 12 at 384^3; 3.0 ->
// 4.1 where the grid has a few full words only, beside the slab counts, which
// take as long.
// The last block writes the band size.
__device__ __forceinline__ void band_emit(uint32_t block, uint32_t blocks,
                                          const uint32_t* __restrict__ bits,
                                          const uint32_t* __restrict__ partials, uint64_t nwords,
                                          uint32_t wx, uint32_t rx,
                                          uint32_t* __restrict__ word_off,
                                          uint32_t* __restrict__ band_index, uint64_t cap,
                                          uint32_t* __restrict__ total, int scanned) {
    __shared__ uint32_t part[8];
    const uint64_t w = (uint64_t)block * blockDim.x + threadIdx.x;
    const bool live = w < nwords;
    const uint32_t b = live ? bits[w] : 0u;
    const uint32_t c = (uint32_t)__popc(b);
    // offset of this block: the counts of the blocks before it (or, when
    // `scanned`, partials already holds the exclusive offsets)
    uint32_t before = 0;
    if (scanned) {
        before = threadIdx.x == 0 ? partials[block] : 0u;
    } else {
        // at most 4096 blocks: up to 16 counts per thread, loaded together
        uint32_t pv[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const uint32_t i = threadIdx.x + 256u * k;
            pv[k] = i < block ? partials[i] : 0u;
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) before += pv[k];
    }
    before = wave_sum(before);
    // exclusive scan of the words' counts inside the block
    const uint32_t incl = wave_inclusive_sum(c);
    const uint32_t wave = threadIdx.x >> 6;
    if (__lane_id() == 63) {
        part[wave] = incl;
        part[4 + wave] = before;
    }
    __syncthreads();
    uint32_t lo = part[4] + part[5] + part[6] + part[7];  // the block's first output slot
    uint32_t wave_off = 0, block_total = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        if (k < (int)wave) wave_off += part[k];
        block_total += part[k];
    }
    const uint32_t o = lo + wave_off + incl - c;
    if (live) word_off[w] = o;
    if (block == blocks - 1 && threadIdx.x == 0) *total = lo + block_total;
    const uint64_t row = w / wx;
    const uint32_t vbase = (uint32_t)(row * rx) + (uint32_t)(w % wx) * 32u;
    // four words at a time, 16 lanes each: lane l of the 16 takes bits 2l and 2l + 1
    const uint64_t nonzero = __ballot(b != 0u);
    const uint32_t bit = 2u * (threadIdx.x & 15u), sub = (threadIdx.x & 63u) >> 4;
    for (uint32_t i0 = 0; i0 < 64u; i0 += 16u) {
        if (!((nonzero >> i0) & 0xFFFFu)) continue;
        uint32_t word[4], base[4], off[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            const int from = (int)(i0 + 4u * i + sub);
            word[i] = (uint32_t)__shfl((int)b, from, 64);
            base[i] = (uint32_t)__shfl((int)vbase, from, 64) + bit;
            off[i] = (uint32_t)__shfl((int)o, from, 64);
        }
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
            const uint32_t k = off[i] + (uint32_t)__popc(word[i] & ((1u << bit) - 1u));
            const uint32_t first = (word[i] >> bit) & 1u;
            if (first && k < cap) band_index[k] = base[i];
            if (((word[i] >> bit) & 2u) && k + first < cap) band_index[k + first] = base[i] + 1u;
        }
    }
}

// Per axis: virtual cell of every scalar vertex, and each virtual cell's
// vertex interval [lo, hi).  Layout of `maps`:
//   vc_x[rx] vc_y[ry] vc_z[rz] lo_x[vcx] hi_x[vcx] lo_y[vcy] hi_y[vcy] lo_z[vcz] hi_z[vcz]
struct AxisMaps {
    uint32_t *vc[3], *lo[3], *hi[3];
    uint32_t* row_any;   // bit (z ry + y): scalar row (y, z) holds a band vertex
    uint64_t row_words;  // words of row_any
};

// blockIdx.y = 0, 1, 2: the maps of axis x, y, z; blockIdx.y = 3: the row
// occupancy bits, one wave per 64 rows (each wave writes its two words);
// blockIdx.y = 4: clears the per-cell band counts cnt[ncells]; blockIdx.y = 5: the
// band vertices of every 256 mask words (partials), for k_band_lists.
__global__ __launch_bounds__(256) void k_axis_maps(GridDev sc, GridDev sp, int radius, AxisMaps m,
                                                   const uint32_t* __restrict__ bits, uint32_t wx,
                                                   uint32_t* __restrict__ cnt, uint64_t ncells,
                                                   uint64_t nwords,
                                                   uint32_t* __restrict__ partials) {
    __shared__ uint32_t part[4];
    const uint32_t axis = blockIdx.y;
    if (axis == 5) {
        const uint32_t groups = (uint32_t)((nwords + 255) / 256);
        for (uint32_t g = blockIdx.x; g < groups; g += gridDim.x) {
            const uint64_t w = (uint64_t)g * 256u + threadIdx.x;
            const uint32_t c = wave_sum(w < nwords ? (uint32_t)__popc(bits[w]) : 0u);
            if (__lane_id() == 0) part[threadIdx.x >> 6] = c;
            __syncthreads();
            if (threadIdx.x == 0) partials[g] = part[0] + part[1] + part[2] + part[3];
            __syncthreads();
        }
        return;
    }
    if (axis == 4) {
        for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < ncells;
             i += (uint64_t)gridDim.x * blockDim.x)
            cnt[i] = 0u;
        return;
    }
    if (axis == 3) {
        const uint64_t rows = (uint64_t)sc.ry * sc.rz;
        for (uint64_t r0 = (uint64_t)blockIdx.x * blockDim.x + (threadIdx.x & ~63u); r0 < rows;
             r0 += (uint64_t)gridDim.x * blockDim.x) {
            const uint64_t r = r0 + __lane_id();
            uint32_t any = 0;
            if (r < rows)
                for (uint32_t w = 0; w < wx; ++w) any |= bits[r * wx + w];
            const uint64_t b = __ballot(any != 0);
            if (__lane_id() == 0) {
                const uint64_t k = r0 >> 5;
                m.row_any[k] = (uint32_t)b;
                if (k + 1 < m.row_words) m.row_any[k + 1] = (uint32_t)(b >> 32);
            }
        }
        return;
    }
    const uint32_t res = axis == 0 ? sc.rx : (axis == 1 ? sc.ry : sc.rz);
    const float smin = axis == 0 ? sc.minx : (axis == 1 ? sc.miny : sc.minz);
    const float pmin = axis == 0 ? sp.minx : (axis == 1 ? sp.miny : sp.minz);
    const int pres = (int)(axis == 0 ? sp.rx : (axis == 1 ? sp.ry : sp.rz));
    const uint32_t nvc = (uint32_t)(pres + 2 * radius);
    auto vc_of = [&](uint32_t v) -> uint32_t {
        const float q = cell_coord(vertex_coord(v, smin, sc.cell), pmin, sp.cell);
        int c = trunc_clamped(q, pres + radius);
        c = clampi(c, -radius, pres - 1 + radius);
        return (uint32_t)(c + radius);
    };
    // first vertex whose virtual cell is >= c (the map is non-decreasing:
    // vertex positions, the cell coordinate, truncation and clamping all are)
    auto first_at_least = [&](uint32_t c) -> uint32_t {
        uint32_t lo = 0, hi = res;
        while (lo < hi) {
            const uint32_t mid = (lo + hi) >> 1;
            if (vc_of(mid) < c) lo = mid + 1;
            else hi = mid;
        }
        return lo;
    };
    // threads [0, res): the vertex -> cell map; [res, res + nvc): each virtual
    // cell's vertex interval [lo, hi), empty (lo = hi) when no vertex maps to it
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < res + nvc;
         i += gridDim.x * blockDim.x) {
        if (i < res) {
            m.vc[axis][i] = vc_of(i);
        } else {
            const uint32_t c = i - res;
            m.lo[axis][c] = first_at_least(c);
            m.hi[axis][c] = first_at_least(c + 1);
        }
    }
}

// 32 row occupancy bits starting at row `bit0` (bits past the end read 0).
__device__ __forceinline__ uint32_t row_bits32(const AxisMaps& m, uint64_t bit0) {
    const uint64_t w = bit0 >> 5;
    const uint32_t sh = (uint32_t)(bit0 & 31u);
    const uint32_t lo = w < m.row_words ? m.row_any[w] : 0u;
    if (!sh) return lo;
    const uint32_t hi = w + 1 < m.row_words ? m.row_any[w + 1] : 0u;
    return (lo >> sh) | (hi << (32u - sh));
}

// Occupied rows y in [ylo + yb, min(ylo + yb + 32, yhi)) of layer z, bit i = row ylo + yb + i.
__device__ __forceinline__ uint32_t layer_rows(const AxisMaps& m, const GridDev& sc, uint32_t z,
                                               uint32_t ylo, uint32_t yb, uint32_t ny) {
    uint32_t b = row_bits32(m, (uint64_t)z * sc.ry + ylo + yb);
    const uint32_t left = ny - yb;
    if (left < 32u) b &= (1u << left) - 1u;
    return b;
}

// Cell-major band order, counted per slab: the slab (cx, cy, z) is the part of
// virtual cell v = (cz vcy + cy) vcx + cx (cz = vc_z[z]) on scalar layer z.
// Slabs are stored cell by cell and by layer inside a cell:
//   slab(cx, cy, z) = vcx vcy lo_z[cz] + (cy vcx + cx) nz(cz) + (z - lo_z[cz]),
// so a cell's vertices come in ascending id order (layers z, rows y, then x),
// i.e. a 64-vertex chunk is a compact slab of the cell, which keeps the
// candidate culling of the field kernels effective.  The list itself is not
// written: the field kernels read a chunk's vertices from the mask with the
// slab counts (chunk_vertex).  The count pass takes one thread per slab
// (consecutive threads = consecutive cx, which read the same row words); rows
// without band vertices are skipped with the row occupancy bits.  It writes the
// slab's band vertex count and adds it to its cell's count (cnt, cleared by
// k_axis_maps).  Writing the list too took 19 us at 113^3 and 41 us at 384^3,
// and the scan before it 9; listing costs the Yu13 field 5 and 20 us there.
__device__ __forceinline__ void slab_rows(uint32_t block, uint32_t blocks,
                                          const uint32_t* __restrict__ bits, const GridDev& sc,
                                          uint32_t wx, const AxisMaps& m, uint32_t vcx,
                                          uint32_t vcy, uint32_t* __restrict__ slab,
                                          uint32_t* __restrict__ cnt) {
    const uint64_t total = (uint64_t)vcx * vcy * sc.rz;
    for (uint64_t t = (uint64_t)block * blockDim.x + threadIdx.x; t < total;
         t += (uint64_t)blocks * blockDim.x) {
        const uint32_t cx = (uint32_t)(t % vcx);
        const uint32_t cy = (uint32_t)((t / vcx) % vcy);
        const uint32_t z = (uint32_t)(t / ((uint64_t)vcx * vcy));
        const uint32_t cz = m.vc[2][z];
        const uint32_t zlo = m.lo[2][cz], nz = m.hi[2][cz] - zlo;
        const uint64_t first = (uint64_t)vcx * vcy * zlo + ((uint64_t)cy * vcx + cx) * nz;
        const uint64_t idx = first + (z - zlo);
        const uint32_t v = (cz * vcy + cy) * vcx + cx;
        uint32_t o = 0;
        const uint32_t ylo = m.lo[1][cy], yhi = m.hi[1][cy];
        const uint32_t xlo = m.lo[0][cx], xhi = m.hi[0][cx];
        const uint32_t ny = yhi > ylo ? yhi - ylo : 0u;
        const uint32_t w0 = xlo >> 5;
        const uint32_t nw = xhi > xlo ? ((xhi + 31u) >> 5) - w0 : 0u;
        for (uint32_t yb = 0; nw && yb < ny; yb += 32u) {
            uint32_t rows = layer_rows(m, sc, z, ylo, yb, ny);
            while (rows) {
                // up to 4 occupied rows per round; with at most 2 words per
                // row (the common case) their 8 words are loaded together
                uint64_t rw[4];
                bool ok[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    ok[k] = rows != 0u;
                    const uint32_t dy = ok[k] ? (uint32_t)__builtin_ctz(rows) : 0u;
                    rw[k] = ((uint64_t)z * sc.ry + ylo + yb + dy) * wx;
                    rows &= rows - 1u;
                }
                if (nw <= 2u) {
                    uint32_t v0[4], v1[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        v0[k] = ok[k] ? bits[rw[k] + w0] : 0u;
                        v1[k] = ok[k] && nw == 2u ? bits[rw[k] + w0 + 1u] : 0u;
                    }
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        o += __popc(clip_word(v0[k], w0, xlo, xhi));
                        if (nw == 2u) o += __popc(clip_word(v1[k], w0 + 1u, xlo, xhi));
                    }
                } else {
                    for (int k = 0; k < 4; ++k) {
                        if (!ok[k]) break;
                        for (uint32_t j = 0; j < nw; ++j) {
                            const uint32_t w = w0 + j;
                            o += __popc(clip_word(bits[rw[k] + w], w, xlo, xhi));
                        }
                    }
                }
            }
        }
        slab[idx] = o;
        if (o) atomicAdd(&cnt[v], o);
    }
}

// Both lists in one launch: workgroups [0, emit_blocks) write the band index, the
// others count the slabs.  Each waits on chains of loads, so one launch after the
// other took the sum of their times: 10.4 us for 6.0 at 128^3, 14.6 for 12.3 at
// 256^3, and a launch more (a second with the counts now in k_axis_maps).
__global__ __launch_bounds__(256) void k_band_lists(
    uint32_t emit_blocks, const uint32_t* __restrict__ bits, const uint32_t* __restrict__ partials,
    uint64_t nwords, GridDev sc, uint32_t wx, uint32_t* __restrict__ word_off,
    uint32_t* __restrict__ band_index, uint64_t cap, uint32_t* __restrict__ total, int scanned,
    AxisMaps m, uint32_t vcx, uint32_t vcy, uint32_t* __restrict__ slab,
    uint32_t* __restrict__ cnt) {
    if (blockIdx.x < emit_blocks)
        band_emit(blockIdx.x, emit_blocks, bits, partials, nwords, wx, sc.rx, word_off, band_index,
                  cap, total, scanned);
    else
        slab_rows(blockIdx.x - emit_blocks, gridDim.x - emit_blocks, bits, sc, wx, m, vcx, vcy,
                  slab, cnt);
}

}  // namespace

int band_dilation_exact(const fsr_grid_info& sc, float h) {
    // farthest box vertex from any point of the particle's scalar cell:
    // |dx| < 4, |dy| < 4, |dz| < 4 cells
    const double reach = 4.0 * 1.7320508075688772 * (double)sc.cell_size;
    double maxabs = 0.0;
    const double lo[3] = {sc.min_pos.x, sc.min_pos.y, sc.min_pos.z};
    const uint32_t r[3] = {sc.resolution.x, sc.resolution.y, sc.resolution.z};
    for (int a = 0; a < 3; ++a) {
        const double hi = lo[a] + (double)sc.cell_size * (double)r[a];
        maxabs = std::max(maxabs, std::max(std::fabs(lo[a]), std::fabs(hi)));
    }
    // FP32 rounding of the vertex position, the difference and the length
    const double slack = 64.0 * 1.1920928955078125e-7 * std::max(maxabs, (double)h);
    return reach + slack < 1.5 * (double)h ? 1 : 0;
}

fsr_status band_build(fsr_context* ctx, const BandArgs& a, hipStream_t s) {
    const uint32_t wx = row_words(a.sc.rx);
    const uint64_t nwords = (uint64_t)wx * a.sc.ry * a.sc.rz;
    const uint32_t blocks = (uint32_t)((nwords + 255) / 256);
    // S (bytes) -> tmp (x), tmp -> S (y, its first nwords words), S -> bits
    // (z); `sbits` is consumed
    uint32_t* sb = const_cast<uint32_t*>(a.sbits);
    auto tiles = [&](uint32_t tw, uint32_t tyz) {
        return dim3((wx + tw - 1) / tw, (a.sc.ry + tyz - 1) / tyz, (a.sc.rz + tyz - 1) / tyz);
    };
    const dim3 big = tiles(8, 16), small = tiles(4, 8);
    if (a.all_exceptions) {
        // no seeds: the exact path alone sets bits of the mask the caller cleared
    } else if (big.y <= 65535u && big.z <= 65535u) {
        const uint64_t n = (uint64_t)big.x * big.y * big.z, cus = (uint64_t)ctx->num_cus;
        const bool fine = 2 * n < cus;
        auto dilate = fine ? k_dilate_box<4, 8, 512, false>
                           : (n < cus ? k_dilate_box<8, 16, 1024, false>
                                      : k_dilate_box<8, 16, 1024, true>);
        hipLaunchKernelGGL(dilate, fine ? small : big, dim3(fine ? 512 : 1024), 0, s,
                           (const uint8_t*)sb, a.bits, wx, a.sc);
        FSR_LAUNCH_CHECK("k_dilate_box");
    } else {
        hipLaunchKernelGGL(k_dilate_x, dim3(blocks), dim3(256), 0, s, (const uint8_t*)sb, a.tmp,
                           wx, nwords, a.sc.rx);
        FSR_LAUNCH_CHECK("k_dilate_x");
        hipLaunchKernelGGL(k_dilate_rows, dim3(blocks), dim3(256), 0, s, a.tmp, sb, nwords,
                           (uint64_t)wx, a.sc.ry, (uint64_t)a.sc.ry);
        FSR_LAUNCH_CHECK("k_dilate_rows(y)");
        hipLaunchKernelGGL(k_dilate_rows, dim3(blocks), dim3(256), 0, s, sb, a.bits, nwords,
                           (uint64_t)wx * a.sc.ry, a.sc.rz, (uint64_t)a.sc.rz);
        FSR_LAUNCH_CHECK("k_dilate_rows(z)");
    }
    // six workgroups of 4 waves per CU, within the band class's limit
    const uint32_t eb = (uint32_t)persistent_blocks(ctx, 64 * kExcWaves, 6, TUNE_BAND);
    // 1.5 h in double, as the smallest float that is not below it: for a float
    // d, (double)d < L holds exactly when d < that float
    const double L = (double)a.h * 1.5;
    float limit = (float)L;
    if ((double)limit < L) limit = std::nextafter(limit, std::numeric_limits<float>::infinity());
    BandArgs b = a;
    b.d2_limit = limit > 0.0f ? std::nextafter(sqrt_bound(limit, true),
                                               std::numeric_limits<float>::infinity())
                              : -1.0f;
    const uint32_t waves = (uint32_t)kExcWaves * eb;
    const uint32_t per = (a.num_particles + waves - 1u) / waves;
    const uint32_t group = std::min(32u, std::max(8u, (per + 7u) / 8u * 8u));
    hipLaunchKernelGGL(k_band_exceptions, dim3(eb), dim3(64 * kExcWaves), 0, s, b, group);
    FSR_LAUNCH_CHECK("k_band_exceptions");
    return FSR_OK;
}

fsr_status band_compact(fsr_context* ctx, const uint32_t* bits, const GridDev& sc,
                        const GridDev& sp, int radius, Counters* counters, fsr_frame_stats* st,
                        BandCompactOut* out, hipStream_t s) {
    const uint32_t wx = row_words(sc.rx);
    const uint64_t nwords = (uint64_t)wx * sc.ry * sc.rz;
    const uint64_t V = (uint64_t)sc.rx * sc.ry * sc.rz;
    uint32_t *word_off, *band_index;
    FSR_TRY(arena_typed(ctx, A_WORD_OFF, nwords, &word_off));
    FSR_TRY(arena_typed(ctx, A_BAND_INDEX, V, &band_index));
    const uint32_t emit_blocks = (uint32_t)((nwords + 255) / 256);
    uint32_t* partials;
    FSR_TRY(arena_typed(ctx, A_BAND_PARTIALS, emit_blocks, &partials));
    out->band_index = band_index;

    // cell-major work list
    const uint32_t vcx = sp.rx + 2 * radius, vcy = sp.ry + 2 * radius, vcz = sp.rz + 2 * radius;
    const uint64_t nvc = (uint64_t)vcx * vcy * vcz;
    uint32_t *maps, *cnt, *cell_off, *chunk_off, *chunk_cell;
    const uint64_t rows = (uint64_t)sc.ry * sc.rz;
    const uint64_t row_words = 2ull * ((rows + 63) / 64);
    const uint64_t map_len =
        (uint64_t)sc.rx + sc.ry + sc.rz + 2ull * (vcx + vcy + vcz) + row_words;
    FSR_TRY(arena_typed(ctx, A_AXIS_MAPS, map_len, &maps));
    FSR_TRY(arena_typed(ctx, A_CELL_CNT, nvc, &cnt));
    FSR_TRY(arena_typed(ctx, A_CELL_OFF, nvc, &cell_off));
    FSR_TRY(arena_typed(ctx, A_CHUNK_OFF, nvc, &chunk_off));
    const uint64_t max_chunks = V / 64 + nvc + 1;
    FSR_TRY(arena_typed(ctx, A_CHUNK_CELL, max_chunks, &chunk_cell));
    AxisMaps m;
    m.vc[0] = maps;
    m.vc[1] = m.vc[0] + sc.rx;
    m.vc[2] = m.vc[1] + sc.ry;
    m.lo[0] = m.vc[2] + sc.rz;
    m.hi[0] = m.lo[0] + vcx;
    m.lo[1] = m.hi[0] + vcx;
    m.hi[1] = m.lo[1] + vcy;
    m.lo[2] = m.hi[1] + vcy;
    m.hi[2] = m.lo[2] + vcz;
    m.row_any = m.hi[2] + vcz;
    m.row_words = row_words;
    const uint32_t maxres = std::max(sc.rx + vcx, std::max(sc.ry + vcy, sc.rz + vcz));
    const uint32_t map_blocks = (uint32_t)std::max<uint64_t>(
        (maxres + 255) / 256, std::min<uint64_t>((rows + 255) / 256, 1024));
    hipLaunchKernelGGL(k_axis_maps, dim3(map_blocks, 6), dim3(256), 0, s, sc, sp, radius, m, bits,
                       wx, cnt, nvc, nwords, partials);
    FSR_LAUNCH_CHECK("k_axis_maps");
    // up to 4096 blocks each block sums the counts before it (at most 16 words
    // per thread); beyond, the counts are scanned first
    const int scanned = emit_blocks > 4096u ? 1 : 0;
    if (scanned)
        FSR_TRY(scan_exclusive(ctx, SCAN_U32, partials, partials, emit_blocks, nullptr, nullptr,
                               s));
    // slab counts (and cell counts); cell offsets, chunk offsets and the chunk
    // list in one scan
    const uint64_t nslabs = (uint64_t)vcx * vcy * sc.rz;
    uint32_t* slab;
    FSR_TRY(arena_typed(ctx, A_SLAB, nslabs, &slab));
    const uint32_t slab_blocks = (uint32_t)std::min<uint64_t>((nslabs + 255) / 256, 16384);
    hipLaunchKernelGGL(k_band_lists, dim3(emit_blocks + slab_blocks), dim3(256), 0, s, emit_blocks,
                       bits, partials, nwords, sc, wx, word_off, band_index, V,
                       &st->num_band_vertices, scanned, m, vcx, vcy, slab, cnt);
    FSR_LAUNCH_CHECK("k_band_lists");
    FSR_TRY(scan_cells(ctx, cnt, nvc, cell_off, chunk_off, chunk_cell, max_chunks,
                       &counters->num_chunks, s));
    out->cell_off = cell_off;
    out->cell_cnt = cnt;
    out->chunk_off = chunk_off;
    out->chunk_cell = chunk_cell;
    out->bits = bits;
    out->wx = wx;
    out->axis = m.lo[0];  // lo_x, hi_x, lo_y, hi_y, lo_z, hi_z follow one another
    out->slab = slab;
    out->vcx = vcx;
    out->vcy = vcy;
    out->vcz = vcz;
    out->radius = radius;
    out->max_chunks = max_chunks;
    return FSR_OK;
}

}  // namespace fsr
