// Adjoint of the ZB05 field and of the marching-cubes vertex interpolation with
// respect to the particle positions, marching-cubes topology held fixed.  The
// reference has no backward pass; the forward semantics differentiated here are
// those of updateScalarFieldValueZB05 (ReconstructionCUDA.cu:230-289,
// kernelZB05 ReconstructionCUDA.cuh:262-268) and of generateTriangles
// (ReconstructionCUDA.cu:383-463, vertex lerp only).
//
// Vertex term (mc_vertex_backward).  A soup vertex on the edge (a, b) of a cube
// sits at c_a + t (c_b - c_a), t = (iso - phi_a) / (phi_b - phi_a), so
//   dt/dphi_a = (iso - phi_b) / D^2,  dt/dphi_b = -(iso - phi_a) / D^2,  D = phi_b - phi_a
// and an edge with |D| < 1e-7 (t fixed at 0.5) carries no gradient.  Normals
// are treated as constants.  Each emitted cube sums, per corner, the terms of
// its soup vertices on the edges at that corner (8 lanes per cube); each band
// vertex then adds the sums of the (up to) 8 cubes it is a corner of, in a
// fixed order: no floating-point atomics, the result is deterministic.
//
// Field term (field_zb05_backward).  With w_i = t_i^3, t_i = 1 - |x - p_i|^2/R^2,
// W = sum w_i, xbar = sum w_i p_i / W and phi = |x - xbar| - r_p:
//   dphi/dp_j = -(1/W) [ w_j n + (n . (p_j - xbar)) (6/R^2) t_j^2 (x - p_j) ],
//   n = (x - xbar) / |x - xbar|.
// A per-vertex pass folds the upstream gradient g into u = (g/W) n and
// c = (g/W) |x - xbar| (the forward kept x - xbar and W per vertex), so that
//   g dphi/dp_j = -[ w_j u + (c - u . (x - p_j)) (6/R^2) t_j^2 (x - p_j) ].
// The particle gradient is then a gather: a wave owns up to 64 particles of one
// hash cell and walks the band vertices of the 3^3 virtual cells around it (the
// cell-major band list keeps x-adjacent cells contiguous: 9 runs), staging 64
// vertices at a time in LDS as the forward stages particles.  A vertex in
// virtual cell v reads the hash cells clamp(v - 1 .. v + 1), so particle cell q
// is read exactly by the vertices of virtual cells q - 1 .. q + 1.  Neighbour
// lists are not stored: the gather walks the same cell ranges the forward used.
// The pairs are evaluated on the matrix cores (k_field_zb05_backward_mc).
// Results are written in the caller's particle order through the sort
// permutation; particles outside the hash grid get 0.
#include "common.hpp"

#include "mc_tables.h"

namespace fsr {

namespace {

constexpr int kAdjThreads = 256;

__constant__ uint64_t cAdjTri[256] = {FSR_MC_TRI_PACKED_VALUES};

__device__ __forceinline__ uint32_t corner_dx(uint32_t c) { return c >= 4 ? 1u : 0u; }
__device__ __forceinline__ uint32_t corner_dy(uint32_t c) {
    return (c == 2 || c == 3 || c == 6 || c == 7) ? 1u : 0u;
}
__device__ __forceinline__ uint32_t corner_dz(uint32_t c) {
    return (c == 1 || c == 2 || c == 5 || c == 6) ? 1u : 0u;
}

// ---------------------------------------------------------------------------
// vertex term: g_phi[v] += sum over soup vertices on edges at v
// ---------------------------------------------------------------------------
struct McBackArgs {
    const uint32_t* band_index;
    const uint32_t* valid_idx;
    uint32_t* touched;          // bit mask over the grid (band mask layout)
    const uint32_t* bits;
    const uint32_t* word_off;
    const uint32_t* nverts;
    const uint32_t* vert_off;
    const float* phi;
    const float* g_tri;
    float* g_phi;
    float* corner;              // [8 (capacity / 3)] corner sums per emitted cube
    const fsr_frame_stats* st;
    GridDev sc;
    float iso;
    uint32_t capacity;
    int cpu_flavor;
};

// Pass 1, one 8-lane group per emitted cube (lane c = corner c): the terms of
// the cube's soup vertices (table order) on the edges at corner c, summed into
// corner[8 t0 + c], t0 = the cube's first triangle (vert_off / 3, unique per
// cube); and the touched bits of the cube's corners, so that pass 2 skips,
// after one bit test, the band vertices no soup vertex depends on.
__global__ __launch_bounds__(kAdjThreads) void k_mc_corner_terms(McBackArgs a) {
    const uint32_t Q = a.st->num_valid_cubes;
    const uint32_t rx = a.sc.rx, ry = a.sc.ry;
    const uint64_t rxy = (uint64_t)rx * ry;
    const uint32_t wx = row_words(rx);
    const uint32_t c = threadIdx.x & 7u;
    const int g0 = (int)(__lane_id() & ~7u);
    const uint32_t groups = gridDim.x * (blockDim.x / 8u);
    for (uint32_t q = blockIdx.x * (blockDim.x / 8u) + threadIdx.x / 8u; q < Q; q += groups) {
        const uint32_t cb = a.valid_idx[q];
        const uint32_t off = a.vert_off[cb], nv = a.nverts[cb];
        if ((uint64_t)off + nv > a.capacity) continue;  // the forward did not emit it
        const uint32_t vid = a.band_index[cb];
        const uint32_t x = vid % rx, y = (vid / rx) % ry, z = (uint32_t)(vid / rxy);
        const uint32_t dx = corner_dx(c), dy = corner_dy(c), dz = corner_dz(c);
        if (dx == 0u) {
            // corners x and x + 1 of this lane's (y, z) row; both bits may share a word
            const uint64_t row = (uint64_t)(z + dz) * ry + (y + dy);
            const uint64_t w0 = row * wx + (x >> 5);
            const uint32_t bit = x & 31u;
            if (bit < 31u) {
                atomicOr(&a.touched[w0], 3u << bit);
            } else {
                atomicOr(&a.touched[w0], 1u << 31);
                atomicOr(&a.touched[w0 + 1], 1u);
            }
        }
        const uint64_t u = ((uint64_t)z * ry + y) * rx + x;
        const float val = a.phi[u + dx + (uint64_t)dy * rx + (uint64_t)dz * rxy];
        uint32_t f = (val <= a.iso) ? (1u << c) : 0u;
        f |= (uint32_t)__builtin_amdgcn_ds_swizzle((int)f, 0x1F | (1 << 10));
        f |= (uint32_t)__builtin_amdgcn_ds_swizzle((int)f, 0x1F | (2 << 10));
        f |= (uint32_t)__builtin_amdgcn_ds_swizzle((int)f, 0x1F | (4 << 10));
        const uint64_t tri = cAdjTri[f];
        float acc = 0.0f;
        for (uint32_t k = 0; k < nv; ++k) {
            const uint32_t e = (uint32_t)(tri >> (4 * k)) & 0xFu;
            const uint32_t s0 = (e < 8) ? (e & 3u) + (e & 4u) : e - 8u;
            const uint32_t s1 = (e < 8) ? (((e & 3u) + 1u) & 3u) + (e & 4u) : e - 4u;
            // the edge's corner values from their lanes (the whole group runs
            // the same k: nv is the group's)
            const float v0 = __shfl(val, g0 + (int)s0, 64);
            const float v1 = __shfl(val, g0 + (int)s1, 64);
            if (s0 != c && s1 != c) continue;
            const float delta = v1 - v0;
            const bool flat = a.cpu_flavor
                                  ? ((double)delta > -1.0e-7 && (double)delta < 1.0e-7)
                                  : (delta > -1.0e-7f && delta < 1.0e-7f);
            if (flat) continue;
            // d(position)/dt: corner s1 minus corner s0 as the forward evaluates them
            const uint32_t X0 = x + corner_dx(s0), Y0 = y + corner_dy(s0), Z0 = z + corner_dz(s0);
            const uint32_t X1 = x + corner_dx(s1), Y1 = y + corner_dy(s1), Z1 = z + corner_dz(s1);
            float ex, ey, ez;
            if (a.cpu_flavor) {
                ex = (a.sc.minx + (float)X1 * a.sc.cell) - (a.sc.minx + (float)X0 * a.sc.cell);
                ey = (a.sc.miny + (float)Y1 * a.sc.cell) - (a.sc.miny + (float)Y0 * a.sc.cell);
                ez = (a.sc.minz + (float)Z1 * a.sc.cell) - (a.sc.minz + (float)Z0 * a.sc.cell);
            } else {
                ex = vertex_coord(X1, a.sc.minx, a.sc.cell) - vertex_coord(X0, a.sc.minx, a.sc.cell);
                ey = vertex_coord(Y1, a.sc.miny, a.sc.cell) - vertex_coord(Y0, a.sc.miny, a.sc.cell);
                ez = vertex_coord(Z1, a.sc.minz, a.sc.cell) - vertex_coord(Z0, a.sc.minz, a.sc.cell);
            }
            const uint64_t o = 3ull * (off + k);
            const float gt = __builtin_fmaf(a.g_tri[o + 2], ez,
                                            __builtin_fmaf(a.g_tri[o + 1], ey, a.g_tri[o] * ex));
            const float inv_d2 = 1.0f / (delta * delta);
            acc += (s0 == c) ? gt * (a.iso - v1) * inv_d2 : -gt * (a.iso - v0) * inv_d2;
        }
        a.corner[8ull * (off / 3u) + c] = acc;
    }
}

// Pass 2, one thread per band vertex: the corner sums of the (up to) 8 emitted
// cubes it is a corner of, in corner order.
__global__ __launch_bounds__(kAdjThreads) void k_mc_vertex_backward(McBackArgs a) {
    const uint32_t B = a.st->num_band_vertices;
    const uint32_t rx = a.sc.rx, ry = a.sc.ry, rz = a.sc.rz;
    const uint64_t rxy = (uint64_t)rx * ry;
    const uint32_t wx = row_words(rx);
    for (uint32_t b = blockIdx.x * blockDim.x + threadIdx.x; b < B; b += gridDim.x * blockDim.x) {
        const uint32_t vid = a.band_index[b];
        const uint32_t x = vid % rx, y = (vid / rx) % ry, z = (uint32_t)(vid / rxy);
        if (!((a.touched[((uint64_t)z * ry + y) * wx + (x >> 5)] >> (x & 31u)) & 1u)) continue;
        // the cubes whose corner cv is this vertex, level by level over the 8
        // (each level's loads issued together): mask word, band rank, vertex
        // count, offset, corner sum
        uint64_t word[8];
        uint32_t bw[8], sh[8];
        bool ok[8];
#pragma unroll
        for (uint32_t cv = 0; cv < 8; ++cv) {
            const uint32_t ox = corner_dx(cv), oy = corner_dy(cv), oz = corner_dz(cv);
            const uint32_t ux = x - ox, uy = y - oy, uz = z - oz;
            ok[cv] = x >= ox && y >= oy && z >= oz && ux + 1 < rx && uy + 1 < ry && uz + 1 < rz;
            word[cv] = ((uint64_t)uz * ry + uy) * wx + (ux >> 5);
            sh[cv] = ux & 31u;
            bw[cv] = ok[cv] ? a.bits[word[cv]] : 0u;
        }
        uint32_t cb[8];
#pragma unroll
        for (uint32_t cv = 0; cv < 8; ++cv) {
            ok[cv] = ok[cv] && ((bw[cv] >> sh[cv]) & 1u);
            cb[cv] = ok[cv] ? a.word_off[word[cv]] + __popc(bw[cv] & ((1u << sh[cv]) - 1u)) : 0u;
        }
        uint32_t nv[8];
#pragma unroll
        for (uint32_t cv = 0; cv < 8; ++cv) nv[cv] = ok[cv] ? a.nverts[cb[cv]] : 0u;
        uint32_t off[8];
#pragma unroll
        for (uint32_t cv = 0; cv < 8; ++cv) {
            off[cv] = nv[cv] ? a.vert_off[cb[cv]] : 0u;
        }
        float acc = 0.0f;
#pragma unroll
        for (uint32_t cv = 0; cv < 8; ++cv) {
            // a cube the forward did not emit (beyond the soup capacity) adds nothing
            if (nv[cv] && (uint64_t)off[cv] + nv[cv] <= a.capacity)
                acc += a.corner[8ull * (off[cv] / 3u) + cv];
        }
        if (acc != 0.0f) a.g_phi[vid] += acc;
    }
}

// ---------------------------------------------------------------------------
// per band vertex (cell-major slot): u = (g/W) n, c = (g/W) |x - xbar|
// ---------------------------------------------------------------------------
// Per cell-major slot: (u, c) (zero when the vertex carries no gradient) and
// the vertex position, so that the gather below stages a vertex with two
// 16-byte loads and no index arithmetic.
__global__ __launch_bounds__(kAdjThreads) void k_field_coef(const uint32_t* __restrict__ cell_band,
                                                            const float4* __restrict__ saved,
                                                            const float* __restrict__ g_phi,
                                                            const fsr_frame_stats* st, GridDev sc,
                                                            float4* __restrict__ coef,
                                                            float4* __restrict__ vpos) {
    const uint32_t B = st->num_band_vertices;
    const uint32_t rxy = sc.rx * sc.ry;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < B; i += gridDim.x * blockDim.x) {
        const float4 s = saved[i];
        const uint32_t vid = cell_band[i];
        const float g = g_phi[vid];
        const uint32_t ix = vid % sc.rx, iy = (vid / sc.rx) % sc.ry, iz = vid / rxy;
        vpos[i] = make_float4(vertex_coord(ix, sc.minx, sc.cell), vertex_coord(iy, sc.miny, sc.cell),
                              vertex_coord(iz, sc.minz, sc.cell), 0.0f);
        float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
        const float len = __builtin_sqrtf(__builtin_fmaf(s.z, s.z, __builtin_fmaf(s.y, s.y, s.x * s.x)));
        if (s.w > 0.0f && len > 0.0f && g != 0.0f) {
            const float gw = g / s.w;
            const float k = gw / len;
            c = make_float4(k * s.x, k * s.y, k * s.z, gw * len);
        }
        coef[i] = c;
    }
}

// ---------------------------------------------------------------------------
// particle gather
// ---------------------------------------------------------------------------
struct FieldBackArgs {
    const float4* sorted;
    const fsr_index_range* ranges;
    const uint32_t* perm;
    const uint32_t* chunk_cell;
    const uint32_t* chunk_off;
    const uint32_t* num_chunks;
    uint32_t* next;               // per-XCD fetch counters (ItemFetch)
    const uint32_t* cell_off;     // virtual cell -> first cell-major slot
    const uint32_t* cell_cnt;
    const float4* coef;           // cell-major slot -> (u, c)
    const float4* vpos;           // cell-major slot -> vertex position
    GridDev sp;
    uint32_t vcx, vcy;
    int radius;
    float radius_sq;
    float* g_pos;                 // float3[N], caller order
};

// The gather evaluates its pairs in 16 x 16 particle/vertex tiles on the
// matrix cores (as the forward field): per 16 staged vertices and 16
// particles of the chunk
//   1. v_mfma_f32_16x16x4_f32: t = c0_p + (2 p'/R^2).x' - |x'|^2/R^2 with A =
//      (x', y', z', 1) of the vertices, B = (2p'/R^2, c0_p) of the particles,
//      C = -|x'|^2/R^2; a second one gives kd = u.p' + (c - u.x') with A =
//      (u, c - u.x') of the vertices and B = (p', 1);
//   2. t clamped to [0, 1], w = t^3 and kk = kd t^2 (4 VALU ops per pair);
//   3. rank-1 v_mfma_f32_4x4x1_16b_f32 updates: sum w (u, c - u.x') (the
//      last component unused) and sum kk (x', 1).
// Vertices whose coefficient is zero, or that lie at least 1.00005 R from the
// bounding box of the chunk's particles, add exactly 0 to every particle and
// are dropped at staging (order-preserving compaction, as in the forward).
// The queue is a ring of kAdjQueue entries: 63 waiting + 256 new, 256 being read.
constexpr int kAdjQueue = 512;
constexpr int kAdjStride = kAdjQueue + 16;
// rows: x', y', z', 1, ux, uy, uz, c - u.x', -|x'|^2/R^2
constexpr int kAdjOne = 3, kAdjU = 4, kAdjQ = 8, kAdjRows = 9;
typedef float v4f __attribute__((ext_vector_type(4)));

template <int M>
__device__ __forceinline__ float adj_swz_xor(float v) {
    return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x1F | (M << 10)));
}

// n staged vertices (a multiple of 16, from `rows`) against one 16-particle tile.
__device__ __forceinline__ void adj_tile(const float* __restrict__ rows, uint32_t n, float bt,
                                         float bk, v4f& gu, v4f& gx) {
    const uint32_t lane = __lane_id();
    const float* a1p = rows + (lane >> 4) * kAdjStride + (lane & 15u);
    const float* k1p = rows + (kAdjU + (lane >> 4)) * kAdjStride + (lane & 15u);
    const float* a2p = rows + (lane & 3u) * kAdjStride + 4u * (lane >> 4);
    const float* u2p = rows + (kAdjU + (lane & 3u)) * kAdjStride + 4u * (lane >> 4);
    const float* cqp = rows + kAdjQ * kAdjStride + 4u * (lane >> 4);
    const v4f zero = v4f{0.f, 0.f, 0.f, 0.f};
    for (uint32_t tb = 0; tb < n; tb += 16u) {
        const float4 cq = *reinterpret_cast<const float4*>(cqp + tb);
        v4f t = __builtin_amdgcn_mfma_f32_16x16x4f32(a1p[tb], bt, v4f{cq.x, cq.y, cq.z, cq.w}, 0, 0, 0);
        v4f kd = __builtin_amdgcn_mfma_f32_16x16x4f32(k1p[tb], bk, zero, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float tp = __builtin_amdgcn_fmed3f(t[r], 0.0f, 1.0f);
            const float t2 = tp * tp;
            t[r] = t2 * tp;
            kd[r] = kd[r] * t2;
        }
        const float4 au = *reinterpret_cast<const float4*>(u2p + tb);
        const float4 ax = *reinterpret_cast<const float4*>(a2p + tb);
        gu = __builtin_amdgcn_mfma_f32_4x4x1f32(au.x, t[0], gu, 0, 0, 0);
        gu = __builtin_amdgcn_mfma_f32_4x4x1f32(au.y, t[1], gu, 0, 0, 0);
        gu = __builtin_amdgcn_mfma_f32_4x4x1f32(au.z, t[2], gu, 0, 0, 0);
        gu = __builtin_amdgcn_mfma_f32_4x4x1f32(au.w, t[3], gu, 0, 0, 0);
        gx = __builtin_amdgcn_mfma_f32_4x4x1f32(ax.x, kd[0], gx, 0, 0, 0);
        gx = __builtin_amdgcn_mfma_f32_4x4x1f32(ax.y, kd[1], gx, 0, 0, 0);
        gx = __builtin_amdgcn_mfma_f32_4x4x1f32(ax.z, kd[2], gx, 0, 0, 0);
        gx = __builtin_amdgcn_mfma_f32_4x4x1f32(ax.w, kd[3], gx, 0, 0, 0);
    }
}

// A workgroup per chunk: its 4 waves stage a quarter each of a 256-vertex round
// into one LDS ring, in candidate order, and each evaluates one of the chunk's
// 16-particle tiles.  A chunk's work varies from nothing (no band vertex near)
// to some 290 rounds of 64 vertices (a particle at the surface); with a wave per
// chunk a SIMD that drew heavy ones ran long after the others had finished, and
// a frame's few thousand chunks leave no others to level it.  Shared, a heavy
// chunk loads all 4 SIMDs of a CU.  Per round two barriers: counts (which also
// says that the previous batches are evaluated), and entries.  Bound by VALU and
// matrix issue, then by the imbalance that is left.  Ball of n particles, wave
// per chunk -> workgroup per chunk: 16k 354 -> 168 us, 64k 524 -> 297, 125k 760 ->
// 405, 256k (192^3) 817 -> 564, 700k 1149 -> 1072.
__global__ __launch_bounds__(kAdjThreads, 6) void k_field_zb05_backward_mc(FieldBackArgs a) {
    constexpr uint32_t kWaves = kAdjThreads / 64;
    __shared__ __align__(16) float q[kAdjRows * kAdjStride];
    __shared__ float bt_lds[kWaves][4][64];  // per lane: (2p'/R^2, c0)
    __shared__ uint32_t count[kWaves];
    __shared__ uint32_t next_chunk[2];  // by the chunk's parity: see the loop's end
    __shared__ FetchState fetch;
    fetch_init(&fetch);
    const uint32_t lane = __lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t nch = *a.num_chunks;
    const float inv_r2 = 1.0f / a.radius_sq;
    const float cull_r2 = a.radius_sq * 1.0001f;
    float* vb = &bt_lds[wave][0][0];
    for (uint32_t t = threadIdx.x; t < (uint32_t)kAdjQueue; t += kAdjThreads)
        q[kAdjOne * kAdjStride + t] = 1.0f;
    ItemFetch<1, true> items(a.next, nch, &fetch);
    if (wave == 0) {
        const uint32_t first = items.next(0);
        if (lane == 0) next_chunk[0] = first;
    }
    __syncthreads();
    // workgroup-uniform
    uint32_t parity = 0;
    for (uint32_t ch = next_chunk[0]; ch < nch; ch = next_chunk[parity]) {
        const uint32_t c = a.chunk_cell[ch];
        const uint32_t k = ch - a.chunk_off[c];
        const fsr_index_range own = a.ranges[c];
        const uint32_t i = own.start + 64u * k + lane;
        const bool live = i < own.end;
        const uint32_t cnt = min(64u, own.end - (own.start + 64u * k));
        const bool mine = wave < ((cnt + 15u) >> 4);
        const uint32_t qcx = c % a.sp.rx, qcy = (c / a.sp.rx) % a.sp.ry, qcz = c / (a.sp.rx * a.sp.ry);

        // 9 runs of band slots: virtual cells (q + radius) + {-1, 0, 1}^3
        uint32_t len = 0, rs = 0;
        if (lane < 9) {
            const uint32_t vy = qcy + a.radius + (lane % 3) - 1;
            const uint32_t vz = qcz + a.radius + (lane / 3) - 1;
            const uint32_t v0 = (vz * a.vcy + vy) * a.vcx + qcx + a.radius - 1;
            rs = a.cell_off[v0];
            len = a.cell_off[v0 + 2] + a.cell_cnt[v0 + 2] - rs;
        }
        const uint32_t incl = wave_inclusive_sum(len);
        const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        const uint32_t rp = incl - len;
        const uint32_t ro = rs - rp;
        // the slot of this lane's vertex of the 64 that start at nb: one lookup
        // while they lie inside the run that the last ones ended in; lanes past
        // the end take slot 0.  (With one load site and no branch around the box
        // test: 567 -> 543 us for 256k particles, 286 -> 274 for 64k.)
        uint32_t jc = 0, run_off = 0, run_end = 0;
        auto slot_of = [&](uint32_t nb) {
            uint32_t at = run_off + nb + lane;
            if (nb + 64u > run_end) {
                uint32_t off = (uint32_t)__builtin_amdgcn_readlane((int)ro, (int)jc);
                for (uint32_t jj = jc + 1u; jj < 9u; ++jj) {
                    const uint32_t pj = (uint32_t)__builtin_amdgcn_readlane((int)rp, (int)jj);
                    if (pj >= nb + 64u) break;
                    if (nb + lane >= pj) off = (uint32_t)__builtin_amdgcn_readlane((int)ro, (int)jj);
                    jc = jj;
                }
                at = nb + lane < total ? off + nb + lane : 0u;
                run_off = (uint32_t)__builtin_amdgcn_readlane((int)ro, (int)jc);
                run_end = jc < 8u ? (uint32_t)__builtin_amdgcn_readlane((int)rp, (int)jc + 1) : total;
            }
            return at;
        };

        const float ox = __builtin_fmaf((float)qcx, a.sp.cell, a.sp.minx);
        const float oy = __builtin_fmaf((float)qcy, a.sp.cell, a.sp.miny);
        const float oz = __builtin_fmaf((float)qcz, a.sp.cell, a.sp.minz);
        float px = 0.f, py = 0.f, pz = 0.f;
        if (live) {
            const float4 p = a.sorted[i];
            px = p.x - ox; py = p.y - oy; pz = p.z - oz;
        }
        vb[lane] = 2.0f * px * inv_r2;
        vb[64 + lane] = 2.0f * py * inv_r2;
        vb[128 + lane] = 2.0f * pz * inv_r2;
        vb[192 + lane] = 1.0f - __builtin_fmaf(pz, pz, __builtin_fmaf(py, py, px * px)) * inv_r2;
        float bx0, bx1, by0, by1, bz0, bz1;
        wave_range(live, px, &bx0, &bx1);
        wave_range(live, py, &by0, &by1);
        wave_range(live, pz, &bz0, &bz1);
        wave_lds_sync();
        v4f gu = v4f{0.f, 0.f, 0.f, 0.f}, gx = gu;
        // (p', 1) of particle 16 wave + l%16, component l/16, from the LDS copy
        // of 2p'/R^2 (times R^2 / 2) and a 1 for the fourth
        const float bt = vb[64 * (lane >> 4) + 16u * wave + (lane & 15u)];
        const float bk = (lane >> 4) == 3u ? 1.0f : bt * (0.5f * a.radius_sq);
        uint32_t head = 0, fill = 0;
        float4 ncf = make_float4(0.f, 0.f, 0.f, 0.f), nvp = ncf;
        if (64u * wave < total) {
            const uint32_t at = slot_of(64u * wave);
            ncf = a.coef[at];
            nvp = a.vpos[at];
        }
        for (uint32_t base = 0; base < total; base += 256u) {
            const uint32_t nb = base + 64u * wave;
            float4 cf = ncf;
            float xx = nvp.x - ox, xy = nvp.y - oy, xz = nvp.z - oz;
            // (before the next loads, which take the same registers)
            asm volatile("" : "+v"(cf.x), "+v"(cf.y), "+v"(cf.z), "+v"(cf.w), "+v"(xx), "+v"(xy),
                         "+v"(xz));
            if (nb + 256u < total) {
                const uint32_t at = slot_of(nb + 256u);
                ncf = a.coef[at];
                nvp = a.vpos[at];
            }
            const float dx = xx - __builtin_amdgcn_fmed3f(xx, bx0, bx1);
            const float dy = xy - __builtin_amdgcn_fmed3f(xy, by0, by1);
            const float dz = xz - __builtin_amdgcn_fmed3f(xz, bz0, bz1);
            const bool keep =
                nb + lane < total && (cf.x != 0.0f || cf.y != 0.0f || cf.z != 0.0f || cf.w != 0.0f) &&
                __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx)) < cull_r2;
            const uint64_t m = __ballot(keep);
            if (lane == 0) count[wave] = (uint32_t)__popcll(m);
            __syncthreads();
            uint32_t before = 0, added = 0;
#pragma unroll
            for (uint32_t w = 0; w < kWaves; ++w) {
                const uint32_t n = count[w];
                before += w < wave ? n : 0u;
                added += n;
            }
            if (keep) {
                const uint32_t slot = (head + fill + before + mask_rank(m)) & (kAdjQueue - 1);
                q[slot] = xx;
                q[kAdjStride + slot] = xy;
                q[2 * kAdjStride + slot] = xz;
                q[kAdjU * kAdjStride + slot] = cf.x;
                q[(kAdjU + 1) * kAdjStride + slot] = cf.y;
                q[(kAdjU + 2) * kAdjStride + slot] = cf.z;
                q[(kAdjU + 3) * kAdjStride + slot] =
                    cf.w - __builtin_fmaf(cf.z, xz, __builtin_fmaf(cf.y, xy, cf.x * xx));
                q[kAdjQ * kAdjStride + slot] =
                    -(__builtin_fmaf(xz, xz, __builtin_fmaf(xy, xy, xx * xx)) * inv_r2);
            }
            fill += added;
            __syncthreads();
            for (; fill >= 64u; fill -= 64u) {
                if (mine) adj_tile(q + head, 64u, bt, bk, gu, gx);
                head = (head + 64u) & (kAdjQueue - 1);
            }
        }
        // the next chunk, fetched under the last batch; in the other one, as a
        // chunk without candidates has no barrier before this, and a wave may
        // still have to read this one's
        parity ^= 1u;
        if (wave == 0) {
            const uint32_t nx = items.next(0);
            if (lane == 0) next_chunk[parity] = nx;
        }
        if (fill) {
            // pad to 16 with entries that add 0: t < 0, u = 0 (head is a
            // multiple of 64, so the pad does not wrap)
            const uint32_t n = (fill + 15u) & ~15u;
            if (wave == 0 && lane >= fill && lane < n) {
#pragma unroll
                for (int rr = 0; rr < kAdjQ; ++rr)
                    if (rr != kAdjOne) q[rr * kAdjStride + head + lane] = 0.f;
                q[kAdjQ * kAdjStride + head + lane] = -1.0e30f;
            }
            __syncthreads();
            if (mine) adj_tile(q + head, n, bt, bk, gu, gx);
        }
        // the next chunk rewrites the ring from its start
        __syncthreads();
        // the four partial sums of each particle; the lanes of the wave's tile
        // write theirs
        v4f su = gu, sx = gx;
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
            float y = su[cc];
            y += adj_swz_xor<16>(y);
            su[cc] = y + __shfl_xor(y, 32, 64);
            float z = sx[cc];
            z += adj_swz_xor<16>(z);
            sx[cc] = z + __shfl_xor(z, 32, 64);
        }
        if (live && (lane >> 4) == wave) {
            const float s6 = 6.0f * inv_r2;
            const uint64_t o = 3ull * a.perm[i];
            a.g_pos[o + 0] = -__builtin_fmaf(s6, __builtin_fmaf(-sx[3], px, sx[0]), su[0]);
            a.g_pos[o + 1] = -__builtin_fmaf(s6, __builtin_fmaf(-sx[3], py, sx[1]), su[1]);
            a.g_pos[o + 2] = -__builtin_fmaf(s6, __builtin_fmaf(-sx[3], pz, sx[2]), su[2]);
        }
    }
}

}  // namespace

fsr_status mc_vertex_backward(fsr_context* ctx, const float* g_tri_pos, float* g_phi,
                              hipStream_t s) {
    const AdjointState& st = ctx->adj;
    if (!st.tri_capacity) return FSR_OK;  // no soup vertices were emitted
    McBackArgs a;
    a.band_index = st.bc.band_index;
    a.valid_idx = st.valid_idx;
    const uint64_t nwords = (uint64_t)row_words(st.sc.rx) * st.sc.ry * st.sc.rz;
    FSR_TRY(arena_typed(ctx, A_ADJ_TOUCH, nwords, &a.touched));
    FSR_TRY(fill_u32(a.touched, 0u, nwords, s));
    a.bits = st.bits;
    a.word_off = st.word_off;
    a.nverts = st.nverts;
    a.vert_off = st.vert_off;
    a.phi = st.phi;
    a.g_tri = g_tri_pos;
    a.g_phi = g_phi;
    a.st = st.stats;
    a.sc = st.sc;
    a.iso = st.iso;
    a.capacity = st.tri_capacity;
    a.cpu_flavor = st.cpu_flavor;
    FSR_TRY(arena_typed(ctx, A_ADJ_CORNER, 8ull * (st.tri_capacity / 3u) + 8u, &a.corner));
    const int blocks = persistent_blocks(ctx, kAdjThreads, 8, TUNE_MC);
    hipLaunchKernelGGL(k_mc_corner_terms, dim3(blocks), dim3(kAdjThreads), 0, s, a);
    FSR_LAUNCH_CHECK("k_mc_corner_terms");
    hipLaunchKernelGGL(k_mc_vertex_backward, dim3(blocks), dim3(kAdjThreads), 0, s, a);
    FSR_LAUNCH_CHECK("k_mc_vertex_backward");
    return FSR_OK;
}

fsr_status field_zb05_backward(fsr_context* ctx, const float* g_phi, float* g_pos,
                               hipStream_t s) {
    const AdjointState& st = ctx->adj;
    if (st.n == 0) return FSR_OK;
    FSR_TRY(fill_f32(g_pos, 0.0f, 3ull * st.n, s));
    const uint64_t V = (uint64_t)st.sc.rx * st.sc.ry * st.sc.rz;
    const uint32_t C = st.sp.rx * st.sp.ry * st.sp.rz;
    float4* coef;
    FSR_TRY(arena_typed(ctx, A_ADJ_COEF, 2 * V, &coef));  // (u, c), then vertex positions
    float4* vpos = coef + V;
    {
        const int blocks = persistent_blocks(ctx, kAdjThreads, 4, TUNE_MC);
        hipLaunchKernelGGL(k_field_coef, dim3(blocks), dim3(kAdjThreads), 0, s, st.cell_band,
                           st.saved, g_phi, st.stats, st.sc, coef, vpos);
        FSR_LAUNCH_CHECK("k_field_coef");
    }
    // particle chunks per hash cell
    const uint64_t max_chunks = (uint64_t)st.n / 64 + C + 1;
    uint32_t* aux;
    FSR_TRY(arena_typed(ctx, A_ADJ_AUX, C + max_chunks, &aux));
    uint32_t* chunk_off = aux;
    uint32_t* chunk_cell = aux + C;
    uint32_t* total = &st.counters->aux[8];
    uint32_t* next = st.counters->xcd_next;
    FSR_TRY(reset_xcd(st.counters, s));
    FSR_TRY(cell_chunk_list(ctx, st.ranges, nullptr, C, chunk_off, chunk_cell, max_chunks, total, s));
    FieldBackArgs a;
    a.sorted = st.sorted;
    a.ranges = st.ranges;
    a.perm = st.perm;
    a.chunk_cell = chunk_cell;
    a.chunk_off = chunk_off;
    a.num_chunks = total;
    a.next = next;
    a.cell_off = st.bc.cell_off;
    a.cell_cnt = st.bc.cell_cnt;
    a.coef = coef;
    a.vpos = vpos;
    a.sp = st.sp;
    a.vcx = st.bc.vcx;
    a.vcy = st.bc.vcy;
    a.radius = st.bc.radius;
    a.radius_sq = st.radius_sq;
    a.g_pos = g_pos;
    const int blocks = persistent_blocks(ctx, kAdjThreads, 6, TUNE_FIELD);
    hipLaunchKernelGGL(k_field_zb05_backward_mc, dim3(blocks), dim3(kAdjThreads), 0, s, a);
    FSR_LAUNCH_CHECK("k_field_zb05_backward_mc");
    return FSR_OK;
}

}  // namespace fsr
