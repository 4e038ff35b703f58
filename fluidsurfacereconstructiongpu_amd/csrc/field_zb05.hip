// ZB05 (Zhu & Bridson 2005) field on the surface band.
//
// Reference: updateScalarGridValuesCompacted -> updateScalarFieldValueZB05
// (ReconstructionCUDA.cu:308-324, :230-289) with kernelZB05
// (ReconstructionCUDA.cuh:262-268).  For a band vertex x in hash cell c, over
// the particles p of the clamped 3^3 cell block around c:
//   w(p) = (1 - |x - p|^2 / R^2)^3 for |x - p| < R, else 0
//   xbar = sum w p / sum w
//   phi(x) = |x - xbar| - r_p      if sum w > 0, otherwise phi is left as is
// (the caller's fill, 0).  The same field serves the Akinci12 method.
//
// MI355X mapping.  A wave owns a chunk of up to 64 band vertices of one hash
// cell, listed from the band mask in cell-major order (chunk_vertex), so all
// lanes share one candidate block: the 9 x-runs of the 3^3 block (x-adjacent cells are
// contiguous in the sorted particle array).  The wave stages candidates in LDS
// (one coalesced 16-byte load per lane, one candidate per lane) and evaluates
// them against the chunk's vertices in 16 x 16 tiles on the matrix cores:
//   t = 1 - |x - p|^2/R^2 = c_x + a_x . p' - q_p
// with p' = p - o and x' = x - o relative to the cell corner o, a = 2 x'/R^2,
// c_x = 1 - |x'|^2/R^2 and q_p = |p'|^2/R^2, is a K = 4 product (one
// v_mfma_f32_16x16x4_f32 per tile), w = max(t, 0)^3 takes 2 VALU ops per
// pair, and the sums of w and w p' are rank-1 updates of 4 x 4 blocks
// (v_mfma_f32_4x4x1_16b_f32), so a pair costs 2 VALU ops where the scalar
// form needs 11.  Coordinates relative to the cell keep the expansion well
// conditioned and make |x - xbar| free of the cancellation the
// absolute-coordinate sum has.  Candidates are staged in the reference's
// order (z, y, x cells, then range order); each vertex's sums are formed as
// four interleaved partial sums that are added at the end.  Work is
// distributed by ItemFetch: each XCD starts on its own contiguous eighth of the
// chunk list.  A smaller frame's workgroup shares each chunk (field_shared).
//
// Culling: a chunk's vertices are a compact slab of its cell (cell-major order
// is by ascending vertex id), so many block candidates lie farther than R
// from the chunk's bounding box.  At staging every candidate is tested against
// that box with R^2 (1 + 1e-4); survivors are compacted in order (ballot rank)
// into a 128-entry LDS queue that is drained 64 at a time.  A culled candidate
// is at least 1.00005 R from every vertex of the chunk, so its computed t is
// negative (the rounding of t is below 1e-5 there) and its weight exactly 0:
// culling leaves every sum unchanged.
#include <type_traits>

#include "chunk_list.hpp"
#include "common.hpp"

namespace fsr {

namespace {

constexpr int kFieldThreads = 256;

__device__ __forceinline__ int clampi(int v, int lo, int hi) {
    return v < lo ? lo : (v > hi ? hi : v);
}

// Lane exchange i <-> i ^ m within each half-wave (m < 32), with no address
// register: ds_swizzle in bit mode (and-mask 31, xor-mask m).
template <int M>
__device__ __forceinline__ float swz_xor(float v) {
    return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x1F | (M << 10)));
}

// Inclusive sum within each row of 16 lanes (DPP row shifts; lanes whose
// source lies before the row start add 0).
__device__ __forceinline__ uint32_t row16_inclusive_sum(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, true);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, true);
    return v;
}

// x, y, z of a sorted particle (one 12-byte load)
__device__ __forceinline__ float3 load_xyz(const float4* p) {
    return *reinterpret_cast<const float3*>(p);
}

// Division by a launch-constant divisor d with a multiply-high: the
// round-up method of Granlund and Montgomery (1994), exact for every 32-bit
// dividend.  m = floor(2^32 (2^l - d) / d) + 1 with l = ceil(log2 d).
struct FastDiv {
    uint32_t m, s1, s2;
};

FastDiv make_fast_div(uint32_t d) {
    const uint32_t l = d <= 1u ? 0u : 32u - (uint32_t)__builtin_clz(d - 1u);
    FastDiv f;
    f.m = (uint32_t)((((uint64_t)1 << l) - d) * ((uint64_t)1 << 32) / d + 1u);
    f.s1 = l < 1u ? l : 1u;
    f.s2 = l > 0u ? l - 1u : 0u;
    return f;
}

__device__ __forceinline__ uint32_t fast_div(uint32_t n, const FastDiv& f) {
    const uint32_t t = __umulhi(n, f.m);
    return (t + ((n - t) >> f.s1)) >> f.s2;
}

// Divisors of the vertex id: x extent and xy extent of the scalar grid.
struct VertexDiv {
    FastDiv rx, rxy;
};

typedef float v4f __attribute__((ext_vector_type(4)));

// LDS queue, structure of arrays: rows x', y', z', a row of ones and a row of -q
// (rows 0 to 4).  The rows start 16 floats more than a multiple of 64 apart, so
// the 16-entry slices that one matrix operand reads from the first four fall
// into distinct LDS banks.  One wave: a ring of kQueue entries; a workgroup
// that shares a chunk: kCoopQueue (63 waiting + 256 new, 256 being read).
constexpr int kQueue = 128;
constexpr int kRowStride = kQueue + 16;
constexpr int kRowX = 0, kRowY = 1, kRowZ = 2, kRowOne = 3, kRowQ = 4, kRows = 5;
constexpr int kCoopQueue = 512;
constexpr int kCoopStride = kCoopQueue + 16;
constexpr int kFieldWaves = kFieldThreads / 64;
constexpr uint32_t kOlt = 4;  // ordered <, as the compare builtin numbers it

// Sums of w and w p' for the NT 16-vertex tiles of one chunk over n staged
// candidates (n a multiple of 16), on the matrix cores.  Per 16 candidates and
// vertex tile:
//   1. one v_mfma_f32_16x16x4_f32 gives t = c_x + a_x . p' - q_p for the
//      16 x 16 pairs: A = (x', y', z', 1) of the candidates (rows),
//      B = (a_x, a_y, a_z, c_x) of the vertices (columns), C = -q_p;
//      lane l holds t of candidates 4(l/16)+r (r = 0..3) for vertex l%16;
//   2. w = max(t, 0)^3 (2 VALU ops per value: t^3 with a clamp to [0, 1]);
//   3. four v_mfma_f32_4x4x1_16b_f32 (one per r) accumulate, in each 4 x 4
//      block b = l/4, the outer product of (x', y', z', 1) of candidate
//      4(b/4)+r with the weights of vertices 4(b%4)..+3, so lane l collects
//      sum w p' (x, y, z) and sum w for vertex l%16 over the candidates
//      congruent to l/16 in each group of 16.
// The caller adds the four partial sums of a vertex (lanes l%16 + 16m).
template <int NT, int kStride>
__device__ __forceinline__ void accumulate(const float* __restrict__ rows, uint32_t n,
                                           const float (&b1)[NT], v4f (&acc)[NT]) {
    const uint32_t lane = __lane_id();
    const float* a1p = rows + (lane >> 4) * kStride + (lane & 15u);
    const float* a2p = rows + (lane & 3u) * kStride + 4u * (lane >> 4);
    const float* cqp = rows + 4 * kStride + 4u * (lane >> 4);
    for (uint32_t tb = 0; tb < n; tb += 16u) {
        const float a1 = a1p[tb];
        const float4 a2 = *reinterpret_cast<const float4*>(a2p + tb);
        const float4 cq = *reinterpret_cast<const float4*>(cqp + tb);
        const v4f c1 = v4f{cq.x, cq.y, cq.z, cq.w};
        // the tiles' t products back to back, then the weights, then the
        // rank-1 updates (independent across tiles, so no chain stalls)
        v4f w[NT];
#pragma unroll
        for (int T = 0; T < NT; ++T) w[T] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b1[T], c1, 0, 0, 0);
#pragma unroll
        for (int T = 0; T < NT; ++T) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                // max(t, 0)^3 as t^3 clamped to [0, 1] (the clamp bit of the
                // last multiply): t <= 1 up to rounding, and t^3 < 0 for t < 0
                const float t = w[T][r];
                w[T][r] = __builtin_amdgcn_fmed3f(t * t * t, 0.0f, 1.0f);
            }
        }
#pragma unroll
        for (int T = 0; T < NT; ++T) acc[T] = __builtin_amdgcn_mfma_f32_4x4x1f32(a2.x, w[T][0], acc[T], 0, 0, 0);
#pragma unroll
        for (int T = 0; T < NT; ++T) acc[T] = __builtin_amdgcn_mfma_f32_4x4x1f32(a2.y, w[T][1], acc[T], 0, 0, 0);
#pragma unroll
        for (int T = 0; T < NT; ++T) acc[T] = __builtin_amdgcn_mfma_f32_4x4x1f32(a2.z, w[T][2], acc[T], 0, 0, 0);
#pragma unroll
        for (int T = 0; T < NT; ++T) acc[T] = __builtin_amdgcn_mfma_f32_4x4x1f32(a2.w, w[T][3], acc[T], 0, 0, 0);
        // keep that order in the schedule: NT matrix ops, 8 NT VALU ops, 4 NT
        // matrix ops (VALU and matrix ops of one SIMD do not overlap, so
        // fewer switches between them pay)
        __builtin_amdgcn_sched_group_barrier(0x008, NT, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 8 * NT, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 4 * NT, 0);
    }
}

// What the lanes of a wave know about their chunk.
struct Chunk {
    uint32_t cnt, first, vid;    // vertices; first cell-major slot; this lane's vertex id
    bool has_vertex;
    float ox, oy, oz;            // cell corner: the local origin
    float lo[3], hi[3];          // box of the chunk's vertices
    uint32_t nrows, total;       // candidate rows (x-runs) and candidates
    uint32_t rp, ro;             // lane j < nrows: first candidate index of row j, and
                                 // the offset from candidate index to sorted index in it
    uint32_t jc;

    // Row lookup: jc is a row whose first candidate index is at most the first
    // index nb of the round being located (rows only grow with the index).  The
    // rows that start before the round's end are visited with wave-uniform reads
    // of rp and ro; a lane takes the last one that starts at or before its index
    // gg.  Empty rows share their first index with the next row, which is
    // visited after them.
    __device__ __forceinline__ uint32_t row_offset(uint32_t nb, uint32_t gg) {
        uint32_t off = (uint32_t)__builtin_amdgcn_readlane((int)ro, (int)jc);
        for (uint32_t jj = jc + 1u; jj < nrows; ++jj) {
            const uint32_t pj = (uint32_t)__builtin_amdgcn_readlane((int)rp, (int)jj);
            if (pj >= nb + 64u) break;
            if (gg >= pj) off = (uint32_t)__builtin_amdgcn_readlane((int)ro, (int)jj);
            jc = jj;
        }
        return off;
    }
};

// Loads chunk ch: its vertices (listed through `scratch`, 64 words of LDS), their
// operands into vt (rows of 64: x', y', z', a_x, a_y, a_z, c_x), their box, and
// the candidate rows.
__device__ __forceinline__ Chunk load_chunk(const FieldArgs& a, const BandCompactOut& bc,
                                            const VertexDiv& vd, uint32_t ch, float inv_r2,
                                            float* __restrict__ vt, uint32_t* scratch) {
    const uint32_t lane = __lane_id();
    const int r = bc.radius;
    Chunk c;
    const uint32_t v = bc.chunk_cell[ch];
    const int cx = (int)(v % bc.vcx) - r;
    const int cy = (int)((v / bc.vcx) % bc.vcy) - r;
    const int cz = (int)(v / (bc.vcx * bc.vcy)) - r;
    const uint32_t k = ch - bc.chunk_off[v];
    const uint32_t ccount = bc.cell_cnt[v];
    c.first = bc.cell_off[v] + 64u * k;
    c.cnt = min(64u, ccount - 64u * k);
    // the chunk's vertex ids (before the candidate rows, whose registers live
    // through the staging loop)
    c.vid = chunk_vertex(bc, a.sc.rx, a.sc.ry, v, k, c.cnt, scratch);

    // candidate rows of the clamped 3^3 block
    const int x0 = clampi(cx - 1, 0, a.sp.rx - 1), x1 = clampi(cx + 1, 0, a.sp.rx - 1);
    const int y0 = clampi(cy - 1, 0, a.sp.ry - 1), y1 = clampi(cy + 1, 0, a.sp.ry - 1);
    const int z0 = clampi(cz - 1, 0, a.sp.rz - 1), z1 = clampi(cz + 1, 0, a.sp.rz - 1);
    const int ny = y1 - y0 + 1;
    c.nrows = (uint32_t)(ny * (z1 - z0 + 1));
    uint32_t len = 0, rs = 0;
    if (lane < c.nrows) {
        const int yy = y0 + (int)lane % ny, zz = z0 + (int)lane / ny;
        const uint32_t rowc = ((uint32_t)zz * a.sp.ry + yy) * a.sp.rx;
        // the row's 3 cells as clamped offsets (a repeated edge cell leaves
        // the run unchanged), loaded together
        fsr_index_range rg[3];
#pragma unroll
        for (int d = 0; d < 3; ++d) rg[d] = a.ranges[rowc + clampi(cx - 1 + d, x0, x1)];
        uint32_t s = 0xFFFFFFFFu, e = 0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            if (rg[d].start != 0xFFFFFFFFu) {
                if (s == 0xFFFFFFFFu) s = rg[d].start;
                e = rg[d].end;
            }
        }
        if (s != 0xFFFFFFFFu) { rs = s; len = e - s; }
    }
    // nrows <= 9: the prefix over the first 16 lanes is the whole prefix
    const uint32_t incl = row16_inclusive_sum(len);
    c.total = (uint32_t)__builtin_amdgcn_readlane((int)incl, 15);
    c.rp = incl - len;
    c.ro = rs - c.rp;
    c.jc = 0;

    c.ox = __builtin_fmaf((float)cx, a.sp.cell, a.sp.minx);
    c.oy = __builtin_fmaf((float)cy, a.sp.cell, a.sp.miny);
    c.oz = __builtin_fmaf((float)cz, a.sp.cell, a.sp.minz);
    float vx = 0.f, vy = 0.f, vz = 0.f;
    // lanes with a vertex (an id past the grid would mean an empty slot)
    c.has_vertex = lane < c.cnt && c.vid < a.sc.rx * a.sc.ry * a.sc.rz;
    if (c.has_vertex) {
        const uint32_t iz = fast_div(c.vid, vd.rxy);
        const uint32_t rem = c.vid - iz * (a.sc.rx * a.sc.ry);
        const uint32_t iy = fast_div(rem, vd.rx);
        const uint32_t ix = rem - iy * a.sc.rx;
        vx = vertex_coord(ix, a.sc.minx, a.sc.cell) - c.ox;
        vy = vertex_coord(iy, a.sc.miny, a.sc.cell) - c.oy;
        vz = vertex_coord(iz, a.sc.minz, a.sc.cell) - c.oz;
    }
    vt[lane] = vx;
    vt[64 + lane] = vy;
    vt[128 + lane] = vz;
    vt[192 + lane] = 2.0f * vx * inv_r2;
    vt[256 + lane] = 2.0f * vy * inv_r2;
    vt[320 + lane] = 2.0f * vz * inv_r2;
    vt[384 + lane] = 1.0f - __builtin_fmaf(vz, vz, __builtin_fmaf(vy, vy, vx * vx)) * inv_r2;
    wave_range(c.has_vertex, vx, &c.lo[0], &c.hi[0]);
    wave_range(c.has_vertex, vy, &c.lo[1], &c.hi[1]);
    wave_range(c.has_vertex, vz, &c.lo[2], &c.hi[2]);
    return c;
}

// The field at this lane's vertex from its sums (sum w p', sum w).
__device__ __forceinline__ void store_vertex(const FieldArgs& a, const Chunk& c, const v4f& s4,
                                             const float* __restrict__ vt) {
    const uint32_t lane = __lane_id();
    float4 keep_out = make_float4(0.f, 0.f, 0.f, 0.f);
    const float sw = s4[3];
    if (sw > 0.0f) {
        const float inv = 1.0f / sw;
        const float dx = vt[lane] - s4[0] * inv;
        const float dy = vt[64 + lane] - s4[1] * inv;
        const float dz = vt[128 + lane] - s4[2] * inv;
        a.phi[c.vid] = __builtin_sqrtf(__builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx))) -
                       a.particle_radius;
        keep_out = make_float4(dx, dy, dz, sw);
    }
    // for the adjoint: x - xbar and sum w, and the vertex, at its cell-major slot
    if (a.saved) {
        a.saved[c.first + lane] = keep_out;
        a.cell_band[c.first + lane] = c.vid;
    }
}

// One LDS block per wave, so every per-lane LDS address is one base register
// plus an immediate offset; or one per workgroup, in the shared form.
struct WaveLds {
    float queue[kRows * kRowStride];
    // per lane: x', y', z' of its vertex (for the end) and (a_x, a_y, a_z, c_x)
    float vtx[7][64];
};
struct GroupLds {
    float queue[kRows * kCoopStride];
    float vtx[kFieldWaves][7][64];
    uint32_t count[kFieldWaves];
    uint32_t next_chunk[2];  // by the chunk's parity: see the loop's end
};

// The shared form: the 4 waves of a workgroup treat a chunk together, for frames
// with few chunks (see coop_limit).  Each wave stages a quarter of a
// 256-candidate round into one ring, in candidate order, and evaluates one of
// the chunk's 16-vertex tiles: the candidates, their order and every tile's
// operations are those of the wave form, so the field is the same bits.  Per
// round two barriers: counts (which also says that the previous batches are
// evaluated), and entries.
__device__ __forceinline__ void field_shared(const FieldArgs& a, const BandCompactOut& bc,
                                             const VertexDiv& vd, GroupLds& L, uint32_t num_chunks,
                                             float inv_r2, float cull_r2, FetchState* fetch) {
    const uint32_t lane = __lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    float* q = L.queue;
    float* vt = &L.vtx[wave][0][0];
    for (uint32_t t = threadIdx.x; t < (uint32_t)kCoopQueue; t += kFieldThreads)
        q[kRowOne * kCoopStride + t] = 1.0f;
    ItemFetch<1, true> items(a.counters->xcd_field, num_chunks, fetch);
    if (wave == 0) {
        const uint32_t nx = items.next(0);
        if (lane == 0) L.next_chunk[0] = nx;
    }
    __syncthreads();
    // workgroup-uniform
    uint32_t parity = 0;
    for (uint32_t ch = L.next_chunk[0]; ch < num_chunks; ch = L.next_chunk[parity]) {
        Chunk c = load_chunk(a, bc, vd, ch, inv_r2, vt, reinterpret_cast<uint32_t*>(vt));
        wave_lds_sync();
        const uint32_t nt = (c.cnt + 15u) >> 4;
        const bool mine = wave < nt;
        float b1[1] = {vt[192 + 64 * (lane >> 4) + 16u * wave + (lane & 15u)]};
        v4f acc[1] = {v4f{0.f, 0.f, 0.f, 0.f}};
        uint32_t head = 0, fill = 0, n_kept = 0, n_steps = 0;
        float3 next = make_float3(0.f, 0.f, 0.f);
        {
            const uint32_t g = 64u * wave + lane;
            const uint32_t off = c.row_offset(64u * wave, g);
            if (g < c.total) next = load_xyz(a.sorted + (off + g));
        }
        for (uint32_t base = 0; base < c.total; base += 256u) {
            const uint32_t g = base + 64u * wave + lane;
            const float3 p = next;
            if (base + 256u < c.total) {
                const uint32_t off = c.row_offset(base + 256u + 64u * wave, g + 256u);
                if (g + 256u < c.total) next = load_xyz(a.sorted + (off + g + 256u));
            }
            const float px = p.x - c.ox, py = p.y - c.oy, pz = p.z - c.oz;
            const float dx = px - __builtin_amdgcn_fmed3f(px, c.lo[0], c.hi[0]);
            const float dy = py - __builtin_amdgcn_fmed3f(py, c.lo[1], c.hi[1]);
            const float dz = pz - __builtin_amdgcn_fmed3f(pz, c.lo[2], c.hi[2]);
            const bool keep =
                g < c.total &&
                __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx)) < cull_r2;
            const uint64_t m = __ballot(keep);
            if (lane == 0) L.count[wave] = (uint32_t)__popcll(m);
            __syncthreads();
            uint32_t before = 0, added = 0;
#pragma unroll
            for (uint32_t w = 0; w < (uint32_t)kFieldWaves; ++w) {
                const uint32_t n = L.count[w];
                before += w < wave ? n : 0u;
                added += n;
            }
            if (keep) {
                const uint32_t slot = (head + fill + before + mask_rank(m)) & (kCoopQueue - 1);
                q[kRowX * kCoopStride + slot] = px;
                q[kRowY * kCoopStride + slot] = py;
                q[kRowZ * kCoopStride + slot] = pz;
                q[kRowQ * kCoopStride + slot] =
                    -(__builtin_fmaf(pz, pz, __builtin_fmaf(py, py, px * px)) * inv_r2);
            }
            fill += added;
            n_kept += added;
            __syncthreads();
            for (; fill >= 64u; fill -= 64u) {
                if (mine) accumulate<1, kCoopStride>(q + head, 64u, b1, acc);
                head = (head + 64u) & (kCoopQueue - 1);
                n_steps += 4u * nt;
            }
        }
        // the next chunk, fetched under the last batch; in the other one, as a
        // chunk without candidates has no barrier before this, and a wave may
        // still have to read this one's
        parity ^= 1u;
        if (wave == 0) {
            const uint32_t nx = items.next(0);
            if (lane == 0) L.next_chunk[parity] = nx;
        }
        if (fill) {
            // pad to a multiple of 16 with entries of weight 0 (t < 0 for
            // every vertex); head is a multiple of 64, so the pad does not wrap
            const uint32_t n = (fill + 15u) & ~15u;
            if (wave == 0 && lane >= fill && lane < n) {
                q[kRowX * kCoopStride + head + lane] = 0.f;
                q[kRowY * kCoopStride + head + lane] = 0.f;
                q[kRowZ * kCoopStride + head + lane] = 0.f;
                q[kRowQ * kCoopStride + head + lane] = -1.0e30f;
            }
            n_steps += (n >> 4) * nt;
            __syncthreads();
            if (mine) accumulate<1, kCoopStride>(q + head, n, b1, acc);
        }
        // the next chunk rewrites the ring from its start
        __syncthreads();
        // the four partial sums of each vertex; the lanes of the wave's tile
        // write theirs
        v4f s4 = acc[0];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            float x = s4[d];
            x += swz_xor<16>(x);
            s4[d] = x + __shfl_xor(x, 32, 64);
        }
        if (c.has_vertex && (lane >> 4) == wave) store_vertex(a, c, s4, vt);
        if (threadIdx.x == 0) {
            uint32_t* w = a.work + 3u * ch;
            w[0] = c.total;
            w[1] = n_kept;
            w[2] = n_steps;
        }
        // vt holds the vertices until here
        wave_lds_sync();
    }
}

// kShared: the build for smaller frames, whose chunks may be few (their count is
// known on the device only): it has the shared form, taken at up to coop_max
// chunks, and the fetch for short lists.
template <bool kShared>
__global__ __launch_bounds__(kFieldThreads, 6) void k_field_zb05(FieldArgs a, BandCompactOut bc,
                                                              VertexDiv vd, uint32_t coop_max) {
    __shared__ __align__(16) union {
        WaveLds wave[kFieldWaves];
        GroupLds group;
    } lds;
    __shared__ FetchState fetch;
    fetch_init(&fetch);
    const uint32_t lane = __lane_id();
    const uint32_t wave = threadIdx.x >> 6;
    const uint32_t num_chunks = a.counters->num_chunks;
    const float inv_r2 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(1.0f / a.radius_sq)));
    const float cull_r2 = a.radius_sq * 1.0001f;
    // the work record ends with a marker after the last chunk
    if (blockIdx.x == 0 && threadIdx.x == 0) a.work[3u * num_chunks] = 0xFFFFFFFFu;
    if (kShared && num_chunks <= coop_max) {
        field_shared(a, bc, vd, lds.group, num_chunks, inv_r2, cull_r2, &fetch);
        return;
    }
    float* q = lds.wave[wave].queue;
    float* vt = &lds.wave[wave].vtx[0][0];
    q[kRowOne * kRowStride + lane] = 1.0f;
    q[kRowOne * kRowStride + 64 + lane] = 1.0f;

    ItemFetch<kFieldWaves, kShared> items(a.counters->xcd_field, num_chunks, &fetch);
    for (;;) {
        const uint32_t ch = items.next(wave);
        if (ch >= num_chunks) break;
        Chunk c = load_chunk(a, bc, vd, ch, inv_r2, vt, reinterpret_cast<uint32_t*>(q));
        wave_lds_sync();
        const int nt = (int)((c.cnt + 15u) >> 4);
        // The rest of the chunk, compiled once per tile count NT, so that the
        // accumulators keep fixed registers across the staging loop.
        auto run = [&](auto ntc) {
            constexpr int NT = decltype(ntc)::value;
            // matrix operand of the vertex tiles: lane l carries component l/16
            // of (a_x, a_y, a_z, c_x) of vertex 16T + l%16
            float b1[NT];
            v4f acc[NT];
            const float* bsrc = vt + 192 + 64 * (lane >> 4) + (lane & 15u);
#pragma unroll
            for (int T = 0; T < NT; ++T) {
                b1[T] = bsrc[16 * T];
                acc[T] = v4f{0.f, 0.f, 0.f, 0.f};
            }
            // the queue is a ring of kQueue entries; entries [head, head + fill)
            // wait for evaluation, and head is 0 or 64
            uint32_t head = 0, fill = 0;
            // work of the chunk: candidates kept by the box test, tile steps
            uint32_t n_kept = 0, n_steps = 0;
            // this lane's candidate of the next round is loaded one round ahead,
            // so the load overlaps the culling and the accumulation of the
            // current one
            // Two rounds of three lie inside one x-run, whose lanes need no row of
            // their own; that, one load site, and lane masks by compare and scalar
            // operations instead of branches took a round from some 45 VALU
            // operations to 30 (field of a 1M dam break 278 -> 268 us, 2M 419 -> 400,
            // Akinci12 675 -> 643; with the box's upper corner in vector registers,
            // 3 operations fewer, no faster).
            float3 next = make_float3(0.f, 0.f, 0.f);
            uint32_t row_off = 0, row_end = 0;  // of the row that the last round ended in
            auto load_round = [&](uint32_t nb) {
                uint32_t at = row_off + nb + lane;
                if (nb + 64u > row_end) {
                    // not inside one row; lanes past the end read particle 0
                    const uint32_t off = c.row_offset(nb, nb + lane);
                    at = nb + lane < c.total ? off + nb + lane : 0u;
                    row_off = (uint32_t)__builtin_amdgcn_readlane((int)c.ro, (int)c.jc);
                    row_end = c.jc + 1u < c.nrows
                                  ? (uint32_t)__builtin_amdgcn_readlane((int)c.rp, (int)c.jc + 1)
                                  : c.total;
                }
                next = load_xyz(a.sorted + at);
            };
            if (c.total) load_round(0u);
            for (uint32_t base = 0; base < c.total; base += 64u) {
                float px = next.x - c.ox, py = next.y - c.oy, pz = next.z - c.oz;
                // (before the next load: it takes the same registers, and the wait
                // for this one must not cover it)
                asm volatile("" : "+v"(px), "+v"(py), "+v"(pz));
                if (base + 64u < c.total) load_round(base + 64u);
                // distance to the box per axis: p - clamp(p, lo, hi), whose
                // square equals that of max(lo - p, p - hi, 0) exactly
                const float dx = px - __builtin_amdgcn_fmed3f(px, c.lo[0], c.hi[0]);
                const float dy = py - __builtin_amdgcn_fmed3f(py, c.lo[1], c.hi[1]);
                const float dz = pz - __builtin_amdgcn_fmed3f(pz, c.lo[2], c.hi[2]);
                const float d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dy, dy, dx * dx));
                // lane mask straight from the compare, less the last round's lanes
                // past the end
                const uint32_t left = c.total - base;
                const uint64_t m = __builtin_amdgcn_fcmpf(d2, cull_r2, kOlt) &
                                   (left < 64u ? (1ull << left) - 1ull : ~0ull);
                if (__builtin_amdgcn_inverse_ballot_w64(m)) {
                    const uint32_t slot = (head + fill + mask_rank(m)) & (kQueue - 1);
                    q[kRowX * kRowStride + slot] = px;
                    q[kRowY * kRowStride + slot] = py;
                    q[kRowZ * kRowStride + slot] = pz;
                    q[kRowQ * kRowStride + slot] =
                        -(__builtin_fmaf(pz, pz, __builtin_fmaf(py, py, px * px)) * inv_r2);
                }
                fill += (uint32_t)__popcll(m);
                n_kept += (uint32_t)__popcll(m);
                if (fill >= 64u) {
                    n_steps += 4u * NT;
                    wave_lds_sync();
                    accumulate<NT, kRowStride>(q + head, 64u, b1, acc);
                    wave_lds_sync();
                    head ^= 64u;
                    fill -= 64u;
                }
            }
            if (fill) {
                // pad to a multiple of 16 with entries of weight 0 (t < 0 for
                // every vertex); head + 64 <= kQueue, so the pad does not wrap
                const uint32_t n = (fill + 15u) & ~15u;
                if (lane >= fill && lane < n) {
                    q[kRowX * kRowStride + head + lane] = 0.f;
                    q[kRowY * kRowStride + head + lane] = 0.f;
                    q[kRowZ * kRowStride + head + lane] = 0.f;
                    q[kRowQ * kRowStride + head + lane] = -1.0e30f;
                }
                n_steps += (n >> 4) * NT;
                wave_lds_sync();
                accumulate<NT, kRowStride>(q + head, n, b1, acc);
                wave_lds_sync();
            }
            // add the four partial sums of each vertex; lane l then holds the
            // sums of vertex 16T + l%16 in acc[T]
            v4f s4 = acc[0];
            const uint32_t my = lane >> 4;
#pragma unroll
            for (int T = 0; T < NT; ++T) {
#pragma unroll
                for (int d = 0; d < 4; ++d) {
                    float x = acc[T][d];
                    x += swz_xor<16>(x);
                    x += __shfl_xor(x, 32, 64);
                    acc[T][d] = x;
                }
                if (my == (uint32_t)T) s4 = acc[T];
            }
            if (c.has_vertex) store_vertex(a, c, s4, vt);
            if (lane == 0) {
                uint32_t* w = a.work + 3u * ch;
                w[0] = c.total;
                w[1] = n_kept;
                w[2] = n_steps;
            }
        };
        switch (nt) {
            case 1: run(std::integral_constant<int, 1>{}); break;
            case 2: run(std::integral_constant<int, 2>{}); break;
            case 3: run(std::integral_constant<int, 3>{}); break;
            default: run(std::integral_constant<int, 4>{}); break;
        }
    }
}

}  // namespace

fsr_status field_zb05(fsr_context* ctx, const FieldArgs& a, hipStream_t s) {
    // a.counters was cleared when the frame (or the stage call) began, and no
    // other kernel fetches through xcd_field
    // one workgroup per resident slot: 6 per CU (6 waves per SIMD); workgroups
    // beyond the resident ones start late and upset the per-XCD fetch order
    const int blocks = persistent_blocks(ctx, kFieldThreads, 6, TUNE_FIELD);
    FieldArgs fa = a;
    FSR_TRY(arena_typed(ctx, A_FIELD_WORK, 3ull * a.bc->max_chunks + 3, &fa.work));
    VertexDiv vd;
    vd.rx = make_fast_div(a.sc.rx);
    vd.rxy = make_fast_div(a.sc.rx * a.sc.ry);
    auto kernel = few_chunks(ctx, a.num_particles) ? k_field_zb05<true> : k_field_zb05<false>;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kFieldThreads), 0, s, fa, *a.bc, vd,
                       coop_limit(ctx, blocks));
    FSR_LAUNCH_CHECK("k_field_zb05");
    return FSR_OK;
}

}  // namespace fsr
