// The vertices of a field kernel's chunk, listed from the band mask.
#pragma once
#include "common.hpp"

namespace fsr {

// The vertex ids of chunk k of virtual cell v, listed from the band mask in
// the cell-major order (layer z, row y, then x ascending): lane l < cnt receives
// the (64 k + l)-th band vertex of the cell.  The cell's layers (slabs) are consecutive in the slab counts;
// 64 layers at a time, those that overlap [64 k, 64 k + 64) are expanded word
// by word, each lane taking one (layer, row, word) of them, and the wanted
// ranks go to `scratch` (64 LDS words of the wave).
__device__ __forceinline__ uint32_t chunk_vertex(const BandCompactOut& bc, uint32_t rx, uint32_t ry, uint32_t v,
                                 uint32_t k, uint32_t cnt, uint32_t* scratch) {
    const uint32_t lane = __lane_id();
    const uint32_t cxv = v % bc.vcx, cyv = (v / bc.vcx) % bc.vcy, czv = v / (bc.vcx * bc.vcy);
    const uint32_t* lo_x = bc.axis;
    const uint32_t* lo_y = lo_x + 2u * bc.vcx;
    const uint32_t* lo_z = lo_y + 2u * bc.vcy;
    const uint32_t zlo = lo_z[czv], nz = lo_z[bc.vcz + czv] - zlo;
    const uint64_t sbase = (uint64_t)bc.vcx * bc.vcy * zlo + ((uint64_t)cyv * bc.vcx + cxv) * nz;
    const uint32_t ylo = lo_y[cyv], ny = lo_y[bc.vcy + cyv] - ylo;
    const uint32_t xlo = lo_x[cxv], xhi = lo_x[bc.vcx + cxv];
    const uint32_t w0 = xlo >> 5, nw = ((xhi + 31u) >> 5) - w0;
    const uint32_t per = ny * nw;
    const uint32_t lo = 64u * k, hi = lo + 64u;
    // every slot starts empty, so a slot the expansion does not fill reads as
    // "no vertex" rather than as a stale id
    scratch[lane] = 0xFFFFFFFFu;
    wave_lds_sync();
    uint32_t before = 0;  // band vertices of the cell's layers before the group
    for (uint32_t g0 = 0; g0 < nz && before < hi; g0 += 64u) {
        const uint32_t sn = g0 + lane < nz ? bc.slab[sbase + g0 + lane] : 0u;
        const uint32_t sincl = before + wave_inclusive_sum(sn);
        const uint32_t sexcl = sincl - sn;
        const uint64_t hit = __ballot(g0 + lane < nz && sn != 0u && sexcl < hi && sincl > lo);
        if (hit) {
            // the overlapping layers of the group are consecutive: j0 .. j1
            const uint32_t j0 = (uint32_t)__builtin_ctzll(hit);
            const uint32_t j1 = 63u - (uint32_t)__builtin_clzll(hit);
            const uint32_t items = (j1 - j0 + 1u) * per;
            uint32_t rank0 = (uint32_t)__builtin_amdgcn_readlane((int)sexcl, (int)j0);
            for (uint32_t i0 = 0; i0 < items; i0 += 64u) {
                const uint32_t i = i0 + lane;
                uint32_t word = 0, base = 0;
                if (i < items) {
                    const uint32_t js = g0 + j0 + i / per, rem = i % per;
                    const uint32_t y = ylo + rem / nw, w = w0 + rem % nw;
                    const uint64_t row = (uint64_t)(zlo + js) * ry + y;
                    word = clip_word(bc.bits[row * bc.wx + w], w, xlo, xhi);
                    base = (uint32_t)(row * rx) + w * 32u;
                }
                const uint32_t c = (uint32_t)__popc(word);
                const uint32_t incl = wave_inclusive_sum(c);
                uint32_t r = rank0 + incl - c;
                while (word) {
                    if (r >= lo && r < hi) scratch[r - lo] = base + (uint32_t)__builtin_ctz(word);
                    ++r;
                    word &= word - 1u;
                }
                rank0 += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
            }
        }
        before = (uint32_t)__builtin_amdgcn_readlane((int)sincl, 63);
    }
    wave_lds_sync();
    const uint32_t id = lane < cnt ? scratch[lane] : 0xFFFFFFFFu;
    wave_lds_sync();
    return id;
}

}  // namespace fsr
