// oh_iq2.h - the IQ2_XXS codebook and sign masks on the device.
#pragma once
#include "oh_common.h"
#include "../../include/ornith_iq2xxs_grid.h"

static __constant__ uint64_t k_iq2_grid[256] = { ORNITH_IQ2XXS_GRID_VALUES };

namespace {

// The 128 sign patterns of IQ2_XXS as byte masks (the eighth sign is the
// parity of the seven stored ones): entry s7 = {m_lo, m_hi, m_lo & 0x01..,
// m_hi & 0x01..}, m byte j = 0xff where sign j is negative, so that
// (g ^ m) + (m & 0x01..) negates exactly those bytes of a grid entry g.
OH_DEV void iq2_sign_table(uint4 *stab) {
    const int tid = tid_x();
    if (tid < 128) {
        const uint32_t sg = (uint32_t)tid | ((__popc((uint32_t)tid) & 1u) << 7);
        uint32_t m0 = 0, m1 = 0;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            m0 |= ((sg >> j) & 1u) * (0xffu << (8 * j));
            m1 |= ((sg >> (j + 4)) & 1u) * (0xffu << (8 * j));
        }
        stab[tid] = make_uint4(m0, m1, m0 & 0x01010101u, m1 & 0x01010101u);
    }
}

} // namespace
