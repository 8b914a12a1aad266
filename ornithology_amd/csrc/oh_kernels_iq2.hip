// oh_kernels_iq2.hip - the translation unit of the prompt's IQ2_XXS experts:
// the f32 fallback rows (src/ornith_quant.c:660-680 decode, then ot_dot's
// strictly sequential f32 accumulation, src/ornith_rforward.c:119-133) for
// the (token, expert) slots of a chunk, grouped by expert.
#include "oh_dpp.h"
#include "oh_iq2.h"
#include "oh_launch.h"

namespace {

constexpr int kCodeStride = 80;                  // a row's 64 code bytes in LDS, spread over the banks
constexpr int kListThreads = 1024;               // one per expert at most (ne <= 1024)

// A row's terms (db * +-g) * x are added in element order, so a row is one
// chain; a lane walks one row (of gate and of up, PAIR) for up to NT slots of
// its expert at once: the weight db * +-g is formed once, and each slot costs
// its product and its sum. The slots' activations sit 2 elements per lane in
// each 16-lane row and enter the products as DPP broadcasts; a row's code bytes
// go through LDS a super-block at a time, so that each cache line is fetched
// once. Vector instructions bound it: 2 per weight and slot, which the order
// of the sums asks for, and 3.3 per weight; 94% of the issue slots are taken.
// 500 tokens, 512 experts, top 10, 4096 -> 1024 -> 4096 (uneven picks): gate, up
// and silu(gate) * up 3.26 ms, down 1.46 ms, against 8.45 ms for both with a
// lane per (slot, row).
template <int NT, bool PAIR>
OH_DEV void iq2_cols(const oh_iq2rows &a, const uint64_t *grid, const uint4 *stab, uint8_t *codes, int64_t row_bi,
                     int row, const int32_t *slots, int n) {
    constexpr int NR = PAIR ? 2 : 1;
    const int nb = a.in / 256, lane = lane_id();
    const float *xp[NT];
    int slot[NT];
#pragma unroll
    for (int c = 0; c < NT; c++) {
        slot[c] = __builtin_amdgcn_readfirstlane(ldg(slots + (c < n ? c : n - 1)));
        xp[c] = a.x + (size_t)(slot[c] / a.adiv) * a.xstride;
    }
    // a row's next super-block (64 code bytes, one whole line half at a time)
    // is requested while the current one, in LDS, is walked
    uint4 pre[NR][4];
    uint32_t dpre[NR];
    auto fetch = [&](int b) {
#pragma unroll
        for (int r = 0; r < NR; r++) {
            const uint4 *q = (const uint4 *)((r ? a.A2 : a.A) + (row_bi + b) * 64);
#pragma unroll
            for (int k = 0; k < 4; k++) pre[r][k] = ldg(q + k);
            dpre[r] = ldg((const uint16_t *)((r ? a.C2 : a.C) + (row_bi + b) * 2));
        }
    };
    float acc[NR][NT] = {}, dcur[NR];
    float2 xn[NT];
    const unsigned xo = 8u * (unsigned)(lane & 15);
    auto fetch_x = [&](int sb) {
#pragma unroll
        for (int c = 0; c < NT; c++) xn[c] = ldo<float2>(xp[c], xo + 128u * (unsigned)sb);
    };
    fetch(0);
    fetch_x(0);
    for (int sb = 0; sb < 8 * nb; sb++) {
        if (sb % 8 == 0) {
#pragma unroll
            for (int r = 0; r < NR; r++) {
#pragma unroll
                for (int k = 0; k < 4; k++) *(uint4 *)(codes + (r * 64 + lane) * kCodeStride + 16 * k) = pre[r][k];
                dcur[r] = h2f((uint16_t)dpre[r]);
            }
            fetch(sb / 8 + 1 < nb ? sb / 8 + 1 : nb - 1);
        }
        float2 x[NT];
        uint2 w[NR];
        float db[NR];
#pragma unroll
        for (int c = 0; c < NT; c++) x[c] = xn[c];
#pragma unroll
        for (int r = 0; r < NR; r++) {
            w[r] = *(const uint2 *)(codes + (r * 64 + lane) * kCodeStride + 8 * (sb % 8));
            db[r] = dcur[r] * (0.5f + (float)(w[r].y >> 28)) * 0.25f;
        }
        fetch_x(sb + 1 < 8 * nb ? sb + 1 : sb);
        // the sub-block's four codebook entries with their signs
        uint32_t gs[NR][8];
#pragma unroll
        for (int r = 0; r < NR; r++)
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const uint64_t gv = grid[(w[r].x >> (8 * k)) & 0xffu];
                const uint4 sm = stab[(w[r].y >> (7 * k)) & 127u];
                gs[r][2 * k] = ((uint32_t)gv ^ sm.x) + sm.z;
                gs[r][2 * k + 1] = ((uint32_t)(gv >> 32) ^ sm.y) + sm.w;
            }
        auto weight = [&](int r, int e) { return db[r] * (float)(int8_t)(gs[r][e / 4] >> (8 * (e % 4))); };
        float wt[NR], t[NR][NT];
#pragma unroll
        for (int r = 0; r < NR; r++) wt[r] = weight(r, 0);
        static_for<32>([&](auto e_) {
            constexpr int e = e_;
            order();
#pragma unroll
            for (int r = 0; r < NR; r++)
#pragma unroll
                for (int c = 0; c < NT; c++) t[r][c] = row_lane<e / 2>(e % 2 ? x[c].y : x[c].x) * wt[r];
            order();
            if constexpr (e + 1 < 32) {
#pragma unroll
                for (int r = 0; r < NR; r++) wt[r] = weight(r, e + 1);
            }
#pragma unroll
            for (int r = 0; r < NR; r++)
#pragma unroll
                for (int c = 0; c < NT; c++) acc[r][c] += t[r][c];
        });
    }
    if (row >= a.rows) return;
#pragma unroll
    for (int c = 0; c < NT; c++) {
        if (c >= n) break;
        const float v = PAIR ? ref_silu(acc[0][c]) * acc[NR - 1][c] : acc[0][c];
        stg(a.y + (size_t)slot[c] * a.ystride + row, v);
    }
}

// grid (rows / 256, items): up to cols (1, 2, 4 or 8) slots of one expert (three
// or more as four, five or more as eight: the columns that only repeat one cost
// less than forming the weights again). A router's picks are uneven, so an
// expert's pieces are blocks of their own, not a loop in one.
template <bool PAIR>
__global__ void __launch_bounds__(256, 3) oh_k_iq2_slots(oh_iq2rows a) {
    __shared__ uint64_t grid[256];
    __shared__ uint4 stab[128];
    __shared__ __align__(16) uint8_t code_lds[4][(PAIR ? 2 : 1) * 64 * kCodeStride];   // a wave's rows are its own
    const int tid = tid_x();
    if ((int)blockIdx.y >= ldg(a.items)) return;
    const uint32_t it = (uint32_t)ldg(a.items + 1 + (int)blockIdx.y);
    const int e = (int)(it & 1023u), j = ldg(a.off + e) + a.cols * (int)(it >> 10);
    const int rest = ldg(a.off + e + 1) - j, n = rest < a.cols ? rest : a.cols;
    grid[tid] = k_iq2_grid[tid];
    iq2_sign_table(stab);
    __syncthreads();
    const int row = (int)blockIdx.x * 256 + tid;
    uint8_t *codes = code_lds[__builtin_amdgcn_readfirstlane(tid >> 6)];
    const int64_t row_bi = ((int64_t)e * a.rows + (row < a.rows ? row : a.rows - 1)) * (a.in / 256);
    if (n >= 5) iq2_cols<8, PAIR>(a, grid, stab, codes, row_bi, row, a.list + j, n);
    else if (n >= 3) iq2_cols<4, PAIR>(a, grid, stab, codes, row_bi, row, a.list + j, n);
    else if (n == 2) iq2_cols<2, PAIR>(a, grid, stab, codes, row_bi, row, a.list + j, n);
    else iq2_cols<1, PAIR>(a, grid, stab, codes, row_bi, row, a.list + j, n);
}

// inclusive sum over the block's threads
OH_DEV int block_incl_sum(int v, int32_t *sum) {
    const int tid = tid_x();
    for (int d = 1; d < kListThreads; d *= 2) {
        sum[tid] = v;
        __syncthreads();
        if (tid >= d) v += sum[tid - d];
        __syncthreads();
    }
    return v;
}

// The slots p < n in lists by expert idx[p]: off[e] .. off[e + 1] are expert
// e's entries of list (their order does not matter: every slot is computed on
// its own), items[0] the number of pieces of up to cols slots of one
// expert, then (piece << 10 | expert) of each. One block; an expert picked
// twice by one token keeps both entries; an index outside [0, ne) is reported
// and left out.
__global__ void __launch_bounds__(kListThreads)
oh_k_slot_lists(const int32_t *idx, int n, int ne, int cols, int32_t *off, int32_t *list, int32_t *items,
                int32_t *err) {
    __shared__ int32_t cnt[kListThreads], sum[kListThreads];
    const int tid = tid_x();
    cnt[tid] = 0;
    __syncthreads();
    for (int p = tid; p < n; p += kListThreads) {
        const int e = ldg(idx + p);
        if (e >= 0 && e < ne) atomicAdd(&cnt[e], 1);
        else atomicOr(err, OH_ERR_EXPERT_LIST);
    }
    __syncthreads();
    const int mine = cnt[tid], np = (mine + cols - 1) / cols;
    const int end = block_incl_sum(mine, sum), pend = block_incl_sum(np, sum);
    cnt[tid] = end - mine;
    if (tid < ne) stg(off + tid, end - mine);
    if (tid == ne - 1) {
        stg(off + ne, end);
        stg(items, pend);
    }
    for (int k = 0; k < np; k++) stg(items + 1 + pend - np + k, (int32_t)(k << 10 | tid));
    __syncthreads();
    for (int p = tid; p < n; p += kListThreads) {
        const int e = ldg(idx + p);
        if (e >= 0 && e < ne) stg(list + atomicAdd(&cnt[e], 1), (int32_t)p);
    }
}

} // namespace

extern "C" {

hipError_t oh_launch_slot_lists(const int32_t *idx, int n, int ne, int cols, int32_t *off, int32_t *list, int32_t *items,
                                int32_t *err, hipStream_t st) {
    if (ne < 1 || ne > kListThreads || cols < 1 || cols > 8) return hipErrorInvalidValue;
    hipLaunchKernelGGL(oh_k_slot_lists, dim3(1), dim3(kListThreads), 0, st, idx, n, ne, cols, off, list, items, err);
    return hipGetLastError();
}

hipError_t oh_launch_iq2_slots(const oh_iq2rows *a, int max_items, hipStream_t st) {
    const dim3 g((a->rows + 255) / 256, max_items);
    if (a->A2) hipLaunchKernelGGL(oh_k_iq2_slots<true>, g, dim3(256), 0, st, *a);
    else hipLaunchKernelGGL(oh_k_iq2_slots<false>, g, dim3(256), 0, st, *a);
    return hipGetLastError();
}

} // extern "C"
