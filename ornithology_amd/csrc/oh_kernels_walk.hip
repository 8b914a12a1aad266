// oh_kernels_walk.hip - the translation unit of the decode step's exact
// attention walk (the scores are formed before it, oh_layers.hip).
#include "oh_dpp.h"
#include "oh_launch.h"

namespace {

constexpr int kWalkThreads = 512, kWalkProd = kWalkThreads / 64 - 1;   // an adding wave, seven that form products
constexpr int kWalkChunk = kWalkProd;            // tiles of 16 positions per chunk: one per producer
constexpr int kWalkRing = 8;                     // a producer's tiles of codes in flight
constexpr int kWalkBufs = 4;                     // product buffers, a chunk each
static_assert(kWalkThreads == 512, "the block sum below adds eight wave sums");

OH_HD inline int walk_weights(int lim) { return ((lim + 15) / 16 + 2 * kWalkChunk) * 16; }   // whole chunks and one more
OH_HD inline int walk_lds_bytes(int lim) { return 4 * walk_weights(lim) + kWalkBufs * kWalkChunk * 16 * 64 * 4; }

// Query head h, its dimensions 64 dg .. 64 dg + 63 (block h * hd / 64 + dg):
// softmax over its T scores (max, exps, the double sum in exact_body's order,
// inv = 1/sum), then o_i = sum_t (p_t * Vs_t) * code_t,i in position order,
// and o *= sigmoid(gate). The sum over t is one chain of adds, 4 cycles each on
// a wave that issues nothing else: wave 0 does only that (lane = dimension),
// four positions per LDS read and a chunk of tiles read ahead, while the other
// waves form the products, a tile of 16 positions each per chunk, into four
// buffers used in turn (the weights p_t * Vs_t enter them as DPP broadcasts). A head's dimensions are spread over
// hd / 64 blocks, which each repeat its softmax. 16 heads of 256 at 4096 positions
// 33.7 -> 24.5 us, at 700 11.0 -> 9.6 us, against a block per head whose waves formed
// and added their own products; 3.5 us of it are the softmax, 14 the sum (8 cycles
// per position: the adds, their LDS reads, a barrier every 112 positions).
__global__ void __launch_bounds__(kWalkThreads) oh_k_attn_walk(oh_op_attn a, const int32_t *io) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr int NT = kWalkThreads;
    __shared__ double red[NT / 64];
    __shared__ float mred[NT / 64];
    __shared__ uint64_t etab[32];
    const int nh = a.nh, nkv = a.nkv, hd = a.hd, cap = a.cap, ng = hd / 64;
    const int h = (int)blockIdx.x / ng, dg = (int)blockIdx.x % ng, t = tid_x();
    const int T = io[OH_IO_POS] + 1, lim = exact_lim(a.exact_max, hd);
    if (T > lim || h >= nh) return;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6), lane = t & 63;
    float *pb = (float *)smem;                              // the weights, zero past T in the last chunk
    float4 *buf = (float4 *)(smem + 4 * walk_weights(lim)); // [kWalkBufs][kWalkChunk][4][64]: four positions per float4
    const int kvh = h / (nh / nkv);
    const int nt = (T + 15) / 16, nch = (nt + kWalkChunk - 1) / kWalkChunk;
    if (t < 32) etab[t] = k_exp2_tab[t];
    // this thread's scores (positions t, t + NT, ...: at most PT of them,
    // lim <= NT * PT, requested in groups of 8 up to T) and value scales, then
    // the gate and the first chunks' codes: every load issued before any is
    // used, the softmax's first (they return in order)
    constexpr int PT = 16;
    const float *sh = a.scores + (size_t)h * cap;
    float sv[PT], vs[PT];
#pragma unroll
    for (int r0 = 0; r0 < PT; r0 += 8) {
        if (NT * r0 >= T) break;
#pragma unroll
        for (int r = r0; r < r0 + 8; r++) {
            const int i = t + NT * r < T ? t + NT * r : T - 1;
            sv[r] = ldg(sh + i);
            vs[r] = ldg(a.Vs + (size_t)i * nkv + kvh);
        }
    }
    const float gt = ldg(a.gate + (size_t)h * hd + 64 * dg + lane);
    // producer p's codes of chunk c: tile kWalkChunk c + p (the 16 codes of
    // dimension lane in one uint4), a ring of kWalkRing chunks
    const int p = wave > 0 ? wave - 1 : 0;
    const uint8_t *vbase = (const uint8_t *)a.Vq + ((size_t)kvh * (cap / 16) * hd + 64 * dg) * 16;
    uint4 cw[kWalkRing];
    auto fetch = [&](uint4 &q, int c) {
        const int k = kWalkChunk * c + p;
        q = ldo<uint4>(vbase + (size_t)(k < nt ? k : nt - 1) * hd * 16, 16u * (unsigned)lane);
    };
    if (wave > 0) {
#pragma unroll
        for (int c = 0; c < kWalkRing; c++) fetch(cw[c], c);
    }
    float mx = -INFINITY;
#pragma unroll
    for (int r0 = 0; r0 < PT; r0 += 8) {
        if (NT * r0 >= T) break;
#pragma unroll
        for (int r = r0; r < r0 + 8; r++) if (t + NT * r < T) mx = fmaxf(mx, sv[r]);
    }
    mx = wave_max_fast(mx);
    if (lane == 0) mred[wave] = mx;
    lds_barrier();
#pragma unroll
    for (int k = 0; k < NT / 64; k++) mx = fmaxf(mx, mred[k]);
    // the exps in groups of 8 slots (a slot past T is computed on a
    // repeated score and left out of the sum), so those of a group overlap
    double sum = 0.0;
#pragma unroll
    for (int r0 = 0; r0 < PT; r0 += 8) {
        if (NT * r0 >= T) break;
#pragma unroll
        for (int r = r0; r < r0 + 8; r++) sv[r] = ref_expf_sel(sv[r] - mx, etab);
#pragma unroll
        for (int r = r0; r < r0 + 8; r++) sum += t + NT * r < T ? (double)sv[r] : 0.0;
    }
    // the double sum over the block (tree-ordered, as the walk's other
    // forms; the exps are at most 1, so the order moves only the last
    // bits of a double)
    sum = wave_sum_d(sum);
    if (lane == 0) red[wave] = sum;
    lds_barrier();
    sum = ((red[0] + red[1]) + (red[2] + red[3])) + ((red[4] + red[5]) + (red[6] + red[7]));
    const float inv = (float)(1.0 / sum);
#pragma unroll
    for (int r0 = 0; r0 < PT; r0 += 8) {
        if (NT * r0 >= T) break;
#pragma unroll
        for (int r = r0; r < r0 + 8; r++) if (t + NT * r < T) pb[t + NT * r] = sv[r] * inv * vs[r];
    }
    for (int i = T + t; i < 16 * kWalkChunk * nch; i += NT) pb[i] = 0.0f;
    lds_barrier();
    // Intervals between block barriers: in interval i the producers form chunk
    // i and the adding wave, which holds chunk i - 3 in registers, adds it and
    // reads chunk i - 2 in its place. No barrier waits for LDS accesses in
    // flight: a producer's stores of interval i are done once the weights that
    // it reads after them arrive, which interval i + 1 begins with; what the
    // adding wave reads in interval i it adds in interval i + 1, and the buffer
    // is written again in interval i + 2.
    const int ni = nch + 3;
    auto pass = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (wave > 0) {
        float w = pb[16 * p + (lane & 15)];
        for (int c0 = 0; c0 < ni; c0 += kWalkRing) {
#pragma unroll
            for (int u = 0; u < kWalkRing; u++) {
                const int c = c0 + u;
                if (c >= ni) break;
                if (c < nch) {
                    float4 *dst = buf + (size_t)((c % kWalkBufs) * kWalkChunk + p) * 4 * 64 + lane;
                    static_for<4>([&](auto g_) {
                        constexpr int g = g_;
                        float x[4], y[4];
#pragma unroll
                        for (int j = 0; j < 4; j++) x[j] = (float)(int8_t)((g == 0 ? cw[u].x : g == 1 ? cw[u].y : g == 2 ? cw[u].z : cw[u].w) >> (8 * j));
                        order();
                        static_for<4>([&](auto j_) {
                            constexpr int j = j_;
                            y[j] = row_lane<4 * g + j>(w) * x[j];
                        });
                        order();
                        dst[64 * g] = make_float4(y[0], y[1], y[2], y[3]);
                    });
                    asm volatile("" ::: "memory");
                    w = pb[16 * (kWalkChunk * (c + 1) + p) + (lane & 15)];
                    fetch(cw[u], c + kWalkRing);
                    pass();
                } else {
                    lds_barrier();                        // waits for the last chunk's stores
                }
            }
        }
        return;
    }
    // the weights past T are +0; o starts at +0 and a round-to-nearest sum is
    // -0 only when both addends are, so o is never -0 and adding +-0 leaves its
    // bits unchanged: the plain sum equals the reference's zero-skipping one
    __builtin_amdgcn_s_setprio(3);
    float o = 0.0f;
    float4 r[kWalkChunk][4];
    auto read = [&](int c, int s) {
        const float4 *src = buf + (size_t)((c % kWalkBufs) * kWalkChunk + s) * 4 * 64 + lane;
#pragma unroll
        for (int g = 0; g < 4; g++) r[s][g] = src[64 * g];
    };
    pass();
    pass();
#pragma unroll
    for (int s = 0; s < kWalkChunk; s++) read(0, s);
    pass();
    for (int i = 3; i < ni; i++) {
        const int c = i - 2 < nch ? i - 2 : nch - 1;         // (past the end: read, not added)
#pragma unroll
        for (int s = 0; s < kWalkChunk; s++) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                o += r[s][g].x;
                o += r[s][g].y;
                o += r[s][g].z;
                o += r[s][g].w;
            }
            order();
            read(c, s);
            order();
        }
        pass();
    }
    stg(a.out + (size_t)h * hd + 64 * dg + lane, o * ref_sigmoid(gt));
}

} // namespace

extern "C" {

int oh_attn_walk_blocks(int nh, int hd) { return nh * (hd / 64); }
int oh_attn_walk_lds(int lim) { return walk_lds_bytes(lim); }

hipError_t oh_launch_attn_walk(const oh_op_attn *a, const int32_t *io, int blocks, int lds_bytes, hipStream_t st) {
    const hipError_t e = hipFuncSetAttribute((const void *)oh_k_attn_walk, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(oh_k_attn_walk, dim3(blocks), dim3(kWalkThreads), (size_t)lds_bytes, st, *a, io);
    return hipGetLastError();
}

} // extern "C"
