// oh_kernels_delta.hip - the translation unit of the prompt's chunked delta
// scan in the reference's order (the default prompt mode; the recurrence and
// the matrix-core form are in oh_prefill.hip and oh_delta_mfma.hip).
//
// ornith_delta_prefill / delta_chunk (src/ornith_attn.c:215-349): the prompt in
// chunks of kScanC tokens counted from the start of the evaluation; per
// chunk, with S_in the incoming state,
//   p_i = prod_{l<=i} alpha_l, Sk_i = S_in k_i, Sq_i = S_in q_i,
//   u_i = beta_i v_i - beta_i p_i Sk_i - sum_{j<i} beta_i (p_i/p_j)(k_j.k_i) u_j,
//   o_i = p_i Sq_i + sum_{j<=i} (p_i/p_j)(k_j.q_i) u_j,
//   S_out = p_{C-1} S_in + sum_j (p_{C-1}/p_j) u_j k_j^T,
// where p_i/p_j is accumulated as the running product of alpha_{j+1..i}. Every
// float is formed in the reference's order, so the result equals its bits
// (it differs from the token-by-token recurrence in rounding).
//
// Everything that does not depend on the state (the Gram matrices and the
// coefficients beta_i (p_i/p_j)(k_j.k_i), (p_i/p_j)(k_j.q_i), p, ...) is formed
// for all chunks at once by oh_k_delta_coef; the scan over the chunks then does
// only what the state's chain needs.
#include "oh_dpp.h"
#include "oh_launch.h"

namespace {

constexpr int kScanC = 32;                     // tokens per chunk
// floats of one (chunk, value head): M as [i / 4][j][i % 4], W as [i][j], then
// p, beta, beta * p, the state update's ratios, the mask of M's rows that hold
// a zero, padding to 16 bytes
constexpr int kCoefM = 0, kCoefW = kScanC * kScanC, kCoefP = 2 * kScanC * kScanC, kCoefBeta = kCoefP + kScanC,
              kCoefBp = kCoefBeta + kScanC, kCoefEnd = kCoefBp + kScanC, kCoefZero = kCoefEnd + kScanC,
              kCoefN = kCoefZero + 4;

// add(k, mul(k)) for k = 0 .. N - 1 in order, the products two steps ahead
// (the first one, which may need the last chain's result, after the next two)
template <int N, class Mul, class Add>
OH_DEV void chain(Mul &&mul, Add &&add) {
    if constexpr (N > 0) {
        float t[N];
        if constexpr (N > 1) t[1] = mul(std::integral_constant<int, 1>{});
        if constexpr (N > 2) t[2] = mul(std::integral_constant<int, 2>{});
        order();
        t[0] = mul(std::integral_constant<int, 0>{});
        order();
        static_for<N>([&](auto k_) {
            constexpr int k = k_;
            if constexpr (k + 3 < N) t[k + 3] = mul(std::integral_constant<int, k + 3>{});
            order();
            add(k_, t[k]);
            order();
        });
    }
}

OH_DEV float f4(const float4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// ---- the coefficients of every chunk -----------------------------------------------
// A block per (key head, chunk): the Gram matrices kk[i][j] = k_j.k_i and
// kq[i][j] = k_j.q_i (ot_dot order: sequential over the head dimension), a
// thread per (i, four j); then a wave per value head of the key head forms
// its coefficient tables, lane i row i. 49 us for 4096 tokens of 16 key and 32
// value heads of 128 (the Gram matrices alone took 78 us with a thread per
// eight scattered pairs; the products' 16 instructions per three LDS reads
// bound it now).
template <int DK>
__global__ void __launch_bounds__(256)
oh_k_delta_coef(const float *qn, const float *kn, const float *al, const float *be, int T, int nk, int nv,
                float *coef) {
    constexpr int C = kScanC, LD = DK + 4, GS = C + 1, TS = C + 1;
    // keys and queries, then (the Gram matrices are in registers by then) the
    // four waves' tables
    constexpr int kStage = 2 * C * LD, kTabs = 4 * 2 * C * TS;
    __shared__ __align__(16) float stage[kStage > kTabs ? kStage : kTabs];
    __shared__ float kk[C * GS], kq[C * GS];
    float *ks = stage, *qs = stage + C * LD;
    const int kh = (int)blockIdx.x, ch = (int)blockIdx.y, tid = tid_x();
    const int c0 = ch * C, n = T - c0 < C ? T - c0 : C;
    for (int e = tid; e < C * DK / 4; e += 256) {
        const int i = e / (DK / 4), c = e - i * (DK / 4);
        const size_t src = ((size_t)(c0 + (i < n ? i : 0)) * nk + kh) * DK;
        *(float4 *)(ks + i * LD + 4 * c) = ldg((const float4 *)(kn + src) + c);
        *(float4 *)(qs + i * LD + 4 * c) = ldg((const float4 *)(qn + src) + c);
    }
    __syncthreads();
    {
        const int i = tid / 8, jb = tid % 8;              // j = jb + 8 m
        float ak[4] = {}, aq[4] = {};
#pragma unroll 4
        for (int c = 0; c < DK; c += 4) {
            const float4 ki = *(const float4 *)(ks + i * LD + c), qi = *(const float4 *)(qs + i * LD + c);
            float4 kj[4];
#pragma unroll
            for (int m = 0; m < 4; m++) kj[m] = *(const float4 *)(ks + (jb + 8 * m) * LD + c);
#pragma unroll
            for (int x = 0; x < 4; x++)
#pragma unroll
                for (int m = 0; m < 4; m++) {
                    ak[m] += f4(kj[m], x) * f4(ki, x);
                    aq[m] += f4(kj[m], x) * f4(qi, x);
                }
        }
#pragma unroll
        for (int m = 0; m < 4; m++) {
            kk[i * GS + jb + 8 * m] = ak[m];
            kq[i * GS + jb + 8 * m] = aq[m];
        }
    }
    __syncthreads();
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, i = lane & 31;
    float *tm = stage + wave * 2 * C * TS, *tw = tm + C * TS;
    for (int hv = kh + wave * nk; hv < nv; hv += 4 * nk) {
        // the gates of the chunk, one per lane (1 past the prompt's end)
        const float av = i < n ? ldg(al + (size_t)(c0 + i) * nv + hv) : 1.0f;
        const float bi = i < n ? ldg(be + (size_t)(c0 + i) * nv + hv) : 0.0f;
        auto gate = [&](int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(av), l)); };
        float pi = gate(0), ratio = 1.0f, we = 0.0f, r = 1.0f;
        for (int l = 1; l < C; l++) pi = l <= i ? pi * gate(l) : pi;
        // (p_i / p_j) as the running product of alpha_{j+1..i}, j descending;
        // and the state update's ratios, prod alpha_{j+1..n-1}
        bool zero = false;
#pragma unroll 8
        for (int j = C - 1; j >= 0; j--) {
            const float aj = gate(j), an = gate(j + 1 < C ? j + 1 : 0);
            const float gk = kk[i * GS + j], gq = kq[i * GS + j];
            ratio = j < i ? ratio * an : ratio;
            const float m = j < i ? bi * ratio * gk : 0.0f;
            zero = zero || (j < i && i < n && m == 0.0f);
            if (lane < 32) {
                tm[i * TS + j] = m;
                tw[i * TS + j] = j < i ? ratio * gq : j == i ? gq : 0.0f;
            }
            we = j < n && i == j ? r : we;
            r = j < n ? r * aj : r;
        }
        const uint32_t zm = (uint32_t)__ballot(zero);
        wave_lds_sync();
        float *o = coef + ((size_t)ch * nv + hv) * kCoefN;
#pragma unroll
        for (int e4 = 0; e4 < C * C / 4 / 64; e4++) {
            const int e = lane + 64 * e4;
            const int iq = e / C, j = e % C;                 // M: rows 4 iq .. 4 iq + 3 at column j
            stg((float4 *)(o + kCoefM) + e, make_float4(tm[(4 * iq) * TS + j], tm[(4 * iq + 1) * TS + j],
                                                        tm[(4 * iq + 2) * TS + j], tm[(4 * iq + 3) * TS + j]));
            const int wi = e / (C / 4), wj = 4 * (e % (C / 4));
            stg((float4 *)(o + kCoefW) + e, make_float4(tw[wi * TS + wj], tw[wi * TS + wj + 1], tw[wi * TS + wj + 2],
                                                        tw[wi * TS + wj + 3]));
        }
        if (lane < 32) {
            stg(o + kCoefP + i, pi);
            stg(o + kCoefBeta + i, bi);
            stg(o + kCoefBp + i, bi * pi);
            stg(o + kCoefEnd + i, we);
        }
        if (lane < 4) stg(o + kCoefZero + lane, u2f(lane == 0 ? zm : 0u));
        wave_lds_sync();                                  // the tables are reused
    }
}

// ---- the scan -------------------------------------------------------------------------
// A block per 16 rows of one value head's state (256 blocks at 32 heads of
// 128). A lone wave issues a vector instruction every 4 cycles whether or not
// it depends on the last one, so what counts is the number of instructions on
// the block's longest path. In every phase a 16-lane row of a wave (a "group")
// holds the block's 16 state rows, and what is common to them (a key's or
// query's element, a coefficient) sits in one lane of the group and enters the
// products as a DPP broadcast, not as an LDS read of its own.
// Per chunk, three phases with a barrier after each:
//   1 all waves: Sk of two tokens per group, from the whole state row in
//     registers; u starts as beta_i v_i - beta_i p_i Sk_i;
//   2 wave 0: the forward substitution of the 16 rows, 2 instructions per
//     term of one 496-term chain; meanwhile waves 1-3 form Sq, and wave 3 the
//     outputs of the previous chunk;
//   3 all waves: the state update, DK / 16 columns of one row per thread (kept
//     in registers from chunk to chunk), exchanged through LDS.
// 4096 tokens of 32 heads of 128 (MI355X): 2271 -> 711 us, 5.6 us per chunk
// (1003 tokens: 588 -> 198 us). The form before it kept one thread per (row,
// token), read every key element from LDS, formed the coefficient chains in
// the scan and ran substitution, Sq and outputs one after the other, at 256
// VGPRs + 256 AGPRs; this one needs 240 VGPRs and 68 KB of LDS, so that two
// blocks share a CU where there are more than 256 (64 heads of 128).
template <int DK>
__global__ void __launch_bounds__(256, 2)
oh_k_delta_chunked(const float *qn, const float *kn, const float *conv, const float *coef, float *S, float *out,
                   int T, int nk, int nv, int cc, float out_scale) {
    constexpr int C = kScanC, RB = 16, KS = DK + 4, XS = DK + 4, CPL = DK / 16, NV4 = DK / 64, US = C + 4;
    constexpr int NK = C * DK / 4 / 256;                 // key loads per thread and chunk
    __shared__ __align__(16) float kc[2][C * KS];
    __shared__ __align__(16) float cf[2][kCoefN];
    __shared__ __align__(16) float ut[2][RB * US];       // u, [row][token]
    __shared__ float sq[2][C * RB];                      // Sq, [token][row]
    __shared__ __align__(16) float xs[RB * XS];          // the state between phases 3 and 1
    const int tid = tid_x(), wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int r = lane & 15, grp = lane >> 4, g = wave * 4 + grp;
    // blocks go to the 8 XCDs round-robin (XCD = block % 8); with nv % 8 == 0
    // the slabs of a head share one XCD and its L2 copy of the head's inputs
    constexpr int NS = DK / RB;
    const int vb = (int)blockIdx.x;
    const int hv = (nv & 7) == 0 ? ((vb >> 3) / NS) * 8 + (vb & 7) : vb / NS;
    const int slab = (nv & 7) == 0 ? (vb >> 3) % NS : vb % NS, kh = hv % nk;
    const int qd = nk * DK, vd = nv * DK, r0 = hv * DK + slab * RB;

    // this thread's state elements: row r, columns g CPL ..
    float x[CPL];
    float *xr = xs + r * XS + g * CPL;
    float *Sr = S + (size_t)(r0 + r) * DK + g * CPL;
#pragma unroll
    for (int c = 0; c < CPL / 4; c++) {
        const float4 v = ldg((const float4 *)Sr + c);
        x[4 * c] = v.x; x[4 * c + 1] = v.y; x[4 * c + 2] = v.z; x[4 * c + 3] = v.w;
        *(float4 *)(xr + 4 * c) = v;
    }

    // a chunk's keys, coefficients and values, requested into registers a
    // chunk ahead, a whole chunk each time: the buffers are padded to whole
    // chunks, and what is computed for tokens past the prompt's end goes nowhere
    float4 rk[NK], rm, rw, rv = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float v0, v1, nv0 = 0.0f, nv1 = 0.0f;
    auto fetch = [&](int c0, int ch) {
        const int tid_ = again(tid), g_ = again(g);
        const float *kp = kn + ((size_t)c0 * nk + kh) * DK;
#pragma unroll
        for (int m = 0; m < NK; m++) {
            const unsigned e = (unsigned)tid_ + 256u * m, i = e / (DK / 4), c = e - i * (DK / 4);
            rk[m] = ldo<float4>(kp, 4u * (i * (unsigned)(nk * DK) + 4u * c));
        }
        const float *cs = coef + ((size_t)ch * nv + hv) * kCoefN;
        rm = ldo<float4>(cs, 16u * tid_);
        rw = ldo<float4>(cs, 4u * kCoefW + 16u * tid_);
        if (tid_ < (kCoefN - kCoefP) / 4) rv = ldo<float4>(cs, 4u * kCoefP + 16u * tid_);
        const float *vp = conv + (size_t)c0 * cc + 2 * qd + r0;
        nv0 = ldo<float>(vp, 4u * (unsigned)(g_ * cc + r));
        nv1 = ldo<float>(vp, 4u * (unsigned)((g_ + RB) * cc + r));
    };
    auto stage = [&](int b) {
#pragma unroll
        for (int m = 0; m < NK; m++) {
            const int e = tid + 256 * m, i = e / (DK / 4), c = e - i * (DK / 4);
            *(float4 *)(&kc[b][i * KS + 4 * c]) = rk[m];
        }
        *(float4 *)(&cf[b][4 * tid]) = rm;
        *(float4 *)(&cf[b][kCoefW + 4 * tid]) = rw;
        if (tid < (kCoefN - kCoefP) / 4) *(float4 *)(&cf[b][kCoefP + 4 * tid]) = rv;
    };
    // o_i = p_i Sq_i + w_ii u_i + sum_{j<i} w_ij u_j (j descending), scaled by
    // 1/sqrt(dk); one wave, token 4 s + grp in step s
    auto outputs = [&](int b, int c0) {
        const int grp_ = again(grp);
        float *op = out + (size_t)c0 * vd + r0;
        const int n = T - c0 < C ? T - c0 : C;
        const float *W = cf[b] + kCoefW, *p = cf[b] + kCoefP;
        float u[C];
#pragma unroll
        for (int j = 0; j < C / 4; j++) {
            const float4 v = *(const float4 *)(&ut[b][r * US + 4 * j]);
            u[4 * j] = v.x; u[4 * j + 1] = v.y; u[4 * j + 2] = v.z; u[4 * j + 3] = v.w;
        }
        static_for<C / 4>([&](auto s_) {
            constexpr int s = s_;
            const int i = 4 * s + grp_;
            const float wl = W[i * C + r], wh = W[i * C + 16 + r];
            float o = p[i] * sq[b][i * RB + r];
            o += W[i * C + i] * ut[b][r * US + i];
            chain<4 * s + 3>(
                [&](auto k_) {
                    constexpr int j = 4 * s + 2 - k_;
                    return row_lane<(j & 15)>(j < 16 ? wl : wh) * u[j];
                },
                [&](auto k_, float t) {
                    constexpr int j = 4 * s + 2 - k_;
                    const float o2 = o + t;
                    o = j < 4 * s || grp > j - 4 * s ? o2 : o;
                });
            if (i < n) stg((float *)((char *)op + 4u * (unsigned)(i * vd + r)), o * out_scale);
        });
    };

    fetch(0, 0);
    stage(0);
    v0 = nv0; v1 = nv1;
    __syncthreads();
    for (int c0 = 0, ch = 0; c0 < T; c0 += C, ch++) {
        const int n = T - c0 < C ? T - c0 : C, b = ch & 1;
        if (c0 + C < T) fetch(c0 + C, ch + 1);
        // the queries of this chunk's phase 2 (waves 1-3: tokens gq, gq + 12
        // and, the first eight groups, gq + 24)
        const int gq = g - 4;
        float4 q[3][NV4];
        if (wave > 0) {
            const float *qp = qn + ((size_t)c0 * nk + kh) * DK;
            const int gq_ = again(gq);
#pragma unroll
            for (int m = 0; m < 3; m++)
#pragma unroll
                for (int h = 0; h < NV4; h++)
                    if (m < 2 || wave < 3)
                        q[m][h] = ldo<float4>(qp + 64 * h, 4u * (unsigned)((gq_ + 12 * m) * nk * DK + 4 * r));
        }
        // ---- phase 1: Sk of tokens g and g + 16
        float s[DK];
#pragma unroll
        for (int c = 0; c < DK / 4; c++) {
            const float4 v = *(const float4 *)(xs + r * XS + 4 * c);
            s[4 * c] = v.x; s[4 * c + 1] = v.y; s[4 * c + 2] = v.z; s[4 * c + 3] = v.w;
        }
        {
            float4 k0[NV4], k1[NV4];
#pragma unroll
            for (int h = 0; h < NV4; h++) {
                k0[h] = *(const float4 *)(&kc[b][g * KS + 64 * h + 4 * r]);
                k1[h] = *(const float4 *)(&kc[b][(g + RB) * KS + 64 * h + 4 * r]);
            }
            float a0 = 0.0f, a1 = 0.0f;
            static_for<DK>([&](auto c_) {
                constexpr int c = c_;
                const float t0 = row_lane<((c >> 2) & 15)>(f4(k0[c >> 6], c & 3)) * s[c];
                const float t1 = row_lane<((c >> 2) & 15)>(f4(k1[c >> 6], c & 3)) * s[c];
                order();
                a0 += t0;
                a1 += t1;
                order();
            });
            const float *be = cf[b] + kCoefBeta, *bp = cf[b] + kCoefBp;
            ut[b][r * US + g] = be[g] * v0 - bp[g] * a0;
            ut[b][r * US + g + RB] = be[g + RB] * v1 - bp[g + RB] * a1;
        }
        __syncthreads();
        // ---- phase 2
        if (wave == 0) {
            // (I + M) U = T: u_i = (((t_i - m_{i,i-1} u_{i-1}) - m_{i,i-2}
            // u_{i-2}) ...), a term with m = 0 skipped (rows that hold one
            // take the form with the test: subtracting +0 is the skip)
            float u[C];
#pragma unroll
            for (int j = 0; j < C / 4; j++) {
                const float4 v = *(const float4 *)(&ut[b][r * US + 4 * j]);
                u[4 * j] = v.x; u[4 * j + 1] = v.y; u[4 * j + 2] = v.z; u[4 * j + 3] = v.w;
            }
            float4 ml[C / 4], mh[C / 8];
#pragma unroll
            for (int q4 = 0; q4 < C / 4; q4++) {
                ml[q4] = *(const float4 *)(&cf[b][kCoefM + (q4 * C + r) * 4]);
                if (q4 >= C / 8) mh[q4 - C / 8] = *(const float4 *)(&cf[b][kCoefM + (q4 * C + 16 + r) * 4]);
            }
            const uint32_t zm = __builtin_amdgcn_readfirstlane(f2u(cf[b][kCoefZero]));
            if (zm == 0) {
                static_for<C>([&](auto i_) {
                    constexpr int i = i_;
                    chain<i>(
                        [&](auto k_) {
                            constexpr int j = i - 1 - k_;
                            return row_lane<(j & 15)>(j < 16 ? f4(ml[i / 4], i & 3) : f4(mh[i / 4 % (C / 8)], i & 3)) * u[j];
                        },
                        [&](auto, float t) { u[i] = u[i] - t; });
                });
            } else {
                static_for<C>([&](auto i_) {
                    constexpr int i = i_;
                    float ui = u[i];
                    static_for<i>([&](auto j_) {
                        constexpr int j = i - 1 - j_;
                        const float m = row_lane<(j & 15)>(j < 16 ? f4(ml[i / 4], i & 3) : f4(mh[i / 4 % (C / 8)], i & 3));
                        const float t = m != 0.0f ? m * u[j] : 0.0f;
                        ui = ui - t;
                    });
                    u[i] = ui;
                });
            }
            if (grp == 0) {
#pragma unroll
                for (int j = 0; j < C / 4; j++)
                    *(float4 *)(&ut[b][r * US + 4 * j]) = make_float4(u[4 * j], u[4 * j + 1], u[4 * j + 2], u[4 * j + 3]);
            }
        } else {
            float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
            if (wave < 3) {
                static_for<DK>([&](auto c_) {
                    constexpr int c = c_;
                    const float t0 = row_lane<((c >> 2) & 15)>(f4(q[0][c >> 6], c & 3)) * s[c];
                    const float t1 = row_lane<((c >> 2) & 15)>(f4(q[1][c >> 6], c & 3)) * s[c];
                    const float t2 = row_lane<((c >> 2) & 15)>(f4(q[2][c >> 6], c & 3)) * s[c];
                    order();
                    a0 += t0;
                    a1 += t1;
                    a2 += t2;
                    order();
                });
                sq[b][(gq + 24) * RB + r] = a2;
            } else {
                static_for<DK>([&](auto c_) {
                    constexpr int c = c_;
                    const float t0 = row_lane<((c >> 2) & 15)>(f4(q[0][c >> 6], c & 3)) * s[c];
                    const float t1 = row_lane<((c >> 2) & 15)>(f4(q[1][c >> 6], c & 3)) * s[c];
                    order();
                    a0 += t0;
                    a1 += t1;
                    order();
                });
            }
            sq[b][gq * RB + r] = a0;
            sq[b][(gq + 12) * RB + r] = a1;
            if (wave == 3 && ch > 0) outputs(b ^ 1, c0 - C);
        }
        __syncthreads();
        // ---- phase 3: S_out = p_{C-1} S_in + sum_j (p_{C-1}/p_j) u_j k_j^T, j
        // descending; a term with a zero factor is skipped
        {
            float4 ka[2][CPL / 4];                       // lane l: keys l and l + 16, this group's columns
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int c = 0; c < CPL / 4; c++)
                    ka[h][c] = *(const float4 *)(&kc[b][(r + 16 * h) * KS + g * CPL + 4 * c]);
            const float *we = cf[b] + kCoefEnd;
            const float pc = cf[b][kCoefP + n - 1];
            float uw[C], z = 1.0f;
#pragma unroll
            for (int j = 0; j < C / 4; j++) {
                const float4 v = *(const float4 *)(&ut[b][r * US + 4 * j]), e = *(const float4 *)(we + 4 * j);
                uw[4 * j] = e.x * v.x; uw[4 * j + 1] = e.y * v.y; uw[4 * j + 2] = e.z * v.z; uw[4 * j + 3] = e.w * v.w;
            }
#pragma unroll
            for (int j = 0; j < C; j++) z = fminf(z, fabsf(uw[j]));
#pragma unroll
            for (int c = 0; c < CPL; c++) x[c] = x[c] * pc;
            if (n == C && __ballot(z == 0.0f) == 0) {
                static_for<C>([&](auto j_) {
                    constexpr int j = C - 1 - j_;
                    float t[CPL];
                    static_for<CPL>([&](auto c_) {
                        constexpr int c = c_;
                        t[c] = row_lane<(j & 15)>(f4(ka[j >> 4][c >> 2], c & 3)) * uw[j];
                    });
                    order();
#pragma unroll
                    for (int c = 0; c < CPL; c++) x[c] += t[c];
                    order();
                });
            } else {
                static_for<C>([&](auto j_) {
                    constexpr int j = C - 1 - j_;
                    const bool on = j < n && uw[j] != 0.0f;
                    static_for<CPL>([&](auto c_) {
                        constexpr int c = c_;
                        const float y = x[c] + row_lane<(j & 15)>(f4(ka[j >> 4][c >> 2], c & 3)) * uw[j];
                        x[c] = on ? y : x[c];
                    });
                });
            }
#pragma unroll
            for (int c = 0; c < CPL / 4; c++)
                *(float4 *)(xr + 4 * c) = make_float4(x[4 * c], x[4 * c + 1], x[4 * c + 2], x[4 * c + 3]);
            if (c0 + C < T) stage(b ^ 1);
            v0 = nv0; v1 = nv1;
        }
        __syncthreads();
    }
    const int nch = (T + C - 1) / C;
    if (wave == 3) outputs((nch - 1) & 1, (nch - 1) * C);
#pragma unroll
    for (int c = 0; c < CPL / 4; c++)
        stg((float4 *)Sr + c, make_float4(x[4 * c], x[4 * c + 1], x[4 * c + 2], x[4 * c + 3]));
}

template <int DK>
hipError_t launch(const float *qn, const float *kn, const float *conv, const float *al, const float *be, float *coef,
                  float *S, float *out, int T, int nk, int nv, int cc, float out_scale, hipStream_t st) {
    hipLaunchKernelGGL(oh_k_delta_coef<DK>, dim3(nk, (T + kScanC - 1) / kScanC), dim3(256), 0, st, qn, kn, al, be, T, nk,
                       nv, coef);
    hipLaunchKernelGGL(oh_k_delta_chunked<DK>, dim3(nv * (DK / 16)), dim3(256), 0, st, qn, kn, conv, coef, S, out, T, nk,
                       nv, cc, out_scale);
    return hipGetLastError();
}

} // namespace

extern "C" {

int oh_delta_coef_floats(int T, int nv) { return (T + kScanC - 1) / kScanC * nv * kCoefN; }

hipError_t oh_launch_delta_exact(int dk, const float *qn, const float *kn, const float *conv, const float *al,
                                 const float *be, float *coef, float *S, float *out, int T, int nk, int nv, int cc,
                                 float out_scale, hipStream_t st) {
    if (dk == 128) return launch<128>(qn, kn, conv, al, be, coef, S, out, T, nk, nv, cc, out_scale, st);
    if (dk == 64) return launch<64>(qn, kn, conv, al, be, coef, S, out, T, nk, nv, cc, out_scale, st);
    return hipErrorInvalidValue;
}

} // extern "C"
