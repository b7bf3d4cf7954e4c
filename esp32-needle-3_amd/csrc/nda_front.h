/* nda_front.h - the attention front of one (row, kv group) on a work-group:
 * steps 1 to 3 of the front kernel (nda_front.hip), which the decode kernel of
 * small GQA batches runs as its first part (nda_prefill.hip). */
#pragma once

#include "nda_device.h"

namespace nda {

template <int DK, int DV, int REP>
struct FrontShape {
    static constexpr int NC = REP * DK + DK + DV;   // columns of one kv group
    static constexpr int NG = NC / 4;               // four-column groups, one per thread
    static constexpr int W = (NG + 63) / 64;        // waves per work-group
    static constexpr int NH = REP + 1;              // normalised heads: REP q + 1 k
    static constexpr int STRIDE = DK + 4;           // LDS row: 16-byte aligned, banks spread
    static constexpr int HALF = DK / 2;
    static constexpr int TREG = 4;                  // taps held in registers; more are streamed
    static_assert(DK % 4 == 0 && DV % 4 == 0, "four-column groups");
    static_assert(W <= 4, "one group per thread");
};

typedef float float4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float4 ld4(const float *p) { return *reinterpret_cast<const float4 *>(p); }

__device__ __forceinline__ void acc4(float4 &a, const float4 &w, const float4 &x)
{
#pragma clang fp contract(off)
    a.x = a.x + w.x * x.x;
    a.y = a.y + w.y * x.y;
    a.z = a.z + w.z * x.z;
    a.w = a.w + w.w * x.w;
}

// What the front leaves in LDS: the rotated k head after the q ones (q only
// with QLDS, else in q_out) in y, v in v.
template <int DK, int DV, int REP>
struct FrontLds {
    using S = FrontShape<DK, DV, REP>;
    __attribute__((aligned(16))) float y[S::NH * S::STRIDE];    // conv outputs of the q/k heads
    __attribute__((aligned(16))) float sq[S::NH * S::STRIDE];   // their squares
    __attribute__((aligned(16))) float v[DV];
    float inv[S::NH];
};

// All NT threads of the work-group call it (two barriers); a by value: its
// pointers, selected through a reference, went to scratch memory. With a.k_out null
// (store mode) the caller stores k and v after a barrier.
template <int DK, int DV, int REP, int NT, bool QLDS>
__device__ __forceinline__ void front_steps(const FrontArgs a, uint32_t row, uint32_t g, uint32_t seq, uint32_t t,
                                            uint32_t pos, int tid, FrontLds<DK, DV, REP> &lds)
{
#pragma clang fp contract(off)
    using S = FrontShape<DK, DV, REP>;
    static_assert(NT >= 64 * S::W, "one four-column group per thread");
    const uint32_t nkv = a.nkv;
    const uint32_t taps = a.taps;
    const uint32_t nt = min(taps, pos + 1u);
    const uint32_t dq = nkv * REP * DK, dk = nkv * DK, dv = nkv * DV, dcol = dq + dk + dv;
    float *hist = a.hist + ((uint64_t)seq * a.n_layers + a.layer) * taps * dcol;
    const bool store = a.k_out == nullptr;

    // What step 3 reads (this thread's rotary pairs and norm scales) is
    // requested now, beside the tap loads, so the wave waits on one round of
    // loads rather than two.
    constexpr int NE = (S::NH * S::HALF + NT - 1) / NT;   // emit elements per thread
    const float2 *rope = a.rope + (uint64_t)pos * S::HALF;
    float2 cs_e[NE];
    float s1_e[NE], s2_e[NE];
#pragma unroll
    for (int n = 0; n < NE; n++) {
        const int e = tid + n * NT;
        const int h = e / S::HALF, i = e % S::HALF;
        if (e < S::NH * S::HALF) {
            const float *sn = a.norm + (h < REP ? 0 : DK);
            cs_e[n] = rope[i];
            s1_e[n] = sn[i];
            s2_e[n] = sn[i + S::HALF];
        }
    }
    // 1. tap convolution of this thread's four columns
    const bool active = tid < S::NG;
    const int lc = tid * 4;                      // column within the group
    const float *src;
    uint32_t ld, cc, gc;                         // source row length, column in it, column in dcol
    if (lc < REP * DK) {
        src = a.q; ld = dq; cc = g * REP * DK + lc; gc = cc;
    } else if (lc < REP * DK + DK) {
        src = a.k; ld = dk; cc = g * DK + (lc - REP * DK); gc = dq + cc;
    } else {
        src = a.v; ld = dv; cc = g * DV + (lc - REP * DK - DK); gc = dq + dk + cc;
    }
    float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float4 raw = acc;
    if (active) {
        float4 x[S::TREG], w[S::TREG];
        raw = ld4(src + (uint64_t)row * ld + cc);
#pragma unroll
        for (int j = 0; j < S::TREG; j++) {
            if ((uint32_t)j < nt) {
                w[j] = ld4(a.w + (uint64_t)j * dcol + gc);
                if (j == 0)
                    x[j] = raw;
                else if ((uint32_t)j <= t)
                    x[j] = ld4(src + (uint64_t)(row - j) * ld + cc);
                else
                    x[j] = ld4(hist + (uint64_t)((pos - j) % taps) * dcol + gc);
            }
        }
#pragma unroll
        for (int j = 0; j < S::TREG; j++)
            if ((uint32_t)j < nt)
                acc4(acc, w[j], x[j]);
        for (uint32_t j = S::TREG; j < nt; j++) {
            const float4 wj = ld4(a.w + (uint64_t)j * dcol + gc);
            const float4 xj = j <= t ? ld4(src + (uint64_t)(row - j) * ld + cc)
                                     : ld4(hist + (uint64_t)((pos - j) % taps) * dcol + gc);
            acc4(acc, wj, xj);
        }
        // the raw row into the tap history, read again only at the next
        // step's front: streamed past L2 (2-6% off the 4096-row front)
        if (a.hist_write)
            __builtin_nontemporal_store(float4v{raw.x, raw.y, raw.z, raw.w},
                                        reinterpret_cast<float4v *>(hist + (uint64_t)(pos % taps) * dcol + gc));
        if (lc < (REP + 1) * DK) {
            const int o = (lc / DK) * S::STRIDE + lc % DK;
            *reinterpret_cast<float4 *>(lds.y + o) = acc;
            *reinterpret_cast<float4 *>(lds.sq + o) =
                make_float4(acc.x * acc.x, acc.y * acc.y, acc.z * acc.z, acc.w * acc.w);
        } else if (store) {
            *reinterpret_cast<float4 *>(lds.v + (lc - (REP + 1) * DK)) = acc;
        } else {
            *reinterpret_cast<float4 *>(a.v_out + (uint64_t)row * dv + cc) = acc;
        }
    }
    __syncthreads();

    // 2. per-head sum of squares in index order, inverse RMS
    if (tid < S::NH) {
        const float *r = lds.sq + tid * S::STRIDE;
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < DK; i++)
            ss = ss + r[i];
        lds.inv[tid] = 1.0f / __builtin_sqrtf(ss / (float)DK + 1e-6f);
    }
    __syncthreads();

    // 3. (1 + s) * x * inv, rotated by the position's (cos, sin)
#pragma unroll
    for (int n = 0; n < NE; n++) {
        const int e = tid + n * NT;
        if (e >= S::NH * S::HALF)
            break;
        const int h = e / S::HALF, i = e % S::HALF;
        const bool is_q = h < REP;
        float *r = lds.y + h * S::STRIDE;
        const float iv = lds.inv[h];
        const float x1 = (1.0f + s1_e[n]) * r[i] * iv;
        const float x2 = (1.0f + s2_e[n]) * r[i + S::HALF] * iv;
        const float2 cs = cs_e[n];
        const float o1 = x1 * cs.x - x2 * cs.y;
        const float o2 = x2 * cs.x + x1 * cs.y;
        if (is_q && !QLDS) {
            float *qo = a.q_out + (uint64_t)row * dq + (g * REP + h) * DK;
            qo[i] = o1;
            qo[i + S::HALF] = o2;
        } else if (QLDS || store) {
            r[i] = o1;
            r[i + S::HALF] = o2;
        } else {
            float *ko = a.k_out + (uint64_t)row * dk + g * DK;
            ko[i] = o1;
            ko[i + S::HALF] = o2;
        }
    }
}

} // namespace nda
