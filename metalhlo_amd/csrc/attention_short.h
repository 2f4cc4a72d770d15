// Attention of a short prompt, one wave per 32 queries: attention_short.hip, and linear_w32.hip in front of a projection.
#pragma once
#include "attention_common.h"

namespace mhip {

// Causal attention of queries 32 (HALVES - 1) ... + 31 of head bh, which see up to 32 HALVES keys, by one wave; `vt`: HALVES * 32 * D * 2 bytes of LDS of its
// own.  store(query, d, w): four consecutive elements of the result from d on.
template <typename T, int D, int HALVES, typename Store>
__device__ __forceinline__ void short_rows(const FaArgs& a, int bh, char* vt, Store&& store) {
    constexpr int kRows = 32;
    constexpr int ND = D / 32, NS = D / 16, CPR = D / 8, kRowsPerInst = 64 / CPR;
    const int lane = threadIdx.x & 63, lrow = lane & 31, lhalf = lane >> 5;
    const int b_i = bh / a.H, h_i = bh % a.H;
    const int qpos = (HALVES - 1) * kRows + lrow;
    const T* qp = static_cast<const T*>(a.q) + b_i * a.qs[0] + h_i * a.qs[1];
    const T* kp = static_cast<const T*>(a.k) + b_i * a.ks[0] + h_i * a.ks[1];
    const T* vp = static_cast<const T*>(a.v) + b_i * a.vs[0] + h_i * a.vs[1];
    const int q_rs = (int)a.qs[2], k_rs = (int)a.ks[2], v_rs = (int)a.vs[2];
    const __amdgpu_buffer_rsrc_t rq = fa_rsrc(qp, (uint32_t)((((int64_t)a.Sq - 1) * q_rs + D) * 2));
    const __amdgpu_buffer_rsrc_t rk = fa_rsrc(kp, (uint32_t)((((int64_t)a.Skv - 1) * k_rs + D) * 2));
    const __amdgpu_buffer_rsrc_t rv = fa_rsrc(vp, (uint32_t)((((int64_t)a.Skv - 1) * v_rs + D) * 2));
    const int keys = min(a.Skv, HALVES * kRows);           // that some row of this wave sees

    u32x4 qf[NS], kf[HALVES][NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        qf[s] = __builtin_amdgcn_raw_buffer_load_b128(rq, qpos < a.Sq ? (uint32_t)((qpos * q_rs + 16 * s + 8 * lhalf) * 2) : kOobA, 0, 0);
#pragma unroll
        for (int t = 0; t < HALVES; t++) {
            const int key = 32 * t + lrow;
            kf[t][s] = __builtin_amdgcn_raw_buffer_load_b128(rk, key < keys ? (uint32_t)((key * k_rs + 16 * s + 8 * lhalf) * 2) : kOobA, 0, 0);
        }
    }
    // (rows of values past the keys are zeros: a weight of zero times them stays zero)
#pragma unroll
    for (int i = 0; i < HALVES * kRows / kRowsPerInst; i++) {
        const int row = i * kRowsPerInst + lane / CPR, col = (lane % CPR ^ v_swz<D>(row)) * 8;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (fa_lds_void*)(vt + i * 1024), 16, row < keys ? (uint32_t)((row * v_rs + col) * 2) : kOobA, 0, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);                     // (nothing is multiplied before the last of them is on its way)

    // ---- S^T = K Q^T; register i of the tiles (t = i / 16, r = i % 16) is key 32t + 8(r/4) + 4*lhalf + r%4 of query qpos
    f32x16 sacc[HALVES];
#pragma unroll
    for (int t = 0; t < HALVES; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) sacc[t][r] = 0.f;
#pragma unroll
    for (int s = 0; s < NS; s++) {
        if (a.negate_q) {
#pragma unroll
            for (int e = 0; e < 4; e++) qf[s][e] ^= 0x80008000u;
        }
#pragma unroll
        for (int t = 0; t < HALVES; t++) sacc[t] = Mfma32A<T>::run(kf[t][s], qf[s], sacc[t]);
    }
    float sv[16 * HALVES], m = -INFINITY, l = 0.f;
#pragma unroll
    for (int i = 0; i < 16 * HALVES; i++) {
        const int key = 32 * (i >> 4) + 8 * ((i & 15) >> 2) + 4 * lhalf + (i & 3);
        sv[i] = key > qpos || key >= a.Skv ? -INFINITY : sacc[i >> 4][i & 15] * a.c;
        m = fmaxf(m, sv[i]);
    }
    m = half_max(m);
    const float m_use = m == -INFINITY ? 0.f : m;
#pragma unroll
    for (int i = 0; i < 16 * HALVES; i++) {
        sv[i] = weight(sv[i], m_use);
        l += sv[i];
    }
    l = half_sum(l);
    const float inv = l > 1e-10f ? 1.f / l : 0.f;

    // ---- O^T += V^T P^T, the operands as in fa_fwd_kernel
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int ti = lane & 15, tg = lane >> 4;
    const int v_row0 = 4 * (tg >> 1) + (ti >> 2), v_d0 = 16 * (tg & 1) + 4 * (ti & 3);
    f32x16 oacc[ND];
#pragma unroll
    for (int dt = 0; dt < ND; dt++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[dt][r] = 0.f;
#pragma unroll
    for (int u = 0; u < 2 * HALVES; u++) {
        u32x4 pb;
#pragma unroll
        for (int e = 0; e < 4; e++) pb[e] = Mfma32A<T>::pack2(sv[8 * u + 2 * e], sv[8 * u + 2 * e + 1]);
#pragma unroll
        for (int dt = 0; dt < ND; dt++) {
            const int row = 16 * u + v_row0, d0 = 32 * dt + v_d0;
            const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((fa_lds_s16x4*)(vt + v_off<D>(row, d0 >> 3) + (d0 & 7) * 2)));
            const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((fa_lds_s16x4*)(vt + v_off<D>(row + 8, d0 >> 3) + (d0 & 7) * 2)));
            oacc[dt] = Mfma32A<T>::run(u32x4{lo.x, lo.y, hi.x, hi.y}, pb, oacc[dt]);
        }
    }
    if (qpos >= a.Sq) return;
#pragma unroll
    for (int dt = 0; dt < ND; dt++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            u32x2 w;
            w.x = Mfma32A<T>::pack2(oacc[dt][4 * g + 0] * inv, oacc[dt][4 * g + 1] * inv);
            w.y = Mfma32A<T>::pack2(oacc[dt][4 * g + 2] * inv, oacc[dt][4 * g + 3] * inv);
            store(qpos, 32 * dt + 8 * g + 4 * lhalf, w);
        }
}

}  // namespace mhip
