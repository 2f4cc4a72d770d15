// Causal attention of up to 64 queries over up to 64 keys without a mask operand, 16-bit types, head sizes 64 and 128: a short prompt.
//
// What bounds it: latencies.  The kernels for longer sequences walk blocks of 64 keys through LDS behind barriers, which for one
// block is 2 us of latencies one after the other ([1,12,37,64] 4.4 us in a graph, of which a launch is 2.2).  Here a wave owns 32 query rows and
// asks for every query, key and value it will need in its first instructions, queries and keys straight into matrix operands, values
// into LDS of its own: neither a barrier nor a running maximum, 3.3 us.
//
// The products and sums are those of attention.hip's fa_fwd_kernel over one block of keys, in its order: a row has the same bits
// whether its sequence ends here or goes on.  (The 16x16x32 instruction, 16 rows a wave, adds up in another order; us, so | here:
// [1,12,37,64] 3.0 | 3.3, [8,32,64,64] 4.6 | 4.5, [64,32,64,64] 15.9 | 14.6, head size 128 [1,32,40] 4.0 | 4.3, [8,32,64] 6.6 | 6.2.)
#include "attention_common.h"

namespace mhip {
namespace {

constexpr int kRows = 32, kMostWaves = 2;

// The 32 rows of wave HALVES - 1, which see up to 32 HALVES keys.
template <typename T, int D, int HALVES>
__device__ __forceinline__ void short_rows(const FaArgs& a, char* vt) {
    constexpr int ND = D / 32, NS = D / 16, CPR = D / 8, kRowsPerInst = 64 / CPR;
    const int lane = threadIdx.x & 63, lrow = lane & 31, lhalf = lane >> 5;
    const int bh = blockIdx.x, b_i = bh / a.H, h_i = bh % a.H;
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
    T* orow = static_cast<T*>(a.o) + b_i * a.os[0] + h_i * a.os[1] + (int64_t)qpos * a.os[2];
#pragma unroll
    for (int dt = 0; dt < ND; dt++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            u32x2 w;
            w.x = Mfma32A<T>::pack2(oacc[dt][4 * g + 0] * inv, oacc[dt][4 * g + 1] * inv);
            w.y = Mfma32A<T>::pack2(oacc[dt][4 * g + 2] * inv, oacc[dt][4 * g + 3] * inv);
            *reinterpret_cast<u32x2*>(orow + 32 * dt + 8 * g + 4 * lhalf) = w;
        }
}

template <typename T, int D>
__global__ __launch_bounds__(64 * kMostWaves) void fa_short_kernel(FaArgs a) {
    __shared__ __attribute__((aligned(1024))) char smem[(1 + 2) * kRows * D * 2];
    // (a wave that sees half of the keys has half of the work, and is alone where there are no more rows)
    if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == 0) short_rows<T, D, 1>(a, smem);
    else short_rows<T, D, 2>(a, smem + kRows * D * 2);
}

template <typename T>
int launch_type(hipStream_t s, const FaArgs& a, int64_t D) {
    const dim3 grid((unsigned)(a.B * a.H)), block(64 * ((a.Sq + kRows - 1) / kRows));
    if (D == 128) hipLaunchKernelGGL((fa_short_kernel<T, 128>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((fa_short_kernel<T, 64>), grid, block, 0, s, a);
    return check_launch("flash_attention_short");
}

}  // namespace

// us, fa_fwd_kernel | here, in a graph, up to 16 states in turn, D 64: [1,12,16] 4.1 | 2.7, [1,12,64] 4.5 | 3.5, [8,32,64] 5.9 | 4.5, [64,32,64] 17.7 | 14.6;
// D 128: [1,32,40] 5.7 | 4.3, [8,32,64] 8.1 | 6.2, [32,32,64] 18.8 | 16.2; GPT-2 over 37 tokens, behind a projection and with cold caches, 467 | 451.
// Past 64 keys or without the causal rule 16 rows a wave were tried: they read the keys again for every 16 rows ([8,32,100] 6.9 | 7.8, every
// key for every query D 128 [16,32,64] 10.4 | 11.5).
bool fa_short_wanted(const FaArgs& a) { return a.is_causal && a.Sq <= kRows * kMostWaves && a.Skv <= 64; }

int launch_fa_short(hipStream_t s, const FaArgs& a, int64_t D, int dtype) {
    return dtype == MHIP_BF16 ? launch_type<bf16_t>(s, a, D) : launch_type<f16_t>(s, a, D);
}

}  // namespace mhip
