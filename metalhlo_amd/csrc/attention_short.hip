// Causal attention of up to 64 queries over up to 64 keys without a mask operand, 16-bit types, head sizes 64 and 128: a short prompt.
//
// What bounds it: latencies.  The kernels for longer sequences walk blocks of 64 keys through LDS behind barriers, which for one
// block is 2 us of latencies one after the other ([1,12,37,64] 5.3 us, of which a launch is 2.2).  Here a wave owns 16 query rows,
// asks for every key and value it will need in its first instructions, straight into matrix operands as in attention_decode.hip,
// and needs neither LDS nor a barrier nor a running maximum: 3.9 us.
//   S^T = K Q^T     v_mfma_f32_16x16x32: operand row = key; a lane of the result holds four keys of one query.
//   O^T += V^T P^T  operand row = d: lane i loads VE = D / 16 neighbouring d of each of its keys, one byte permute pairs two keys of one
//                   d, tile f holds d = VE i + f, and a lane ends up with 4 VE consecutive d of its query.
#include "attention_common.h"
#include "gemm_lds.h"

namespace mhip {
namespace {

constexpr int kRows = 16, kMostWaves = 4;

template <typename T, int D>
__global__ __launch_bounds__(64 * kMostWaves) void fa_short_kernel(FaArgs a) {
    constexpr int KG = 4;                                // groups of 16 keys
    constexpr int NS = D / 32, VE = D / 16, VDw = VE / 2;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int bh = blockIdx.x, b_i = bh / a.H, h_i = bh % a.H;
    const int q0 = wave * kRows, q = q0 + li;
    const T* qp = static_cast<const T*>(a.q) + b_i * a.qs[0] + h_i * a.qs[1];
    const T* kp = static_cast<const T*>(a.k) + b_i * a.ks[0] + h_i * a.ks[1];
    const T* vp = static_cast<const T*>(a.v) + b_i * a.vs[0] + h_i * a.vs[1];
    const int q_rs = (int)a.qs[2], k_rs = (int)a.ks[2], v_rs = (int)a.vs[2];
    const __amdgpu_buffer_rsrc_t rq = fa_rsrc(qp, (uint32_t)((((int64_t)a.Sq - 1) * q_rs + D) * 2));
    const __amdgpu_buffer_rsrc_t rk = fa_rsrc(kp, (uint32_t)((((int64_t)a.Skv - 1) * k_rs + D) * 2));
    const __amdgpu_buffer_rsrc_t rv = fa_rsrc(vp, (uint32_t)((((int64_t)a.Skv - 1) * v_rs + D) * 2));
    // keys that some row of this wave sees
    const int keys = min(a.Skv, q0 + kRows);

    u32x4 qf[NS], kf[KG][NS];
    uint32_t vf[4 * KG][VDw];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        qf[s] = __builtin_amdgcn_raw_buffer_load_b128(rq, q < a.Sq ? (uint32_t)((q * q_rs + 32 * s + 8 * lg) * 2) : kOobA, 0, 0);
        if (a.negate_q) {
#pragma unroll
            for (int e = 0; e < 4; e++) qf[s][e] ^= 0x80008000u;
        }
    }
#pragma unroll
    for (int j = 0; j < KG; j++)
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const int key = 16 * j + li;
            kf[j][s] = __builtin_amdgcn_raw_buffer_load_b128(rk, key < keys ? (uint32_t)((key * k_rs + 32 * s + 8 * lg) * 2) : kOobA, 0, 0);
        }
#pragma unroll
    for (int t = 0; t < 4 * KG; t++) {
        const int key = 16 * (t >> 2) + 4 * lg + (t & 3);
        const uint32_t off = key < keys ? (uint32_t)((key * v_rs + VE * li) * 2) : kOobA;
        if constexpr (VDw == 4) {
            const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(rv, off, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; e++) vf[t][e] = w[e];
        } else {
            const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(rv, off, 0, 0);
            vf[t][0] = w.x; vf[t][1] = w.y;
        }
    }

    float sv[4 * KG], m = -INFINITY;
#pragma unroll
    for (int j = 0; j < KG; j++) {
        f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NS; s++) s4 = Tile16<T>::run(kf[j][s], qf[s], s4);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int key = 16 * j + 4 * lg + r;
            sv[4 * j + r] = key >= a.Skv || key > q ? -INFINITY : s4[r] * a.c;
            m = fmaxf(m, sv[4 * j + r]);
        }
    }
    m = fmaxf(m, __shfl_xor(m, 16, 64));
    m = half_max(m);
    const float m_use = m == -INFINITY ? 0.f : m;
    float l = 0.f;
#pragma unroll
    for (int t = 0; t < 4 * KG; t++) {
        sv[t] = weight(sv[t], m_use);
        l += sv[t];
    }
    l += __shfl_xor(l, 16, 64);
    l = half_sum(l);
    const float inv = l > 1e-10f ? 1.f / l : 0.f;
    f32x4 o[VE];
#pragma unroll
    for (int f = 0; f < VE; f++) o[f] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < KG / 2; h++) {                   // 32 keys: the ones whose weights the lane has
        u32x4 pb;
#pragma unroll
        for (int e = 0; e < 4; e++) pb[e] = Mfma32A<T>::pack2(sv[8 * h + 2 * e], sv[8 * h + 2 * e + 1]);
#pragma unroll
        for (int f = 0; f < VE; f++) {
            u32x4 w;
#pragma unroll
            for (int e = 0; e < 4; e++)
                w[e] = __builtin_amdgcn_perm(vf[8 * h + 2 * e + 1][f / 2], vf[8 * h + 2 * e][f / 2], (f & 1) ? 0x07060302u : 0x05040100u);
            o[f] = Tile16<T>::run(w, pb, o[f]);
        }
    }
    // lane (li, lg): query li, d = VE (4 lg + r) + f
    if (q >= a.Sq) return;
    T* orow = static_cast<T*>(a.o) + b_i * a.os[0] + h_i * a.os[1] + (int64_t)q * a.os[2] + 4 * VE * lg;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        uint32_t w[VDw];
#pragma unroll
        for (int e = 0; e < VDw; e++) w[e] = Mfma32A<T>::pack2(o[2 * e][r] * inv, o[2 * e + 1][r] * inv);
        if constexpr (VDw == 4) *reinterpret_cast<u32x4*>(orow + VE * r) = u32x4{w[0], w[1], w[2], w[3]};
        else *reinterpret_cast<u32x2*>(orow + VE * r) = u32x2{w[0], w[1]};
    }
}

template <typename T>
int launch_type(hipStream_t s, const FaArgs& a, int64_t D) {
    const dim3 grid((unsigned)(a.B * a.H)), block(64 * ((a.Sq + kRows - 1) / kRows));
    if (D == 128) hipLaunchKernelGGL((fa_short_kernel<T, 128>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((fa_short_kernel<T, 64>), grid, block, 0, s, a);
    return check_launch("flash_attention_short");
}

}  // namespace

// us, fa_flow_kernel or fa_fwd_kernel | here, a launch among others, D 64: [1,12,64] 4.7 | 4.6, [8,32,64] 5.6 | 4.5, [64,32,64] 20.0 | 17.7; D 128: [1,32,40]
// 6.0 | 4.3, [8,32,64] 8.4 | 7.4, [32,32,64] 19.9 | 18.4; GPT-2 over 37 tokens, behind a projection and with cold caches, 466 | 454.  For any number of
// heads, since a sequence keeps its bits whatever is beside it; which is also why there is no such kernel for 65 to 128 keys ([1,12,100] 5.7 | 4.8, [8,32,100]
// 6.9 | 7.8: every 16 rows read the keys again) or without the causal rule ([1,12,64] 4.9 | 4.0, D 128 [16,32,64] 10.4 | 11.5).
bool fa_short_wanted(const FaArgs& a) { return a.is_causal && a.Sq <= kRows * kMostWaves && a.Skv <= 64; }

int launch_fa_short(hipStream_t s, const FaArgs& a, int64_t D, int dtype) {
    return dtype == MHIP_BF16 ? launch_type<bf16_t>(s, a, D) : launch_type<f16_t>(s, a, D);
}

}  // namespace mhip
