// Flash-attention forward for fp32 tensors on the fp32 matrix instruction
// (v_mfma_f32_32x32x2_f32): both products and the softmax in fp32, so the result keeps the
// 1e-5 bar of the scalar kernel it replaces for head sizes 32, 64, 96 and 128 (the reference's
// flagship kernel is fp32: Metal/Kernels/FlashAttentionKernel.swift:489-613).
//
// One workgroup = four waves = 128 query rows of one (batch, head); a wave owns 32 of them
// and walks blocks of 32 keys that the workgroup stages in LDS.  Scores are computed
// transposed, S^T = K . Q^T, so that a lane holds 16 keys of ONE query column per
// accumulator: the row statistics are per-lane loops plus one exchange between the two
// 32-lane halves, and the probabilities are already laid out as the B operand of the second
// product O^T += V^T . P^T (k-step i of that product pairs key 8 (i / 4) + 4 (lane / 32) + i % 4
// of the block with the lane's own register i), so P never moves between lanes.
//
// Rows of q, k, v and o lie where the strides say: a transformer block's head split and merge around this kernel (seven
// copies of 3 us each over [1,128,768], 7 of 5 to 9 us over [4,500,1024]) are then not run.
#include <math.h>

#include <initializer_list>

#include "attention_common.h"

namespace mhip {
namespace {

typedef float f32x2 __attribute__((ext_vector_type(2)));
constexpr int kFBQ = 128;     // query rows per workgroup
constexpr int kFBK = 32;      // keys per block

// Element offset of head bh: `packed` elements a head, or where the strides say.
template <bool VIEWS>
__device__ __forceinline__ int64_t head_at(const FaArgs& a, const int64_t (&strides)[3], int bh, int64_t packed) {
    return VIEWS ? bh / a.H * strides[0] + bh % a.H * strides[1] : bh * packed;
}

// key (within a block) of accumulator register i in the 32-lane half h
__device__ __forceinline__ int f32_key(int i, int h) { return 8 * (i >> 2) + 4 * h + (i & 3); }

// VIEWS: rows lie where the strides say; without it they are packed and every row offset is a constant (strides from memory
// cost the packed tensors 1 to 4 %, [2,8,512,128] 27.7 against 28.8 us).
template <int D, bool CAUSAL, bool HAS_MASK, bool VIEWS>
__global__ __launch_bounds__(256, 2) void fa_f32_mfma_kernel(FaArgs a, float scale) {
    // K rows padded to D + 2 floats (lane = key reads fall on distinct banks), V rows to D + 8
    // (the two halves of a wave read rows four apart)
    constexpr int KS = D + 2, VS = D + 8;
    constexpr int NS = D / 2;            // k-steps of the first product
    constexpr int ND = D / 32;           // 32-column blocks of the output
    constexpr int F4 = kFBK * D / 4 / 256;   // 16-byte pieces of a K (or V) block per thread
    __shared__ __attribute__((aligned(16))) float ks[kFBK * KS];
    __shared__ __attribute__((aligned(16))) float vs[kFBK * VS];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int ln = lane & 31, h = lane >> 5;
    int bh, qb;
    tile_of_workgroup<CAUSAL>(a, blockIdx.x, bh, qb);
    const int q0 = qb * kFBQ + wave * 32;
    const int qpos = q0 + ln;                       // this lane's query row
    const bool q_live = qpos < a.Sq;
    const float* qp = static_cast<const float*>(a.q) + head_at<VIEWS>(a, a.qs, bh, a.Sq * (int64_t)D);
    const float* kp = static_cast<const float*>(a.k) + head_at<VIEWS>(a, a.ks, bh, a.Skv * (int64_t)D);
    const float* vp = static_cast<const float*>(a.v) + head_at<VIEWS>(a, a.vs, bh, a.Skv * (int64_t)D);
    float* op = static_cast<float*>(a.o) + head_at<VIEWS>(a, a.os, bh, a.Sq * (int64_t)D);
    const int64_t q_rs = VIEWS ? a.qs[2] : D, k_rs = VIEWS ? a.ks[2] : D, v_rs = VIEWS ? a.vs[2] : D, o_rs = VIEWS ? a.os[2] : D;
    const float* mp = HAS_MASK ? static_cast<const float*>(a.mask) + (int64_t)(bh / a.H) * a.mask_sb +
                                     (int64_t)(bh % a.H) * a.mask_sh + (int64_t)qpos * a.Skv
                               : nullptr;

    // Q^T fragments: k-step s holds Q[qpos][2 s + h]
    float qf[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) qf[s] = q_live ? qp[qpos * q_rs + 2 * s + h] : 0.f;

    int nkv = (a.Skv + kFBK - 1) / kFBK;
    if (CAUSAL) {
        const int last_q = min(qb * kFBQ + kFBQ, a.Sq) - 1;
        nkv = min(nkv, last_q / kFBK + 1);
    }
    const int last_wave_q = min(q0 + 32, a.Sq) - 1;   // causal: blocks past it add nothing for this wave

    f32x16 o[ND];
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[d][i] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;            // l_run: this lane's 16 keys of every block

    // this thread's pieces of a block: piece p covers floats 4 p .. 4 p + 3 of the [32][D] block
    f32x4 kr[F4], vr[F4];
    auto fetch = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < F4; j++) {
            const int p = j * 256 + tid, row = p / (D / 4), col = (p % (D / 4)) * 4;
            const int key = blk * kFBK + row;
            if (key < a.Skv) {
                kr[j] = *reinterpret_cast<const f32x4*>(kp + key * k_rs + col);
                vr[j] = *reinterpret_cast<const f32x4*>(vp + key * v_rs + col);
            } else {
                kr[j] = f32x4{0.f, 0.f, 0.f, 0.f};
                vr[j] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
    };
    auto stage = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < F4; j++) {
            const int p = j * 256 + tid, row = p / (D / 4), col = (p % (D / 4)) * 4;
            float* kd = ks + row * KS + col;           // 8-byte aligned: two stores
            *reinterpret_cast<f32x2*>(kd) = f32x2{kr[j].x, kr[j].y};
            *reinterpret_cast<f32x2*>(kd + 2) = f32x2{kr[j].z, kr[j].w};
            *reinterpret_cast<f32x4*>(vs + row * VS + col) = vr[j];
        }
    };

    if (nkv > 0) fetch(0);
    for (int blk = 0; blk < nkv; blk++) {
        __syncthreads();                               // the previous block has been read by every wave
        stage();
        __syncthreads();
        if (blk + 1 < nkv) fetch(blk + 1);             // in flight while this block is worked on
        const int kb = blk * kFBK;
        if (CAUSAL && kb > last_wave_q) continue;      // (uniform within the wave; the barriers stay in step)

        // ---- S^T = K . Q^T
        f32x16 sacc;
#pragma unroll
        for (int i = 0; i < 16; i++) sacc[i] = 0.f;
#pragma unroll
        for (int s = 0; s < NS; s++)
            sacc = __builtin_amdgcn_mfma_f32_32x32x2f32(ks[ln * KS + 2 * s + h], qf[s], sacc, 0, 0, 0);

        // ---- scale, mask, block maximum (log2 domain unless there is a mask)
        float t[16];
        float m_blk = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int key = kb + f32_key(i, h);
            float sv = sacc[i] * scale;
            bool keep = key < a.Skv && q_live;
            if (CAUSAL) keep = keep && key <= qpos;
            if (HAS_MASK) { if (keep) sv += mp[key]; }
            t[i] = keep ? (HAS_MASK ? sv : sv * kLog2e) : -INFINITY;
            m_blk = fmaxf(m_blk, t[i]);
        }
        m_blk = half_max(m_blk);
        // (a reference maximum that moves only when the block exceeds it by 2^8: see moved_reference)
        const float m_new = moved_reference<HAS_MASK>(m_run, m_blk);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        // (v_exp_f32 itself, about 1 ulp: the library exp2f wraps it in five more instructions that
        // only serve results below 2^-126, which are zeros here either way)
        const float alpha = weight<HAS_MASK>(m_run, m_use);
        m_run = m_new;
        float psum = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            t[i] = weight<HAS_MASK>(t[i], m_use);
            psum += t[i];
        }
        l_run = l_run * alpha + psum;
        if (__any(alpha != 1.f)) {                     // rare once the reference has settled
#pragma unroll
            for (int d = 0; d < ND; d++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[d][i] *= alpha;
        }

        // ---- O^T += V^T . P^T
#pragma unroll
        for (int d = 0; d < ND; d++)
#pragma unroll
            for (int i = 0; i < 16; i++)
                o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vs[f32_key(i, h) * VS + 32 * d + ln], t[i], o[d], 0, 0, 0);
    }

    // ---- normalise and store: register group i / 4 of block d holds columns
    // 32 d + 8 (i / 4) + 4 h .. + 3 of row qpos
    const float l_tot = half_sum(l_run);
    const float inv = l_tot > 1e-10f ? 1.f / l_tot : 0.f;
    if (q_live) {
        float* orow = op + qpos * o_rs;
#pragma unroll
        for (int d = 0; d < ND; d++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const f32x4 w = {o[d][4 * g] * inv, o[d][4 * g + 1] * inv, o[d][4 * g + 2] * inv, o[d][4 * g + 3] * inv};
                *reinterpret_cast<f32x4*>(orow + 32 * d + 8 * g + 4 * h) = w;
            }
    }
}

// The same products with the KEYS dealt over the waves: a workgroup owns 32 query rows, wave w takes blocks w, w + 4, ...
// of 32 keys and its own softmax state, and the four meet in LDS at the end.  Four times as many workgroups, each
// with a quarter of the chain; K and V go from memory straight to the operand registers (a lane's 16 bytes of
// its key's row serve four issues: k = 8 j + 4 h + e on both operands), so there is no barrier in the loop, and
// each set of registers is loaded again as soon as its product has read it, half a block ahead of its use.
template <int D, bool CAUSAL, bool HAS_MASK, bool VIEWS>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void fa_f32_split_kernel(FaArgs a, float scale) {
    constexpr int NS = D / 8, ND = D / 32;
    __shared__ float part[4][32][33];
    __shared__ float ml[2][4][32];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ln = lane & 31, h = lane >> 5;
    int bh, qb;
    tile_of_workgroup<CAUSAL>(a, blockIdx.x, bh, qb);
    const int q0 = qb * 32, qpos = q0 + ln;
    const bool q_live = qpos < a.Sq;
    const float* qp = static_cast<const float*>(a.q) + head_at<VIEWS>(a, a.qs, bh, a.Sq * (int64_t)D);
    const int64_t q_rs = VIEWS ? a.qs[2] : D, o_rs = VIEWS ? a.os[2] : D;
    const int k_rs = VIEWS ? (int)a.ks[2] : D, v_rs = VIEWS ? (int)a.vs[2] : D;
    const __amdgpu_buffer_rsrc_t rk = fa_rsrc(static_cast<const float*>(a.k) + head_at<VIEWS>(a, a.ks, bh, a.Skv * (int64_t)D), (uint32_t)((((int64_t)a.Skv - 1) * k_rs + D) * 4));
    const __amdgpu_buffer_rsrc_t rv = fa_rsrc(static_cast<const float*>(a.v) + head_at<VIEWS>(a, a.vs, bh, a.Skv * (int64_t)D), (uint32_t)((((int64_t)a.Skv - 1) * v_rs + D) * 4));
    const float* mp = HAS_MASK ? static_cast<const float*>(a.mask) + (int64_t)(bh / a.H) * a.mask_sb +
                                     (int64_t)(bh % a.H) * a.mask_sh + (int64_t)min(qpos, a.Sq - 1) * a.Skv
                               : nullptr;
    // (a lane's keys of a block are four runs of four, loaded whole; in the last block of a row that is no multiple of four a
    // run may leave the mask: element by element)
    const bool whole_runs = a.Skv % 4 == 0;
    f32x4 qf[NS];
#pragma unroll
    for (int j = 0; j < NS; j++)
        qf[j] = q_live ? *reinterpret_cast<const f32x4*>(qp + qpos * q_rs + 8 * j + 4 * h) : f32x4{0.f, 0.f, 0.f, 0.f};

    int nkv = (a.Skv + kFBK - 1) / kFBK;
    if (CAUSAL) nkv = min(nkv, qb + 1);

    // (keys past the end lie beyond the buffers' extents and read zero)
    f32x4 kr[NS];
    float vr[ND][16];
    auto load_k = [&](int blk) __attribute__((always_inline)) {
        const uint32_t off = (uint32_t)((blk * kFBK + ln) * (k_rs * 4) + 16 * h);
#pragma unroll
        for (int j = 0; j < NS; j++) kr[j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, off + 32 * j, 0, 0));
    };
    // (a key's row is part of the vector offset: a scalar offset is outside the bounds check, and keys past the end must read zero)
    auto load_v = [&](int blk) __attribute__((always_inline)) {
        const uint32_t off = (uint32_t)((blk * kFBK + 4 * h) * (v_rs * 4) + 4 * ln);
#pragma unroll
        for (int i = 0; i < 16; i++)
#pragma unroll
            for (int d = 0; d < ND; d++)
                vr[d][i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rv, off + (uint32_t)((8 * (i >> 2) + (i & 3)) * (v_rs * 4) + 128 * d), 0, 0));
    };

    f32x16 o[ND];
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[d][i] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;
    if (wave < nkv) { load_k(wave); load_v(wave); }
    for (int blk = wave; blk < nkv; blk += 4) {
        const int kb = blk * kFBK;
        f32x4 mrun[HAS_MASK ? 4 : 1];
        const bool mask_runs = HAS_MASK && (whole_runs || kb + kFBK <= a.Skv);
        if (mask_runs) {
#pragma unroll
            for (int g = 0; g < 4; g++) __builtin_memcpy(&mrun[HAS_MASK ? g : 0], mp + min(kb + 8 * g + 4 * h, a.Skv - 4), 16);
        }
        f32x16 sacc;
#pragma unroll
        for (int i = 0; i < 16; i++) sacc[i] = 0.f;
#pragma unroll
        for (int j = 0; j < NS; j++)
#pragma unroll
            for (int e = 0; e < 4; e++) sacc = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[j][e], qf[j][e], sacc, 0, 0, 0);
        if (blk + 4 < nkv) load_k(blk + 4);
        float t[16];
        float m_blk = -INFINITY;
        const bool edge = (CAUSAL && kb + kFBK - 1 > q0) || kb + kFBK > a.Skv;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const int key = kb + f32_key(i, h);
            float sv = sacc[i] * scale;
            const bool keep = !edge || (key < a.Skv && (!CAUSAL || key <= qpos));
            if (HAS_MASK) sv += mask_runs ? mrun[HAS_MASK ? i >> 2 : 0][i & 3] : key < a.Skv ? mp[key] : 0.f;
            t[i] = keep ? (HAS_MASK ? sv : sv * kLog2e) : -INFINITY;
            m_blk = fmaxf(m_blk, t[i]);
        }
        m_blk = half_max(m_blk);
        const float m_new = moved_reference<HAS_MASK>(m_run, m_blk);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = weight<HAS_MASK>(m_run, m_use);
        m_run = m_new;
        float psum = 0.f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            t[i] = weight<HAS_MASK>(t[i], m_use);
            psum += t[i];
        }
        l_run = l_run * alpha + psum;
        if (__any(alpha != 1.f)) {
#pragma unroll
            for (int d = 0; d < ND; d++)
#pragma unroll
                for (int i = 0; i < 16; i++) o[d][i] *= alpha;
        }
#pragma unroll
        for (int i = 0; i < 16; i++)
#pragma unroll
            for (int d = 0; d < ND; d++) o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[d][i], t[i], o[d], 0, 0, 0);
        if (blk + 4 < nkv) load_v(blk + 4);
    }

    // ---- the waves' states, 32 columns of the output at a time
    l_run = half_sum(l_run);
    if (h == 0) { ml[0][wave][ln] = m_run; ml[1][wave][ln] = l_run; }
    float* op = static_cast<float*>(a.o) + head_at<VIEWS>(a, a.os, bh, a.Sq * (int64_t)D);
    const int col = threadIdx.x & 31, row0 = threadIdx.x >> 5;
#pragma unroll
    for (int d = 0; d < ND; d++) {
        if (d) __syncthreads();
#pragma unroll
        for (int i = 0; i < 16; i++) part[wave][ln][f32_key(i, h)] = o[d][i];
        __syncthreads();
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const int q = row0 + 8 * p;
            float m = -INFINITY, l = 0.f, sum = 0.f;
#pragma unroll
            for (int w = 0; w < 4; w++) m = fmaxf(m, ml[0][w][q]);
            const float m_use = m == -INFINITY ? 0.f : m;
#pragma unroll
            for (int w = 0; w < 4; w++) {
                const float al = weight<HAS_MASK>(ml[0][w][q], m_use);
                l = fmaf(ml[1][w][q], al, l);
                sum = fmaf(part[w][q][col], al, sum);
            }
            if (q0 + q < a.Sq) op[(q0 + q) * o_rs + 32 * d + col] = sum * (l > 1e-10f ? 1.f / l : 0.f);
        }
    }
}

template <int D, bool V>
int launch_f32(hipStream_t s, FaArgs a, float scale, bool causal, bool has_mask) {
    // Keys over the waves while tiles of 128 rows leave compute units idle or nearly so (us, 128 rows | split, causal):
    // 12 tiles [1,12,128,64] 16.2 | 7.6; 64 [2,8,512,64] 48 | 16, D 128 83 | 29; 128 [1,8,2048,64] 175 | 50, D 128 302 | 114.
    // From 256 on every wave re-reading K and V costs more than the shorter chain gives (256 tiles of D 96 40 | 48, 1024 of
    // D 128 621 | 738), except where rows are short or keys many: 1024 tiles of D 32 174 | 165, 384 of [4,12,1000,64] 100 | 78
    // (768 of [16,12,512,64] 81 | 95).
    const int64_t tiles = (int64_t)a.B * a.H * ((a.Sq + kFBQ - 1) / kFBQ);
    const bool split = ((int64_t)a.Skv + kFBQ) * (a.ks[2] > a.vs[2] ? a.ks[2] : a.vs[2]) * 4 < 0x7FFFFFFFLL &&
                       (tiles < 256 || (D == 32 && tiles <= 1024) || (D == 64 && tiles <= 512 && a.Skv >= 768));
    const int rows = split ? 32 : kFBQ;
    a.nqb = (a.Sq + rows - 1) / rows;
    set_tile_order(a);
    const int64_t grid = (int64_t)a.B * a.H * a.nqb;
    if (grid > 0x7FFFFFFFLL) return fail(MHIP_ERR_UNSUPPORTED, "flash_attention: grid too large");
#define MHIP_FA32(C, M)                                                                                                     \
    do {                                                                                                                    \
        if (split) hipLaunchKernelGGL((fa_f32_split_kernel<D, C, M, V>), dim3((unsigned)grid), dim3(256), 0, s, a, scale);  \
        else hipLaunchKernelGGL((fa_f32_mfma_kernel<D, C, M, V>), dim3((unsigned)grid), dim3(256), 0, s, a, scale);         \
    } while (0)
    if (causal && has_mask) MHIP_FA32(true, true);
    else if (causal) MHIP_FA32(true, false);
    else if (has_mask) MHIP_FA32(false, true);
    else MHIP_FA32(false, false);
#undef MHIP_FA32
    return check_launch("flash_attention_f32");
}

}  // namespace

// fp32, [B,H,S,D] with strides that are multiples of 4 elements, head size a multiple of 32 up to 128, 16-byte aligned tensors.
// MHIP_FA_F32_MFMA=2 keeps the scalar kernel for packed tensors, the only ones it reads.
bool fa_f32_mfma_eligible(const FaArgs& a, int64_t D, bool packed) {
    if (packed && tune_int("MHIP_FA_F32_MFMA", 1) == 2) return false;
    if (D % 32 != 0 || D > 128 || a.Skv < 1) return false;
    const uintptr_t all = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k) |
                          reinterpret_cast<uintptr_t>(a.v) | reinterpret_cast<uintptr_t>(a.o);
    if ((all & 15) != 0) return false;
    for (const int64_t* st : {a.qs, a.ks, a.vs, a.os})
        for (int i = 0; i < 3; i++)
            if (st[i] % 4 != 0) return false;
    return true;
}

int launch_fa_f32_mfma(hipStream_t s, const FaArgs& a, int64_t D, float scale, bool packed) {
    const bool causal = a.is_causal != 0, has_mask = a.mask != nullptr;
    switch (D) {
        case 32: return packed ? launch_f32<32, false>(s, a, scale, causal, has_mask) : launch_f32<32, true>(s, a, scale, causal, has_mask);
        case 64: return packed ? launch_f32<64, false>(s, a, scale, causal, has_mask) : launch_f32<64, true>(s, a, scale, causal, has_mask);
        case 96: return packed ? launch_f32<96, false>(s, a, scale, causal, has_mask) : launch_f32<96, true>(s, a, scale, causal, has_mask);
        default: return packed ? launch_f32<128, false>(s, a, scale, causal, has_mask) : launch_f32<128, true>(s, a, scale, causal, has_mask);
    }
}

}  // namespace mhip
