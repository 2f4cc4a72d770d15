// Flash-attention forward without a mask operand for 16-bit head sizes 64 and 128: the products and the recurrence of
// attention.hip's fa_fwd_kernel (same tiles, same order of every sum, same bits), one block of keys further apart.
//
// A block of 64 keys costs a wave 16 matrix instructions of 32 cycles (D 64) and about 170 others, 32 of them
// exponentials of 8: about 950 cycles where the two kinds run side by side, 1500 one after the other, and a barrier, LDS
// latencies and the way to the row's maximum on top.  fa_fwd_kernel issues them one after the other and lets the three waves
// of a SIMD make up for it; with fewer tiles there is one wave, and a block takes it 0.87 us.  Here the scores of block i + 1
// are formed BETWEEN the maximum and the exponentials of block i, and the product with V of every sixteen keys as soon as their
// weights exist, in segments that the scheduler may not cross: 0.68 us, of which the four segments are 0.43.
#include <type_traits>

#include "attention_common.h"

namespace mhip {
namespace {

// A ring of NB tiles for K and for V; K's tiles are a block ahead of V's.
//
// Nothing may be spilled: a reload waits for every load in flight, the tiles just asked for among them.  With head size 128 and no
// causal rule the compiler does not fit a wave into the 256 registers of two workgroups a unit (9 spilled, [1,12,1024] 34.3 us);
// one workgroup a unit has 512 (25.3; fa_fwd_kernel 26.4).
template <typename T, int D, bool CAUSAL>
__global__ __launch_bounds__(256, D == 128 && !CAUSAL ? 1 : 2) void fa_flow_kernel(FaArgs a) {
    constexpr int NB = 2;
    constexpr int CPR = D / 8;                  // 16-byte chunks per row
    constexpr int kTile = kBKV * D * 2;         // bytes of one K (or V) tile
    constexpr int kRowsPerInst = 64 / CPR;      // tile rows one wave-wide LDS-DMA load fills
    constexpr int kInst = kBKV / kRowsPerInst / 4;   // such loads per wave per tile
    constexpr int ND = D / 32, NS = D / 16;
    constexpr int NQ = 2 * NS;                  // matrix instructions of the scores
    __shared__ __attribute__((aligned(1024))) char smem[2 * NB * kTile];

    int bh, qb;
    tile_of_workgroup<CAUSAL, false>(a, blockIdx.x, bh, qb);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lrow = lane & 31, lhalf = lane >> 5;
    const int qblk0 = qb * kBQ;
    const int qw = qblk0 + wave * 32;          // first query row of this wave
    const int qpos = qw + lrow;

    const int b_i = bh / a.H, h_i = bh % a.H;
    const T* qp = static_cast<const T*>(a.q) + b_i * a.qs[0] + h_i * a.qs[1];
    const T* kp = static_cast<const T*>(a.k) + b_i * a.ks[0] + h_i * a.ks[1];
    const T* vp = static_cast<const T*>(a.v) + b_i * a.vs[0] + h_i * a.vs[1];
    T* op = static_cast<T*>(a.o) + b_i * a.os[0] + h_i * a.os[1];
    const int q_rs = (int)a.qs[2], k_rs = (int)a.ks[2], v_rs = (int)a.vs[2];      // row pitches in elements
    const __amdgpu_buffer_rsrc_t rq = fa_rsrc(qp, (uint32_t)((((int64_t)a.Sq - 1) * q_rs + D) * 2));
    int nkv = (a.Skv + kBKV - 1) / kBKV;
    if (CAUSAL) nkv = min(nkv, (min(qblk0 + kBQ, a.Sq) - 1) / kBKV + 1);
    // (the last block's loads ask for blocks behind it: nothing is fetched past the keys this workgroup sees)
    const int keys = CAUSAL ? min(a.Skv, nkv * kBKV) : a.Skv;
    const __amdgpu_buffer_rsrc_t rk = fa_rsrc(kp, (uint32_t)((((int64_t)keys - 1) * k_rs + D) * 2));
    const __amdgpu_buffer_rsrc_t rv = fa_rsrc(vp, (uint32_t)((((int64_t)keys - 1) * v_rs + D) * 2));

    // ---- Q^T operand: lane = query column, 8 consecutive d per k-step
    u32x4 qf[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        qf[s] = __builtin_amdgcn_raw_buffer_load_b128(rq, qpos < a.Sq ? (uint32_t)((qpos * q_rs + 16 * s + 8 * lhalf) * 2) : kOobA, 0, 0);
        if (a.negate_q) {
            qf[s].x ^= 0x80008000u; qf[s].y ^= 0x80008000u;
            qf[s].z ^= 0x80008000u; qf[s].w ^= 0x80008000u;
        }
    }

    // blocks that this wave multiplies: the rest of the workgroup's it only helps to load
    const int mine = CAUSAL ? min(nkv, (qw + 31) / kBKV + 1) : nkv;

    // ---- global -> LDS without a register stop: every wave-wide load fills 1 KB of a tile (lane l lands at byte 16 l of
    // that KB); the swizzle is applied by choosing which global chunk each lane fetches.  Keys past the end lie
    // beyond the descriptors' extents and put zeros into LDS.  Every step issues the same number of loads (the waits
    // count them), blocks past the last one included.
    const int ld_row = wave * kRowsPerInst + lane / CPR, ld_pos = lane % CPR;
    const uint32_t koff0 = (uint32_t)((ld_row * k_rs + ((ld_pos ^ k_swz<D>(ld_row)) << 3)) * 2);
    const uint32_t voff0 = (uint32_t)((ld_row * v_rs + ((ld_pos ^ v_swz<D>(ld_row)) << 3)) * 2);
    const uint32_t ring = fa_lds_address(smem);
    auto slot = [](int blk) __attribute__((always_inline)) { return (NB & (NB - 1)) == 0 ? blk & (NB - 1) : blk % NB; };
    auto load_k = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kInst; i++)
            fa_load_to_lds(rk, ring + (uint32_t)(slot(blk) * kTile + (i * 4 + wave) * 1024), koff0 + (uint32_t)(blk * kBKV + i * 4 * kRowsPerInst) * (uint32_t)(k_rs * 2));
    };
    auto load_v = [&](int blk) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < kInst; i++)
            fa_load_to_lds(rv, ring + (uint32_t)((NB + slot(blk)) * kTile + (i * 4 + wave) * 1024), voff0 + (uint32_t)(blk * kBKV + i * 4 * kRowsPerInst) * (uint32_t)(v_rs * 2));
    };
    // loads land in program order: K of the next block but one and V of the next have landed when only the pairs issued behind
    // them are in flight
    auto tiles_ready = [&]() __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NB - 2) * 2 * kInst) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    // V^T fragment addresses: lane i of a 16-lane group supplies key row i/4 and d columns 4*(i%4)..+3 of its group's
    // 16-column block.
    const int ti = lane & 15, tg = lane >> 4;
    const int v_row0 = 4 * (tg >> 1) + (ti >> 2), v_d0 = 16 * (tg & 1) + 4 * (ti & 3);      // + 16u (+ 8), + 32 dt
    auto v_frag = [&](const char* vt, int u, int dt) __attribute__((always_inline)) {
        const int row = 16 * u + v_row0, d0 = 32 * dt + v_d0;
        const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((fa_lds_s16x4*)(vt + v_off<D>(row, d0 >> 3) + (d0 & 7) * 2)));
        const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((fa_lds_s16x4*)(vt + v_off<D>(row + 8, d0 >> 3) + (d0 & 7) * 2)));
        return u32x4{lo.x, lo.y, hi.x, hi.y};
    };
    auto k_frag = [&](const char* kt, int m) __attribute__((always_inline)) {      // operand of score instruction m
        return *reinterpret_cast<const u32x4*>(kt + k_off<D>(32 * (m & 1) + lrow, 2 * (m >> 1) + lhalf));
    };

    f32x16 oacc[ND];
#pragma unroll
    for (int i = 0; i < ND; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[i][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;   // reference maximum in the log2 domain (see moved_reference), running sum
    f32x16 even[2], odd[2], zero;           // scores of the block at hand and of the next
#pragma unroll
    for (int r = 0; r < 16; r++) zero[r] = 0.f;

    load_k(0);
#pragma unroll
    for (int p = 0; p < NB - 1; p++) { load_k(p + 1); load_v(p); }
    tiles_ready();
#pragma unroll
    for (int m = 0; m < NQ; m++) even[m & 1] = Mfma32A<T>::run(k_frag(smem, m), qf[m >> 1], m < 2 ? zero : even[m & 1]);

    // Block `it`, whose scores are in `cur`; those of the block behind it go to `next` (behind the last block of this wave of
    // whatever K holds: they are dropped).
    auto step = [&](int it, f32x16(&cur)[2], f32x16(&next)[2]) __attribute__((always_inline)) {
        // K of block it + 1 and V of block it have landed; every wave has read the tiles whose places are reused
        if (it) tiles_ready();
        else {
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        load_k(it + NB);
        load_v(it + NB - 1);
        if (it >= mine) return;
        const int kv0 = it * kBKV;
        const char* kt = smem + slot(it + 1) * kTile;
        const char* vt = smem + (NB + slot(it)) * kTile;
        constexpr int Q = NQ / 4;                       // score instructions of a quarter
        u32x4 kf[2][Q];
        auto read_k = [&](int j) __attribute__((always_inline)) {
#pragma unroll
            for (int m = 0; m < Q; m++) kf[j & 1][m] = k_frag(kt, j * Q + m);
        };
        auto quarter = [&](int j) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < Q; i++) {
                const int m = j * Q + i;
                next[m & 1] = Mfma32A<T>::run(kf[j & 1][i], qf[m >> 1], m < 2 ? zero : next[m & 1]);
            }
        };
        read_k(0);
        read_k(1);

        // Register i of the pair (t = i/16, r = i%16) is key kv0 + 32t + 8(r/4) + 4*lhalf + r%4 of query column qpos.
        float scale_s = a.c;
        const bool boundary = (CAUSAL && kv0 + kBKV - 1 > qw) || kv0 + kBKV > a.Skv;
        if (boundary) {
            // scores to the log2 domain first, then mask
#pragma unroll
            for (int i = 0; i < 32; i++) {
                const int key = kv0 + 32 * (i >> 4) + 8 * ((i & 15) >> 2) + 4 * lhalf + (i & 3);
                cur[i >> 4][i & 15] = (CAUSAL && key > qpos) || key >= a.Skv ? -INFINITY : cur[i >> 4][i & 15] * a.c;
            }
            scale_s = 1.f;
        }
        // the maximum over raw scores otherwise (the scale is positive), scale and shift in one fma in front of the exp2
        float mloc = cur[0][0];
#pragma unroll
        for (int i = 1; i < 32; i++) mloc = fmaxf(mloc, cur[i >> 4][i & 15]);
        quarter(0);
#pragma unroll
        for (int i = 0; i < Q; i++) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
            __builtin_amdgcn_sched_group_barrier(0x002, 16 / Q, 1);
        }
        mloc = half_max(mloc);
        const float m_new = moved_reference(m_run, mloc * scale_s);
        const float m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
        m_run = m_new;
        const float shift = boundary ? -m_use : -m_new;
        // the accumulator only needs rescaling when some row's maximum moved
        if (__any(alpha != 1.f)) {
#pragma unroll
            for (int i = 0; i < ND; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) oacc[i][r] *= alpha;
        }
        float lsum = 0.f;
        u32x4 pb[2];
        auto weights = [&](int u) __attribute__((always_inline)) {
            float w[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                w[i] = __builtin_amdgcn_exp2f(fmaf(cur[u >> 1][8 * (u & 1) + i], scale_s, shift));
                lsum += w[i];
            }
#pragma unroll
            for (int e = 0; e < 4; e++) pb[u & 1][e] = Mfma32A<T>::pack2(w[2 * e], w[2 * e + 1]);
        };
        // the operands of the next segment on their way, then one matrix instruction after the other, each with as much
        // arithmetic behind it as it lasts
        auto interleave = [&](auto ds_tag, auto n_tag) __attribute__((always_inline)) {
            constexpr int kDs = decltype(ds_tag)::value, N = decltype(n_tag)::value;
            __builtin_amdgcn_sched_group_barrier(0x100, kDs, 0);
#pragma unroll
            for (int i = 0; i < N; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x402, 28 / N, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        u32x4 vf[2][ND];
        __builtin_amdgcn_sched_barrier(0);
        // ---- four segments: a quarter of the next scores, sixteen keys' weights, the product with V of the keys before
#pragma unroll
        for (int u = 0; u < 4; u++) {
            if (u < 2) read_k(u + 2);
#pragma unroll
            for (int dt = 0; dt < ND; dt++) vf[u & 1][dt] = v_frag(vt, u, dt);
            if (u > 0) {
#pragma unroll
                for (int dt = 0; dt < ND; dt++) oacc[dt] = Mfma32A<T>::run(vf[1 - (u & 1)][dt], pb[1 - (u & 1)], oacc[dt]);
            }
            if (u < 3) quarter(u + 1);
            weights(u);
            if (u == 0) interleave(std::integral_constant<int, Q + 2 * ND>{}, std::integral_constant<int, Q>{});
            else if (u == 1) interleave(std::integral_constant<int, Q + 2 * ND>{}, std::integral_constant<int, ND + Q>{});
            else if (u == 2) interleave(std::integral_constant<int, 2 * ND>{}, std::integral_constant<int, ND + Q>{});
            else interleave(std::integral_constant<int, 2 * ND>{}, std::integral_constant<int, ND>{});
        }
#pragma unroll
        for (int dt = 0; dt < ND; dt++) oacc[dt] = Mfma32A<T>::run(vf[1][dt], pb[1], oacc[dt]);
        l_run = l_run * alpha + lsum;
    };
    // (two blocks a turn save 32 copies each; with head size 128 they cost registers that are not there)
    for (int it = 0; it < nkv; it++) {
        step(it, even, odd);
        if (D == 64) {
            if (++it < nkv) step(it, odd, even);
        } else {
#pragma unroll
            for (int t = 0; t < 2; t++) even[t] = odd[t];
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may land in LDS after the workgroup ends

    // ---- normalise and store: lane holds 4 consecutive d per register group
    // (half_sum with the lane's half counted anew: kept from the start it was the one register too many of head size 128, causal)
    const unsigned lsum = __builtin_bit_cast(unsigned, l_run);
    const auto lr = __builtin_amdgcn_permlane32_swap(lsum, lsum, false, false);
    const int el = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    const float l_tot = l_run + __builtin_bit_cast(float, (el & 32) ? lr[0] : lr[1]);
    const float inv = l_tot > 1e-10f ? 1.f / l_tot : 0.f;
    if (qpos < a.Sq) {
        T* orow = op + (int64_t)qpos * a.os[2];
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
}

template <typename T, int D>
int launch_form(hipStream_t s, const FaArgs& a, unsigned grid) {
    if (a.is_causal) hipLaunchKernelGGL((fa_flow_kernel<T, D, true>), dim3(grid), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((fa_flow_kernel<T, D, false>), dim3(grid), dim3(256), 0, s, a);
    return check_launch("flash_attention");
}

}  // namespace

// 16-bit q, k, v, o of head size 64 or 128 with 16-byte aligned rows and no mask, while the workgroups that a compute unit keeps
// hold all tiles: two, or one with head size 128 and no causal rule (see the kernel).  Beyond that the third workgroup of D 64 that
// fa_fwd_kernel keeps on a unit is worth more, and so it is, for more than one workgroup a unit, where the longest tile has
// few blocks of keys: what is fetched ahead is then most of what there is.  us, fa_fwd_kernel | this one:
//   D 64   causal  [1,12,1024] (96 tiles) 18.1 | 15.5, [4,8,1000] (256) 18.4 | 16.1, [3,12,1000] (288) 18.8 | 16.5, [8,8,1000] (512) 19.7 | 17.8,
//                  [1,8,4096] (256) 57.4 | 47.3, [9,8,1000] (576) 20.7 | 20.1, [10,8,1000] (640) 21.3 | 22.5; by blocks of keys [8,32,16] (256, 1 block)
//                  4.5 | 4.6, [1,12,100] (12, 2) 6.0 | 5.8, [16,32,128] (512, 2) 10.0 | 10.3, [8,32,256] (512, 4) 10.7 | 10.9, [4,32,500] (512, 8) 13.3 | 12.6
//          else    [1,12,1024] 17.4 | 14.8, [8,8,1000] 26.6 | 25.0, [9,8,1000] 32.9 | 34.1, 300 queries over 3000 keys (48) 42.2 | 34.3; [1,12,64] (12, 1)
//                  4.3 | 4.1, [8,32,64] (256, 1) 4.7 | 4.5, [16,32,64] over 37 keys (512, 1) 5.2 | 5.4, [8,32,192] (512, 3) 10.0 | 9.7
//   D 128  causal  [1,8,512] (32) 15.8 | 15.0, [2,8,1000] (128) 25.8 | 24.4, [2,4,4096] (256) 85.2 | 80.4, [6,8,1000] (384) 27.9 | 26.6, [8,8,1000] (512)
//                  33.9 | 33.9; [8,32,128] (256, 2) 10.7 | 10.9, [2,32,192] (128, 3) 9.3 | 8.9, [12,32,128] (384, 2) 13.9 | 14.6
//          else    [1,8,512] 15.7 | 15.2, [2,8,1000] 26.6 | 25.6, [2,4,4096] 88.2 | 84.3, 100 queries over 2000 keys (256) 65.6 | 56.9, [6,8,1000] (384)
//                  37.8 | 49.4; [8,32,128] (256, 2) 10.9 | 11.2
bool fa_flow_wanted(const FaArgs& a, int64_t D) {
    const int64_t tiles = (int64_t)a.B * a.H * ((a.Sq + kBQ - 1) / kBQ), cus = compute_units();
    const int blocks = ((a.is_causal && a.Sq < a.Skv ? a.Sq : a.Skv) + kBKV - 1) / kBKV;
    if (tiles <= cus) return blocks >= (D == 128 ? 3 : a.is_causal ? 2 : 1);
    return tiles <= 2 * cus && (a.is_causal ? blocks >= 5 : D == 64 && blocks >= 3);
}

int launch_fa_flow(hipStream_t s, FaArgs a, int64_t D, int dtype) {
    a.nqb = (a.Sq + kBQ - 1) / kBQ;
    set_tile_order(a);
    const unsigned grid = (unsigned)(a.B * a.H * a.nqb);
    if (dtype == MHIP_BF16) return D == 64 ? launch_form<bf16_t, 64>(s, a, grid) : launch_form<bf16_t, 128>(s, a, grid);
    return D == 64 ? launch_form<f16_t, 64>(s, a, grid) : launch_form<f16_t, 128>(s, a, grid);
}

}  // namespace mhip
