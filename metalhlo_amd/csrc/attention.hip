// Flash-attention forward for gfx950: O = softmax(scale * Q K^T + mask, causal) V.
//
// MFMA path (16-bit types, D a multiple of 8 up to 128).  A workgroup of four waves owns 128
// query rows of one (batch, head); each wave owns 32 of them.  Keys/values are
// walked in blocks of 64, staged in LDS and double-buffered.
//
// The scores are computed TRANSPOSED, S^T = K . Q^T, with v_mfma_f32_32x32x16:
// in the accumulator layout every lane then holds 16 keys of ONE query column,
// so the online-softmax row statistics are plain per-lane loops plus a single
// exchange between the two 32-lane halves, and the probabilities can be fed
// straight back as the B operand of O^T += V^T . P^T without any cross-lane
// movement.  V is transposed (and its keys put in the order that B operand
// needs) in registers on the way into LDS.  Softmax state and both
// accumulations are fp32; the output is rounded once.
//
// Head sizes other than 64 and 128 lie in LDS rows of 64 or 128 (the pieces behind the row's end are zeros) and
// skip the matrix steps of whole blocks of 32 d that do not exist.  Their probabilities go through the second product
// with all of their fp32 bits, as three bf16 parts; f16 values as two bf16 parts, which holds them exactly too.
//
// On B4 H12 S1000 causal against the scalar path: bf16 D 96 729 -> 34.3 us, D 32 346 -> 20.2; f16 D 96 51.8, D 32 25.7
// (two products per part, and V split in registers).  Parts are cut off, not rounded: a conversion to bf16 pairs costs
// as much as four simple instructions (35.6 and 20.6 us with it), and what is left is exact either way.  Share of the
// results that are not the number nearest to the 64-bit one, scalar path / here, D 96: bf16 0.0003 / 0.0002, f16 0.0027 /
// 0.0016; with two parts of the weights bf16 was at 0.0023.
//
// Everything else (unaligned tensors, larger heads) takes a wave-per-query scalar path.
#include <type_traits>

#include "attention_common.h"

namespace mhip {

template <typename T> struct alignas(4) Pair16 { T v[2]; };

// One query row by one wave, q, k, v, o packed: per block of 64 keys, lanes own keys for the scores, then own head-dim
// columns for the weighted sum.  The recurrence is the reference's (FlashAttentionKernel.swift:589-598) applied per
// block of keys; a causally hidden key is never read.  `qs` (256 floats) and `ps` (64): LDS of the wave's own.
template <typename T>
__device__ inline void fa_row(const FaArgs& a, int64_t bh, int qpos, int D, float scale, float* qs, float* ps) {
    const int lane = threadIdx.x & 63;
    const T* qp = static_cast<const T*>(a.q) + (bh * a.Sq + qpos) * D;
    const T* kp = static_cast<const T*>(a.k) + bh * a.Skv * D;
    const T* vp = static_cast<const T*>(a.v) + bh * a.Skv * D;
    const T* mp = a.mask ? static_cast<const T*>(a.mask) + (bh / a.H) * a.mask_sb +
                               (bh % a.H) * a.mask_sh + (int64_t)qpos * a.Skv
                         : nullptr;
    for (int d = lane; d < D; d += 64) qs[d] = Elem<T>::to_f32(qp[d]);
    __builtin_amdgcn_wave_barrier();
    float oacc[4] = {0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;
    const int kv_end = a.is_causal ? min(a.Skv, qpos + 1) : a.Skv;
    for (int kv0 = 0; kv0 < kv_end; kv0 += 64) {
        const int key = kv0 + lane;
        float s = -INFINITY;
        if (key < kv_end) {
            float acc = 0.f;
            const T* kr = kp + (int64_t)key * D;
            for (int d = 0; d < D; d++) acc = fmaf(qs[d], Elem<T>::to_f32(kr[d]), acc);
            s = acc * scale;
            if (mp) s += Elem<T>::to_f32(mp[key]);
        }
        const float m_new = fmaxf(m_run, wave_max(s));
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        const float alpha = expf(m_run - m_use);
        const float p = expf(s - m_use);
        m_run = m_new;
        l_run = l_run * alpha + wave_sum(p);
        ps[lane] = p;
        __builtin_amdgcn_wave_barrier();
        const int nk = min(64, kv_end - kv0);
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int d = lane + 64 * j;
            if (d < D) {
                float acc = oacc[j] * alpha;
                for (int t = 0; t < nk; t++)
                    acc = fmaf(ps[t], Elem<T>::to_f32(vp[(int64_t)(kv0 + t) * D + d]), acc);
                oacc[j] = acc;
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
    const float inv = l_run > 1e-10f ? 1.f / l_run : 0.f;
    T* orow = static_cast<T*>(a.o) + (bh * a.Sq + qpos) * D;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const int d = lane + 64 * j;
        if (d < D) orow[d] = Elem<T>::from_f32(oacc[j] * inv);
    }
}

// Eight f16 numbers as bf16 pairs hi + lo, exactly: 8 of the 11 significant bits and the other 3.
__device__ __forceinline__ void split_f16(u32x4& v, u32x4& lo) {
    typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
    auto narrow = [](f16x2 h) {        // (both fit bf16: truncation is exact)
        return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, (float)h[1]), __builtin_bit_cast(uint32_t, (float)h[0]), 0x07060302u);
    };
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const uint32_t w = v[e];
        const f16x2 h = __builtin_bit_cast(f16x2, w & 0xFFF8FFF8u), l = __builtin_bit_cast(f16x2, w) - h;
        v[e] = narrow(h);
        lo[e] = narrow(l);
    }
}

// NB: depth of the K and of the V ring in LDS.  Two everywhere: with head size 64 a ring of three or
// four measured 8 to 13 % slower (B8 H12 S1024: 38.5 / 40.5 against 35.7 us) -- it costs the third
// resident workgroup per CU, which hides more latency than the deeper prefetch does.

// D = row length in LDS, DR = head size rounded up to 32; PART = a head size of a.D < D or any but 64 and 128.
template <typename T, int D, int DR, bool PART, bool CAUSAL, bool HAS_MASK, int NB>
__global__ __launch_bounds__(256, 2) void fa_fwd_kernel(FaArgs a) {
    const int head = PART ? a.D : D;
    constexpr int CPR = D / 8;                  // 16-byte chunks per row
    constexpr int kTile = kBKV * D * 2;         // bytes of one K (or V) tile
    constexpr int kRowsPerInst = 64 / CPR;      // tile rows one wave-wide LDS-DMA load fills
    constexpr int kInst = kBKV / kRowsPerInst / 4;   // such loads per wave per tile
    constexpr int ND = DR / 32, NS = DR / 16;
    constexpr bool kSplitV = PART && std::is_same<T, f16_t>::value;
    constexpr int kLoadsPerTile = 2 * kInst;    // per wave
    __shared__ __attribute__((aligned(1024))) char smem[2 * NB * kTile];   // K ring, then V ring

    // ---- which (batch*head, query block): see tile_of_workgroup
    int bh, qb;
    tile_of_workgroup<CAUSAL>(a, blockIdx.x, bh, qb);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
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
    const __amdgpu_buffer_rsrc_t rq = fa_rsrc(qp, (uint32_t)((((int64_t)a.Sq - 1) * q_rs + head) * 2));
    const __amdgpu_buffer_rsrc_t rk = fa_rsrc(kp, (uint32_t)((((int64_t)a.Skv - 1) * k_rs + head) * 2));
    const __amdgpu_buffer_rsrc_t rv = fa_rsrc(vp, (uint32_t)((((int64_t)a.Skv - 1) * v_rs + head) * 2));

    // ---- Q^T operand: lane = query column, 8 consecutive d per k-step ------
    u32x4 qf[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const uint32_t off = qpos < a.Sq && (!PART || 16 * s + 8 * lhalf < head) ? (uint32_t)((qpos * q_rs + 16 * s + 8 * lhalf) * 2) : kOobA;
        qf[s] = __builtin_amdgcn_raw_buffer_load_b128(rq, off, 0, 0);
        if (a.negate_q) {
            qf[s].x ^= 0x80008000u; qf[s].y ^= 0x80008000u;
            qf[s].z ^= 0x80008000u; qf[s].w ^= 0x80008000u;
        }
    }

    int nkv = (a.Skv + kBKV - 1) / kBKV;
    if (CAUSAL) {
        const int last_q = min(qblk0 + kBQ, a.Sq) - 1;
        nkv = min(nkv, last_q / kBKV + 1);
    }

    // ---- global -> LDS without a register stop: every wave-wide load fills 1 KB
    // of a tile (lane l lands at byte 16*l of that KB); the swizzle is applied by
    // choosing which global chunk each lane fetches.  Keys past the end read 0.
    const int ld_row = lane / CPR, ld_pos = lane % CPR;
    // (a block past the last one this workgroup needs is loaded all the same: the waits below
    // count loads, so every step issues the same number.)  Each lane's offsets inside block 0
    // are computed once; a step adds the block's offset.  Keys past the end need no test: their
    // offsets lie beyond the extent of the buffer descriptors above, and such loads put zeros
    // into LDS (V rows of zeros, so that a probability of zero times them stays zero).
    // (The swizzles repeat every sixteen rows and a wave's loads of a tile are 4 * kRowsPerInst
    // = 16 or 32 rows apart, so load i differs from load 0 by a constant.)
    const int wave_s = __builtin_amdgcn_readfirstlane(wave);
    const int ld_row0 = wave_s * kRowsPerInst + ld_row;
    const int kcol = (ld_pos ^ k_swz<D>(ld_row0)) << 3, vcol = (ld_pos ^ v_swz<D>(ld_row0)) << 3;
    // (a piece behind the row's end stays out of bounds whatever block is added: extents are below 2 GB)
    const uint32_t koff0 = PART && kcol >= head ? kOobA : (uint32_t)((ld_row0 * k_rs + kcol) * 2);
    const uint32_t voff0 = PART && vcol >= head ? kOobA : (uint32_t)((ld_row0 * v_rs + vcol) * 2);
    auto load_tile = [&](int kv0, int buf) {
#pragma unroll
        for (int i = 0; i < kInst; i++) {
            const int blk = i * 4 + wave_s;               // which KB of the tile
            const int row = kv0 + i * 4 * kRowsPerInst;   // (scalar)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (fa_lds_void*)(smem + buf * kTile + blk * 1024), 16,
                                                     koff0 + (uint32_t)(row * k_rs * 2), 0, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (fa_lds_void*)(smem + (NB + buf) * kTile + blk * 1024), 16,
                                                     voff0 + (uint32_t)(row * v_rs * 2), 0, 0, 0);
        }
    };
    // loads land in program order: the next block has landed when only the NB - 2 blocks issued
    // behind it are still in flight
    auto tiles_ready = [&]() {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NB - 2) * kLoadsPerTile) : "memory");
        __builtin_amdgcn_s_barrier();
    };

    // V^T fragment addresses: lane i of a 16-lane group supplies key row i/4 and
    // d columns 4*(i%4)..+3 of its group's 16-column block.
    const int ti = lane & 15, tg = lane >> 4;
    const int v_row0 = 4 * (tg >> 1) + (ti >> 2);                   // + 16u (+ 8)
    const int v_d0 = 16 * (tg & 1) + 4 * (ti & 3);                  // + 32 dt

    f32x16 oacc[ND];
#pragma unroll
    for (int i = 0; i < ND; i++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[i][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;   // reference maximum in the log2 domain (see moved_reference), running sum

#pragma unroll
    for (int p = 0; p < NB - 1; p++) load_tile(p * kBKV, p);
    tiles_ready();

    // A lane's keys of a block are eight runs of four, which it loads whole (8 bytes need no alignment) in front of the
    // products that hide the latency: bf16 B2 H8 S512 D64 40.7 -> 17.7 us.  In the last block of a row that is no multiple
    // of four a run may leave the mask; that block loads element by element.
    const T* mp = HAS_MASK ? static_cast<const T*>(a.mask) + (int64_t)b_i * a.mask_sb + (int64_t)h_i * a.mask_sh + (int64_t)min(qpos, a.Sq - 1) * a.Skv : nullptr;
    const bool whole_runs = a.Skv % 4 == 0;
    // log2(e) times a mask near bf16's lowest number is -inf.  A row with no other key than such ones so far (m_run is
    // -inf) shares itself between those of the largest mask, here its value; the first ordinary key drops them.
    constexpr bool kDeep = HAS_MASK && std::is_same<T, bf16_t>::value;
    float deep = -INFINITY;

    // Two blocks a turn where there is no mask, their places in the rings then constants of the LDS addresses: 14 of 165 vector instructions of a block less.  us, one | two, head
    // size 64: causal [4,16,4096] 165.4 | 163.0, [8,12,1024] 22.4 | 22.1, [16,12,512] 16.0 | 15.6, full [4,16,4096] 308.2 | 300.3, [8,12,1024] 34.5 | 34.0; of 128 within 0.5 %; in parts, [12,2048]
    // causal and full, of 96 56.6 | 54.2 and 57.3 | 55.3, f16 93.7 | 90.9 and 93.7 | 92.7, of 32 35.4 | 34.0 and 33.5 | 33.9.  (Blocks as a function that the loop calls cost the masked forms up to 10 %,
    // [2,16,4096] of 64 291 | 320, and the forms without a mask 8 to 31 spilled scalars.)
    static_assert(NB == 2, "two blocks a turn");
    constexpr int kTurn = HAS_MASK ? 1 : NB;
    for (int turn = 0; turn < nkv; turn += kTurn)
#pragma unroll
    for (int u = 0; u < kTurn; u++) {
        const int it = turn + u, cur = kTurn == NB ? u : it % NB, kv0 = it * kBKV;
        if (u && it >= nkv) break;
        load_tile(kv0 + (NB - 1) * kBKV, (cur + NB - 1) % NB);

        const bool wave_active = !CAUSAL || kv0 <= qw + 31;
        if (wave_active) {
            const char* kt = smem + cur * kTile;
            const char* vt = smem + (NB + cur) * kTile;
            u32x2 mrun[HAS_MASK ? 8 : 1];
            const bool mask_runs = HAS_MASK && (whole_runs || kv0 + kBKV <= a.Skv);
            if (mask_runs) {
#pragma unroll
                for (int g = 0; g < 8; g++) __builtin_memcpy(&mrun[HAS_MASK ? g : 0], mp + min(kv0 + 8 * g + 4 * lhalf, a.Skv - 4), 8);
            }
            // ---- S^T = K . Q^T ---------------------------------------------
            f32x16 sacc[2];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) sacc[t][r] = 0.f;
            // two workgroups share a SIMD: let a wave in a matrix phase issue ahead of
            // the other wave's softmax arithmetic
            __builtin_amdgcn_s_setprio(2);
#pragma unroll
            for (int s = 0; s < NS; s++) {
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    const u32x4 kf = *reinterpret_cast<const u32x4*>(kt + k_off<D>(32 * t + lrow, 2 * s + lhalf));
                    sacc[t] = Mfma32A<T>::run(kf, qf[s], sacc[t]);
                }
            }
            __builtin_amdgcn_s_setprio(0);
            float sv[32];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 16; r++) sv[t * 16 + r] = sacc[t][r];
            // Register i of the pair (t = i/16, r = i%16) is key
            // kv0 + 32t + 8(r/4) + 4*lhalf + r%4 of query column qpos.
            const bool boundary = (CAUSAL && kv0 + kBKV - 1 > qw) || kv0 + kBKV > a.Skv;
            float m_new;
            if (HAS_MASK || boundary) {
                // general form: scores to the log2 domain first, then mask
#pragma unroll
                for (int i = 0; i < 32; i++) sv[i] *= a.c;
                if (HAS_MASK) {
                    if (mask_runs) {
#pragma unroll
                        for (int i = 0; i < 32; i++) {
                            const uint32_t w = mrun[HAS_MASK ? i >> 2 : 0][i >> 1 & 1];       // (keys past the end: any value, masked below)
                            sv[i] = fmaf(Elem<T>::to_f32(__builtin_bit_cast(Pair16<T>, w).v[i & 1]), kLog2e, sv[i]);
                        }
                    } else {
#pragma unroll
                        for (int i = 0; i < 32; i++) {
                            const int key = kv0 + 32 * (i >> 4) + 8 * ((i & 15) >> 2) + 4 * lhalf + (i & 3);
                            if (key < a.Skv) sv[i] += Elem<T>::to_f32(mp[key]) * kLog2e;
                        }
                    }
                }
                if (boundary) {
#pragma unroll
                    for (int i = 0; i < 32; i++) {
                        const int key = kv0 + 32 * (i >> 4) + 8 * ((i & 15) >> 2) + 4 * lhalf + (i & 3);
                        if ((CAUSAL && key > qpos) || key >= a.Skv) sv[i] = -INFINITY;
                    }
                }
                float mloc = sv[0];
#pragma unroll
                for (int i = 1; i < 32; i++) mloc = fmaxf(mloc, sv[i]);
                mloc = half_max(mloc);
                m_new = moved_reference(m_run, mloc);
                const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
#pragma unroll
                for (int i = 0; i < 32; i++) sv[i] = __builtin_amdgcn_exp2f(sv[i] - m_use);
            } else {
                // interior block: max over raw scores (the scale is positive), and
                // scale + shift folded into one fma in front of the exp2
                float mloc = sv[0];
#pragma unroll
                for (int i = 1; i < 32; i++) mloc = fmaxf(mloc, sv[i]);
                mloc = half_max(mloc);
                m_new = moved_reference(m_run, mloc * a.c);
                const float neg_m = -m_new;     // finite: an interior block has no masked score
#pragma unroll
                for (int i = 0; i < 32; i++) sv[i] = __builtin_amdgcn_exp2f(fmaf(sv[i], a.c, neg_m));
            }
            const float m_use2 = (m_new == -INFINITY) ? 0.f : m_new;
            float alpha = __builtin_amdgcn_exp2f(m_run - m_use2);
            m_run = m_new;
            if (kDeep && __any(m_new == -INFINITY)) {
                // (read again, element by element: rare, and the loop above keeps its registers; a NaN score stays one)
                auto mask_at = [&](int i) {
                    const int key = kv0 + 32 * (i >> 4) + 8 * ((i & 15) >> 2) + 4 * lhalf + (i & 3);
                    const float m = key >= a.Skv || (CAUSAL && key > qpos) ? -INFINITY : Elem<T>::to_f32(mp[key]);
                    return m * kLog2e == -INFINITY ? m : -INFINITY;
                };
                float most = deep;
#pragma unroll
                for (int i = 0; i < 32; i++) most = fmaxf(most, mask_at(i));
                most = half_max(most);
                if (m_new == -INFINITY) {
                    alpha = most == deep ? 1.f : 0.f;
                    deep = most;
#pragma unroll
                    for (int i = 0; i < 32; i++)
                        if (most != -INFINITY && mask_at(i) == most) sv[i] += 1.f;      // (exp2(-inf) so far)
                }
            }
            float lsum = 0.f;
#pragma unroll
            for (int i = 0; i < 32; i++) lsum += sv[i];
            l_run = l_run * alpha + lsum;
            // the accumulator only needs rescaling when some row's maximum moved
            if (__any(alpha != 1.f)) {
#pragma unroll
                for (int i = 0; i < ND; i++)
#pragma unroll
                    for (int r = 0; r < 16; r++) oacc[i][r] *= alpha;
            }
            // ---- O^T += V^T . P^T.  B operand: slot j of step u is register 8u + j; A operand: slot j of step u is
            // key 16u + 8(j/4) + 4*lhalf + j%4, i.e. two transposing reads 8 keys apart
            auto v_frag = [&](int u, int dt) {
                const int row = 16 * u + v_row0;
                const int d0 = 32 * dt + v_d0;
                const char* p0 = vt + v_off<D>(row, d0 >> 3) + (d0 & 7) * 2;
                const char* p1 = vt + v_off<D>(row + 8, d0 >> 3) + (d0 & 7) * 2;
                const u32x2 lo = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((fa_lds_s16x4*)p0));
                const u32x2 hi = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((fa_lds_s16x4*)p1));
                return u32x4{lo.x, lo.y, hi.x, hi.y};
            };
            if constexpr (PART) {
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    u32x4 p[3];
#pragma unroll
                    for (int part = 0; part < 3; part++)
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            float &x = sv[8 * u + 2 * e], &y = sv[8 * u + 2 * e + 1];
                            const uint32_t xb = __builtin_bit_cast(uint32_t, x), yb = __builtin_bit_cast(uint32_t, y);
                            p[part][e] = __builtin_amdgcn_perm(yb, xb, 0x07060302u);
                            x -= __builtin_bit_cast(float, xb & 0xFFFF0000u);
                            y -= __builtin_bit_cast(float, yb & 0xFFFF0000u);
                        }
                    u32x4 vf[ND], vl[ND];
#pragma unroll
                    for (int dt = 0; dt < ND; dt++) {
                        vf[dt] = v_frag(u, dt);
                        if (kSplitV) split_f16(vf[dt], vl[dt]);
                    }
#pragma unroll
                    for (int part = 2; part >= 0; part--)
#pragma unroll
                        for (int dt = 0; dt < ND; dt++) {
                            if (kSplitV) oacc[dt] = Mfma32A<bf16_t>::run(vl[dt], p[part], oacc[dt]);
                            oacc[dt] = Mfma32A<bf16_t>::run(vf[dt], p[part], oacc[dt]);
                        }
                }
            } else {
                u32x4 pb[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    pb[u].x = Mfma32A<T>::pack2(sv[8 * u + 0], sv[8 * u + 1]);
                    pb[u].y = Mfma32A<T>::pack2(sv[8 * u + 2], sv[8 * u + 3]);
                    pb[u].z = Mfma32A<T>::pack2(sv[8 * u + 4], sv[8 * u + 5]);
                    pb[u].w = Mfma32A<T>::pack2(sv[8 * u + 6], sv[8 * u + 7]);
                }
                __builtin_amdgcn_s_setprio(2);
#pragma unroll
                for (int u = 0; u < 4; u++)
#pragma unroll
                    for (int dt = 0; dt < ND; dt++) oacc[dt] = Mfma32A<T>::run(v_frag(u, dt), pb[u], oacc[dt]);
            }
            __builtin_amdgcn_s_setprio(0);
        }
        if (it + 1 < nkv) tiles_ready();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // nothing may land in LDS after the workgroup ends

    // ---- normalise and store: lane holds 4 consecutive d per register group -
    const float l_tot = half_sum(l_run);
    const float inv = l_tot > 1e-10f ? 1.f / l_tot : 0.f;
    // PART: a product with an infinity or a NaN in V reaches every row whose wave met that key, through a weight of zero
    // too, and a sum in parts of the weight has no sign for an infinity.  Such rows (a sum that is not finite) are formed
    // again the scalar way, in the LDS that the tiles no longer need.  So are rows of scores beyond 2^28 without a
    // mask: the fused multiply-add of an interior block and the rounded product of a boundary block are then apart by more
    // than a weight can stand.
    bool whole = true;
    if (PART) {
        float probe = 0.f * l_tot;
#pragma unroll
        for (int i = 0; i < ND; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) probe = fmaf(oacc[i][r], 0.f, probe);
        whole = half_sum(probe) == 0.f && (HAS_MASK || m_run == -INFINITY || fabsf(m_run) < 0x1p28f);
        __syncthreads();
    }
    if (qpos < a.Sq && whole) {
        T* orow = op + (int64_t)qpos * a.os[2];
#pragma unroll
        for (int dt = 0; dt < ND; dt++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                u32x2 w;
                w.x = Mfma32A<T>::pack2(oacc[dt][4 * g + 0] * inv, oacc[dt][4 * g + 1] * inv);
                w.y = Mfma32A<T>::pack2(oacc[dt][4 * g + 2] * inv, oacc[dt][4 * g + 3] * inv);
                if (!PART || 32 * dt + 8 * g + 4 * lhalf < head) *reinterpret_cast<u32x2*>(orow + 32 * dt + 8 * g + 4 * lhalf) = w;
            }
    }
    if (PART) {
        uint32_t again = (uint32_t)__ballot(!whole && qpos < a.Sq);       // (the lower half holds a bit per row)
        float* mem = reinterpret_cast<float*>(smem) + wave_s * 320;
        for (; again; again &= again - 1)
            fa_row<T>(a, bh, qw + __builtin_ctz(again), head, a.negate_q ? -a.scale : a.scale, mem, mem + 256);
    }
}

// ---------------------------------------------------------------------------
// Scalar path: one wave per query row, any type, D <= 256.
// ---------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void fa_scalar_kernel(FaArgs a, int D, float scale) {
    __shared__ float qs[4][256];
    __shared__ float ps[4][64];
    const int wave = threadIdx.x >> 6;
    const int64_t row = (int64_t)blockIdx.x * 4 + wave;      // over B*H*Sq
    if (row < (int64_t)a.B * a.H * a.Sq) fa_row<T>(a, row / a.Sq, (int)(row % a.Sq), D, scale, qs[wave], ps[wave]);
}

template <typename T, int D, int DR = D, bool PART = false>
static int launch_fa(hipStream_t s, FaArgs a, bool causal, bool has_mask) {
    a.nqb = (a.Sq + kBQ - 1) / kBQ;
    const int64_t bh = (int64_t)a.B * a.H;
    set_tile_order(a);
    const int64_t grid = bh * a.nqb;
    if (grid > 0x7FFFFFFFLL) return fail(MHIP_ERR_UNSUPPORTED, "flash_attention: grid too large");
    constexpr int NB = 2;
#define MHIP_FA(C, M)                                                                       \
    hipLaunchKernelGGL((fa_fwd_kernel<T, D, DR, PART, C, M, NB>), dim3((unsigned)grid), dim3(256), 0, s, a)
    if (causal && has_mask) MHIP_FA(true, true);
    else if (causal) MHIP_FA(true, false);
    else if (has_mask) MHIP_FA(false, true);
    else MHIP_FA(false, false);
#undef MHIP_FA
    return check_launch("flash_attention");
}

template <typename T>
static int launch_fa_part(hipStream_t s, const FaArgs& a, bool causal, bool has_mask) {
    if (a.D <= 32) return launch_fa<T, 64, 32, true>(s, a, causal, has_mask);
    if (a.D <= 64) return launch_fa<T, 64, 64, true>(s, a, causal, has_mask);
    if (a.D <= 96) return launch_fa<T, 128, 96, true>(s, a, causal, has_mask);
    return launch_fa<T, 128, 128, true>(s, a, causal, has_mask);
}

template <typename T>
static int launch_fa_scalar(hipStream_t s, FaArgs a, int D, float scale) {
    const int64_t rows = (int64_t)a.B * a.H * a.Sq;
    const int64_t grid = (rows + 3) / 4;
    if (grid > 0x7FFFFFFFLL) return fail(MHIP_ERR_UNSUPPORTED, "flash_attention: grid too large");
    hipLaunchKernelGGL((fa_scalar_kernel<T>), dim3((unsigned)grid), dim3(256), 0, s, a, D, scale);
    return check_launch("flash_attention_scalar");
}

}  // namespace mhip

namespace mhip {
// attention_pipe.hip: head size 128, four waves x 64 query rows, matrix / softmax overlap in one wave.
bool fa_pipe_eligible(const FaArgs& a, int64_t D, int dtype, bool has_mask, int variant);
int launch_fa_pipe(hipStream_t s, const FaArgs& a, int dtype, bool causal, int pair);
// attention_decode.hip: up to sixteen query rows over a long cache.
bool fa_decode_eligible(const FaArgs& a);
int64_t fa_decode_workspace(int64_t bh, int64_t Sq, int64_t Skv, int64_t D);
int launch_fa_decode(hipStream_t s, const FaArgs& a, int64_t D, int dtype, void* workspace, int64_t workspace_bytes);
// attention_flow.hip: head sizes 64 and 128 without a mask, few tiles.
bool fa_flow_wanted(const FaArgs& a, int64_t D);
int launch_fa_flow(hipStream_t s, FaArgs a, int64_t D, int dtype);
// attention_short.hip: few keys.
bool fa_short_wanted(const FaArgs& a);
int launch_fa_short(hipStream_t s, const FaArgs& a, int64_t D, int dtype);
// attention_f32.hip: fp32 tensors on the fp32 matrix instruction.
bool fa_f32_mfma_eligible(const FaArgs& a, int64_t D, bool packed);
int launch_fa_f32_mfma(hipStream_t s, const FaArgs& a, int64_t D, float scale, bool packed);
}  // namespace mhip

using namespace mhip;

// `strides`: NULL (packed [B,H,S,D]) or twelve element strides {batch, head, row} x {q, k, v, o}.
static int fa_entry(const char* name, void* stream, const void* q, const void* k, const void* v, const void* mask, void* o,
                    int64_t B, int64_t H, int64_t Sq, int64_t Skv, int64_t D, float scale, int is_causal,
                    int64_t mask_stride_b, int64_t mask_stride_h, int dtype, const int64_t* strides, void* workspace = nullptr,
                    int64_t workspace_bytes = 0, bool any_views = false) {
    if (B < 0 || H < 0 || Sq < 0 || Skv < 0 || D <= 0)
        return fail(MHIP_ERR_INVALID_ARGUMENT, "%s: bad size", name);
    if (D > 256) return fail(MHIP_ERR_UNSUPPORTED, "%s: head_dim %lld > 256", name, (long long)D);
    if (B == 0 || H == 0 || Sq == 0) return MHIP_OK;
    if (!q || !o || (Skv > 0 && (!k || !v)))
        return fail(MHIP_ERR_INVALID_ARGUMENT, "%s: NULL tensor pointer", name);
    if (Sq > 0x7FFFFFFF || Skv > 0x7FFFFFFF || B * H > 0x7FFFFFFF)
        return fail(MHIP_ERR_UNSUPPORTED, "%s: dimension exceeds 2^31-1", name);
    hipStream_t s = as_stream(stream);
    FaArgs a;
    a.q = q; a.k = k; a.v = v; a.mask = mask; a.o = o;
    a.D = (int)D;
    a.B = (int)B; a.H = (int)H; a.Sq = (int)Sq; a.Skv = (int)Skv;
    a.c = fabsf(scale) * kLog2e;
    a.scale = fabsf(scale);
    a.negate_q = scale < 0.f;
    a.is_causal = is_causal ? 1 : 0;
    a.mask_sb = mask_stride_b; a.mask_sh = mask_stride_h;
    a.nqb = 0; a.pair_tiles = 0; a.cu_group = 1;
    const int64_t packed[12] = {H * Sq * D, Sq * D, D, H * Skv * D, Skv * D, D, H * Skv * D, Skv * D, D, H * Sq * D, Sq * D, D};
    bool is_packed = true;
    int64_t max_row = D, max_span = 0;
    for (int i = 0; i < 12; i++) {
        const int64_t st = strides ? strides[i] : packed[i];
        if (st < 0) return fail(MHIP_ERR_INVALID_ARGUMENT, "%s: negative stride", name);
        (i < 3 ? a.qs : i < 6 ? a.ks : i < 9 ? a.vs : a.os)[i % 3] = st;
        is_packed = is_packed && st == packed[i];
    }
    const int64_t* rows[4] = {a.qs, a.ks, a.vs, a.os};
    bool strides_aligned = true;
    for (int t = 0; t < 4; t++) {
        if (rows[t][2] < D) return fail(MHIP_ERR_INVALID_ARGUMENT, "%s: row stride smaller than head_dim", name);
        strides_aligned = strides_aligned && rows[t][0] % 8 == 0 && rows[t][1] % 8 == 0 && rows[t][2] % 8 == 0;
        max_row = rows[t][2] > max_row ? rows[t][2] : max_row;
        const int64_t n = (t == 0 || t == 3) ? Sq : Skv;
        const int64_t span = (n > 0 ? (n - 1) * rows[t][2] : 0) + D;
        max_span = span > max_span ? span : max_span;
    }
    const bool is16 = dtype == MHIP_BF16 || dtype == MHIP_F16;
    const bool aligned = ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k) |
                           reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(o)) & 15) == 0;
    const bool fits = max_span * 2 < 0x7FFFFFFFLL;
    if (is16 && aligned && strides_aligned && fits && Skv > 0 && (D == 64 || D == 128)) {
        const bool hm = mask != nullptr;
        // 0 = no tuned choice; 1 = 128-row kernel; 2 / 3 = 256-row pipelined kernel, causal tiles unpaired / paired
        const int variant = is_packed ? tuned_attention_variant(dtype, B * H, Sq, Skv, D, is_causal != 0) : 0;
        if (variant == 0 && fa_decode_eligible(a) && B * H <= 0x7FFFFFFF) return launch_fa_decode(s, a, D, dtype, workspace, workspace_bytes);
        if (variant == 0 && !hm && fa_short_wanted(a)) return launch_fa_short(s, a, D, dtype);
        if (is_packed && fa_pipe_eligible(a, D, dtype, hm, variant))
            return launch_fa_pipe(s, a, dtype, is_causal != 0, variant == 2 ? 0 : variant == 3 ? 1 : -1);
        if (!hm && fa_flow_wanted(a, D)) return launch_fa_flow(s, a, D, dtype);
        if (dtype == MHIP_BF16)
            return D == 128 ? launch_fa<bf16_t, 128>(s, a, is_causal, hm)
                            : launch_fa<bf16_t, 64>(s, a, is_causal, hm);
        return D == 128 ? launch_fa<f16_t, 128>(s, a, is_causal, hm)
                        : launch_fa<f16_t, 64>(s, a, is_causal, hm);
    }
    // (with rows of a multiple of 8 elements every piece of 16 bytes is aligned)
    if (is16 && (is_packed || (any_views && strides_aligned)) && aligned && fits && Skv > 0 && D % 8 == 0 && D < 128)
        return dtype == MHIP_BF16 ? launch_fa_part<bf16_t>(s, a, is_causal, mask != nullptr) : launch_fa_part<f16_t>(s, a, is_causal, mask != nullptr);
    if (any_views && !is_packed && Skv > 0 && dtype == MHIP_F32 && fa_f32_mfma_eligible(a, D, false)) return launch_fa_f32_mfma(s, a, D, scale, false);
    if (!is_packed)
        return fail(MHIP_ERR_UNSUPPORTED, "%s: strided layouts need bf16 / f16, head_dim 64 or 128, 16-byte aligned pointers and "
                                          "strides that are multiples of 8 elements", name);
    switch (dtype) {
        case MHIP_F32:
            if (fa_f32_mfma_eligible(a, D, true)) return launch_fa_f32_mfma(s, a, D, scale, true);
            return launch_fa_scalar<float>(s, a, (int)D, scale);
        case MHIP_BF16: return launch_fa_scalar<bf16_t>(s, a, (int)D, scale);
        case MHIP_F16: return launch_fa_scalar<f16_t>(s, a, (int)D, scale);
        default: return fail(MHIP_ERR_UNSUPPORTED, "%s: dtype %d", name, dtype);
    }
}

extern "C" int mhip_flash_attention(void* stream, const void* q, const void* k, const void* v,
                                    const void* mask, void* o, int64_t B, int64_t H, int64_t Sq,
                                    int64_t Skv, int64_t D, float scale, int is_causal,
                                    int64_t mask_stride_b, int64_t mask_stride_h, int dtype) {
    return fa_entry("mhip_flash_attention", stream, q, k, v, mask, o, B, H, Sq, Skv, D, scale, is_causal, mask_stride_b,
                    mask_stride_h, dtype, nullptr);
}

extern "C" int mhip_flash_attention_strided(void* stream, const void* q, const void* k, const void* v,
                                            const void* mask, void* o, int64_t B, int64_t H, int64_t Sq,
                                            int64_t Skv, int64_t D, float scale, int is_causal,
                                            int64_t mask_stride_b, int64_t mask_stride_h, int dtype,
                                            const int64_t* strides) {
    return fa_entry("mhip_flash_attention_strided", stream, q, k, v, mask, o, B, H, Sq, Skv, D, scale, is_causal,
                    mask_stride_b, mask_stride_h, dtype, strides);
}

extern "C" int mhip_flash_attention_views(void* stream, const void* q, const void* k, const void* v, const void* mask, void* o,
                                          int64_t B, int64_t H, int64_t Sq, int64_t Skv, int64_t D, float scale, int is_causal,
                                          int64_t mask_stride_b, int64_t mask_stride_h, int dtype, const int64_t* strides) {
    return fa_entry("mhip_flash_attention_views", stream, q, k, v, mask, o, B, H, Sq, Skv, D, scale, is_causal, mask_stride_b,
                    mask_stride_h, dtype, strides, nullptr, 0, true);
}

extern "C" int mhip_flash_attention_ws(void* stream, const void* q, const void* k, const void* v, const void* mask, void* o,
                                       int64_t B, int64_t H, int64_t Sq, int64_t Skv, int64_t D, float scale, int is_causal,
                                       int64_t mask_stride_b, int64_t mask_stride_h, int dtype, const int64_t* strides,
                                       void* workspace, int64_t workspace_bytes) {
    if (workspace_bytes < 0 || (reinterpret_cast<uintptr_t>(workspace) & 15) != 0)
        return fail(MHIP_ERR_INVALID_ARGUMENT, "mhip_flash_attention_ws: the workspace must be 16-byte aligned");
    return fa_entry("mhip_flash_attention_ws", stream, q, k, v, mask, o, B, H, Sq, Skv, D, scale, is_causal, mask_stride_b,
                    mask_stride_h, dtype, strides, workspace, workspace_bytes);
}

extern "C" int64_t mhip_flash_attention_workspace(int64_t B, int64_t H, int64_t Sq, int64_t Skv, int64_t D, int is_causal, int dtype) {
    if (B <= 0 || H <= 0 || Skv <= 0 || is_causal || (dtype != MHIP_BF16 && dtype != MHIP_F16)) return 0;
    return fa_decode_workspace(B * H, Sq, Skv, D);
}
