// Attention of a few query rows (a decode step, Sq <= 16) over a long key / value cache, 16-bit types, head
// sizes 64 and 128: the time is that of reading K and V once.
//
// A query tile of 128 rows would be almost all padding, and its one workgroup per head walks the keys through
// LDS stages with little in flight.  Here every wave of a workgroup takes blocks of 32 keys of its own, loads
// them straight into matrix operands (no LDS, no barrier in the loop) one block ahead, and keeps its own
// softmax state; the waves meet at the end in LDS, and the parts of a split key range in a workspace, where the last
// workgroup of a head to arrive puts them together (arrive.h).
//
//   S^T = K Q^T     v_mfma_f32_16x16x32: operand row = key, so a lane loads 16 bytes of one key's row; a lane
//                   of the result holds four keys of one query.
//   O^T += V^T P^T  operand row = d: lane i loads VE = D / 16 neighbouring d of each of its eight keys, and one
//                   byte permute per register pairs two keys of one d; tile f then holds d = VE i + f.  The
//                   eight keys of a lane are the ones whose probabilities it just computed.
#include <type_traits>

#include "arrive.h"
#include "attention_common.h"

namespace mhip {
namespace {

template <typename T> struct Mfma16A;
template <> struct Mfma16A<bf16_t> {
    __device__ static f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    }
};
template <> struct Mfma16A<f16_t> {
    __device__ static f32x4 run(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
};

constexpr int kKeys = 32;        // keys per block
constexpr int kMaxSq = 16;
// A part of a split key range is a multiple of this.  us, multiples of 128 | 256 keys, one query (eight): 32 heads over 512 keys, head size 128,
// 6.7 | 8.0 (7.2 | 8.6), 12 over 640, 64, 5.2 | 7.5 (5.6 | 7.7), 24 over 1024, 64, 6.2 | 6.7 (6.3 | 6.9), 8 over 1536, 64, 6.7 | 6.9 (6.8 | 6.9), 8 over
// 2048, 128, 8.7 | 8.5 (9.1 | 9.4), 8 over 4096, 64, 11.7 | 9.0 (12.5 | 9.0); 12 over 300 6.0 | 4.7 (whole).
constexpr int part_keys(int64_t Skv) { return Skv >= 512 && Skv <= 1024 ? 128 : 256; }

// domain of scores and reference (see moved_reference): f16's lowest number is far from fp32's
template <typename T, bool HAS_MASK>
constexpr bool kNatural = HAS_MASK && std::is_same<T, bf16_t>::value;

template <typename T, int D, bool HAS_MASK, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void fa_decode_kernel(FaArgs a, float* part, int per_part, uint64_t* words, uint64_t tag) {
    constexpr bool NAT = kNatural<T, HAS_MASK>;
    constexpr int NS = D / 32, NF = D / 16, VDw = NF / 2;      // k steps of Q K^T, tiles of O^T, dwords of a lane's V piece
    __shared__ __attribute__((aligned(16))) float sums[WAVES][NF][64][4];
    __shared__ float ml[2][WAVES][kMaxSq];
    __shared__ int last;
    // (the arguments in one go: 1 x 8 heads over 4096 keys 9.40 -> 9.18 us, 8 x 32 over 512 12.94 -> 12.76)
    asm volatile("" ::"s"(a.q), "s"(a.k), "s"(a.v), "s"(a.o), "s"(a.H), "s"(a.Sq), "s"(a.Skv), "s"(a.c), "s"(a.negate_q), "s"(a.qs[0]), "s"(a.qs[1]), "s"(a.ks[0]), "s"(a.ks[1]),
                 "s"(a.vs[0]), "s"(a.vs[1]), "s"((int)a.qs[2]), "s"((int)a.ks[2]), "s"((int)a.vs[2]), "s"(part), "s"(per_part), "s"(words), "s"(tag));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lg = lane >> 4;
    const int bh = blockIdx.x, b_i = bh / a.H, h_i = bh % a.H;
    const T* qp = static_cast<const T*>(a.q) + b_i * a.qs[0] + h_i * a.qs[1];
    const T* kp = static_cast<const T*>(a.k) + b_i * a.ks[0] + h_i * a.ks[1];
    const T* vp = static_cast<const T*>(a.v) + b_i * a.vs[0] + h_i * a.vs[1];
    const int q_rs = (int)a.qs[2], k_rs = (int)a.ks[2], v_rs = (int)a.vs[2];
    const __amdgpu_buffer_rsrc_t rq = fa_rsrc(qp, (uint32_t)((((int64_t)a.Sq - 1) * q_rs + D) * 2));
    const __amdgpu_buffer_rsrc_t rk = fa_rsrc(kp, (uint32_t)((((int64_t)a.Skv - 1) * k_rs + D) * 2));
    const __amdgpu_buffer_rsrc_t rv = fa_rsrc(vp, (uint32_t)((((int64_t)a.Skv - 1) * v_rs + D) * 2));
    const T* mp = HAS_MASK ? static_cast<const T*>(a.mask) + (int64_t)b_i * a.mask_sb + (int64_t)h_i * a.mask_sh : nullptr;

    uint64_t seen = 0;
    if (part && threadIdx.x == 0) seen = arrive_look(words + bh);
    u32x4 qf[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        qf[s] = __builtin_amdgcn_raw_buffer_load_b128(rq, li < a.Sq ? (uint32_t)((li * q_rs + 32 * s + 8 * lg) * 2) : kOobA, 0, 0);
        if (a.negate_q) {
#pragma unroll
            for (int e = 0; e < 4; e++) qf[s][e] ^= 0x80008000u;
        }
    }

    // this workgroup's keys [k0, k1); block n of wave w is keys k0 + 32 (WAVES n + w) ...  (keys past the end of
    // the cache lie beyond the buffers' extents and read zero)
    const int k0 = (int)blockIdx.y * per_part, k1 = min(a.Skv, k0 + per_part);
    struct Block { u32x4 k[2][NS]; uint32_t v[8][VDw]; };
    const uint32_t koff = (uint32_t)((li * k_rs + 8 * lg) * 2), voff = (uint32_t)((4 * lg * v_rs + NF * li) * 2);
    auto load = [&](Block& blk, int key) {
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int s = 0; s < NS; s++)
                blk.k[j][s] = __builtin_amdgcn_raw_buffer_load_b128(rk, koff + (uint32_t)(((key + 16 * j) * k_rs + 32 * s) * 2), 0, 0);
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const uint32_t off = voff + (uint32_t)((key + 16 * (t >> 2) + (t & 3)) * v_rs * 2);
            if constexpr (VDw == 4) {
                const u32x4 w = __builtin_amdgcn_raw_buffer_load_b128(rv, off, 0, 0);
#pragma unroll
                for (int e = 0; e < 4; e++) blk.v[t][e] = w[e];
            } else {
                const u32x2 w = __builtin_amdgcn_raw_buffer_load_b64(rv, off, 0, 0);
                blk.v[t][0] = w.x; blk.v[t][1] = w.y;
            }
        }
    };

    f32x4 oacc[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) oacc[f] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;          // of query li; the sum is this lane's keys only
    auto attend = [&](const Block& blk, int key) {
        float sv[8];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            f32x4 s4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < NS; s++) s4 = Mfma16A<T>::run(blk.k[j][s], qf[s], s4);
#pragma unroll
            for (int r = 0; r < 4; r++) sv[4 * j + r] = s4[r] * (NAT ? a.scale : a.c);
        }
        if (HAS_MASK) {
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const int kk = key + 16 * (t >> 2) + 4 * lg + (t & 3);
                if (li < a.Sq && kk < a.Skv) sv[t] += Elem<T>::to_f32(mp[(int64_t)li * a.Skv + kk]) * (NAT ? 1.f : kLog2e);
            }
        }
        if (key + kKeys > k1) {
#pragma unroll
            for (int t = 0; t < 8; t++)
                if (key + 16 * (t >> 2) + 4 * lg + (t & 3) >= k1) sv[t] = -INFINITY;
        }
        float mloc = sv[0];
#pragma unroll
        for (int t = 1; t < 8; t++) mloc = fmaxf(mloc, sv[t]);
        mloc = fmaxf(mloc, __shfl_xor(mloc, 16, 64));
        mloc = half_max(mloc);
        const float m_new = moved_reference<NAT>(m_run, mloc), m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = weight<NAT>(m_run, m_use);
        m_run = m_new;
        float lsum = 0.f;
#pragma unroll
        for (int t = 0; t < 8; t++) {
            sv[t] = weight<NAT>(sv[t], m_use);
            lsum += sv[t];
        }
        l_run = l_run * alpha + lsum;
        if (__any(alpha != 1.f)) {
#pragma unroll
            for (int f = 0; f < NF; f++) oacc[f] *= alpha;
        }
        u32x4 pb;
#pragma unroll
        for (int e = 0; e < 4; e++) pb[e] = Mfma32A<T>::pack2(sv[2 * e], sv[2 * e + 1]);
#pragma unroll
        for (int f = 0; f < NF; f++) {
            u32x4 vf;
#pragma unroll
            for (int e = 0; e < 4; e++)
                vf[e] = __builtin_amdgcn_perm(blk.v[2 * e + 1][f / 2], blk.v[2 * e][f / 2], (f & 1) ? 0x07060302u : 0x05040100u);
            oacc[f] = Mfma16A<T>::run(vf, pb, oacc[f]);
        }
    };
    // Blocks of this wave, in a ring; of eight waves with head size 128 wave w starts w eighths of the way round.  Workgroups that walk side by side from the start of their
    // keys are a power of two apart where caches are as long as one, and meet in the same banks of the memory; so a workgroup itself is in eight places at a time.  us, from the first
    // block | so, one query: 256 heads over 4096 keys 93.9 | 90.8, over 2048 47.7 | 47.3, 96 over 4096 38.9 | 37.6, 64 over 8192 50.0 | 48.9, 192 over 3000
    // 52.9 | 51.8, 256 over 4000 91.2 | 88.7, 48 over 4096 22.7 | 21.7.  The place depends on nothing but the wave, so that a head's bits do not say where in the launch it is (a start that a hash
    // of the head chooses: 89.8, 47.3, 37.5, 49.4, 51.6, 88.6, 21.5).  Four waves of two workgroups a unit lose by it, 512 heads over 4096 177 | 180; eight waves with a run of blocks each
    // instead 96.4 for 256 heads; head size 64, whose rows are a line each, by a ring from a hash, 128 over 8192 48.4 | 49.4.
    constexpr int kStride = WAVES * kKeys;
    const int base = k0 + wave * kKeys;
    if (base < k1) {
        int left = (k1 - base + kStride - 1) / kStride, key = base;
        if (WAVES == 8 && D == 128 && left >= 4) key += left * wave / WAVES * kStride;
        Block cur;
        load(cur, key);
        for (;;) {
            Block nxt;
            const int next = key + kStride < k1 ? key + kStride : base;
            const bool more = --left > 0;
            if (more) load(nxt, next);
            attend(cur, key);
            if (!more) break;
            cur = nxt;
            key = next;
        }
    }

    if (part && threadIdx.x == 0) arrive_claim(words + bh, seen, tag);
    // ---- the waves' states
    l_run += __shfl_xor(l_run, 16, 64);
    l_run = half_sum(l_run);
    if (lg == 0) { ml[0][wave][li] = m_run; ml[1][wave][li] = l_run; }
#pragma unroll
    for (int f = 0; f < NF; f++) *reinterpret_cast<f32x4*>(sums[wave][f][lane]) = oacc[f];
    __syncthreads();
    T* op = static_cast<T*>(a.o) + b_i * a.os[0] + h_i * a.os[1];
    if (!part) {
        for (int idx = threadIdx.x; idx < a.Sq * D; idx += 64 * WAVES) {
            const int q = idx / D, d = idx % D, f = d % NF, i = d / NF;
            float m = -INFINITY, l = 0.f, o = 0.f;
#pragma unroll
            for (int w = 0; w < WAVES; w++) m = fmaxf(m, ml[0][w][q]);
            const float m_use = m == -INFINITY ? 0.f : m;
#pragma unroll
            for (int w = 0; w < WAVES; w++) {
                const float al = weight<NAT>(ml[0][w][q], m_use);
                l = fmaf(ml[1][w][q], al, l);
                o = fmaf(sums[w][f][(i >> 2) * 16 + q][i & 3], al, o);
            }
            op[(int64_t)q * a.os[2] + d] = Elem<T>::from_f32(o * (l > 1e-10f ? 1.f / l : 0.f));
        }
        return;
    }

    // ---- this part of the keys: [part][bh][Sq] x 4 NF groups of four sums, as the accumulators hold them (group 4 f + g: d = NF (4 g + e) + f), then
    // [part][bh][Sq] pairs of reference maximum and sum
    constexpr int kGroups = 4 * NF;
    const int parts = gridDim.y;
    const __amdgpu_buffer_rsrc_t rp = parts_rsrc(part), rl = parts_rsrc(part + (int64_t)parts * gridDim.x * a.Sq * D);
    auto row_of = [&](int p, int q) __attribute__((always_inline)) { return (p * (int)gridDim.x + bh) * a.Sq + q; };
    for (int idx = threadIdx.x; idx < a.Sq * kGroups; idx += 64 * WAVES) {
        const int q = idx / kGroups, group = idx % kGroups;
        float m = -INFINITY, l = 0.f;
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WAVES; w++) m = fmaxf(m, ml[0][w][q]);
        const float m_use = m == -INFINITY ? 0.f : m;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            const float al = weight<NAT>(ml[0][w][q], m_use);
            l = fmaf(ml[1][w][q], al, l);
            const f32x4 v = *reinterpret_cast<const f32x4*>(sums[w][group >> 2][(group & 3) * 16 + q]);
#pragma unroll
            for (int e = 0; e < 4; e++) o[e] = fmaf(v[e], al, o[e]);
        }
        store_part(rp, (uint32_t)((row_of(blockIdx.y, q) * kGroups + group) * 16), o);
        if (group == 0)
            __builtin_amdgcn_raw_buffer_store_b64(u32x2{__builtin_bit_cast(uint32_t, m), __builtin_bit_cast(uint32_t, l)}, rl, (uint32_t)(row_of(blockIdx.y, q) * 8), 0, kAgentScope);
    }
    if (!arrive_last(words + bh, parts, &last)) return;

    // ---- the last part of the head to arrive, four sums a thread.  (One element of O a thread, with the weights formed for each of them, 16 queries of
    // 8 heads over 16384 keys of head size 128 took 67.4 us, 32 so, and with a launch of
    // its own behind it 48.2.)
    auto put = [&](int q, int group, int e, float v) __attribute__((always_inline)) {
        op[(int64_t)q * a.os[2] + NF * (4 * (group & 3) + e) + (group >> 2)] = Elem<T>::from_f32(v);
    };
    // Up to sixteen parts: every thread asks for its row's references and sums too, and all is there after one latency.
    auto few = [&](auto most_tag) __attribute__((always_inline)) {
        constexpr int kMost = decltype(most_tag)::value;
        for (int idx = threadIdx.x; idx < a.Sq * kGroups; idx += 64 * WAVES) {
            const int q = idx / kGroups, group = idx % kGroups;
            u32x2 state[kMost];
            f32x4 v[kMost], o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int p = 0; p < kMost; p++) {
                state[p] = __builtin_amdgcn_raw_buffer_load_b64(rl, p < parts ? (uint32_t)(row_of(p, q) * 8) : kOobA, 0, kAgentScope);
                v[p] = load_part(rp, p < parts ? (uint32_t)((row_of(p, q) * kGroups + group) * 16) : kOobA);
            }
            float pm[kMost], m = -INFINITY, l = 0.f;
#pragma unroll
            for (int p = 0; p < kMost; p++) {
                const uint32_t bits = state[p].x;
                pm[p] = p < parts ? __builtin_bit_cast(float, bits) : -INFINITY;
                m = fmaxf(m, pm[p]);
            }
            const float m_use = m == -INFINITY ? 0.f : m;
#pragma unroll
            for (int p = 0; p < kMost; p++) {
                const uint32_t bits = state[p].y;
                const float al = weight<NAT>(pm[p], m_use);
                l = fmaf(__builtin_bit_cast(float, bits), al, l);
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = fmaf(v[p][e], al, o[e]);
            }
            const float inv = l > 1e-10f ? 1.f / l : 0.f;
#pragma unroll
            for (int e = 0; e < 4; e++) put(q, group, e, o[e] * inv);
        }
    };
    if (parts <= 4) return few(std::integral_constant<int, 4>{});
    if (parts <= 8) return few(std::integral_constant<int, 8>{});
    if (parts <= 16) return few(std::integral_constant<int, 16>{});
    // More: a row's weights are formed once, a lane a part (64 at most), while the first loads are on their way, and the parts are dealt over
    // threads where there are few queries.
    constexpr int kSlots = 64 * WAVES / kGroups;
    float* const weights = &sums[0][0][0][0];                // [kMaxSq][64]
    float* const inverse = weights + kMaxSq * 64;            // [kMaxSq]
    float* const shares = inverse + 64;                      // [sharers][Sq][D]
    static_assert((kMaxSq * 64 + 64 + (kSlots > kMaxSq ? kSlots : kMaxSq) * D) * 4 <= (int)sizeof(sums), "in place of the waves' sums");
    int together = 1;                                        // queries at a time, a power of two
    while (together < a.Sq && together < kSlots) together *= 2;
    const int sharers = min(kSlots / together, 4), group = threadIdx.x % kGroups, slot = threadIdx.x / kGroups, first = slot / together;
    constexpr int kLoads = 16;
    f32x4 v[kLoads];
    // sixteen loads of 16 bytes in flight: parts first, first + step, ... of a row
    auto ask = [&](int q, int group, int first, int step) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < kLoads; u++) {
            const int p = first + u * step;
            v[u] = load_part(rp, p < parts && q < a.Sq ? (uint32_t)((row_of(p, q) * kGroups + group) * 16) : kOobA);
        }
    };
    u32x2 state[kMaxSq / WAVES];
#pragma unroll
    for (int j = 0; j < kMaxSq / WAVES; j++) {
        const int q = wave + j * WAVES;
        state[j] = __builtin_amdgcn_raw_buffer_load_b64(rl, lane < parts && q < a.Sq ? (uint32_t)(row_of(lane, q) * 8) : kOobA, 0, kAgentScope);
    }
    int q = first < sharers ? slot % together : a.Sq;
    ask(q, group, first, sharers);
#pragma unroll
    for (int j = 0; j < kMaxSq / WAVES; j++) {
        const int qw = wave + j * WAVES;
        if (qw >= a.Sq) break;
        const uint32_t m_bits = state[j].x, l_bits = state[j].y;
        const float pm = lane < parts ? __builtin_bit_cast(float, m_bits) : -INFINITY, m = wave_max(pm);
        const float al = lane < parts ? weight<NAT>(pm, m == -INFINITY ? 0.f : m) : 0.f;
        const float l = wave_sum(__builtin_bit_cast(float, l_bits) * al);
        weights[qw * 64 + lane] = al;
        if (lane == 0) inverse[qw] = l > 1e-10f ? 1.f / l : 0.f;
    }
    __syncthreads();
    for (; q < a.Sq; q += together) {
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
        for (int p0 = first;;) {
#pragma unroll
            for (int u = 0; u < kLoads; u++) {
                const float al = weights[q * 64 + min(p0 + u * sharers, 63)];
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = fmaf(v[u][e], al, o[e]);
            }
            p0 += kLoads * sharers;
            if (p0 >= parts) break;
            ask(q, group, p0, sharers);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            if (sharers == 1) put(q, group, e, o[e] * inverse[q]);
            else shares[(first * a.Sq + q) * D + NF * (4 * (group & 3) + e) + (group >> 2)] = o[e];
        }
        if (q + together < a.Sq) ask(q + together, group, first, sharers);
    }
    if (sharers == 1) return;
    __syncthreads();
    for (int idx = threadIdx.x; idx < a.Sq * D; idx += 64 * WAVES) {
        float o = shares[idx] + shares[a.Sq * D + idx];       // (two threads share four sums, or four)
        if (sharers == 4) o += shares[2 * a.Sq * D + idx] + shares[3 * a.Sq * D + idx];
        op[(int64_t)(idx / D) * a.os[2] + idx % D] = Elem<T>::from_f32(o * inverse[idx / D]);
    }
}

// How a launch's keys are dealt: parts of the range, keys a part, waves of a workgroup.
struct DecodePlan { int parts, per, waves; };

DecodePlan decode_plan(int64_t bh, int64_t Skv) {
    auto dealt = [&](int64_t want, int waves) {
        const int64_t unit = part_keys(Skv), most = Skv / unit, n = want < most ? want : most;
        const int parts = n < 2 ? 1 : n > 64 ? 64 : (int)n;
        return DecodePlan{parts, parts == 1 ? (int)Skv : (int)(((Skv + parts - 1) / parts + unit - 1) / unit * unit), waves};
    };
    // Workgroups of eight waves, one a compute unit, where 256 units divided among the heads leave fewer than a quarter of them over and more than four waves of a workgroup get
    // a block of keys (a part being 256 keys at least, or 128, and parts 64 at most, few heads over few keys do not fill the units either way): half as many parts to write and
    // to put together as with two workgroups of four waves a unit, which is what the others take.  us, four | eight waves, one query: 8 heads over 16384 keys of head size 128
    // 23.0 | 17.7 (eight queries 26.3 | 19.2), 32 over 4096 15.8 | 14.7, 192 over 700 16.3 | 13.2, 64 over 200 6.0 | 5.1, 256 over 4096 93.9 | 93.2, of 64 48.8 | 46.1, 12 over 5632
    // of 64 11.3 | 9.1, 12 over 300 5.1 | 4.8; sixteen queries, 256 over 250 of 128 10.5 | 11.2, 16 over 2048 11.5 | 11.6, nine of 128 over 512 11.7 | 10.9 (their number is left out of the rule, so that
    // a row's bits do not follow from it); of more heads a second turn ([32,12,1000] of 64, four queries, 21.2 | 22.6, 512 over 4096 177 | 179); parts of 128 keys 24 over 1024 of 64 6.1 | 6.4.
    if (bh <= 256 && 256 / bh * bh >= 192) {
        const DecodePlan p = dealt(256 / bh, 8);
        if (p.per > 4 * kKeys) return p;
    }
    return dealt((512 + bh - 1) / bh, 4);
}

template <typename T, int D, int WAVES>
int launch_waves(hipStream_t s, const FaArgs& a, float* part, const DecodePlan& plan) {
    const int64_t bh = (int64_t)a.B * a.H;
    const dim3 grid((unsigned)bh, (unsigned)((a.Skv + plan.per - 1) / plan.per));
    uint64_t* words = reinterpret_cast<uint64_t*>(part + (int64_t)plan.parts * bh * a.Sq * (D + 2));
    const uint64_t tag = plan.parts > 1 ? launch_tag() : 0;
    if (plan.parts == 1) part = nullptr;
    if (a.mask) hipLaunchKernelGGL((fa_decode_kernel<T, D, true, WAVES>), grid, dim3(64 * WAVES), 0, s, a, part, plan.per, words, tag);
    else hipLaunchKernelGGL((fa_decode_kernel<T, D, false, WAVES>), grid, dim3(64 * WAVES), 0, s, a, part, plan.per, words, tag);
    return check_launch("flash_attention_decode");
}

template <typename T, int D>
int launch(hipStream_t s, const FaArgs& a, float* part, const DecodePlan& plan) {
    return plan.waves == 8 ? launch_waves<T, D, 8>(s, a, part, plan) : launch_waves<T, D, 4>(s, a, part, plan);
}

}  // namespace

// (checked by the caller: 16-bit, aligned, extents below 2 GB, Skv > 0, D 64 or 128)
bool fa_decode_eligible(const FaArgs& a) { return a.Sq <= kMaxSq && !a.is_causal; }

int64_t fa_decode_workspace(int64_t bh, int64_t Sq, int64_t Skv, int64_t D) {
    if (Sq < 1 || Sq > kMaxSq || (D != 64 && D != 128)) return 0;
    const int parts = decode_plan(bh, Skv).parts;
    return parts == 1 ? 0 : parts * bh * Sq * (D + 2) * 4 + bh * 8;
}

int launch_fa_decode(hipStream_t s, const FaArgs& a, int64_t D, int dtype, void* workspace, int64_t workspace_bytes) {
    const int64_t bh = (int64_t)a.B * a.H, need = fa_decode_workspace(bh, a.Sq, a.Skv, D);
    DecodePlan plan = decode_plan(bh, a.Skv);
    if (!workspace || need > workspace_bytes) { plan.parts = 1; plan.per = a.Skv; }
    float* part = static_cast<float*>(workspace);
    if (dtype == MHIP_BF16) return D == 128 ? launch<bf16_t, 128>(s, a, part, plan) : launch<bf16_t, 64>(s, a, part, plan);
    return D == 128 ? launch<f16_t, 128>(s, a, part, plan) : launch<f16_t, 64>(s, a, part, plan);
}

}  // namespace mhip
