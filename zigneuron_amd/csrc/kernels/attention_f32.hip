// Fused single-pass attention for gfx950 on the fp32 matrix cores:
// O = softmax(scale * Q K^T) V per problem (one head, [seq_len x d_k] row
// major), the contract of cpuAttentionForward (src/backend.zig:3197-3222),
// without writing the [seq_len x seq_len] scores to memory.
//
// Each wave owns 32 queries and walks the keys in blocks of BKV, keeping a
// running row maximum and row sum (the online softmax): for every block
//   S^T = K_blk . (c Q)^T        (v_mfma_f32_32x32x2f32, K-dim = head dim)
//   m'  = max(m, max_key S^T),  P^T = exp2(S^T - m'),  c = scale*log2(e)
//   O^T = O^T * exp2(m - m') + V_blk^T . P^T,   l = l * exp2(m - m') + sum P
// and at the end O = O^T^T / l.
//
// Computing the transposed products makes the data flow register-only:
//  * the S^T accumulator (lane j + 32h, register r: key 8(r/4) + 4h + r%4 of a
//    32-key block, query j) is, register for register, the B operand of the
//    V^T . P^T product under the K order used by every kernel here (lane half
//    h, step t of K group g covers k = 8g + 4h + t);
//  * every value of query j lives in lanes j and j + 32, so the softmax
//    needs one cross-half exchange per block (the block maximum) and the
//    O^T rescale is lane-local.
// Q stays in registers for the whole walk; K and V blocks go HBM -> LDS by
// DMA (buffer_load ... lds, two stages, the same staging as the GEMM), K
// stored key-major [BKV][DP], V stored [BKV][DP] and read with the
// X-contiguous fragment rule (head dim d = FD*i + f for lane i, block f).
// Head dims are zero-padded to DP; keys past seq_len get score -inf.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../zn_kernel_args.h"

#include "zn_mfma_stage.h"
#include "zn_split.h"

#include <type_traits>

namespace {

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }

// One key block of the walk: S^T = K_blk . Q^T, the online-softmax update of
// (m, l, O^T) and O^T += V_blk^T . P^T.  MASK: the block runs past seq_len
// (only the last one can), its missing keys get score -inf.
template <int DP, int BKV, bool MASK>
__device__ __forceinline__ void attention_block(const float *lk, const float *lv, const float (&qf)[DP / 8][4],
                                                zn_f32x16 (&o)[DP / 32], float &m, float &l, int kv0, int S,
                                                int lane) {
    constexpr int FD = DP / 32;   // 32-row blocks of O^T (head dim)
    constexpr int FS = BKV / 32;  // 32-row blocks of S^T (keys)
    const int h = lane >> 5;
    zn_f32x16 s[FS];
#pragma unroll
    for (int f = 0; f < FS; ++f)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[f][r] = 0.0f;
#pragma unroll
    for (int g = 0; g < DP / 8; ++g) {
        float kf[FS][4];
        read_frags_dma<BKV, DP, FS, true>(lk, 0, 8 * g, lane, kf);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int f = 0; f < FS; ++f) s[f] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[f][t], qf[g][t], s[f], 0, 0, 0);
    }

    // scores are already in the log2 domain (Q was scaled by scale*log2(e))
    float mb = -INFINITY;
#pragma unroll
    for (int f = 0; f < FS; ++f)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if constexpr (MASK)
                if (kv0 + 32 * f + 8 * (r / 4) + 4 * h + (r % 4) >= S) s[f][r] = -INFINITY;
            mb = fmaxf(mb, s[f][r]);
        }
    mb = fmaxf(mb, __shfl_xor(mb, 32));
    const float mn = fmaxf(m, mb);  // finite: every block holds at least one key
    const float alpha = exp2_fast(m - mn);
    float rs = 0.0f;
#pragma unroll
    for (int f = 0; f < FS; ++f)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float e = exp2_fast(s[f][r] - mn);
            s[f][r] = e;
            rs += e;
        }
    l = l * alpha + rs;
    m = mn;
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {  // some query's maximum moved
#pragma unroll
        for (int f = 0; f < FD; ++f)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[f][r] *= alpha;
    }

    // O^T += V_blk^T . P^T; P^T is the S^T accumulator, register 4g + t
#pragma unroll
    for (int fs = 0; fs < FS; ++fs)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            float vf[FD][4];
            read_frags_x<DP, BKV, FD>(lv, 0, 32 * fs + 8 * g, lane, vf);
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int f = 0; f < FD; ++f)
                    o[f] = __builtin_amdgcn_mfma_f32_32x32x2f32(vf[f][t], s[fs][4 * g + t], o[f], 0, 0, 0);
        }
}

// Grid: blockIdx.x = problem, blockIdx.y = block of NW*32 queries, so the
// query blocks of one problem share an XCD and its L2 copy of K and V.
template <int DP, int BKV, int NW, int W>
__device__ __forceinline__ void attention_tile(const ZnAttnArgs &p) {
    constexpr int NT = NW * kWave;
    constexpr int FD = DP / 32;
    static_assert(DP % 32 == 0 && BKV % 32 == 0, "whole 32x32 blocks");
    typedef DmaStage<BKV, DP, NT, true, W> SK;   // K block, [key][d]
    typedef DmaStage<DP, BKV, NT, false, W> SV;  // V block, [key][d]
    __shared__ __attribute__((aligned(1024))) float lds_k[2][SK::kFloats];
    __shared__ __attribute__((aligned(1024))) float lds_v[2][SV::kFloats];

    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int j = lane & 31, h = lane >> 5;
    const int S = p.seq_len, D = p.d_k;
    const int64_t base = (int64_t)blockIdx.x * p.stride;
    const float *gq = p.q + base;
    const int q = (int)blockIdx.y * (NW * 32) + wave * 32 + j;  // this lane's query

    // Q^T fragments, the B operand of S^T = K . Q^T: qf[g][t] = Q[q][8g + 4h + t] * scale*log2(e).
    float qf[DP / 8][4];
#pragma unroll
    for (int g = 0; g < DP / 8; ++g) {
        const int f0 = 8 * g + 4 * h;
        if constexpr (W == 16) {
            zn_f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
            if (q < S && f0 < D) v = *reinterpret_cast<const zn_f32x4 *>(gq + (int64_t)q * D + f0);
#pragma unroll
            for (int t = 0; t < 4; ++t) qf[g][t] = v[t] * p.scale_log2;
        } else {
#pragma unroll
            for (int t = 0; t < 4; ++t)
                qf[g][t] = (q < S && f0 + t < D) ? gq[(int64_t)q * D + f0 + t] * p.scale_log2 : 0.0f;
        }
    }

    zn_f32x16 o[FD];
#pragma unroll
    for (int f = 0; f < FD; ++f)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[f][r] = 0.0f;
    float m = -INFINITY;  // running maximum of this query's scaled scores (log2 domain)
    float l = 0.0f;       // this lane's share of the running sum

    const uint32_t bytes = (uint32_t)((int64_t)S * D * 4);
    const __amdgpu_buffer_rsrc_t rk = make_rsrc(p.k + base, bytes);
    const __amdgpu_buffer_rsrc_t rv = make_rsrc(p.v + base, bytes);
    const int nblk = (S + BKV - 1) / BKV;
    const int nfull = S / BKV;  // blocks with no missing keys
    SK::issue(rk, lds_k[0], D, 0, 0, S, D, wave, lane);
    SV::issue(rv, lds_v[0], D, 0, 0, D, S, wave, lane);
    for (int b = 0; b < nblk; ++b) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's part of block b is in LDS
        __syncthreads();  // every wave's part is; every wave is done with block b - 1
        const int cur = b & 1;
        if (b + 1 < nblk) {
            SK::issue(rk, lds_k[cur ^ 1], D, (b + 1) * BKV, 0, S, D, wave, lane);
            SV::issue(rv, lds_v[cur ^ 1], D, 0, (b + 1) * BKV, D, S, wave, lane);
        }
        if (b < nfull)
            attention_block<DP, BKV, false>(lds_k[cur], lds_v[cur], qf, o, m, l, b * BKV, S, lane);
        else
            attention_block<DP, BKV, true>(lds_k[cur], lds_v[cur], qf, o, m, l, b * BKV, S, lane);
    }

    // O[q][d] = O^T[d][q] / l.  Register r of block f holds d = FD*(8(r/4) + 4h + r%4) + f:
    // for each r/4 the lane owns the 4*FD consecutive head dims starting at FD*(8(r/4) + 4h).
    l += __shfl_xor(l, 32);
    if (q < S) {
        float *orow = p.out + base + (int64_t)q * D;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int d0 = FD * (8 * g + 4 * h);
            float vals[4 * FD];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int f = 0; f < FD; ++f) vals[FD * t + f] = o[f][4 * g + t] / l;
            if constexpr (W == 16) {
#pragma unroll
                for (int c = 0; c < FD; ++c)
                    if (d0 + 4 * c < D)
                        *reinterpret_cast<zn_f32x4 *>(orow + d0 + 4 * c) =
                            zn_f32x4{vals[4 * c], vals[4 * c + 1], vals[4 * c + 2], vals[4 * c + 3]};
            } else {
#pragma unroll
                for (int e = 0; e < 4 * FD; ++e)
                    if (d0 + e < D) orow[d0 + e] = vals[e];
            }
        }
    }
}

// ---------------------------------------------------------------- split form
// The same walk on the bf16 matrix cores, every operand value split into
// three bf16 parts (zn_split.h): S^T = K . (cQ)^T and O^T += V^T . P^T on
// v_mfma_f32_16x16x32_bf16.  Q is split once per workgroup into registers; K
// and V blocks of 32 keys are loaded through registers, split and written to
// LDS (two stages), V transposed on the way.  In the order of a slice used
// here (chunk c: k = 4c .. 4c + 3 and 16 + 4c .. 16 + 4c + 3) the two 16-key
// S^T accumulators of a lane are its chunk of the P^T operand, so P stays in
// registers as before.
//
// A walk whose scores or sums are not finite (an Inf or NaN input, or
// magnitudes whose scaled products overflow) is done again by its wave alone
// on the fp32 matrix cores, straight from memory (attention_plain).
//
// Few problems leave most of the chip idle: then blockIdx.z takes a range of
// the keys, and zn_attention_combine merges the ranges' (O, m, l).
template <int DP, int NW, int FQ, int BKV>
struct AttnSplit {
    static constexpr int NT = NW * kWave;
    static constexpr int SL = DP / 32, DB = DP / 16;  // 32-deep slices and 16-row blocks of the head dim
    static constexpr int KB = BKV / 32;               // 32-key slices of a block
    static constexpr int kPart = DP * 2 * BKV;        // bytes of one bf16 part of a K (or V) block
    static constexpr int kStage = 6 * kPart;
    static constexpr int kUnits = DP * BKV / 4;       // staging units of 8 values: K, then V
    static constexpr int UPT = (kUnits + NT - 1) / NT;
    static_assert(kUnits / 2 % kWave == 0, "a wave's units are all of K or all of V");

    __device__ static __forceinline__ int slot(int r, int c) { return r * 64 + ((c ^ (-(r >> 2) & 3)) << 4); }
    __device__ static __forceinline__ float max_over_quads(float x) {
        // the 4 lanes of a query: li, li + 16, li + 32, li + 48
        const auto a = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
        x = fmaxf(__builtin_bit_cast(float, a[0]), __builtin_bit_cast(float, a[1]));
        const auto b = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, x), false, false);
        return fmaxf(__builtin_bit_cast(float, b[0]), __builtin_bit_cast(float, b[1]));
    }

    __device__ static __forceinline__ void run(const ZnAttnArgs &p, char *lds) {
        const int tid = threadIdx.x, lane = tid & (kWave - 1);
        const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
        const int li = lane & 15, lh = lane >> 4;
        const int S = p.seq_len, D = p.d_k;
        const int64_t base = (int64_t)blockIdx.x * p.stride;
        const int q0 = (int)blockIdx.y * (NW * FQ * 16) + wave * FQ * 16;
        const int kbeg = (int)blockIdx.z * p.keys_per_split;
        const int kend = min(S, kbeg + p.keys_per_split);
        const uint32_t bytes = (uint32_t)((int64_t)S * D * 4);
        const __amdgpu_buffer_rsrc_t rq = make_rsrc(p.q + base, bytes);
        const __amdgpu_buffer_rsrc_t rk = make_rsrc(p.k + base, bytes);
        const __amdgpu_buffer_rsrc_t rv = make_rsrc(p.v + base, bytes);

        // staging units of this thread: byte offset of the first load at key kbeg, LDS position
        uint32_t off0[UPT];
        int lpos[UPT];
        bool is_v[UPT];
#pragma unroll
        for (int j = 0; j < UPT; ++j) {
            const int u = j * NT + tid;
            is_v[j] = __builtin_amdgcn_readfirstlane(u) >= kUnits / 2;
            if (!is_v[j]) {
                const int key = u / (DP / 8), dc = u % (DP / 8);  // chunk dc % 4 of slice dc / 4
                const int d = 32 * (dc / 4) + 4 * (dc % 4);
                off0[j] = (uint32_t)((kbeg + key) * D + d) * 4u;
                lpos[j] = (dc / 4) * (BKV * 64) + slot(key, dc % 4);
            } else {
                const int v = u - kUnits / 2, d = v % DP, ks = v / DP / 4, c = v / DP % 4;  // key slice and chunk
                off0[j] = d < D ? (uint32_t)((kbeg + 32 * ks + 4 * c) * D + d) * 4u : kOutOfRange;
                lpos[j] = 3 * kPart + ks * (DP * 64) + slot(d, c);
            }
        }
        const uint32_t row = (uint32_t)D * 4u;
        float g[UPT][8];
        auto load = [&](int b, int j) {
            if (j * NT + tid >= kUnits) return;  // whole waves
            const uint32_t off = off0[j] == kOutOfRange ? kOutOfRange : off0[j] + (uint32_t)b * (BKV * row);
            if (!is_v[j]) {
                const zn_f32x4 v0 = __builtin_bit_cast(zn_f32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, off, 0, 0));
                const zn_f32x4 v1 = __builtin_bit_cast(zn_f32x4, __builtin_amdgcn_raw_buffer_load_b128(rk, off + 64, 0, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    g[j][e] = v0[e];
                    g[j][4 + e] = v1[e];
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const uint32_t o = off == kOutOfRange ? off : off + (e < 4 ? e : 12 + e) * row;
                    g[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rv, o, 0, 0));
                }
            }
        };
        auto stage = [&](int st, int j) {
            if (j * NT + tid >= kUnits) return;
            zn_u32x4 w[3];
            split8(g[j], w);
#pragma unroll
            for (int q = 0; q < 3; ++q) *reinterpret_cast<zn_u32x4 *>(lds + st * kStage + lpos[j] + q * kPart) = w[q];
        };
        const int fr = slot(li, lh);
        auto read_k = [&](int st, int sl, int kb, int q) {
            return __builtin_bit_cast(zn_bf16x8, *reinterpret_cast<const zn_u32x4 *>(lds + st * kStage + q * kPart + sl * (BKV * 64) + kb * (16 * 64) + fr));
        };
        auto read_v = [&](int st, int ks, int db, int q) {
            return __builtin_bit_cast(zn_bf16x8, *reinterpret_cast<const zn_u32x4 *>(lds + st * kStage + (3 + q) * kPart + ks * (DP * 64) + db * (16 * 64) + fr));
        };

#pragma unroll
        for (int j = 0; j < UPT; ++j) load(0, j);
        // Q^T fragments: query 16f + li, chunk lh of slice sl, times scale * log2(e)
        zn_bf16x8 qf[FQ][SL][3];
#pragma unroll
        for (int f = 0; f < FQ; ++f)
#pragma unroll
            for (int sl = 0; sl < SL; ++sl) {
                const int q = q0 + 16 * f + li, d = 32 * sl + 4 * lh;
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int de = d + (e < 4 ? e : 12 + e);
                    const uint32_t off = q < S && de < D ? (uint32_t)(q * D + de) * 4u : kOutOfRange;
                    x[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rq, off, 0, 0)) * p.scale_log2;
                }
                zn_u32x4 w[3];
                split8(x, w);
#pragma unroll
                for (int r = 0; r < 3; ++r) qf[f][sl][r] = __builtin_bit_cast(zn_bf16x8, w[r]);
            }

        zn_f32x4 o[FQ][DB];
        float m[FQ], l[FQ];  // running maximum (log2 domain), this lane's share of the running sum
#pragma unroll
        for (int f = 0; f < FQ; ++f) {
#pragma unroll
            for (int d = 0; d < DB; ++d) o[f][d] = zn_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            m[f] = -INFINITY;
            l[f] = 0.0f;
        }
#pragma unroll
        for (int j = 0; j < UPT; ++j) stage(0, j);
        constexpr int kPA[6] = {2, 1, 0, 1, 0, 0}, kPB[6] = {0, 1, 2, 0, 1, 0};
        const int nblk = (kend - kbeg + BKV - 1) / BKV;
        // MASK: the range's last block, its missing keys get score -inf
        auto block = [&](int b, auto mc) {
            constexpr bool MASK = decltype(mc)::value;
            const int st = b & 1;
            __syncthreads();  // block b is in LDS; every wave is done with block b - 1
#pragma unroll
            for (int j = 0; j < UPT; ++j) load(b + 1, j);
            zn_f32x4 s[FQ][2 * KB];
#pragma unroll
            for (int f = 0; f < FQ; ++f)
#pragma unroll
                for (int kb = 0; kb < 2 * KB; ++kb) s[f][kb] = zn_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int kp = 0; kp < KB; ++kp)
#pragma unroll
                for (int sl = 0; sl < SL; ++sl) {
                    zn_bf16x8 kf[2][3];
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                        for (int q = 0; q < 3; ++q) kf[kb][q] = read_k(st, sl, 2 * kp + kb, q);
#pragma unroll
                    for (int pr = 0; pr < 6; ++pr)
#pragma unroll
                        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                            for (int f = 0; f < FQ; ++f)
                                s[f][2 * kp + kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kb][kPA[pr]], qf[f][sl][kPB[pr]],
                                                                                            s[f][2 * kp + kb], 0, 0, 0);
                }
            zn_bf16x8 pf[FQ][KB][3];
            const int left = kend - kbeg - b * BKV;  // keys of this range from this block on
#pragma unroll
            for (int f = 0; f < FQ; ++f) {
                float mb = -INFINITY;
#pragma unroll
                for (int kb = 0; kb < 2 * KB; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        if (MASK && 16 * kb + 4 * lh + r >= left) s[f][kb][r] = -INFINITY;
                        mb = fmaxf(mb, s[f][kb][r]);
                    }
                const float mn = fmaxf(m[f], max_over_quads(mb) * kSplitUnscale);
                const float alpha = exp2_fast(m[f] - mn);
                float rs = 0.0f;
#pragma unroll
                for (int kb = 0; kb < 2 * KB; ++kb)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        s[f][kb][r] = exp2_fast(__builtin_fmaf(s[f][kb][r], kSplitUnscale, -mn));
                        rs += s[f][kb][r];
                    }
                l[f] = l[f] * alpha + rs;
                m[f] = mn;
                if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {
#pragma unroll
                    for (int d = 0; d < DB; ++d) o[f][d] *= alpha;
                }
#pragma unroll
                for (int ks = 0; ks < KB; ++ks) {
                    float e8[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) e8[e] = s[f][2 * ks + e / 4][e % 4];
                    zn_u32x4 w[3];
                    split8(e8, w);
#pragma unroll
                    for (int q = 0; q < 3; ++q) pf[f][ks][q] = __builtin_bit_cast(zn_bf16x8, w[q]);
                }
            }
#pragma unroll
            for (int d = 0; d < DB; ++d) {
#pragma unroll
                for (int ks = 0; ks < KB; ++ks) {
                    zn_bf16x8 vf[3];
#pragma unroll
                    for (int q = 0; q < 3; ++q) vf[q] = read_v(st, ks, d, q);
#pragma unroll
                    for (int pr = 0; pr < 6; ++pr)
#pragma unroll
                        for (int f = 0; f < FQ; ++f)
                            o[f][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[kPA[pr]], pf[f][ks][kPB[pr]], o[f][d], 0, 0, 0);
                }
                // the next block's staging, spread over the products
#pragma unroll
                for (int j = 0; j < UPT; ++j)
                    if (j * DB / UPT == d) stage(st ^ 1, j);
            }
        };
        const int nfull = (kend - kbeg) / BKV;
        for (int b = 0; b < nfull; ++b) block(b, std::false_type());
        if (nfull < nblk) block(nfull, std::true_type());
        bool bad = false;
#pragma unroll
        for (int f = 0; f < FQ; ++f) {
            bad |= !(l[f] < INFINITY);
#pragma unroll
            for (int d = 0; d < DB; ++d)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    bad |= !(__builtin_fabsf(o[f][d][r]) < INFINITY);
                    o[f][d][r] *= kSplitUnscale;
                }
        }
        if (__builtin_amdgcn_ballot_w64(bad)) plain(p, rq, rk, rv, q0, kbeg, kend, lane, o, m, l);
#pragma unroll
        for (int f = 0; f < FQ; ++f) {
            float sum = l[f] + __shfl_xor(l[f], 16);
            sum += __shfl_xor(sum, 32);
            const int q = q0 + 16 * f + li;
            if (q >= S) continue;
            if (p.splits > 1) {
                // [problem][query][range]: D rounded up to 4 of O, then m and l
                const int ld = ((D + 3) & ~3) + 4;
                float *dst = p.part + (((int64_t)blockIdx.x * S + q) * p.splits + blockIdx.z) * ld;
#pragma unroll
                for (int d = 0; d < DB; ++d)
                    if (16 * d + 4 * lh < D) *reinterpret_cast<zn_f32x4 *>(dst + 16 * d + 4 * lh) = o[f][d];
                if (lh == 0) {
                    dst[ld - 4] = m[f];
                    dst[ld - 3] = sum;
                }
                continue;
            }
            float *orow = p.out + base + (int64_t)q * D;
#pragma unroll
            for (int d = 0; d < DB; ++d) {
                const int col = 16 * d + 4 * lh;
                if (col + 4 <= D) {
                    *reinterpret_cast<zn_f32x4u *>(orow + col) = o[f][d] / sum;
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (col + r < D) orow[col + r] = o[f][d][r] / sum;
                }
            }
        }
    }

    // The wave's queries on the fp32 matrix cores, 16 keys at a time, K and V read from memory.
    __device__ static __forceinline__ void plain(const ZnAttnArgs &p, __amdgpu_buffer_rsrc_t rq, __amdgpu_buffer_rsrc_t rk,
                                                 __amdgpu_buffer_rsrc_t rv, int q0, int kbeg, int kend, int lane,
                                                 zn_f32x4 (&o)[FQ][DB], float (&m)[FQ], float (&l)[FQ]) {
        const int li = lane & 15, lh = lane >> 4;
        const int S = p.seq_len, D = p.d_k;
        auto get = [&](__amdgpu_buffer_rsrc_t r, int x, int d, int lim) {
            const uint32_t off = x < lim && d < D ? (uint32_t)(x * D + d) * 4u : kOutOfRange;
            return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
        };
#pragma unroll
        for (int f = 0; f < FQ; ++f) {
            const int q = q0 + 16 * f + li;
#pragma unroll
            for (int d = 0; d < DB; ++d) o[f][d] = zn_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            m[f] = -INFINITY;
            l[f] = 0.0f;
            for (int k0 = kbeg; k0 < kend; k0 += 16) {
                zn_f32x4 s = {0.0f, 0.0f, 0.0f, 0.0f};
                for (int d = 0; d < D; d += 4)
                    s = __builtin_amdgcn_mfma_f32_16x16x4f32(get(rk, k0 + li, d + lh, kend), get(rq, q, d + lh, S) * p.scale_log2, s, 0, 0, 0);
                float mb = -INFINITY;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (k0 + 4 * lh + r >= kend) s[r] = -INFINITY;
                    mb = fmaxf(mb, s[r]);
                }
                const float mn = fmaxf(m[f], max_over_quads(mb));
                const float ref = mn == -INFINITY ? 0.0f : mn;  // nothing but -inf scores so far
                const float alpha = exp2_fast(m[f] - ref);
                float rs = 0.0f;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    s[r] = exp2_fast(s[r] - ref);
                    rs += s[r];
                }
                l[f] = l[f] * alpha + rs;
                m[f] = mn;
#pragma unroll
                for (int d = 0; d < DB; ++d) {
                    o[f][d] *= alpha;
#pragma unroll
                    for (int r = 0; r < 4; ++r)  // k index lh of step r: key k0 + 4 lh + r
                        o[f][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(get(rv, k0 + 4 * lh + r, 16 * d + li, kend), s[r], o[f][d], 0, 0, 0);
                }
            }
        }
    }
};

}  // namespace

// zn_attention_d<DP>[_v]: head dims up to DP (zero-padded), 4 waves = 128
// queries per workgroup, blockIdx.x = problem, blockIdx.y = query block.  _v: 16-byte loads and stores
// (d_k % 4 == 0, 16-byte aligned Q, K, V and O).
#define ZN_ATTN_KERNEL(DP, BKV, W, SUFFIX)                                                   \
    extern "C" __global__ __launch_bounds__(256, 2) void zn_attention_d##DP##SUFFIX(ZnAttnArgs p) { \
        attention_tile<DP, BKV, 4, W>(p);                                                    \
    }
#define ZN_ATTN_DIM(DP, BKV)          \
    ZN_ATTN_KERNEL(DP, BKV, 16, _v)   \
    ZN_ATTN_KERNEL(DP, BKV, 4, )

ZN_ATTN_DIM(32, 64)
ZN_ATTN_DIM(64, 64)

// zn_attention_s<DP>: the split form, head dims up to DP, any alignment;
// NW waves of FQ x 16 queries.
#define ZN_ATTN_SPLIT(DP, NW, FQ, BKV)                                                                         \
    extern "C" __global__ __launch_bounds__(NW * 64, 2) void zn_attention_s##DP(ZnAttnArgs p) {           \
        typedef AttnSplit<DP, NW, FQ, BKV> T;                                                                  \
        __shared__ __attribute__((aligned(1024))) char lds[2 * T::kStage];                                \
        T::run(p, lds);                                                                                   \
    }
ZN_ATTN_SPLIT(32, 4, 2, 64)
ZN_ATTN_SPLIT(64, 8, 2, 64)
ZN_ATTN_SPLIT(96, 8, 1, 32)
ZN_ATTN_SPLIT(128, 8, 1, 32)

// out[query] = sum over ranges z of 2^(m_z - M) O_z / sum of 2^(m_z - M) l_z,
// M = max m_z, the ranges in ascending order.  One wave per query: lane z
// takes range z's m and l, lane d the head dims d and d + 64, whose range
// loads are all independent (splits <= 32; MI355X, 1000 queries of 80 dims in
// 16 ranges: one thread per element walking m, l and O took 12 us).
constexpr int kMaxAttnSplits = 32;
extern "C" __global__ __launch_bounds__(256) void zn_attention_combine(ZnAttnArgs p) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t q = (int64_t)blockIdx.x * 4 + threadIdx.x / kWave;
    if (q >= (int64_t)p.batch * p.seq_len) return;
    const int ld = ((p.d_k + 3) & ~3) + 4;
    const float *src = p.part + q * p.splits * ld;
    float ov[2][kMaxAttnSplits];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int z = 0; z < kMaxAttnSplits; ++z) {
            ov[i][z] = 0.0f;
            if (z < p.splits && lane + 64 * i < p.d_k) ov[i][z] = src[z * ld + lane + 64 * i];
        }
    const bool in = lane < p.splits;
    const float m = in ? src[lane * ld + ld - 4] : -INFINITY;
    const float l = in ? src[lane * ld + ld - 3] : 0.0f;
    float mx = m;
#pragma unroll
    for (int s = 1; s < kMaxAttnSplits; s <<= 1) mx = fmaxf(mx, __shfl_xor(mx, s));
    const float w = exp2_fast(m - (mx == -INFINITY ? 0.0f : mx));
    const float wl = in ? w * l : 0.0f;
    float sum = 0.0f, o[2] = {0.0f, 0.0f};
#pragma unroll
    for (int z = 0; z < kMaxAttnSplits; ++z)
        if (z < p.splits) {
            const float wz = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), z));
            sum += __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, wl), z));
            o[0] += wz * ov[0][z];
            o[1] += wz * ov[1][z];
        }
    float *row = p.out + q / p.seq_len * p.stride + q % p.seq_len * p.d_k;
#pragma unroll
    for (int i = 0; i < 2; ++i)
        if (lane + 64 * i < p.d_k) row[lane + 64 * i] = o[i] / sum;
}
