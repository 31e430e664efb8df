// fp32 GEMM on the bf16 matrix cores of gfx950, operands split into three
// bf16 parts (zn_split.h).
#ifndef ZN_GEMM_SPLIT_H
#define ZN_GEMM_SPLIT_H

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../zn_kernel_args.h"

#include "gemm_core.h"
#include "zn_split.h"

namespace {

// One workgroup of NW waves: a 16 FM NW x BN tile of C, wave w its rows
// 16 FM w .. 16 FM (w + 1) - 1, K in slices of 32.
//  * Any row alignment: K-contiguous operands are loaded 16 bytes at a time
//    at 4-byte aligned offsets (each descriptor spans its operand exactly and
//    is checked per dword), X-contiguous ones a dword a lane, 64 neighbouring
//    x at once; k past the end is set to zero in registers.
//  * A never passes through LDS: each lane loads and splits the values of its
//    own fragments, since no other wave reads those rows.  B is split by the
//    thread that loads it and written to one of two LDS stages (6 bytes a
//    value; the writes run at 64 bytes a clock, so leaving A out of them
//    gained more than its row-per-lane loads cost: 8192^3 NN on 256x128 tiles
//    5.5 -> 4.9 ms).
//  * Fragments are read with ds_read_b128, free of bank conflicts (slot);
//    with the plain XOR of the fp32 tiles they took 8.1 clocks, now 4.8.
//  * FLUSH: the six products of a slice are summed from zero and then added
//    to the tile's sums, one rounding of the long sum per 32 of K instead of
//    six (K 512: 1.2e-7 against 3.4e-7).  The 256x256 tile has no registers
//    for it (it spills 240 of them) and keeps one chain, itself a little
//    closer to 64 bits than the fp32 kernels.  Tiles of one kind give a value
//    the same bits, so the 128x128 one has a chain form too (sc), for a part
//    of a product whose whole runs on 256x256.
//  * What bounds it: the vector instructions beside the products, 6.5 to split
//    a value and 1.1 a product on 256x256 tiles, 3.1 on 128x128 (a product
//    alone takes 16 clocks of its matrix core; four vector instructions beside
//    it made that 29 in a loop of nothing else).  Counters: at 8192^3 the
//    matrix cores are busy 74% of the time, in one round of 128x128 tiles 35 to
//    38%.  Larger tiles split each value for more products: 256x256 4.2-4.4 ms
//    at 8192^3 (the fp32 tile 7.35), 256x128 4.8, 128x128 5.2, 128x64 6.0.
//    Loads two and four slices ahead, XCD-blocked tile orders and four columns
//    at a time changed nothing.
//  * Registers: 256x256 spills 112 bytes around its loop and in the epilogue,
//    none inside it.
//  * Sums that are not finite: the wave does its tile again on the fp32
//    matrix cores (plain), about five times slower.  Its finite values then
//    have that arithmetic's bits; taking only the others from there changes
//    how the main loop is scheduled (NN and NT on 128x128 2 to 3% slower).
template <int NW, int FM, int BN, bool AK, bool BKC, bool FLUSH, int GC, int AB, int NV, int G = kGNone, bool GU = false>
struct SplitTile {
    static constexpr int NT = NW * kWave;
    static constexpr int BM = 16 * FM * NW, BK = 32;
    static constexpr int FN = BN / 16, NG = FN / GC;  // column blocks, in groups of GC
    static constexpr int UB = BN * 4 / NT;  // B staging units of 8 k per thread
    static constexpr int kRowBytes = 64;    // 32 bf16
    static constexpr int kPartB = BN * kRowBytes;
    static constexpr int kStage = 3 * kPartB;
    static_assert(BN * 4 % NT == 0 && BN % kWave == 0, "whole units per thread; a wave's X-contiguous loads share one k");

    static constexpr bool GATHER_K = G == kGNhwc || G == kGTransposed;  // convolutions: B gathered K-contiguously
    static constexpr bool GATHER_X = G == kGNhwcW;                      // ... or X-contiguously
    static_assert(G == kGNone || (GATHER_K && BKC) || (GATHER_X && !BKC), "the NHWC gathers");
    // GU: every slice of K lies in one filter tap (GATHER_K: channels are a multiple of 32), or every aligned run of 4 of
    // K in one output row (GATHER_X: out_w a multiple of 4).  A kernel of its own for each, and offsets made without a
    // branch: a branch inside a step ends the region that interleave() orders.
    static constexpr int kNoRow = -(1 << 30);  // an image row that no tap reaches

    // slot of chunk c (8 k, 16 bytes) of LDS row r: the chunks of 4 rows fill the 64 banks, and the rotation spreads the
    // 16 rows of each of the hardware's four 16-lane groups of a ds_read_b128 (lanes 0-3, 12-15, 20-27; ...) over them
    __device__ static __forceinline__ int slot(int r, int c) { return r * kRowBytes + ((c ^ (-(r >> 2) & 3)) << 4); }

    // Instruction order of one group of N products: the splitting of the next slice, the fragment reads, the stage
    // writes and the loads spread evenly between them, NV vector instructions to a product (left alone the compiler
    // puts a unit's fifty in one run: 8192^3 NT 4.61 -> 4.13 ms on 256x256 with 5, 5.15 -> 4.75 ms on 256x128 with 3).
    template <int N>
    __device__ static __forceinline__ void interleave() {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);   // MFMA
            __builtin_amdgcn_sched_group_barrier(0x2, NV, 0);  // VALU
            if (i % 2 == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // LDS read
            if (i % 4 == 1) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // LDS write
            if (i % 4 == 3) __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);   // load
        }
    }

    __device__ static __forceinline__ void run(const ZnGemmArgs &p, char *lds) {
        const int tid = threadIdx.x, lane = tid & (kWave - 1);
        const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
        const int li = lane & 15, lh = lane >> 4;
        int tm, tn, slice;
        tile_coords(p, tm, tn, slice);
        const int m0 = tm * BM + wave * 16 * FM, n0 = tn * BN;
        const int64_t bz = blockIdx.y;
        const int kbeg = slice * p.k_chunk;
        const int kend = min(p.k, kbeg + p.k_chunk);
        const int ktiles = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;
        const int lda = (int)p.lda, ldb = (int)p.ldb;
        const uint32_t a_bytes = (uint32_t)(AK ? (p.m - 1) * lda + p.k : (p.k - 1) * lda + p.m) * 4u;
        const ZnConvGeom &cg = p.conv;
        const uint32_t b_bytes =
            (uint32_t)(GATHER_K   ? cg.channels * cg.in_h * cg.in_w
                       : GATHER_X ? cg.images * cg.channels * cg.in_h * cg.in_w
                       : BKC      ? (p.n - 1) * ldb + p.k
                                  : (p.k - 1) * ldb + p.n) * 4u;
        const __amdgpu_buffer_rsrc_t ra = make_rsrc(p.a + bz * p.stride_a, a_bytes);
        const __amdgpu_buffer_rsrc_t rb = make_rsrc(p.b + bz * p.stride_b, b_bytes);

        // Chunk c of a slice holds k = 4c .. 4c + 3 and 16 + 4c .. 16 + 4c + 3.
        // A: this lane's rows 16f + li, chunk lh.  B: staging units (row, chunk).
        uint32_t offa[FM], offb[UB];
        int lpos[UB], kq[UB];
        int gh[UB], gw[UB];  // gathers: image row and column of the unit's pixel (K) or tap (X), before the other's share
#pragma unroll
        for (int f = 0; f < FM; ++f) {
            const int x = m0 + 16 * f + li;
            offa[f] = x < p.m ? (uint32_t)(AK ? x * lda + kbeg + 4 * lh : x + 4 * lh * lda) * 4u : kOutOfRange;
        }
#pragma unroll
        for (int j = 0; j < UB; ++j) {
            const int u = j * NT + tid;
            const int row = BKC ? u / 4 : u % BN, c = BKC ? u % 4 : u / BN;
            const int x = n0 + row;
            kq[j] = BKC ? 4 * c : __builtin_amdgcn_readfirstlane(4 * c);
            offb[j] = x < p.n ? (uint32_t)(BKC ? x * ldb + kbeg + 4 * c : x) * 4u : kOutOfRange;
            lpos[j] = slot(row, c);
            if constexpr (GATHER_K) {
                const int oh = zn_udiv(x, cg.ow_mul, cg.ow_shift), ow = x - oh * cg.out_w;
                const int ih = G == kGNhwc ? oh * cg.stride_h - cg.pad_h : oh + cg.pad_h;
                gw[j] = G == kGNhwc ? ow * cg.stride_w - cg.pad_w : ow + cg.pad_w;
                gh[j] = x < p.n ? ih : kNoRow;
                offb[j] = (uint32_t)((ih * cg.in_w + gw[j]) * cg.channels + (GU ? kq[j] : 0)) * 4u;
            }
            if constexpr (GATHER_X) {
                const int khw = zn_udiv(x, cg.div1_mul, cg.div1_shift), ic = x - khw * cg.div1;
                const int kh = zn_udiv(khw, cg.kw_mul, cg.kw_shift), kw = khw - kh * cg.k_w;
                gh[j] = x < p.n ? kh - cg.pad_h : kNoRow;
                gw[j] = kw - cg.pad_w;
                offb[j] = (uint32_t)(((kh - cg.pad_h) * cg.in_w + gw[j]) * cg.channels + ic) * 4u;
            }
        }
        float ga[FM][8], gb[UB][8];  // the raw values of the next slice
        auto load_k = [&](__amdgpu_buffer_rsrc_t r, uint32_t off0, int s, float(&g)[8]) {
            const uint32_t off = off0 + (uint32_t)s * (BK * 4u);
            const zn_f32x4 v0 = __builtin_bit_cast(zn_f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
            const zn_f32x4 v1 = __builtin_bit_cast(zn_f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off + 64, 0, 0));
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                g[e] = v0[e];
                g[4 + e] = v1[e];
            }
        };
        auto load_a = [&](int s, int f, float(&g)[8], bool tail) {
            if constexpr (AK) {
                load_k(ra, offa[f], s, g);
            } else {
                const int k0 = kbeg + s * BK;
                if (!tail || k0 + BK <= kend) {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        g[e] = __builtin_bit_cast(
                            float, __builtin_amdgcn_raw_buffer_load_b32(
                                       ra, offa[f], (uint32_t)(k0 * lda) * 4u + (uint32_t)((e < 4 ? e : 12 + e) * lda) * 4u, 0));
                } else {
                    // k rows past the end: the last row (zeroed below)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const int k = min(k0 + 4 * lh + (e < 4 ? e : 12 + e), kend - 1) - 4 * lh;
                        const uint32_t off = offa[f] == kOutOfRange ? kOutOfRange : offa[f] + (uint32_t)(k * lda) * 4u;
                        g[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, off, 0, 0));
                    }
                }
            }
        };
        // byte offset of the value `at` places from unit j's pixel, under tap (kh, kw), or out of range in the padding
        auto gather_k = [&](int j, int kh, int kw, uint32_t at) {
            const int ih = G == kGNhwc ? gh[j] + kh : gh[j] - kh, iw = G == kGNhwc ? gw[j] + kw : gw[j] - kw;
            const bool ok = ((unsigned)ih < (unsigned)cg.in_h) & ((unsigned)iw < (unsigned)cg.in_w);
            const uint32_t off = offb[j] + at * 4u;
            return ok ? off : kOutOfRange;
        };
        auto tap_k = [&](int k, int &kh, int &kw) {  // places from a pixel to the one under k's tap, at k's channel
            const int khw = zn_udiv(k, cg.div1_mul, cg.div1_shift);
            kh = zn_udiv(khw, cg.kw_mul, cg.kw_shift);
            kw = khw - kh * cg.k_w;
            const int px = kh * cg.in_w + kw;
            return (uint32_t)((G == kGNhwc ? px : -px) * cg.channels + k - khw * cg.div1);
        };
        auto load_b = [&](int s, int j, float(&g)[8]) {
            if constexpr (GATHER_K) {
                // 4 consecutive channels of one tap a load (channels are a multiple of 4); GU: the tap on the scalar unit
                const int k0 = kbeg + s * BK;
                uint32_t off[2];
                int kh, kw;
                if constexpr (GU) {
                    const uint32_t at = tap_k(k0, kh, kw);
                    off[0] = gather_k(j, kh, kw, at);
                    off[1] = off[0] + 64;
                } else {
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const int k = k0 + kq[j] + 16 * h;
                        const uint32_t at = tap_k(k, kh, kw), o = gather_k(j, kh, kw, at);
                        off[h] = k < kend ? o : kOutOfRange;
                    }
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const zn_f32x4 v = __builtin_bit_cast(zn_f32x4, __builtin_amdgcn_raw_buffer_load_b128(rb, off[h], 0, 0));
#pragma unroll
                    for (int e = 0; e < 4; ++e) g[4 * h + e] = v[e];
                }
            } else if constexpr (GATHER_X) {
                // 64 channels-under-a-tap of one output pixel a load; the pixel is wave-uniform.  GU: one decode for each 4
                // consecutive pixels, which share their row.
                const int plane = cg.channels * cg.in_h * cg.in_w;
                uint32_t off[8];
                // pixel k (the last ones instead of those past the end, which meet zeros of A): its first row and column of
                // the image, and the place of that value
                auto pixel = [&](int k, int &oh, int &ow) {
                    k = min(k, kend - (GU ? 4 : 1));
                    const int q = zn_udiv(k, cg.ow_mul, cg.ow_shift);
                    const int b = zn_udiv(q, cg.oh_mul, cg.oh_shift);
                    ow = (k - q * cg.out_w) * cg.stride_w;
                    oh = (q - b * cg.out_h) * cg.stride_h;
                    return (uint32_t)(b * plane + (oh * cg.in_w + ow) * cg.channels) * 4u;
                };
                const int k0 = kbeg + s * BK + kq[j];
                if constexpr (GU) {
                    const uint32_t next = (uint32_t)(cg.stride_w * cg.channels) * 4u;
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        int oh, ow;
                        const uint32_t at = pixel(k0 + 16 * h, oh, ow);
                        const bool row = (unsigned)(gh[j] + oh) < (unsigned)cg.in_h;
                        const uint32_t o = row ? offb[j] + at : kOutOfRange;
                        const int iw = gw[j] + ow;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const uint32_t oe = o + e * next;
                            off[4 * h + e] = (unsigned)(iw + e * cg.stride_w) < (unsigned)cg.in_w ? oe : kOutOfRange;
                        }
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        int oh, ow;
                        const uint32_t at = pixel(k0 + (e < 4 ? e : 12 + e), oh, ow);
                        const bool ok = ((unsigned)(gh[j] + oh) < (unsigned)cg.in_h) & ((unsigned)(gw[j] + ow) < (unsigned)cg.in_w);
                        const uint32_t o = offb[j] + at;
                        off[e] = ok ? o : kOutOfRange;
                    }
                }
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    g[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, off[e], 0, 0));
            } else if constexpr (BKC) {
                load_k(rb, offb[j], s, g);
            } else {
                const int k0 = kbeg + s * BK + kq[j];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int k = min(k0 + (e < 4 ? e : 12 + e), kend - 1);  // rows past the end meet zeros of A
                    g[e] = __builtin_bit_cast(
                        float, __builtin_amdgcn_raw_buffer_load_b32(rb, offb[j], (uint32_t)k * (uint32_t)ldb * 4u, 0));
                }
            }
        };
        auto split_unit = [&](float(&g)[8], int s, int kc, bool mask, zn_u32x4(&w)[3]) {
            if (mask && kbeg + (s + 1) * BK > kend) {
                const int rem = kend - (kbeg + s * BK + kc);
#pragma unroll
                for (int e = 0; e < 8; ++e) g[e] = (e < 4 ? e : 12 + e) < rem ? g[e] : 0.0f;
            }
            split8(g, w);
        };
        zn_u32x4 fa[AB][FM][3];
        auto stage_b = [&](int st, int s, int j, float(&g)[8], bool tail) {
            zn_u32x4 w[3];
            split_unit(g, s, kq[j], BKC && tail, w);
            char *dst = lds + st * kStage + lpos[j];
#pragma unroll
            for (int q = 0; q < 3; ++q) *reinterpret_cast<zn_u32x4 *>(dst + q * kPartB) = w[q];
        };
        const int frb = slot(li, lh);  // the rotation repeats every 16 rows
        zn_u32x4 fb[2][GC][3];
        auto read_b = [&](int st, int f, int q) {
            return *reinterpret_cast<const zn_u32x4 *>(lds + st * kStage + q * kPartB + frb + f * 16 * kRowBytes);
        };

        zn_f32x4 acc[FM][FN], tmp[2][GC][FM];
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) {
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = zn_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int c = 0; c < GC; ++c) tmp[1][c][fm] = zn_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }

        if (ktiles > 0) {
#pragma unroll
            for (int j = 0; j < UB; ++j) load_b(0, j, gb[j]);
#pragma unroll
            for (int f = 0; f < FM; ++f) load_a(0, f, ga[f], true);
#pragma unroll
            for (int j = 0; j < UB; ++j) {
                stage_b(0, 0, j, gb[j], true);
                load_b(1, j, gb[j]);
            }
#pragma unroll
            for (int f = 0; f < FM; ++f) {
                split_unit(ga[f], 0, 4 * lh, true, fa[0][f]);
                load_a(1, f, ga[f], true);
            }
            __syncthreads();
#pragma unroll
            for (int c = 0; c < GC; ++c)
#pragma unroll
                for (int q = 0; q < 3; ++q) fb[0][c][q] = read_b(0, c, q);
        }
        // (part of A, part of B) in the order they are added
        constexpr int kPA[6] = {0, 1, 2, 0, 1, 0}, kPB[6] = {2, 1, 0, 1, 0, 0};
        auto step = [&](int kt, auto sc, auto tc) {
            constexpr int S = decltype(sc)::value, SA = S % AB;
            constexpr bool TAIL = decltype(tc)::value;  // slice kt + 1 may end past K
            constexpr int kLast = NG - 1;
#pragma unroll
            for (int gr = 0; gr < NG; ++gr) {
                if (gr == kLast) __syncthreads();  // slice kt + 1 is in LDS; every wave has read slice kt
                zn_u32x4(&b)[GC][3] = fb[gr & 1];
                zn_u32x4(&bn)[GC][3] = fb[(gr & 1) ^ 1];
#pragma unroll
                for (int pr = 0; pr < 6; ++pr) {
#pragma unroll
                    for (int c = 0; c < GC; ++c)
#pragma unroll
                        for (int fm = 0; fm < FM; ++fm) {
                            zn_f32x4 &t = FLUSH ? tmp[gr & 1][c][fm] : acc[fm][gr * GC + c];
                            const zn_f32x4 c0 = FLUSH && pr == 0 ? zn_f32x4{0.0f, 0.0f, 0.0f, 0.0f} : t;
                            t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(zn_bf16x8, b[c][kPB[pr]]),
                                                                        __builtin_bit_cast(zn_bf16x8, fa[SA][fm][kPA[pr]]), c0,
                                                                        0, 0, 0);
                        }
                    if (pr < 3) {
#pragma unroll
                        for (int c = 0; c < GC; ++c)
                            bn[c][pr] = gr < kLast ? read_b(S, (gr + 1) * GC + c, pr) : read_b(S ^ 1, c, pr);
                    }
                    if (FLUSH && pr == 1) {
#pragma unroll
                        for (int c = 0; c < GC; ++c)
#pragma unroll
                            for (int fm = 0; fm < FM; ++fm)
                                acc[fm][(gr + NG - 1) % NG * GC + c] += tmp[(gr & 1) ^ 1][c][fm];
                    }
                }
                // this lane's share of the next B slice and its next A fragments, spread over the groups
#pragma unroll
                for (int j = 0; j < UB; ++j)
                    if (j * kLast / (AB == 2 ? UB + FM : UB) == gr) {
                        stage_b(S ^ 1, kt + 1, j, gb[j], TAIL);
                        load_b(kt + 2, j, gb[j]);
                    }
#pragma unroll
                for (int f = 0; f < FM; ++f)
                    if ((AB == 2 ? (UB + f) * kLast / (UB + FM) : kLast) == gr) {
                        split_unit(ga[f], kt + 1, 4 * lh, TAIL, fa[(SA + 1) % AB][f]);
                        load_a(kt + 2, f, ga[f], TAIL);
                    }
                interleave<6 * GC * FM>();
            }
        };
        static_assert(NG % 2 == 0, "the fragment and sum buffers alternate over whole slices");
        // The loop's steps load and stage whole slices and hold no branches; the last ones (at least those that load or
        // stage the last slice) mask it.
        int kt = 0;
        for (; kt + 4 < ktiles; kt += 2) {  // its second step loads slice kt + 3
            step(kt, std::integral_constant<int, 0>(), std::false_type());
            step(kt + 1, std::integral_constant<int, 1>(), std::false_type());
        }
        for (; kt < ktiles; kt += 2) {
            step(kt, std::integral_constant<int, 0>(), std::true_type());
            if (kt + 1 < ktiles) step(kt + 1, std::integral_constant<int, 1>(), std::true_type());
        }
        bool bad = false;
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) {
                if (FLUSH && fn / GC == NG - 1 && ktiles > 0) acc[fm][fn] += tmp[1][fn % GC][fm];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    bad |= !(__builtin_fabsf(acc[fm][fn][r]) < INFINITY);
                    acc[fm][fn][r] *= kSplitUnscale;
                }
            }
        if (__builtin_amdgcn_ballot_w64(bad)) plain(p, ra, rb, acc, m0, n0, kbeg, kend, lane);
        store(p, acc, bz, m0, n0, lane, slice);
    }

    // The wave's sums on the fp32 matrix cores: a value that is not finite, or so large that its scaled split or sums
    // overflow, makes the split sums infinite or NaN.
    __device__ static __forceinline__ void plain(const ZnGemmArgs &p, __amdgpu_buffer_rsrc_t ra, __amdgpu_buffer_rsrc_t rb,
                                                 zn_f32x4 (&acc)[FM][FN], int mw, int nw, int kbeg, int kend, int lane) {
        const int li = lane & 15, lh = lane >> 4;
        const int lda = (int)p.lda, ldb = (int)p.ldb;
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) acc[fm][fn] = zn_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        for (int k = kbeg; k < kend; k += 4) {
            const int kk = k + lh;
            float a[FM], b[FN];
#pragma unroll
            for (int f = 0; f < FM; ++f) {
                const int x = mw + 16 * f + li;
                const uint32_t off = x < p.m && kk < kend ? (uint32_t)(AK ? x * lda + kk : kk * lda + x) * 4u : kOutOfRange;
                a[f] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ra, off, 0, 0));
            }
#pragma unroll
            for (int f = 0; f < FN; ++f) {
                const int x = nw + 16 * f + li;
                const bool in = x < p.n && kk < kend;
                uint32_t off;
                if constexpr (G == kGNone) {
                    off = in ? (uint32_t)(BKC ? x * ldb + kk : kk * ldb + x) * 4u : kOutOfRange;
                } else {
                    // only the gathered operand's own extent is bounded: the col matrix it stands for has pixels x taps
                    // values, whose offsets may pass 2^31 and meet kOutOfRange
                    const ZnConvGeom &cg = p.conv;
                    const int px = GATHER_X ? kk : x, tap = GATHER_X ? x : kk;
                    const int khw = zn_udiv(tap, cg.div1_mul, cg.div1_shift), ic = tap - khw * cg.div1;
                    const int kh = zn_udiv(khw, cg.kw_mul, cg.kw_shift), kw = khw - kh * cg.k_w;
                    const int q = zn_udiv(px, cg.ow_mul, cg.ow_shift), ow = px - q * cg.out_w;
                    const int img = GATHER_X ? zn_udiv(q, cg.oh_mul, cg.oh_shift) : 0, oh = q - img * cg.out_h;
                    const int ih = G == kGTransposed ? q + cg.pad_h - kh : (GATHER_X ? oh : q) * cg.stride_h - cg.pad_h + kh;
                    const int iw = G == kGTransposed ? ow + cg.pad_w - kw : ow * cg.stride_w - cg.pad_w + kw;
                    const bool ok = in && (unsigned)ih < (unsigned)cg.in_h && (unsigned)iw < (unsigned)cg.in_w;
                    off = ok ? (uint32_t)(((img * cg.in_h + ih) * cg.in_w + iw) * cg.channels + ic) * 4u : kOutOfRange;
                }
                b[f] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rb, off, 0, 0));
            }
#pragma unroll
            for (int fm = 0; fm < FM; ++fm)
#pragma unroll
                for (int fn = 0; fn < FN; ++fn)
                    acc[fm][fn] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[fn], a[fm], acc[fm][fn], 0, 0, 0);
        }
    }

    // Columns col .. col + 3 of a row of n, zeros past its end
    __device__ static __forceinline__ zn_f32x4 load4(const float *row, int col, int n) {
        if (col + 4 <= n) return *reinterpret_cast<const zn_f32x4u *>(row + col);
        zn_f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = col + r < n ? row[col + r] : 0.0f;
        return v;
    }
    // The bias and a row's old values are all requested before the first is used: one at a time they cost a memory
    // round trip each (4096 x 1024 x 1024 with bias and tanh 79 us against 63 us for the plain product).
    template <int ACT>
    __device__ static __forceinline__ void store_act(const ZnGemmArgs &p, const zn_f32x4 (&acc)[FM][FN], int64_t bz, int mw,
                                                     int nw, int lane) {
        const int li = lane & 15, lh = lane >> 4;
        float *gc = p.c + bz * p.stride_c;
        zn_f32x4 bias[FN];
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) {
            bias[fn] = zn_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            if (p.bias && !p.bias_rows) bias[fn] = load4(p.bias, nw + 16 * fn + 4 * lh, p.n);
        }
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) {
            const int row = mw + 16 * fm + li;
            if (row >= p.m) continue;
            float *crow = gc + (int64_t)row * p.ldc;
            const float rb = p.bias && p.bias_rows ? p.bias[row] : 0.0f;
            zn_f32x4 old[FN];
            if (p.accumulate) {
#pragma unroll
                for (int fn = 0; fn < FN; ++fn) old[fn] = load4(crow, nw + 16 * fn + 4 * lh, p.n);
            }
#pragma unroll
            for (int fn = 0; fn < FN; ++fn) {
                zn_f32x4 v = acc[fm][fn];
                if (p.accumulate) v = old[fn] + v;
                if (p.bias) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = v[r] + (p.bias_rows ? rb : bias[fn][r]);
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = zn_activate(v[r], ACT);
                store4(crow, nw + 16 * fn + 4 * lh, p.n, v);
            }
        }
    }
    // 4-byte aligned 16-byte stores: C rows need not be whole float4s
    __device__ static __forceinline__ void store4(float *crow, int col, int n, const zn_f32x4 &v) {
        if (col + 4 <= n) {
            *reinterpret_cast<zn_f32x4u *>(crow + col) = v;
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (col + r < n) crow[col + r] = v[r];
        }
    }
    __device__ static __forceinline__ void store(const ZnGemmArgs &p, const zn_f32x4 (&acc)[FM][FN], int64_t bz, int mw,
                                                 int nw, int lane, int slice) {
        const bool split = p.splits > 1;
        if (split || (!p.accumulate && !p.bias && p.act == 0)) {
            const int li = lane & 15, lh = lane >> 4;
            float *gc = split ? p.ws + ((int64_t)bz * p.splits + slice) * (int64_t)p.m * p.n : p.c + bz * p.stride_c;
            const int64_t ldc = split ? (int64_t)p.n : p.ldc;
#pragma unroll
            for (int fm = 0; fm < FM; ++fm) {
                const int row = mw + 16 * fm + li;
                if (row >= p.m) continue;
                float *crow = gc + (int64_t)row * ldc;
#pragma unroll
                for (int fn = 0; fn < FN; ++fn) store4(crow, nw + 16 * fn + 4 * lh, p.n, acc[fm][fn]);
            }
            return;
        }
        switch (p.act) {
        case 1: store_act<1>(p, acc, bz, mw, nw, lane); break;
        case 2: store_act<2>(p, acc, bz, mw, nw, lane); break;
        case 3: store_act<3>(p, acc, bz, mw, nw, lane); break;
        default: store_act<0>(p, acc, bz, mw, nw, lane); break;
        }
    }
};

}  // namespace

#endif
