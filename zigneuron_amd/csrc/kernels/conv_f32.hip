// Exported implicit-GEMM convolution kernels for gfx950 (forward, input and
// weight gradients), on the GEMM core of gemm_core.h with gathered B operands.
// The 64x64 kernels of the three gathers that load only by DMA (transposed,
// NHWC forward, NHWC weight gradient) run the pinned three-stage loop at
// BK 16 (24 KB of LDS, six workgroups per CU): on MI355X, C5 forward
// 160.3 -> 156.6 us, a 4 x 128 x 14 x 14 -> 256 convolution 21.9 -> 19.8 us
// forward and 50.6 -> 46.5 us backward, bit-identical results.  The host's
// K granularity for the 64x64 tile (32: split-K chunks, the NHWC forward's
// one-tap slices) is a multiple of that BK.
#include "gemm_core.h"
#include "gemm_split.h"

// Implicit-GEMM convolution, per image b = blockIdx.y:
// out_b[OC][OH*OW] = W[OC][K] . im2col(input_b)^T (+ bias[oc]), an NN GEMM
// whose B operand is gathered from the NCHW input (ZnConvGeom).  _v: W rows
// are 16-byte aligned; _g: the input is gathered in chunks of 4 pixels with
// 16-byte loads (stride_w == 1, out_w % 4 == 0), otherwise element by element.
#define ZN_CONV_KERNEL(TILE, BM, BN, BK, WM, WN, MINB, WA, G, SUFFIX)                             \
    extern "C" __global__ __launch_bounds__(WM *WN * 64, MINB) void zn_conv_nn_##TILE##SUFFIX(ZnGemmArgs p) { \
        gemm_tile_dma<BM, BN, BK, WM, WN, true, false, WA, 4, G>(p);                              \
    }
#define ZN_CONV_TILE(TILE, BM, BN, BK, WM, WN, MINB)                                              \
    ZN_CONV_KERNEL(TILE, BM, BN, BK, WM, WN, MINB, 16, kGIm2col, _v)                             \
    ZN_CONV_KERNEL(TILE, BM, BN, BK, WM, WN, MINB, 4, kGIm2col, )                                \
    ZN_CONV_KERNEL(TILE, BM, BN, BK, WM, WN, MINB, 16, kGIm2col4, _v_g)                          \
    ZN_CONV_KERNEL(TILE, BM, BN, BK, WM, WN, MINB, 4, kGIm2col4, _g)

ZN_CONV_TILE(x, 256, 128, 16, 4, 2, 1)
ZN_CONV_TILE(l, 128, 128, 16, 2, 2, 4)
ZN_CONV_TILE(n, 128, 64, 16, 2, 1, 1)
ZN_CONV_TILE(m, 64, 64, 32, 2, 2, 1)
ZN_CONV_TILE(s, 32, 32, 32, 1, 1, 1)

// Input gradient of a stride-1 convolution, per image b = blockIdx.y:
// grad_input_b[C][H*W] = W'[C][K] . B^T, NT, W' = weights regrouped as
// [ic][(kh*kW + kw)*OC + oc] and B gathered from grad_output rows
// (ConvTGatherStage).  _v: W' rows are 16-byte aligned.
#define ZN_CONVT_KERNEL(TILE, LOOP, BM, BN, BK, WM, WN, MINB, WA, SUFFIX)                       \
    extern "C" __global__ __launch_bounds__(WM *WN * 64, MINB) void zn_convt_nt_##TILE##SUFFIX(ZnGemmArgs p) { \
        LOOP<BM, BN, BK, WM, WN, true, true, WA, 16, kGTransposed>(p); \
    }
#define ZN_CONVT_TILE(TILE, LOOP, BM, BN, BK, WM, WN, MINB) \
    ZN_CONVT_KERNEL(TILE, LOOP, BM, BN, BK, WM, WN, MINB, 16, _v) \
    ZN_CONVT_KERNEL(TILE, LOOP, BM, BN, BK, WM, WN, MINB, 4, )

ZN_CONVT_TILE(x, gemm_tile_dma, 256, 128, 16, 4, 2, 1)
ZN_CONVT_TILE(l, gemm_tile_dma, 128, 128, 16, 2, 2, 4)
ZN_CONVT_TILE(n, gemm_tile_dma, 128, 64, 16, 2, 1, 1)
ZN_CONVT_TILE(m, gemm_tile_pinned, 64, 64, 16, 2, 2, 2)
ZN_CONVT_TILE(s, gemm_tile_dma, 32, 32, 32, 1, 1, 1)

// Weight gradient of a convolution with stride_w == 1 and out_w % 4 == 0:
// grad_W[OC][taps] = go2^T . col with K = the output pixels of all images,
// A = grad_output read as [pixels][OC] rows (X-contiguous, like TN) and
// B = col gathered from the NCHW input (ConvWGatherStage).  _v: OC % 4 == 0
// and grad_output 16-byte aligned.
#define ZN_CONVW_KERNEL(TILE, BM, BN, BK, WM, WN, MINB, WA, SUFFIX)                                \
    extern "C" __global__ __launch_bounds__(WM *WN * 64, MINB) void zn_convw_tn_##TILE##SUFFIX(ZnGemmArgs p) { \
        gemm_tile_dma<BM, BN, BK, WM, WN, false, true, WA, 16, kGWeight>(p);                     \
    }
#define ZN_CONVW_TILE(TILE, BM, BN, BK, WM, WN, MINB)                                              \
    ZN_CONVW_KERNEL(TILE, BM, BN, BK, WM, WN, MINB, 16, _v)                                       \
    ZN_CONVW_KERNEL(TILE, BM, BN, BK, WM, WN, MINB, 4, )

ZN_CONVW_TILE(x, 256, 128, 16, 4, 2, 1)
ZN_CONVW_TILE(l, 128, 128, 16, 2, 2, 4)
ZN_CONVW_TILE(n, 128, 64, 16, 2, 1, 1)
ZN_CONVW_TILE(m, 64, 64, 32, 2, 2, 1)
ZN_CONVW_TILE(s, 32, 32, 32, 1, 1, 1)

// Convolution forward on an NHWC copy of the input, per image b = blockIdx.y:
// out_b[OC][OH*OW] = W[OC][K] . B^T (+ bias[oc]), NT, W in the im2col K order
// and B gathered 4 channels at a time (ConvNhwcGatherStage, C % 4 == 0, any
// stride).  _v: W rows are 16-byte aligned.
#define ZN_CONVF_KERNEL(TILE, LOOP, BM, BN, BK, WM, WN, MINB, WA, SUFFIX)                       \
    extern "C" __global__ __launch_bounds__(WM *WN * 64, MINB) void zn_convf_nt_##TILE##SUFFIX(ZnGemmArgs p) { \
        LOOP<BM, BN, BK, WM, WN, true, true, WA, 16, kGNhwc>(p); \
    }
#define ZN_CONVF_TILE(TILE, LOOP, BM, BN, BK, WM, WN, MINB) \
    ZN_CONVF_KERNEL(TILE, LOOP, BM, BN, BK, WM, WN, MINB, 16, _v) \
    ZN_CONVF_KERNEL(TILE, LOOP, BM, BN, BK, WM, WN, MINB, 4, )

ZN_CONVF_TILE(x, gemm_tile_dma, 256, 128, 16, 4, 2, 1)
ZN_CONVF_TILE(l, gemm_tile_dma, 128, 128, 16, 2, 2, 4)
ZN_CONVF_TILE(n, gemm_tile_dma, 128, 64, 16, 2, 1, 1)
ZN_CONVF_TILE(m, gemm_tile_pinned, 64, 64, 16, 2, 2, 2)
ZN_CONVF_TILE(s, gemm_tile_dma, 32, 32, 32, 1, 1, 1)

// Weight gradient from an NHWC copy of the input: grad_W[OC][taps] =
// go2^T . col, TN, K = the output pixels of all images, B gathered 4 channels
// at a time (ConvNhwcWGatherStage, C % 4 == 0, any stride).  _v: OC % 4 == 0
// and grad_output 16-byte aligned.
#define ZN_CONVWN_KERNEL(TILE, LOOP, BM, BN, BK, WM, WN, MINB, WA, SUFFIX)                      \
    extern "C" __global__ __launch_bounds__(WM *WN * 64, MINB) void zn_convwn_tn_##TILE##SUFFIX(ZnGemmArgs p) { \
        LOOP<BM, BN, BK, WM, WN, false, false, WA, 16, kGNhwcW>(p); \
    }
#define ZN_CONVWN_TILE(TILE, LOOP, BM, BN, BK, WM, WN, MINB) \
    ZN_CONVWN_KERNEL(TILE, LOOP, BM, BN, BK, WM, WN, MINB, 16, _v) \
    ZN_CONVWN_KERNEL(TILE, LOOP, BM, BN, BK, WM, WN, MINB, 4, )

ZN_CONVWN_TILE(x, gemm_tile_dma, 256, 128, 16, 4, 2, 1)
ZN_CONVWN_TILE(l, gemm_tile_dma, 128, 128, 16, 2, 2, 4)
ZN_CONVWN_TILE(n, gemm_tile_dma, 128, 64, 16, 2, 1, 1)
ZN_CONVWN_TILE(m, gemm_tile_pinned, 64, 64, 16, 2, 2, 2)
// 128x128 on the register-staged loop (16-byte grad_output rows only): one
// round of tiles x K slices
extern "C" __global__ __launch_bounds__(512, 1) void zn_convwn_tn_r_v(ZnGemmArgs p) {
    gemm_tile_wide<128, 128, 16, 2, 4, false, false, kGNhwcW>(p);
}
ZN_CONVWN_TILE(s, gemm_tile_dma, 32, 32, 32, 1, 1, 1)

// The NHWC forward, the transposed convolution and the NHWC weight gradient
// on the bf16 matrix cores (gemm_split.h): 128x128 tiles (cr), and 64x128
// ones (ch) for few output rows; _u: one decode of the gather for each slice
// of K (the filter tap) or 4 of it (the output row), and no branch inside a
// step (C5's weight gradient GEMM 140 -> 128 us: 315 scalar instructions a
// slice before, 80 now).  cr of the forward and the input gradient: one
// column block at a time fits 128 registers, two workgroups to a CU (C5's
// forward GEMM 123 -> 106 us; without _u 40 bytes spill, three of the values
// inside the loop); the weight gradient, one round of workgroups,
// would spill there (217 us), and ch measured the same with either.
#define ZN_CONV_SPLIT(NAME, NW, AK, BKC, G, GU, GC, MINB)                                        \
    extern "C" __global__ __launch_bounds__(NW * 64, MINB) void NAME(ZnGemmArgs p) {             \
        typedef SplitTile<NW, 1, 128, AK, BKC, true, GC, 2, 3, G, GU> T;                         \
        __shared__ __attribute__((aligned(1024))) char lds[2 * T::kStage];                       \
        T::run(p, lds);                                                                          \
    }
#define ZN_CONV_SPLIT_TILE(TILE, NW, GC, MINB, WGC, WMINB)                                       \
    ZN_CONV_SPLIT(zn_convfs_nt_##TILE, NW, true, true, kGNhwc, false, GC, MINB)                  \
    ZN_CONV_SPLIT(zn_convfs_nt_##TILE##_u, NW, true, true, kGNhwc, true, GC, MINB)               \
    ZN_CONV_SPLIT(zn_convts_nt_##TILE, NW, true, true, kGTransposed, false, GC, MINB)            \
    ZN_CONV_SPLIT(zn_convts_nt_##TILE##_u, NW, true, true, kGTransposed, true, GC, MINB)         \
    ZN_CONV_SPLIT(zn_convwns_tn_##TILE, NW, false, false, kGNhwcW, false, WGC, WMINB)            \
    ZN_CONV_SPLIT(zn_convwns_tn_##TILE##_u, NW, false, false, kGNhwcW, true, WGC, WMINB)
ZN_CONV_SPLIT_TILE(cr, 8, 1, 4, 2, 2)
ZN_CONV_SPLIT_TILE(ch, 4, 2, 2, 2, 2)
