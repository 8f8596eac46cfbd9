// sk_bp.hip -- the per-call backprojector kernels.
//
//   k_bp  B.r   (futhark/backprojection.fut:20-93).  Pixel-parallel gather, no atomics: a
//               block owns a 16 x 16*PPT pixel tile and walks the lines in order, staging
//               for each block of 32 lines the tile's rho-window of the sinogram in LDS
//               together with the per-bin intercepts r/cost.
//   k_bp_images B.r of 2, 4 or 8 images per workgroup on 16 x 32 tiles (fast mode, 1 to 4 candidates
//               per pixel; 2 and 8 images with two candidates only).
//
// The work item itself lives in sk_kern.h (shared with the persistent kernels).
#include "sk_kern.h"

namespace sk {

// Waves per SIMD the registers are held to: 8 where the candidates of a lane's pixels fit 64
// registers beside the loop (NC * PPT <= 8 candidates), else 5; the general path is not held.
constexpr int bp_waves_per_simd(int nc, int ppt) { return nc == 0 ? 1 : (nc * ppt <= 8 ? 8 : 5); }

// Grid: (tiles across, tiles down, images).  Dynamic LDS: BP_LB * W float2.
template <bool EXACT, int MODE, int WEIGHTS, int NC, bool DR1, int PPT>
__global__ __launch_bounds__(256, bp_waves_per_simd(NC, PPT)) void k_bp(BpParams P) {
  extern __shared__ float2 win[];
  __shared__ BpLineLds lsh[BP_LB];
  int tx = blockIdx.x, ty = blockIdx.y;
  if (P.order) {
    const unsigned t = P.order[blockIdx.y * gridDim.x + blockIdx.x];
    tx = (int)(t & 0xffffu);
    ty = (int)(t >> 16);
  }
  bp_item<EXACT, MODE, WEIGHTS, NC, DR1, PPT>(P, tx, ty, blockIdx.z, win, lsh);
}

// The hoisted fast path for S images at once on 16 x 32 tiles: grid (tiles across, tiles down,
// images / S).  Dynamic LDS: BP_LB * W * (1 + S) floats.  One image issues 13 VALU per pixel and
// line for the index, the positions and the lengths of the two candidates and 2 FMAs; S images
// share the 13 and read 8 + 8 S bytes of LDS instead of 16 S.  64 images of 512^2, 512 angles:
// 3.41 ms one at a time (16 x 64 tiles), 2.37, 1.61 and 1.45 ms for S = 2, 4 and 8, which is LDS
// bandwidth next (16 x 64 tiles with S = 4 hold 127 registers and leave 3 workgroups per CU:
// 1.69 ms; 16 x 16: 1.79).
constexpr int BP_IMAGES_PPT = 2;

template <int MODE, int WEIGHTS, int NC, int S>
__global__ __launch_bounds__(256, S == 8 ? 3 : (S == 4 ? 5 : 7)) void k_bp_images(BpParams P) {
  extern __shared__ float4 win4[];
  __shared__ BpLineLds lsh[BP_LB];
  int tx = blockIdx.x, ty = blockIdx.y;
  if (P.order) {
    const unsigned t = P.order[blockIdx.y * gridDim.x + blockIdx.x];
    tx = (int)(t & 0xffffu);
    ty = (int)(t >> 16);
  }
  bp_item<false, MODE, WEIGHTS, NC, false, BP_IMAGES_PPT, S>(P, tx, ty, blockIdx.z, (float2*)win4, lsh);
}

int bp_pixels_per_lane(int variant) { return variant == 1 ? 2 : (variant == 2 ? 4 : 1); }

BpParams bp_params(const Geom* g, const BpArgs& a, int ppt) {
  const unsigned* order =
      g->d_bp_order ? g->d_bp_order + g->bp_order_off[ppt == 1 ? 0 : (ppt == 2 ? 1 : 2)] : nullptr;
  return BpParams{g->d_lines, g->A, g->R, g->N, g->ncand, bp_window_bins(ppt, g->drho, g->ncand), a.batch,
                  g->n_steep, g->rho0, g->drho, 1.0f / g->drho, a.sino, a.out, a.outT, a.colinv, g->d_inter, order};
}

template <bool EXACT, int MODE, int WEIGHTS, int NC, bool DR1, int PPT>
static void bp_go(const Geom* g, const BpArgs& a, hipStream_t s) {
  const BpParams P = bp_params(g, a, PPT);
  const int TH = 16 * PPT;
  dim3 grid((g->N + BP_TW - 1) / BP_TW, (g->N + TH - 1) / TH, a.batch);
  const size_t lds = sizeof(float2) * BP_LB * (size_t)P.W;
  hipLaunchKernelGGL((k_bp<EXACT, MODE, WEIGHTS, NC, DR1, PPT>), grid, dim3(256), lds, s, P);
}

template <int MODE, int WEIGHTS, int NC, int S>
static void bp_go_images(const Geom* g, const BpArgs& a, hipStream_t s) {
  const BpParams P = bp_params(g, a, BP_IMAGES_PPT);
  const int TH = 16 * BP_IMAGES_PPT;
  const dim3 grid((g->N + BP_TW - 1) / BP_TW, (g->N + TH - 1) / TH, (a.batch + S - 1) / S);
  const size_t lds = sizeof(float) * BP_LB * (size_t)P.W * (1 + S);
  hipLaunchKernelGGL((k_bp_images<MODE, WEIGHTS, NC, S>), grid, dim3(256), lds, s, P);
}

template <int MODE, int WEIGHTS>
static void bp_go_images_s(int images, const Geom* g, const BpArgs& a, hipStream_t s) {
  if (g->bp_nc == 1)
    bp_go_images<MODE, WEIGHTS, 1, 4>(g, a, s);
  else if (g->bp_nc == 3)
    bp_go_images<MODE, WEIGHTS, 3, 4>(g, a, s);
  else if (g->bp_nc == 4)
    bp_go_images<MODE, WEIGHTS, 4, 4>(g, a, s);
  else if (images == 8)
    bp_go_images<MODE, WEIGHTS, 2, 8>(g, a, s);
  else if (images == 4)
    bp_go_images<MODE, WEIGHTS, 2, 4>(g, a, s);
  else
    bp_go_images<MODE, WEIGHTS, 2, 2>(g, a, s);
}

// Images per workgroup of the fast backprojector, 1 = the one-image kernels.  Below about a
// workgroup per CU more images only lengthen each one (the walk over the lines is serial).  us for 1,
// 2 and 4 images per workgroup: 512^2, 804 angles (512 tiles of 16 x 32): 2 images 245, 200, 224; 3
// images 318, 274, 224; 640^2, 450: 2 images 187, 141, 165; 4 images 328, 223, 166.  Eight share more
// but fit 3 workgroups per CU (4 images: 5), so a launch pays where it ends within the first 768 or
// where the rounds are many; us for 4 and 8 per workgroup, 8 images, 400 angles: 512^2 with 358 (512
// workgroups of 8) 166 and 145; 608^2 (722) 248 and 200; 640^2 (800) 255 and 291; 768^2 (1152) 311 and
// 320; 896^2 (1568) 425 and 459; 1024^2 (2048) 530 and 501.  Bins off about unit width (1, 3 or 4
// candidates) have the 4-image kernel only.
int bp_images(const Geom* g, int batch) {
  if (!g->bp_nc) return 1;
  const int TH = 16 * BP_IMAGES_PPT;
  const long tiles = (long)((g->N + BP_TW - 1) / BP_TW) * ((g->N + TH - 1) / TH);
  if (g->bp_nc != 2) return batch >= 3 && tiles * ((batch + 3) / 4) >= 256 ? 4 : 1;
  const long eights = tiles * ((batch + 7) / 8);
  if (batch >= 7 && ((eights >= 512 && eights <= 768) || eights >= 1920)) return 8;
  if (batch >= 3 && tiles * ((batch + 3) / 4) >= 256) return 4;
  if (batch >= 2 && tiles * ((batch + 1) / 2) >= 384) return 2;
  return 1;
}

// A^T by the general kernel: where the candidate index is not safe, and few lines of few pixels, which
// the hoisted kernel's set-up of a block and its loop per kind of line outweigh.  us hoisted and
// general: 256^2, 8 lines 6.1 and 5.3; 512^2, 4 lines 6.0 and 4.5, 12 lines 7.7 and 7.5; bins of
// 0.4, 4 lines of 512^2 7.1 and 6.4.  From 2^20 pixels the hoisted kernel is the faster one
// (four 512^2 images, 8 lines 9.7 and 13.5).
static bool adj_general(const Geom* g, int batch) {
  const long pixels = (long)batch * g->N * g->N;
  const int few = g->ncand > 2 ? 5 : (pixels <= 1L << 18 ? 12 : 8);
  return !g->index_safe || (pixels < 1L << 20 && g->A <= few);
}

template <bool EXACT, int MODE, int WEIGHTS, int PPT>
static void bp_go_nc(const Geom* g, const BpArgs& a, hipStream_t s) {
  if constexpr (EXACT) {
    if (g->bp_two_cand)
      bp_go<true, MODE, WEIGHTS, 2, true, PPT>(g, a, s);
    else
      bp_go<true, MODE, WEIGHTS, 0, false, PPT>(g, a, s);
  } else {
    if constexpr (WEIGHTS == W_ADJ) {
      if (adj_general(g, a.batch)) {
        if (g->bp_two_cand)
          bp_go<false, MODE, W_ADJ, 2, true, 1>(g, a, s);
        else
          bp_go<false, MODE, W_ADJ, 0, false, 1>(g, a, s);
        return;
      }
    }
    switch (g->bp_nc) {
      case 1: bp_go<false, MODE, WEIGHTS, 1, false, PPT>(g, a, s); break;
      case 2: bp_go<false, MODE, WEIGHTS, 2, false, PPT>(g, a, s); break;
      case 3: bp_go<false, MODE, WEIGHTS, 3, false, PPT>(g, a, s); break;
      case 4: bp_go<false, MODE, WEIGHTS, 4, false, PPT>(g, a, s); break;
      default: bp_go<false, MODE, WEIGHTS, 0, false, 1>(g, a, s);  // the fastest height of this path
    }
  }
}

template <bool EXACT, int MODE, int WEIGHTS>
static void bp_go_v(int variant, const Geom* g, const BpArgs& a, hipStream_t s) {
  if ((EXACT && WEIGHTS != W_REF) || variant == 0)
    bp_go_nc<EXACT, MODE, WEIGHTS, 1>(g, a, s);
  else if (variant == 1)
    bp_go_nc<EXACT, MODE, WEIGHTS, 2>(g, a, s);
  else
    bp_go_nc<EXACT, MODE, WEIGHTS, 4>(g, a, s);
}

template <int MODE, int WEIGHTS>
static void bp_go_ex(bool ex, int variant, const Geom* g, const BpArgs& a, hipStream_t s) {
  if (ex)
    bp_go_v<true, MODE, WEIGHTS>(variant, g, a, s);
  else
    bp_go_v<false, MODE, WEIGHTS>(variant, g, a, s);
}

// The tile height of a geometry that was not tuned, on a context whose option is 0: the tallest of
// 64 and 32 rows that leaves 1024 tiles (4 workgroups per CU), else 16.  Taller tiles share a
// line's constants among more pixels, but the walk over the lines is serial and needs workgroups
// enough to hide it: 512^2, 358 angles: 72, 84, 123 us for 16, 32, 64 rows; 768^2, 537: 199, 171,
// 196; 1024^2, 716: 403, 321, 314; 2048^2, 1433: 3008, 2383, 2179.  Four candidates a pixel keep
// 64-row tiles from 8 waves per SIMD (1024^2, 716 angles, bins of 0.4: 821, 786, 1051).  Exact mode's
// divisions hide the rest at 16 rows (1024^2, 700: 989, 1040, 1148).
static int bp_variant_default(const Geom* g, int batch) {
  const long across = (g->N + BP_TW - 1) / BP_TW;
  for (int v = g->bp_nc == 4 ? 1 : 2; v > 0; --v) {
    const int rows = 16 * bp_pixels_per_lane(v);
    if (across * ((g->N + rows - 1) / rows) * batch >= 1024) return v;
  }
  return 0;
}

int launch_bp(Ctx* c, const Geom* g, BpMode mode, BpWeights w, const BpArgs& a, hipStream_t s) {
  const bool ex = c->exact != 0;
  int v = g->bp_variant >= 0 ? g->bp_variant : (c->bp_variant || ex ? c->bp_variant : bp_variant_default(g, a.batch));
  if (sizeof(float2) * BP_LB * (size_t)bp_window_bins(bp_pixels_per_lane(v), g->drho, g->ncand) > 60 * 1024)
    v = 0;
  if (sizeof(float2) * BP_LB * (size_t)bp_window_bins(1, g->drho, g->ncand) > 60 * 1024)
    return fail(c, SK_EINVAL, "backprojection window exceeds LDS (deltarho too small)");
  if (w == W_ADJ && mode != BP_PLAIN) return fail(c, SK_EINVAL, "adjoint weights support plain mode only");
  const int images = ex || mode == BP_ONES_INV || (w == W_ADJ && adj_general(g, a.batch)) ? 1 : bp_images(g, a.batch);
  if (images > 1) {
    if (w == W_ADJ)
      bp_go_images_s<BP_PLAIN, W_ADJ>(images, g, a, s);
    else if (mode == BP_SIRT)
      bp_go_images_s<BP_SIRT, W_REF>(images, g, a, s);
    else
      bp_go_images_s<BP_PLAIN, W_REF>(images, g, a, s);
  } else if (w == W_REF) {
    switch (mode) {
      case BP_PLAIN: bp_go_ex<BP_PLAIN, W_REF>(ex, v, g, a, s); break;
      case BP_ONES_INV: bp_go_ex<BP_ONES_INV, W_REF>(ex, 0, g, a, s); break;
      case BP_SIRT: bp_go_ex<BP_SIRT, W_REF>(ex, v, g, a, s); break;
    }
  } else {
    bp_go_ex<BP_PLAIN, W_ADJ>(ex, v, g, a, s);
  }
  return launched(c, "backprojection kernel");
}

}  // namespace sk
