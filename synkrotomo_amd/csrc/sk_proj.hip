// sk_proj.hip -- the per-call forward projector kernels and the projectors' C-ABI entry points
// (the backprojector kernels: sk_bp.hip).
//
//   k_fp  A.x   (futhark/forwardprojection.fut:21-84).  Ray-parallel: one lane per ray (or
//               two, variant 1), a wavefront = 64 consecutive bins of one line.  All lanes
//               of a wave step the same frame row together, so the two gathers per step
//               land in one or two cache lines of that row; each row is addressed through
//               a buffer descriptor whose range check returns 0 outside the row, the
//               reference's contribution of an out-of-bounds pixel.  The row range is
//               clipped per wave to the rows where any of its rays can touch the image
//               (skipped rows contribute exactly +0 in the reference).  Flat lines read a
//               transposed copy of the image, the reference's own frame trick
//               (forwardprojection.fut:80-82).
//   k_fp_staged A.x, staged (variants 5, 6): a workgroup = 256 consecutive bins of one
//               line.  It walks the frame rows in blocks of FPS_ROWS (12): the four waves load the
//               block's image-row segment (the columns any of its rays can touch) with
//               coalesced dword loads into LDS, then every lane forms its ray's row steps
//               from LDS.  Same per-step expressions as k_fp (bitwise equal results).
//   k_fp_grouped A.x, grouped staged (variant 7): a workgroup = 64 consecutive bins of four
//               lines adjacent in slope, 16 bins of each line per wave, so the staged segment
//               of a block is two to four chunks of 64 columns instead of six; blocks of 16
//               rows.  Same walk, for 1, 2 or 4 images at once.
//   k_fp_lds    A.x of images up to 80 x 80: the whole image in LDS, the per-wave walk from there.
//   k_fp_listed, k_bpt_rays  the rays of B^T that A.x does not give (launch_fp_bpt).
//
// The work items themselves live in sk_kern.h (shared with the persistent kernels).
// With SK_OPT_EXACT the results are bitwise those of the sequential FP32 restatement of
// the reference.  By default (fast mode) the per-step quotients use the hardware
// reciprocal, the forward projector accumulates the fractions of each row's length and
// scales by the line length once per ray, and the backprojector folds the line length into
// the staged sinogram value; pixel indices and candidate sets are unchanged.
#include "sk_kern.h"

namespace sk {

// ------------------------------------------------------------------------ kernels
__global__ __launch_bounds__(256) void k_transpose(const float* __restrict__ in,
                                                   float* __restrict__ out, int N) {
  __shared__ float t[32][33];
  const size_t off = (size_t)blockIdx.z * N * N;
  const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int k = ty; k < 32; k += 8) {
    const int y = by + k, x = bx + tx;
    if (x < N && y < N) t[k][tx] = in[off + (size_t)y * N + x];
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const int y = bx + k, x = by + tx;
    if (x < N && y < N) out[off + (size_t)y * N + x] = t[tx][k];
  }
}

// Workgroup -> (line, bin block) orders.  ORDER 0: grid (bin blocks, lines, images).
// ORDER 1: grid (lines, bin blocks, images): the workgroups resident together are one bin
// block of (nearly) every angle -- one ring of the image at a time, with each row touched by
// the rays of many neighbouring angles while it is cached.  (Permuting the lines so that
// each XCD gets a contiguous run of angles measured 1.2x slower, and giving each XCD whole
// bin blocks 1.6x slower, from the imbalance between short edge rays and long central ones.)
template <bool EXACT, int MODE, int WEIGHTS, bool DR1, int RPT, int ORDER = 0>
__global__ __launch_bounds__(FP_BLOCK) void k_fp(FpParams P) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (ORDER == 0)
    fp_item<EXACT, MODE, WEIGHTS, DR1, RPT>(P, blockIdx.y, blockIdx.x * FP_WAVES + wave, blockIdx.z);
  else
    fp_item<EXACT, MODE, WEIGHTS, DR1, RPT>(P, blockIdx.x, blockIdx.y * FP_WAVES + wave, blockIdx.z);
}

// B^T of the listed (degenerate) lines: every row of 64 bins with the backprojector's lengths.  Few
// rays and two gathers a row, so latency bounds it: LISTED_WAVES waves of a workgroup take a run of
// the rows each, four rows' loads in flight, and their sums are added in order.  B^T of 8 images of
// 512^2, 360 angles, two of them such lines: 355 us with one wave walking all rows, 201 us like this
// (A.x: 185).  Grid (bins / 64, listed lines, images).
constexpr int LISTED_WAVES = 16;
template <bool DR1>
__global__ __launch_bounds__(64 * LISTED_WAVES) void k_fp_listed(FpParams P, const int* __restrict__ list) {
  __shared__ float part[LISTED_WAVES][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const Line L = P.lines[list[blockIdx.y]];
  const int N = P.N, h = N >> 1;
  const int first = blockIdx.x * 64, r = first + lane, last = min(first + 63, P.R - 1);
  const float icpt = (P.rho0 + (float)r * P.drho) / L.cost;  // forwardprojection.fut:33-34
  int a0, a1, b0, b1;
  row_clip(L.slope, (P.rho0 + (float)first * P.drho) / L.cost, h, a0, a1);
  row_clip(L.slope, (P.rho0 + (float)last * P.drho) / L.cost, h, b0, b1);
  const int i0 = __builtin_amdgcn_readfirstlane(min(a0, b0)), i1 = __builtin_amdgcn_readfirstlane(max(a1, b1));
  const int run = (max(i1 - i0, 0) + LISTED_WAVES - 1) / LISTED_WAVES;
  const int w0 = i0 + run * wave, w1 = min(w0 + run, i1);
  const float* src = ((L.flags & LINE_FLAT) ? P.imgT : P.img) + (size_t)blockIdx.z * N * N;
  float sum = 0.0f;
  for (int i = w0; i < w1; i += 4) {
    float xbot[4], vb[4], vt[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {  // rows past the run: an empty descriptor reads 0
      xbot[q] = (float)(i + q) * L.slope + icpt;
      const __amdgpu_buffer_rsrc_t row = row_rsrc(src + (size_t)(i + h + q) * N, i + q < w1 ? N : 0);
      vb[q] = row_load(row, (int)floorf(xbot[q]) + h);
      vt[q] = row_load(row, (int)floorf(xbot[q] + L.slope) + h);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (i + q >= w1) break;  // uniform
      const float xtop = xbot[q] + L.slope;
      const int Xb = (int)floorf(xbot[q]), Xt = (int)floorf(xtop);
      auto term = [&](int X, float v) {
        const float len = bp_entry<false, DR1>(L, X, (float)(i + q), xbot[q], xtop, r, P.ncand, P.rho0, P.drho);
        return (unsigned)(X + h) < (unsigned)N ? len * v : 0.0f;
      };
      sum = sum + (term(Xb, vb[q]) + (Xb == Xt ? 0.0f : term(Xt, vt[q])));
    }
  }
  part[wave][lane] = sum;
  __syncthreads();
  if (wave != 0 || r >= P.R) return;
  for (int w = 1; w < LISTED_WAVES; ++w) sum = sum + part[w][lane];
  P.out[(size_t)blockIdx.z * P.A * P.R + (size_t)L.orig * P.R + r] = sum;
}

// B^T of the rays for which A.x does not do, with the backprojector's lengths; one thread a ray of a
// line that is not degenerate, the row sums in order.  A.x forms a row as vb + f*(vo - vb):
// - A ray that leaves most of a row's length outside gets its short part from 1 - f, 6e-8 off however
//   short, and divided by a row sum of 1e-3 (the gradient of a SIRT step) that is 6e-5 of the
//   result: rays that cross less than two pixels' length.  The outermost corners of a line lie at
//   distance h*(|cost| + |sint|) from the axis, and a chord d nearer than that is d/|cost*sint|
//   long.  d only picks the rays (FP32: on a nearly axis-parallel line its error can exceed the
//   whole range of short chords); the rows come from the ray's own intercept, and a ray that
//   crosses more of them than a short chord can is left as it is, A.x being right for it.
// - A pixel that is not finite, or two whose difference overflows, reach every ray that passes beside
//   them (0*inf), and A.x is then not finite, whatever follows: those rays are walked again.
// Nearly every ray costs its load and a handful of VALU, the few walked ones the latency of their
// loads, four rows in flight.  8 images of 512^2, 360 angles: 8 us of 201.  Grid (bins / 256,
// lines, images).
constexpr int RIM_ROWS = 32;  // a short chord: 3 rows, one more at each end, and 2e-6*h/|slope| <= 17 for rounding
template <bool DR1>
__global__ __launch_bounds__(256) void k_bpt_rays(FpParams P) {
  const Line L = P.lines[blockIdx.y];
  const int r = (int)(blockIdx.x * 256 + threadIdx.x);
  if (r >= P.R || (L.flags & LINE_DEGEN)) return;
  const int N = P.N, h = N >> 1;
  float* out = P.out + (size_t)blockIdx.z * P.A * P.R + (size_t)L.orig * P.R + r;
  const bool finite = (__builtin_bit_cast(unsigned, *out) & 0x7f800000u) != 0x7f800000u;
  const float rho = P.rho0 + (float)r * P.drho;
  const float d = (float)h * (fabsf(L.cost) + fabsf(L.sint)) - fabsf(rho);
  if (finite && d > 2.0f * fabsf(L.cost * L.sint)) return;
  const float icpt = rho / L.cost;  // forwardprojection.fut:33-34
  int i0, i1;
  row_span(L.slope, icpt, h, i0, i1);
  if (finite && (i0 >= i1 || i1 - i0 > RIM_ROWS)) return;
  const float* src = ((L.flags & LINE_FLAT) ? P.imgT : P.img) + (size_t)blockIdx.z * N * N;
  float sum = 0.0f;
  for (int i = i0; i < i1; i += 4) {
    float xbot[4], vb[4], vt[4];
    int Xb[4], Xt[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      xbot[q] = (float)(i + q) * L.slope + icpt;
      Xb[q] = (int)floorf(xbot[q]);
      Xt[q] = (int)floorf(xbot[q] + L.slope);
      const float* row = src + (size_t)(i + q + h) * N + h;
      vb[q] = i + q < i1 && (unsigned)(Xb[q] + h) < (unsigned)N ? row[Xb[q]] : 0.0f;
      vt[q] = i + q < i1 && (unsigned)(Xt[q] + h) < (unsigned)N ? row[Xt[q]] : 0.0f;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (i + q >= i1) break;
      auto part = [&](int X, float v) {
        const float len = bp_entry<false, DR1>(L, X, (float)(i + q), xbot[q], xbot[q] + L.slope, r, P.ncand, P.rho0, P.drho);
        return (unsigned)(X + h) < (unsigned)N ? len * v : 0.0f;
      };
      sum = sum + (part(Xb[q], vb[q]) + (Xb[q] == Xt[q] ? 0.0f : part(Xt[q], vt[q])));
      const int Xm = (Xb[q] + Xt[q]) / 2;  // as fp_item: the pixel between two ends that rounded apart
      if (abs(Xt[q] - Xb[q]) == 2 && (unsigned)(Xm + h) < (unsigned)N)
        sum = sum + part(Xm, src[(size_t)(i + q + h) * N + h + Xm]);
    }
  }
  *out = sum;
}

// --------------------------------------------------------- small images (fast mode)
// The whole image in LDS: cell (y, x) at fpl_origin(N) + y*pitch + x, with zeros two cells wide
// around it (a row's right border is the next row's left one).  The pitch is odd, so lanes along a
// column fall into different banks as well.
constexpr int FPL_MAX_N = 80;  // 28 KB of LDS
__host__ __device__ constexpr int fpl_pitch(int N) { return (N + 2) | 1; }
__host__ __device__ constexpr int fpl_origin(int N) { return 2 * fpl_pitch(N) + 2; }
__host__ __device__ constexpr int fpl_cells(int N) { return fpl_origin(N) + (N + 2) * fpl_pitch(N); }

// Rows [i0, i1) of one ray per lane; column c of frame row i is cells[(c * cs + i * rs)].  Columns
// are held to [-2, N], whose cells c and c + 1 past the image are 0 like a load outside it.
template <bool POS, bool NT>
__device__ __forceinline__ float fpl_rows(const float* cells, int N, int h, int i0, int i1, int cs, int rs,
                                          float slope, float icpt, float rslope) {
  float sum = 0.0f, fi = (float)i0;  // exact
  const int cofs = h - (POS ? 0 : 1);
  const float* row = cells + (i0 + h) * rs;
  auto step = [&](const float* at, float f) {
    const float xb = f * slope + icpt, xt = xb + slope;
    const int c = min(max(floor_to_int(xb) + cofs, -2), N) * cs;
    const float va = at[c], vc = at[c + cs];
    return POS ? fp_row_add<true, NT>(sum, xb, xt, va, vc, rslope) : fp_row_add<false, NT>(sum, xb, xt, vc, va, rslope);
  };
#pragma unroll 4
  for (int i = i0; i < i1; ++i, fi += 1.0f, row += rs) sum = step(row, fi);
  return sum;
}

// One image of a small geometry: a wave per 64 bins of a line, four to a workgroup, all bins of all
// lines in turn; grid (workgroups, images).  The walk (row range, fractions, order of the sums) is
// fp_item's, with the two pixels of a row from LDS: no load latency per row, and no transposed copy --
// where one is at hand anyway (SIRT's update writes it; B^T reads it) the per-wave kernel needs
// 2 us less (a SIRT iteration of 32^2, 22 angles 12.0 us against 13.5, of 64^2, 89 angles 23.9
// against 25.7).  What is left is launch, the copy and a serial walk of N rows at one wave per SIMD: 64^2 and 90
// angles, calls back to back, 7.9 us against 9.0 for the transposed copy and the per-wave kernel
// (6.7 at 16^2, where only the launch is left).
__global__ __launch_bounds__(256) void k_fp_lds(FpParams P) {
  extern __shared__ float lds[];
  const int N = P.N, Q = fpl_pitch(N), h = N >> 1, origin = fpl_origin(N), end = origin + N * Q;
  const float* img = P.img + (size_t)blockIdx.y * N * N;
  {
    const int dj = 256 / N, dk = 256 - dj * N;
    int y = (int)threadIdx.x / N, x = (int)threadIdx.x - y * N;
#pragma unroll 8
    for (int e = threadIdx.x; e < N * N; e += 256) {
      lds[origin + y * Q + x] = img[e];
      x += dk;
      y += dj;
      if (x >= N) {
        x -= N;
        ++y;
      }
    }
    for (int e = threadIdx.x; e < origin; e += 256) lds[e] = 0.0f;
    for (int e = end + threadIdx.x; e < fpl_cells(N); e += 256) lds[e] = 0.0f;
    for (int r = threadIdx.x; r < N; r += 256)
      for (int e = N; e < Q; ++e) lds[origin + r * Q + e] = 0.0f;
  }
  __syncthreads();
  const int blocks = (P.R + 63) / 64;
  const int item = __builtin_amdgcn_readfirstlane(blockIdx.x * FP_WAVES + (threadIdx.x >> 6));
  const int j = item / blocks, first = (item - j * blocks) * 64;
  if (j >= P.A) return;
  const int r = first + (threadIdx.x & 63), last = min(first + 63, P.R - 1);
  const Line L = P.lines[j];
  const float icpt = (P.rho0 + (float)r * P.drho) / L.cost;  // forwardprojection.fut:33-34
  int a0, a1, b0, b1;
  row_clip(L.slope, (P.rho0 + (float)first * P.drho) / L.cost, h, a0, a1);
  row_clip(L.slope, (P.rho0 + (float)last * P.drho) / L.cost, h, b0, b1);
  const int i0 = __builtin_amdgcn_readfirstlane(min(a0, b0)), i1 = __builtin_amdgcn_readfirstlane(max(a1, b1));
  const bool flat = L.flags & LINE_FLAT, nt = L.flags & LINE_NEWTON;
  const int cs = flat ? Q : 1, rs = flat ? 1 : Q;
  const float rslope = nt ? 1.0f / fabsf(L.slope) : 0.0f;
  const float* cells = lds + origin;
  float s;
  if (L.flags & LINE_SLOPE_POS)
    s = nt ? fpl_rows<true, true>(cells, N, h, i0, i1, cs, rs, L.slope, icpt, rslope)
           : fpl_rows<true, false>(cells, N, h, i0, i1, cs, rs, L.slope, icpt, 0.0f);
  else
    s = nt ? fpl_rows<false, true>(cells, N, h, i0, i1, cs, rs, L.slope, icpt, rslope)
           : fpl_rows<false, false>(cells, N, h, i0, i1, cs, rs, L.slope, icpt, 0.0f);
  if (r >= P.R) return;
  P.out[(size_t)blockIdx.y * P.A * P.R + (size_t)L.orig * P.R + r] = s * L.lbase;
}

// ------------------------------------------------------------- staged A.x (fast mode)
// A workgroup holds FPS_RAYS consecutive bins of one line, one ray per lane.  Frame rows go
// in blocks of FPS_ROWS: for each row the columns any of the workgroup's rays can touch (a
// segment of at most FPS_MAXW floats starting one column left of the lowest ray) are staged
// in LDS with coalesced loads, zeros outside the image and past the last row, and every
// lane reads its two pixels of the row from LDS.  The gathers thus leave the texture path,
// which bounds the per-wave kernel.  The row arithmetic (fp_row_add, xbot from the
// broadcast i*slope) is that of the per-wave kernel, and rows where a ray is outside the
// image add exactly 0 in both, so the two give bitwise equal results.  NBUF = 2 double-
// buffers the staged block (one barrier per block), NBUF = 1 halves the LDS per workgroup
// (two barriers per block).
// Grid: (lines, bin blocks of FPS_RAYS, images).  Dynamic LDS: NBUF * FPS_CS * FPS_MAXW floats.
template <int MODE, int NBUF>
__global__ __launch_bounds__(FPS_RAYS) void k_fp_staged(FpParams P) {
  extern __shared__ float4 seg4[];
  fps_item<MODE, NBUF>(P, blockIdx.x, blockIdx.y, blockIdx.z, (float*)seg4);
}

// Grouped staged A.x (variant 7) of S images at once: grid (line groups, bin blocks of FPG_BINS,
// images / S).  CPLMAX: the largest chunk count of the geometry's groups.  Dynamic LDS:
// fpg_lds_floats.
// One image: VALU issue bounds it (13 per row and ray off the exact step, 10 on it, and 45 per
// block and wave of staging and block bounds; 1.3 per CU-clock).  More images share a row's
// position, address and fraction, so each adds 3 VALU and its 8 bytes of LDS reads per row and
// ray; at S = 4 the LDS is busy 65% of the time.  64 images of 512^2, 512 angles: 3.01 ms
// one image at a time, 2.24 ms for S = 2, 1.75 ms for S = 4.
// Waves per SIMD the registers are held to: one image, what its LDS (17, 26 and 35 KB at 2, 3 and 4 chunks)
// lets run together; at 8 the residual's pointers spilled 16 to 19 scalar registers from 3 chunks on.
constexpr int fpg_waves_per_simd(int s, int cpl) {
  return s == 4 ? 4 : (cpl == 2 ? 8 : (cpl == 3 ? 6 : (s == 1 ? 4 : 5)));
}

template <int MODE, int S, int CPLMAX>
__global__ __launch_bounds__(FPS_RAYS, fpg_waves_per_simd(S, CPLMAX)) void k_fp_grouped(FpParams P) {
  extern __shared__ float4 seg4[];
  const int4 grp = P.groups[blockIdx.x];
  const int cpl = grp.x >> 24;  // uniform
  if (CPLMAX == 2 || cpl <= 2)
    fpg_item<MODE, 2, S>(P, grp, blockIdx.y, blockIdx.z, (float*)seg4);
  else if (CPLMAX == 3 || cpl == 3)
    fpg_item<MODE, CPLMAX >= 3 ? 3 : 2, S>(P, grp, blockIdx.y, blockIdx.z, (float*)seg4);
  else
    fpg_item<MODE, CPLMAX >= 4 ? 4 : 2, S>(P, grp, blockIdx.y, blockIdx.z, (float*)seg4);
}

// ------------------------------------------------------------------------ launchers
int launched(Ctx* c, const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(c, e, what);
  return SK_OK;
}

int launch_transpose(Ctx* c, const float* in, float* out, int N, int batch, hipStream_t s) {
  dim3 grid((N + 31) / 32, (N + 31) / 32, batch);
  hipLaunchKernelGGL(k_transpose, grid, dim3(256), 0, s, in, out, N);
  return launched(c, "transpose kernel");
}

FpParams fp_params(const Geom* g, const FpArgs& a) {
  return FpParams{g->d_lines, g->A, g->R, g->N, g->ncand, a.batch, g->rho0, g->drho,
                  a.img, a.imgT, a.out, a.b, a.rowinv, g->d_fpg, g->d_fp_steps, g->fpg_cpl};
}

// fp variants: 0/1/2 = 1/2/4 rays per lane, bin blocks fastest; 3/4 = 1/2 rays per lane,
// lines fastest.
int fp_rays_per_lane(int variant) {
  return (variant == 1 || variant == 4) ? 2 : (variant == 2 ? 4 : 1);
}

template <bool EXACT, int MODE, int WEIGHTS, bool DR1, int RPT, int ORDER = 0>
static void fp_go(const Geom* g, const FpArgs& a, hipStream_t s) {
  const int per_block = FP_BLOCK * RPT;
  const unsigned nb = (unsigned)((g->R + per_block - 1) / per_block);
  const dim3 grid = ORDER ? dim3(g->A, nb, a.batch) : dim3(nb, g->A, a.batch);
  hipLaunchKernelGGL((k_fp<EXACT, MODE, WEIGHTS, DR1, RPT, ORDER>), grid, dim3(FP_BLOCK), 0, s,
                     fp_params(g, a));
}

// Exact mode runs one ray per lane (its IEEE divisions make more rays per lane no faster) in
// either grid order.
template <bool EXACT, int MODE>
static void fp_go_v(int variant, const Geom* g, const FpArgs& a, hipStream_t s) {
  if (variant == 3 || (EXACT && variant == 4))
    fp_go<EXACT, MODE, W_REF, true, 1, 1>(g, a, s);
  else if (!EXACT && variant == 1)
    fp_go<EXACT, MODE, W_REF, true, 2>(g, a, s);
  else if (!EXACT && variant == 2)
    fp_go<EXACT, MODE, W_REF, true, 4>(g, a, s);
  else if (!EXACT && variant == 4)
    fp_go<EXACT, MODE, W_REF, true, 2, 1>(g, a, s);
  else
    fp_go<EXACT, MODE, W_REF, true, 1>(g, a, s);
}

template <int MODE, int NBUF>
static void fp_go_staged(const Geom* g, const FpArgs& a, hipStream_t s) {
  const unsigned nb = (unsigned)((g->R + FPS_RAYS - 1) / FPS_RAYS);
  const size_t lds = sizeof(float) * NBUF * FPS_CS * (size_t)FPS_MAXW;
  hipLaunchKernelGGL((k_fp_staged<MODE, NBUF>), dim3(g->A, nb, a.batch), dim3(FPS_RAYS), lds, s,
                     fp_params(g, a));
}

template <int MODE, int S>
static void fp_go_grouped_s(const Geom* g, const FpArgs& a, hipStream_t s) {
  const unsigned nb = (unsigned)((g->R + FPG_BINS - 1) / FPG_BINS);
  const size_t lds = sizeof(float) * fpg_lds_floats(FpgShape<S>::nbuf, S, g->fpg_cpl, FpgShape<S>::xstep);
  const dim3 grid(g->n_fpg, nb, (a.batch + S - 1) / S);
  const FpParams P = fp_params(g, a);
  if (g->fpg_cpl == 2)
    hipLaunchKernelGGL((k_fp_grouped<MODE, S, 2>), grid, dim3(FPS_RAYS), lds, s, P);
  else if (g->fpg_cpl == 3)
    hipLaunchKernelGGL((k_fp_grouped<MODE, S, 3>), grid, dim3(FPS_RAYS), lds, s, P);
  else
    hipLaunchKernelGGL((k_fp_grouped<MODE, S, 4>), grid, dim3(FPS_RAYS), lds, s, P);
}

// Images per workgroup: 4 (from three images on: a fourth that repeats costs less than a second
// pass) or 2 where that leaves at least two workgroups per CU, else 1.  Below that the chip is
// not full and more images per workgroup only lengthen it: 256^2, 179 angles (270 workgroups an
// image), 4 images: 36.0, 30.3 and 32.3 us for 1, 2 and 4; 8 images: 62.6, 45.2, 40.8; 128^2, 89
// angles (69), 2 images: 13.3, 13.8; 512^2, 358 angles (1080), 3 images: 127.5, 126.1, 110.0.
int fpg_images(const Geom* g, int batch) {
  const long per = (long)g->n_fpg * ((g->R + FPG_BINS - 1) / FPG_BINS);
  if (batch >= 3 && per * ((batch + 3) / 4) >= 512) return 4;
  if (batch >= 2 && per * ((batch + 1) / 2) >= 512) return 2;
  return 1;
}

template <int MODE>
static void fp_go_grouped(const Geom* g, const FpArgs& a, hipStream_t s) {
  switch (fpg_images(g, a.batch)) {
    case 4: fp_go_grouped_s<MODE, 4>(g, a, s); break;
    case 2: fp_go_grouped_s<MODE, 2>(g, a, s); break;
    default: fp_go_grouped_s<MODE, 1>(g, a, s);
  }
}

// Workgroups of four 64-bin waves that a call has.
static long fp_workgroups(const Geom* g, int batch) {
  return ((long)g->A * ((g->R + 63) / 64) + FP_WAVES - 1) / FP_WAVES * batch;
}

// The kernel of a geometry that was not tuned, on a context whose option is 0: the grouped one (7, and
// below it what a geometry without line groups, or exact mode, falls back to), where it is not
// slower than one ray per lane (0 bins fastest, 3 lines fastest).  us for 0, 3 and 7, one image
// unless said, R = sqrt(2) N / drho:
// - 256^2 and 179 angles 29.5, 22.7, 20.9; 512^2 and 358 90, 94, 60; 2048^2 and 1433 3662, -, 1750.
// - Below 128^2 a ray takes a few rows only and the per-wave kernel is as fast (64^2, 100 angles: 9.0 and
//   9.5 for 3 and 7), with a tenth of the code to fetch on a first call, until a batch fills the chip
//   (3 and 7: 96^2 and 150 angles 11.6, 11.1; 16 images 32, 20; 64 images 99, 40).
// - Bins below 1: neighbouring lanes share pixels and the per-wave gathers cost less.  One image per
//   workgroup and one round of workgroups: bins of 0.75, 362^2 and 506 angles 50, 47.5, 62.4; 724^2 and 253
//   90, 91, 119; of 0.5, 512^2 and 716 145, 133, 140; past 4096 workgroups 1024^2 and 1433 938, 894, 822.
//   Several images share the staging again (256^2 and 179, bins of 0.5, 4 images: 7 at 0.71 of 0).
// - A detector that ends several image widths from the axis: bins that see nothing, whose workgroups cost
//   the most where lines run fastest (256^2 and 256 angles, bins of 1, R = 14481: 48, 70, 83; 512^2 and
//   512, bins of 2, R = 14481, 4 images: 415, 1063, 1061), and line groups that spread more the farther
//   off their bins lie, so with narrow bins from little more than the image's diagonal on (512^2 and 179,
//   bins of 0.5, R = 5792, four times what is seen: 76, 64, 119; 256^2 and 128, bins of 1, the axis 2000 from
//   the first one: 27, -, 41).
// - Few lines: those of a group lie far apart, so its rows are wide and each wave waits for more columns
//   than its rays meet.  One line: 256^2 14.6 us, 17.6 grouped.  Up to ten lines, from 128 workgroups of
//   the per-wave kernel: 256^2, 6 angles, 64 images, bins of 2 34, 48; 130^2, 4 angles, 64 images 18, 25.  Bins
//   below 1, by the farthest bin's pixels per line (centred detectors: 8 pixels of width per line), times of 7
//   over 0: 256^2, 12 angles, bins of 0.36, 64 images 1.5; 512^2, 16 images, 32 angles 1.2, 64 angles 0.6;
//   4 images, 179 angles, a detector of six times what is seen 1.9.
// - Bins below 1 of a geometry without line groups: one line at a time, staged (6), is no faster (1024^2, 48
//   angles, bins of 0.5, 32 images: 1141 and 1947).
static int fp_variant_default(const Geom* g, int batch) {
  // the farthest bin from the axis, in image widths (0.71 sees the whole image)
  const double reach = fmax(fabs((double)g->rho0), fabs(g->rho0 + (double)g->R * g->drho)) / g->N;
  const bool narrow = g->drho < 1.0f && fpg_images(g, batch) == 1;
  if (reach > (narrow ? 0.9 : 6.0)) return 0;
  const long workgroups = fp_workgroups(g, batch);
  if (g->N < 128 && workgroups < 512) return 3;
  if (narrow && workgroups < 4096) return 3;
  if (g->A == 1 || (g->A <= 10 && workgroups >= 128) || (g->drho < 1.0f && (g->N * reach > 6.0 * g->A || !g->d_fpg))) return 0;
  return 7;
}

// Whether A.x with no transposed copy at hand (FpArgs: imgT = img) takes k_fp_lds, and needs none, the
// same way as the rule above: the image is small enough to be copied by every workgroup (us with it and
// with the better of the other two and their transposed copy: 64^2 and 90 angles 7.9, 9.0; 80^2 and 126
// 9.4, 10.2; 96^2 and 150 12.0, 11.1; 120^2 and 190 13.4, 13.0), and no more than the three workgroups
// per CU or so that hide it (64^2 and 90 angles: 4 images 8.0, 9.4; 16 images, 720 workgroups, 10.9,
// 13.8; with half bins, 1440 workgroups, 15.4, 12.8).  Without flat lines there is no copy to save.
bool fp_in_lds(const Ctx* c, const Geom* g, int batch) {
  return !c->exact && g->fp_variant < 0 && !c->fp_variant && g->N <= FPL_MAX_N && g->n_steep < g->A &&
         fp_workgroups(g, batch) <= 768;
}

int launch_fp(Ctx* c, const Geom* g, FpMode mode, const FpArgs& a, hipStream_t s) {
  const bool ex = c->exact != 0;
  if (mode == FP_PLAIN && a.imgT == a.img && fp_in_lds(c, g, a.batch)) {
    const dim3 grid((unsigned)fp_workgroups(g, 1), a.batch);
    hipLaunchKernelGGL(k_fp_lds, grid, dim3(256), sizeof(float) * fpl_cells(g->N), s, fp_params(g, a));
    return launched(c, "forward projection kernel");
  }
  int v = g->fp_variant >= 0 ? g->fp_variant : (c->fp_variant ? c->fp_variant : fp_variant_default(g, a.batch));
  if (v == 7) {
    if (!ex && g->d_fpg && mode != FP_ONES_INV) {
      if (mode == FP_PLAIN)
        fp_go_grouped<FP_PLAIN>(g, a, s);
      else
        fp_go_grouped<FP_SIRT>(g, a, s);
      return launched(c, "forward projection kernel");
    }
    v = 6;  // no group table for this geometry: the one-line staged kernel
  }
  if (v == 5 || v == 6) {
    if (!ex && g->fps_w > 0 && g->fps_w <= FPS_MAXW && mode != FP_ONES_INV) {
      if (mode == FP_PLAIN)
        v == 5 ? fp_go_staged<FP_PLAIN, 2>(g, a, s) : fp_go_staged<FP_PLAIN, 1>(g, a, s);
      else
        v == 5 ? fp_go_staged<FP_SIRT, 2>(g, a, s) : fp_go_staged<FP_SIRT, 1>(g, a, s);
      return launched(c, "forward projection kernel");
    }
    v = 3;  // exact mode, or a geometry whose segments do not fit: the per-wave kernel
  }
  switch (mode) {
    case FP_PLAIN: ex ? fp_go_v<true, FP_PLAIN>(v, g, a, s) : fp_go_v<false, FP_PLAIN>(v, g, a, s); break;
    case FP_ONES_INV:
      ex ? fp_go<true, FP_ONES_INV, W_REF, true, 1>(g, a, s) : fp_go<false, FP_ONES_INV, W_REF, true, 1>(g, a, s);
      break;
    case FP_SIRT: ex ? fp_go_v<true, FP_SIRT>(v, g, a, s) : fp_go_v<false, FP_SIRT>(v, g, a, s); break;
  }
  return launched(c, "forward projection kernel");
}

// B^T.v.  Fast mode: on a line that is not degenerate the backprojector's length of a ray in a
// pixel is the forward projector's (both are the part of the row's x-range inside the pixel over
// the range, and a ray with a nonzero length lies within sqrt(2)/2 of the pixel's centre, so it is
// one of the pixel's candidates): those lines are A.v, by whichever kernel A.x runs, but for the
// short rays at the image's corners and those that are not finite (k_bpt_rays).  The degenerate lines (theta ~ 0, pi/2: a ray on
// a pixel edge counts in A and not in B) are walked again with the backprojector's own lengths, one
// launch over their table indices.  8 images of 512^2, 360 angles: 1249 us with every line on that
// walk (60 VALU a row and two dependent global gathers), 201 us like this.  Small images take few
// rows, and one launch of that walk is as fast as two or three (us, walk and this: with degenerate
// lines 16^2 and 22 angles 8.2, 11.2; 24^2 and 33 angles 11.3, 12.5; 32^2 and 44 angles 14.8, 13.5;
// without them 8.2, 8.9; 11.3, 9.9) until a batch fills the chip (16^2, 256 images: 23.7, 17.4).
static bool bpt_walks(const Geom* g, int batch) {
  return !g->index_safe || (g->N < (g->n_degen ? 32 : 24) && fp_workgroups(g, batch) <= 768);
}

int launch_fp_bpt(Ctx* c, const Geom* g, const FpArgs& a, hipStream_t s) {
  const bool dr1 = g->drho == 1.0f;
  if (c->exact || bpt_walks(g, a.batch)) {
    if (c->exact)
      dr1 ? fp_go<true, FP_PLAIN, W_ADJ, true, 1>(g, a, s) : fp_go<true, FP_PLAIN, W_ADJ, false, 1>(g, a, s);
    else
      dr1 ? fp_go<false, FP_PLAIN, W_ADJ, true, 1>(g, a, s) : fp_go<false, FP_PLAIN, W_ADJ, false, 1>(g, a, s);
    return launched(c, "backprojection-transpose kernel");
  }
  int rc = launch_fp(c, g, FP_PLAIN, a, s);
  if (rc) return rc;
  const FpParams P = fp_params(g, a);
  const dim3 rays((unsigned)((g->R + 255) / 256), (unsigned)g->A, (unsigned)a.batch);
  if (dr1)
    hipLaunchKernelGGL((k_bpt_rays<true>), rays, dim3(256), 0, s, P);
  else
    hipLaunchKernelGGL((k_bpt_rays<false>), rays, dim3(256), 0, s, P);
  rc = launched(c, "backprojection-transpose kernel");
  if (rc || !g->n_degen) return rc;
  const dim3 grid((unsigned)((g->R + 63) / 64), (unsigned)g->n_degen, (unsigned)a.batch);
  if (dr1)
    hipLaunchKernelGGL((k_fp_listed<true>), grid, dim3(64 * LISTED_WAVES), 0, s, P, g->d_degen);
  else
    hipLaunchKernelGGL((k_fp_listed<false>), grid, dim3(64 * LISTED_WAVES), 0, s, P, g->d_degen);
  return launched(c, "backprojection-transpose kernel");
}

}  // namespace sk

using namespace sk;

static int check_common(sk_ctx* ctx, sk_geom* g, int batch, const void* p1, const void* p2) {
  if (!ctx) return SK_EINVAL;
  Ctx* c = &ctx->c;
  if (!g) return fail(c, SK_EINVAL, "geometry is NULL");
  if (batch < 1 || batch > 65535) return fail(c, SK_EINVAL, "batch must be in [1, 65535]");
  if (!p1 || !p2) return fail(c, SK_EINVAL, "device pointer is NULL");
  if (g->g.device != c->device) return fail(c, SK_EINVAL, "geometry belongs to another device");
  SK_HIP(c, hipSetDevice(c->device));
  return SK_OK;
}

extern "C" {

int sk_fp(sk_ctx* ctx, sk_geom* g, int batch, const float* d_img, float* d_sino, void* stream) {
  int rc = check_common(ctx, g, batch, d_img, d_sino);
  if (rc) return rc;
  Ctx* c = &ctx->c;
  const Geom& G = g->g;
  hipStream_t s = (hipStream_t)stream;
  const float* imgT = d_img;
  if (G.n_steep < G.A && !fp_in_lds(c, &G, batch)) {
    void* ws = nullptr;
    rc = scratch(c, sizeof(float) * (size_t)batch * G.N * G.N, s, &ws);
    if (rc) return rc;
    rc = launch_transpose(c, d_img, (float*)ws, G.N, batch, s);
    if (rc) return rc;
    imgT = (const float*)ws;
  }
  FpArgs a{d_img, imgT, d_sino, nullptr, nullptr, batch};
  return launch_fp(c, &G, FP_PLAIN, a, s);
}

int sk_bp(sk_ctx* ctx, sk_geom* g, int batch, const float* d_sino, float* d_img, void* stream) {
  int rc = check_common(ctx, g, batch, d_sino, d_img);
  if (rc) return rc;
  BpArgs a{d_sino, d_img, nullptr, nullptr, batch};
  return launch_bp(&ctx->c, &g->g, BP_PLAIN, W_REF, a, (hipStream_t)stream);
}

int sk_bp_transpose(sk_ctx* ctx, sk_geom* g, int batch, const float* d_img, float* d_sino,
                    void* stream) {
  int rc = check_common(ctx, g, batch, d_img, d_sino);
  if (rc) return rc;
  Ctx* c = &ctx->c;
  const Geom& G = g->g;
  hipStream_t s = (hipStream_t)stream;
  const float* imgT = d_img;
  if (G.n_steep < G.A) {
    void* ws = nullptr;
    rc = scratch(c, sizeof(float) * (size_t)batch * G.N * G.N, s, &ws);
    if (rc) return rc;
    rc = launch_transpose(c, d_img, (float*)ws, G.N, batch, s);
    if (rc) return rc;
    imgT = (const float*)ws;
  }
  FpArgs a{d_img, imgT, d_sino, nullptr, nullptr, batch};
  return launch_fp_bpt(c, &G, a, s);
}

int sk_bp_adjoint(sk_ctx* ctx, sk_geom* g, int batch, const float* d_sino, float* d_img,
                  void* stream) {
  int rc = check_common(ctx, g, batch, d_sino, d_img);
  if (rc) return rc;
  BpArgs a{d_sino, d_img, nullptr, nullptr, batch};
  return launch_bp(&ctx->c, &g->g, BP_PLAIN, W_ADJ, a, (hipStream_t)stream);
}

}  // extern "C"
