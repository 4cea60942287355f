// 3-D worlds: the two inner axes of a pass in one kernel.  A workgroup holds one H x W plane of a world's
// half spectrum in LDS, so a step is three passes over memory instead of five:
//
//   plane_fwd:  real plane -> rows along W -> columns along H -> half spectra   (rows_fwd + lines along H)
//   (lines along D, convolution: lx_fft.hip)
//   plane_inv:  half spectra -> columns along H -> rows along W -> growth, weighted sum, update
//                                                                               (lines along H + rows_inv)
//
// Transforms run over lane groups with the cross-lane step between registers (no exchange scratch, so that
// a plane of 96 x 96 takes 40 KB and four workgroups share a CU).  A plane's rows have stride 4 mod 8
// complex: the 8 rows x 4 columns that 32 lanes read at once lie in different banks.
// Measured, us, the passes they replace -> these: 16 worlds of 96^3, forward 46 -> 27 (115 MB: 4.3 TB/s), inverse
// with field and potential written 111 -> 64 (284 MB: 4.4 TB/s); 8 worlds, a chained reverse step 72 -> 48 (143 MB).
#include <algorithm>

#include "lx_pass.h"

namespace {

// complex elements per plane row: >= W / 2 + 1, 4 mod 8
constexpr int plane_stride(int W) { return (W / 2 + 1 - 4 + 7) / 8 * 8 + 4; }
constexpr size_t plane_lds(int H, int W) {  // the plane, then the tables of both axes (one if they are equal)
  return (size_t(H) * plane_stride(W) + H + (H == W ? 0 : W)) * sizeof(float2);
}
// threads: a lane group per row pair, 256 at most (96 x 96: 103 and 128 VGPRs, four workgroups of four waves
// per CU; 384 threads in one round of row pairs left two workgroups of six)
constexpr int plane_threads(int H, int W) {
  return H / 2 * row_tpr(W) < 64 ? 64 : (H / 2 * row_tpr(W) > 256 ? 256 : (H / 2 * row_tpr(W) + 63) / 64 * 64);
}

// A plane's transforms are spread over lanes as the rows' and the lines' of the passes are (lx_fft.hip), so that a
// step rounds alike whichever takes it: columns of 96 points on 4 lanes (one round of 64 groups for 49 columns
// instead of two of 32: a step of 16 worlds of 96^3 133 -> 129 us, gradients of 8 1517 -> 1481 us).
template <int L, int T = row_tpr(L)>
struct PlaneFft {
  static constexpr int TPR = T, P = L / TPR;
  // frequency held by register e of lane t
  static LX_DEV int freq(int t, int e) { return e + P * bitrev_n(t, TPR); }
};

// exp(-2 pi i j / L) tables of both axes into LDS
template <int H, int W>
LX_DEV void plane_tables(float2* twh, float2* tww, const float2* gh, const float2* gw) {
  for (int i = threadIdx.x; i < H; i += plane_threads(H, W)) twh[i] = gh[i];
  if constexpr (H != W)
    for (int i = threadIdx.x; i < W; i += plane_threads(H, W)) tww[i] = gw[i];
}

// Forward transform of a row pair held as x = a + i b (x[m] = point TPR m + t) into the pair's two plane
// rows of half spectra: A[k] = (Z[k] + conj Z[W-k]) / 2, B[k] = (Z[k] - conj Z[W-k]) / 2i.
template <int W>
LX_DEV void pair_forward(float2* x, int t, int lane, const float2* tw, float2* row0) {
  using F = PlaneFft<W>;
  constexpr int TPR = F::TPR, P = F::P, WH = W / 2 + 1, RS = plane_stride(W), NI = (WH + TPR - 1) / TPR;
  fft_lanes<P, TPR, false>(x, t, lane, tw);
  wave_lds_fence();
#pragma unroll
  for (int e = 0; e < P; ++e) row0[F::freq(t, e)] = x[e];  // W <= 2 RS: both rows hold Z
  wave_lds_fence();
  float2 z[NI], zn[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int k = min(t + TPR * i, WH - 1);
    z[i] = row0[k];
    zn[i] = row0[k == 0 ? 0 : W - k];
  }
  wave_lds_fence();
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int k = t + TPR * i;
    if (k < WH) {
      row0[k] = make_float2(0.5f * (z[i].x + zn[i].x), 0.5f * (z[i].y - zn[i].y));
      row0[RS + k] = make_float2(0.5f * (z[i].y + zn[i].y), 0.5f * (zn[i].x - z[i].x));
    }
  }
}

// Inverse transform of the pair's two plane rows: x[m] = (a, b) at point TPR m + t, unnormalised.
template <int W>
LX_DEV void pair_inverse(float2* x, int t, int lane, const float2* tw, const float2* row0) {
  using F = PlaneFft<W>;
  constexpr int TPR = F::TPR, P = F::P, RS = plane_stride(W);
#pragma unroll
  for (int e = 0; e < P; ++e) {
    const int f = F::freq(t, e);
    const bool mirror = f >= W / 2;
    const float sg = mirror ? -1.f : 1.f;
    const int col = mirror ? W - f : f;
    const float2 ya = row0[col], yb = row0[RS + col];
    float2 z = make_float2(fmaf(-sg, yb.y, ya.x), fmaf(sg, ya.y, yb.x));
    if (f == 0 || f == W / 2) z = make_float2(ya.x, yb.x);
    x[e] = z;
  }
  fft_lanes<P, TPR, true>(x, t, lane, tw);
}

// Columns of the plane in LDS -> half spectra of the plane in memory
template <int H, int W>
LX_DEV void columns_out(const float2* plane, const float2* tw, float2* S) {
  using F = PlaneFft<H, line_tpr(H, 1)>;
  constexpr int TPR = F::TPR, P = F::P, WH = W / 2 + 1, RS = plane_stride(W), NC = plane_threads(H, W) / TPR;
  using SG = Strided<TPR>;  // a wave's lanes: neighbouring columns side by side
#pragma unroll 1
  for (int r = 0; r < (WH + NC - 1) / NC; ++r) {
    int lane = threadIdx.x & 63;  // opaque per column, as the rounds of plane_inv
    __asm__ volatile("" : "+v"(lane));
    const int t = SG::point(lane), c0 = r * NC + (threadIdx.x >> 6) * SG::G + SG::line(lane);
    const int c = min(c0, WH - 1);  // every lane stays in: the network crosses lanes
    float2 x[P];
#pragma unroll
    for (int m = 0; m < P; ++m) x[m] = plane[(TPR * m + t) * RS + c];
    fft_strided<P, TPR, false>(x, t, lane, tw);
    if (c0 < WH) {
#pragma unroll
      for (int e = 0; e < P; ++e) S[F::freq(t, e) * WH + c] = x[e];
    }
  }
}

// Half spectra of the plane in memory -> columns transformed back in LDS
template <int H, int W>
LX_DEV void columns_in(float2* plane, const float2* tw, const float2* U) {
  using F = PlaneFft<H, line_tpr(H, 2)>;
  constexpr int TPR = F::TPR, P = F::P, WH = W / 2 + 1, RS = plane_stride(W), NC = plane_threads(H, W) / TPR;
  using SG = Strided<TPR>;  // a wave's lanes: neighbouring columns side by side
#pragma unroll 1
  for (int r = 0; r < (WH + NC - 1) / NC; ++r) {
    int lane = threadIdx.x & 63;  // opaque per column, as the rounds of plane_inv
    __asm__ volatile("" : "+v"(lane));
    const int t = SG::point(lane), c0 = r * NC + (threadIdx.x >> 6) * SG::G + SG::line(lane);
    const int c = min(c0, WH - 1);
    float2 x[P];
#pragma unroll
    for (int e = 0; e < P; ++e) x[e] = U[F::freq(t, e) * WH + c];
    __builtin_amdgcn_sched_barrier(0);
    fft_strided<P, TPR, true>(x, t, lane, tw);
    if (c0 < WH) {
#pragma unroll
      for (int m = 0; m < P; ++m) plane[(TPR * m + t) * RS + c] = x[m];
    }
  }
}

struct PlaneTables {
  const float2* h;
  const float2* w;
};

template <int H, int W>
__global__ __launch_bounds__(plane_threads(H, W)) void plane_fwd_kernel(const float* __restrict__ A,
                                                                       float2* __restrict__ S, PlaneTables tb) {
  using F = PlaneFft<W>;
  constexpr int TPR = F::TPR, P = F::P, WH = W / 2 + 1, RS = plane_stride(W);
  extern __shared__ __align__(16) float2 lds[];
  float2* plane = lds;
  float2 *twh = lds + H * RS, *tww = H == W ? twh : twh + H;
  const int lane = threadIdx.x & 63, t = threadIdx.x % TPR;
  A += int64_t(blockIdx.x) * H * W;
  constexpr int NG = plane_threads(H, W) / TPR, ROUNDS = (H / 2 + NG - 1) / NG;
  plane_tables<H, W>(twh, tww, tb.h, tb.w);
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int pr = threadIdx.x / TPR + r * NG;
    const float* a0 = A + 2 * min(pr, H / 2 - 1) * W;
    float2 x[P];
#pragma unroll
    for (int m = 0; m < P; ++m) x[m] = make_float2(a0[TPR * m + t], a0[W + TPR * m + t]);
    if (r == 0) __syncthreads();  // the tables
    if (pr < H / 2) pair_forward<W>(x, t, lane, tww, plane + 2 * pr * RS);
  }
  __syncthreads();
  columns_out<H, W>(plane, twh, S + int64_t(blockIdx.x) * H * WH);
}

// The inverse planes.  One channel and one kernel: the update follows in the same kernel.  Otherwise the
// potentials are written (to the caller's, or over the planes' own spectra) and points_kernel takes them.
struct PlaneInv {
  const float2* U;
  float* pot;            // potentials, plane p at pot + p pot_stride; NULL: none (update only)
  int64_t pot_stride;
  const float* A;        // update
  float* A_out;
  float* field;
  const float* gf;
  const float* w;
  const float* dt;
  int64_t gf_bs, w_bs, dt_bs;
  int D, kind, state_fn, average, update, sel;
  float dt_val;
  LxAdjFinish fin;
  int fin_blocks;
};

struct Growth {
  int kind;
  float m, s, inv_s, inv_9s2;
  LX_DEV Growth(int kind_, float m_, float s_)
      : kind(kind_), m(m_), s(s_), inv_s(1.f / s_), inv_9s2(1.f / (9.f * (s_ * s_))) {}
  template <int KIND>
  LX_DEV void four(float4& u) const {
    u.x = growth_pre<KIND>(m, s, inv_s, inv_9s2, u.x);
    u.y = growth_pre<KIND>(m, s, inv_s, inv_9s2, u.y);
    u.z = growth_pre<KIND>(m, s, inv_s, inv_9s2, u.z);
    u.w = growth_pre<KIND>(m, s, inv_s, inv_9s2, u.w);
  }
  LX_DEV void operator()(float4& u) const {  // kind is uniform over the block
    switch (kind) {
      case LX_GF_POLY_QUAD4: four<LX_GF_POLY_QUAD4>(u); break;
      case LX_GF_GAUSSIAN: four<LX_GF_GAUSSIAN>(u); break;
      case LX_GF_GAUSSIAN_TARGET: four<LX_GF_GAUSSIAN_TARGET>(u); break;
      case LX_GF_STEP: four<LX_GF_STEP>(u); break;
      case LX_GF_STAIRCASE: four<LX_GF_STAIRCASE>(u); break;
      case LX_GF_TRIANGLE: four<LX_GF_TRIANGLE>(u); break;
      default: break;
    }
  }
};

LX_DEV float4 add_weighted(float4 G, float w, float4 g) {
  return make_float4(add_nc(G.x, mul_nc(w, g.x)), add_nc(G.y, mul_nc(w, g.y)), add_nc(G.z, mul_nc(w, g.z)),
                     add_nc(G.w, mul_nc(w, g.w)));
}
LX_DEV float4 step_four(int state_fn, float4 v, float4 g, float dt) {
  return make_float4(step_value(state_fn, v.x, g.x, dt), step_value(state_fn, v.y, g.y, dt),
                     step_value(state_fn, v.z, g.z, dt), step_value(state_fn, v.w, g.w, dt));
}

// A wave's lanes transform the row pairs of its own lane groups and then take four neighbouring points
// each of the same rows (16-byte accesses), so that only the columns need the workgroup's barriers.
template <int H, int W>
__global__ __launch_bounds__(plane_threads(H, W)) void plane_inv_kernel(PlaneInv a, PlaneTables tb) {
  using F = PlaneFft<W>;
  constexpr int TPR = F::TPR, P = F::P, WH = W / 2 + 1, RS = plane_stride(W), NT = plane_threads(H, W);
  constexpr int GW = 64 / TPR;                    // row pairs of a wave per round
  constexpr int NG = NT / TPR, ROUNDS = (H / 2 + NG - 1) / NG;
  constexpr int QW = GW * 2 * (W / 4), IT = (QW + 63) / 64;  // four-point items of a wave's rows, of a lane
  extern __shared__ __align__(16) float2 lds[];
  float2* plane = lds;
  float2 *twh = lds + H * RS, *tww = H == W ? twh : twh + H;
  const int wave = threadIdx.x >> 6;
  if (int(blockIdx.x) >= int(gridDim.x) - a.fin_blocks) {
    const int64_t i = int64_t(int(blockIdx.x) - (int(gridDim.x) - a.fin_blocks)) * (NT / 64) + wave;
    if (i < lx_adj_finish_outputs(a.fin)) lx_adj_finish_wave(a.fin, i);
    return;
  }
  const int64_t p = blockIdx.x, in_plane = p * H * W;
  const int b = int(p / a.D);
  plane_tables<H, W>(twh, tww, tb.h, tb.w);
  float wk = 1.f, gm = 0.f, gs = 1.f, dtw = 1.f;
  if (a.update && !a.sel) {
    wk = a.w[b * a.w_bs];
    gm = a.gf[b * a.gf_bs];
    gs = a.gf[b * a.gf_bs + 1];
    dtw = a.dt ? a.dt[b * a.dt_bs] : a.dt_val;
  }
  const Growth growth(a.sel ? int(LX_GF_IDENTITY) : a.kind, gm, gs);
  __syncthreads();  // the tables
  columns_in<H, W>(plane, twh, a.U + p * H * WH);
  __syncthreads();
  const float inv_n = 1.f / float(int64_t(H) * W * a.D);
#pragma unroll 1
  for (int r = 0; r < ROUNDS; ++r) {
    // opaque per round: addresses and twiddles are not hoisted out of the loop and kept live
    int lane = threadIdx.x & 63;
    __asm__ volatile("" : "+v"(lane));
    const int t = lane % TPR;
    const int pr = threadIdx.x / TPR + r * NG;
    const int first = r * NG + wave * GW;  // the wave's first pair of the round
    if (first >= H / 2) break;             // wave-uniform
    // the lane's i-th four points: row and column (row >= H: none)
    auto item = [&](int i, int& row, int& col) {
      const int q = lane + 64 * i;
      row = q < QW ? 2 * first + q / (W / 4) : H;
      col = q % (W / 4) * 4;
      return row < H;
    };
    float2* row0 = plane + 2 * min(pr, H / 2 - 1) * RS;
    float2 x[P];
    pair_inverse<W>(x, t, lane, tww, row0);
    __builtin_amdgcn_sched_barrier(0);
    wave_lds_fence();
    if (pr < H / 2) {  // the potentials replace the rows: row j's at the start of plane row j
      float *u0 = reinterpret_cast<float*>(row0), *u1 = reinterpret_cast<float*>(row0 + RS);
#pragma unroll
      for (int m = 0; m < P; ++m) {
        u0[TPR * m + t] = x[m].x * inv_n;
        u1[TPR * m + t] = x[m].y * inv_n;
      }
    }
    wave_lds_fence();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 2
    for (int i = 0; i < IT; ++i) {
      int row, col;
      if (!item(i, row, col)) continue;
      float4 v;
      if (a.update) v = *reinterpret_cast<const float4*>(a.A + in_plane + row * W + col);
      float4 u = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(plane + row * RS) + col);
      const int64_t o = row * W + col;
      if (a.pot) *reinterpret_cast<float4*>(a.pot + p * a.pot_stride + o) = u;
      if (!a.update) continue;
      float4 g = make_float4(0.f, 0.f, 0.f, 0.f);
      if (wk != 0.f || a.pot) {  // a kernel without weight counts (times 0) only where its potential is wanted
        growth(u);
        g = add_weighted(g, wk, u);
      }
      if (a.average) {
        const float den = add_nc(0.f, wk);
        g = make_float4(g.x / den, g.y / den, g.z / den, g.w / den);
      }
      if (a.field) *reinterpret_cast<float4*>(a.field + in_plane + o) = g;
      *reinterpret_cast<float4*>(a.A_out + in_plane + o) = step_four(a.state_fn, v, g, dtw);
    }
  }
}

// The update from the potentials of several kernels: growth, weighted sum in the kernels' order, state.
// One block per 256 four-point items of one channel image, then of the image gridDim.y further on (images are
// any number, a grid's y dimension is at most kGridY).
struct Points {
  const float* pot;  // kernel k of world b, plane d at pot + ((b K + k) D + d) pot_stride
  int64_t pot_stride;
  const float* A;
  float* A_out;
  float* field;
  const float* gf;
  const float* w;
  const float* dt;
  uint64_t kinds, cins;
  int64_t gf_bs, w_bs, dt_bs;
  int64_t images;
  int D, cells, C, K, state_fn, average, sel, want_all;  // cells: of a plane; want_all: potentials are the caller's
  float dt_val;
};

constexpr int64_t kGridY = 65535;

LX_DEV void points_of(const Points& a, int64_t img) {
  const int64_t b = img / a.C;
  const int c = int(img - b * a.C);
  const int64_t q = int64_t(blockIdx.x) * 256 + threadIdx.x;  // four-point item of the image
  const int per_plane = a.cells / 4;
  if (q >= int64_t(a.D) * per_plane) return;
  const int d = int(q / per_plane);
  const int64_t o = (q - int64_t(d) * per_plane) * 4, io = img * a.D * a.cells + q * 4;
  const float* w = a.sel ? nullptr : a.w + b * a.w_bs;
  const float* gf = a.sel ? nullptr : a.gf + b * a.gf_bs;
  const float4 v = *reinterpret_cast<const float4*>(a.A + io);
  float4 G = make_float4(0.f, 0.f, 0.f, 0.f);
  float den = 0.f;
  for (int k = 0; k < a.K; ++k) {
    const float wk = a.sel ? ((int(a.cins >> (4 * k)) & 15) == c ? 1.f : 0.f) : w[c * a.K + k];
    den = add_nc(den, wk);
    if (wk == 0.f) {
      // a kernel that feeds no channel counts (times 0) in channel 0 where its potential is wanted
      bool skip = a.sel || c != 0 || !a.want_all;
      for (int cc = 1; cc < a.C && !skip; ++cc) skip = w[cc * a.K + k] != 0.f;
      if (skip) continue;
    }
    float4 u = *reinterpret_cast<const float4*>(a.pot + ((b * a.K + k) * a.D + d) * a.pot_stride + o);
    if (!a.sel) Growth(int(a.kinds >> (4 * k)) & 15, gf[2 * k], gf[2 * k + 1])(u);
    G = add_weighted(G, wk, u);
  }
  if (a.average) G = make_float4(G.x / den, G.y / den, G.z / den, G.w / den);
  if (a.field) *reinterpret_cast<float4*>(a.field + io) = G;
  const float dtw = a.sel ? 1.f : a.dt ? a.dt[b * a.dt_bs] : a.dt_val;
  *reinterpret_cast<float4*>(a.A_out + io) = step_four(a.state_fn, v, G, dtw);
}

__global__ __launch_bounds__(256) void points_kernel(Points a) {
  for (int64_t img = blockIdx.y; img < a.images; img += gridDim.y) points_of(a, img);
}

// One channel, one kernel, reverse: the planes of rows_fwd_adj_kernel (lx_fft.hip) and of the lines beside
// it.  BRIDGE: the adjoint potential of the later step (half spectra after the lines along D) is transformed
// back and added to lambda; then the pointwise reverse of this step turns its potential into dL/dU, which is
// transformed and replaces the plane's spectra.  lambda, the potential (and the state where the update needs
// it) are read and lambda written once; the gradient scalars are one partial sum per plane.
struct PlaneAdj {
  float2* X;
  const float* U;
  float* lam;
  const float* A;
  float* part;  // [B][per][4]: dm, ds, dw, ddt
  const float* gf;
  const float* w;
  const float* dt;
  int64_t gf_bs, w_bs, dt_bs;
  int D, kind, mode, average, accumulate;  // mode 0: lambda passes through, 1: the true clip, 2: v2
};

template <int H, int W, bool BRIDGE>
__global__ __launch_bounds__(plane_threads(H, W)) void plane_adj_kernel(PlaneAdj a, PlaneTables tb) {
  using F = PlaneFft<W>;
  constexpr int TPR = F::TPR, P = F::P, WH = W / 2 + 1, RS = plane_stride(W), NT = plane_threads(H, W);
  constexpr int GW = 64 / TPR, NG = NT / TPR, ROUNDS = (H / 2 + NG - 1) / NG;
  constexpr int QW = GW * 2 * (W / 4), IT = (QW + 63) / 64;
  extern __shared__ __align__(16) float2 lds[];
  __shared__ float red[4][NT / 64];
  float2* plane = lds;
  float2 *twh = lds + H * RS, *tww = H == W ? twh : twh + H;
  const int wave = threadIdx.x >> 6;
  const int64_t p = blockIdx.x, in_plane = p * H * W;
  const int b = int(p / a.D);
  plane_tables<H, W>(twh, tww, tb.h, tb.w);
  const float w = a.w[b * a.w_bs], gm = a.gf[b * a.gf_bs], gs = a.gf[b * a.gf_bs + 1], dtw = a.dt[b * a.dt_bs];
  const float inv_s = 1.f / gs, inv_9s2 = 1.f / (9.f * (gs * gs)), inv_n = 1.f / float(int64_t(H) * W * a.D);
  const float coef = a.average ? w / w : w, inv_den = a.average ? 1.f / w : 1.f;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  __syncthreads();  // the tables
  if constexpr (BRIDGE) {
    columns_in<H, W>(plane, twh, a.X + p * H * WH);
    __syncthreads();
  }
#pragma unroll 1
  for (int r = 0; r < ROUNDS; ++r) {
    int lane = threadIdx.x & 63;  // opaque per round, as in plane_inv
    __asm__ volatile("" : "+v"(lane));
    const int t = lane % TPR;
    const int pr = threadIdx.x / TPR + r * NG;
    const int first = r * NG + wave * GW;
    if (first >= H / 2) break;  // wave-uniform
    float2* row0 = plane + 2 * min(pr, H / 2 - 1) * RS;
    float *u0 = reinterpret_cast<float*>(row0), *u1 = reinterpret_cast<float*>(row0 + RS);
    if constexpr (BRIDGE) {
      float2 x[P];
      pair_inverse<W>(x, t, lane, tww, row0);
      wave_lds_fence();
      if (pr < H / 2) {
#pragma unroll
        for (int m = 0; m < P; ++m) {
          u0[TPR * m + t] = x[m].x * inv_n;
          u1[TPR * m + t] = x[m].y * inv_n;
        }
      }
      wave_lds_fence();
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll 2
    for (int i = 0; i < IT; ++i) {
      const int q = lane + 64 * i, row = 2 * first + q / (W / 4), col = q % (W / 4) * 4;
      if (q >= QW || row >= H) continue;
      const int64_t o = in_plane + row * W + col;
      const float4 U4 = *reinterpret_cast<const float4*>(a.U + o);
      const float4 L4 = *reinterpret_cast<const float4*>(a.lam + o);
      float4 A4 = make_float4(0.f, 0.f, 0.f, 0.f);
      if (a.mode != 0) A4 = *reinterpret_cast<const float4*>(a.A + o);
      float4* at = reinterpret_cast<float4*>(reinterpret_cast<float*>(plane + row * RS) + col);
      float4 inc = make_float4(0.f, 0.f, 0.f, 0.f);
      if constexpr (BRIDGE) inc = *at;
      const float Uv[4] = {U4.x, U4.y, U4.z, U4.w}, Av[4] = {A4.x, A4.y, A4.z, A4.w};
      const float Iv[4] = {inc.x, inc.y, inc.z, inc.w};
      float Lv[4] = {L4.x, L4.y, L4.z, L4.w}, du[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float L = Lv[e];
        if constexpr (BRIDGE) L = add_nc(L, Iv[e]);
        float dgdu, dgdm, dgds;
        const float g = growth_rcp(a.kind, gm, gs, inv_s, inv_9s2, Uv[e]);
        growth_grad(a.kind, gm, gs, inv_s, inv_9s2, Uv[e], dgdu, dgdm, dgds);
        const float wg = mul_nc(w, g);
        const float G = a.average ? wg / w : wg;
        float dz = L;
        if (a.mode == 1) {
          const float z = add_nc(Av[e], mul_nc(dtw, G));
          dz = (z > 0.f && z < 1.f) ? L : 0.f;
        }
        const float dG = dtw * dz;
        const float dg = dG * coef;
        du[e] = dg * dgdu;
        acc[0] += dg * dgdm;
        acc[1] += dg * dgds;
        acc[2] += dG * (a.average ? (g - G) * inv_den : g);
        acc[3] += a.mode == 2 ? dz * (G - Av[e]) : dz * G;
        Lv[e] = a.mode == 2 ? dz * (1.f - dtw) : dz;
      }
      if (BRIDGE || a.mode != 0) *reinterpret_cast<float4*>(a.lam + o) = make_float4(Lv[0], Lv[1], Lv[2], Lv[3]);
      *at = make_float4(du[0], du[1], du[2], du[3]);
    }
    wave_lds_fence();
    __builtin_amdgcn_sched_barrier(0);
    if (pr < H / 2) {
      float2 x[P];
#pragma unroll
      for (int m = 0; m < P; ++m) x[m] = make_float2(u0[TPR * m + t], u1[TPR * m + t]);
      wave_lds_fence();
      pair_forward<W>(x, t, lane, tww, row0);
    }
  }
  wave_sum_n(acc);
  if ((threadIdx.x & 63) == 0)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[i][wave] = acc[i];
  __syncthreads();
  columns_out<H, W>(plane, twh, a.X + p * H * WH);
  if (threadIdx.x < 4) {
    float sum = red[threadIdx.x][0];
#pragma unroll
    for (int v = 1; v < NT / 64; ++v) sum += red[threadIdx.x][v];
    float* dst = a.part + p * 4 + threadIdx.x;
    *dst = a.accumulate ? *dst + sum : sum;
  }
}

// The convolution along D of worlds that share one kernel's spectrum: a lane group takes one line of NB
// worlds in turn, so the line's spectrum is read once for all of them (every world's own group re-read it
// from L2: as many bytes as the lines themselves), and the next world's line is loaded while this one is
// transformed.  16 worlds of 96^3: 38.7 -> 32.1 us (115 MB: 3.6 TB/s).
struct SharedConv {
  const float2* S;
  float2* U;
  const float2* Kh;
  const float2* tw;
  const float2* twl;
  float2* FA;
  int64_t img_elems;
  int lines, st, B, NB;  // lines of an image: contiguous, points st apart
  float csign;
};

template <int L>
__global__ __launch_bounds__(256) void shared_conv_kernel(SharedConv a) {
  using LC = Lanes<L>;
  constexpr int TPR = LC::TPR, P = LC::P;
  using SG = Strided<TPR>;
  __shared__ __align__(16) float2 xch_all[LC::XL ? 256 / TPR * strided_scratch<L, TPR>() : 2];
  const int t = SG::point(threadIdx.x & 63), own = (threadIdx.x >> 6) * SG::G + SG::line(threadIdx.x & 63);
  float2* xch = xch_all + (LC::XL ? own * strided_scratch<L, TPR>() : 0);
  const int line = int(blockIdx.x) * (256 / TPR) + own;
  const bool live = line < a.lines;
  const int off = live ? line : 0, b0 = int(blockIdx.y) * a.NB, b1 = min(b0 + a.NB, a.B);
  float2 kv[P], x[P], nx[P];
  const float2* src = a.S + int64_t(b0) * a.img_elems + off;
#pragma unroll
  for (int m = 0; m < P; ++m) x[m] = src[(TPR * m + t) * a.st];
#pragma unroll
  for (int e = 0; e < P; ++e) {
    kv[e] = a.Kh[freq_of<L>(t, e) * a.st + off];
    kv[e].y *= a.csign;
  }
#pragma unroll 1
  for (int b = b0; b < b1; ++b) {
    int lane = threadIdx.x & 63;  // opaque per world: twiddles and addresses are not kept live
    __asm__ volatile("" : "+v"(lane));
    const int t = SG::point(lane);
    auto fft = [&](auto inv_c) {
      constexpr bool INV = decltype(inv_c)::value;
      if constexpr (LC::XL) fft_xlds<P, TPR, INV>(x, t, a.twl + t * twl_row(P), xch);
      else fft_strided<P, TPR, INV>(x, t, lane, a.tw);
    };
    src += a.img_elems;
    if (b + 1 < b1) {
#pragma unroll
      for (int m = 0; m < P; ++m) nx[m] = src[(TPR * m + t) * a.st];
    }
    __builtin_amdgcn_sched_barrier(0);
    fft(std::false_type{});
    if (a.FA && live) {
      float2* fa = a.FA + int64_t(b) * a.img_elems + off;
#pragma unroll
      for (int e = 0; e < P; ++e) fa[freq_of<L>(t, e) * a.st] = x[e];
    }
#pragma unroll
    for (int e = 0; e < P; ++e) x[e] = cmul(x[e], kv[e]);
    wave_lds_fence();
    fft(std::true_type{});
    wave_lds_fence();
    float2* dst = a.U + int64_t(b) * a.img_elems + off;
    if (live) {
#pragma unroll
      for (int m = 0; m < P; ++m) dst[(TPR * m + t) * a.st] = x[m];
    }
#pragma unroll
    for (int m = 0; m < P; ++m) x[m] = nx[m];
  }
}

int launched(const char* what) {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? LX_OK : lx_fail(LX_EDEVICE, "%s launch: %s", what, hipGetErrorString(e));
}

template <typename F>
bool by_side(int n, F&& f) {
  switch (n) {
    case 32: f(IntC<32>{}); return true;
    case 48: f(IntC<48>{}); return true;
    case 64: f(IntC<64>{}); return true;
    case 96: f(IntC<96>{}); return true;
    case 128: f(IntC<128>{}); return true;
    default: return false;
  }
}

// f(IntC<H>, IntC<W>) for planes these kernels take: sides 32 to 128
template <typename F>
bool by_plane(int H, int W, F&& f) {
  bool ok = false;
  by_side(H, [&](auto h) { ok = by_side(W, [&](auto w) { f(h, w); }); });
  return ok;
}

// a kernel's dynamic LDS beyond 64 KB (planes of 128 x 128) is asked for before its launches
template <typename K>
int allow_lds(K kernel, size_t bytes) {
  if (bytes <= 65536) return LX_OK;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                          int(bytes)) != hipSuccess)
    return lx_fail(LX_EDEVICE, "plane kernels: %zu bytes of LDS refused", bytes);
  return LX_OK;
}

int plane_tables_of(int H, int W, hipStream_t st, PlaneTables* tb) {
  LxPassTables h, w;
  if (int rc = lx_pass_tables(H, st, &h)) return rc;
  if (int rc = lx_pass_tables(W, st, &w)) return rc;
  tb->h = h.tw;
  tb->w = w.tw;
  return LX_OK;
}

}  // namespace

bool lx_plane_takes(int H, int W) { return by_plane(H, W, [](auto, auto) {}); }

// A plane is one workgroup's: a chain of up to 64 points a lane whatever the number of planes, where rows and lines
// spread over the chip (and a few worlds' rows have kernels of their own).  Small planes are no slower at any count,
// large ones once most CUs have one.  Measured, us of these kernels against rows and lines for 16, 64, 128, 160, 256,
// 512 planes: forward of 96 x 96 7.6 / 8.9, 8.5 / 9.6, 9.2 / 11.2, 9.8 / 12.2, 10.4 / 13.1, 12.6 / 19.5, of 128 x 96
// 9.4 / 8.7, 10.3 / 9.7, 11.7 / 11.6, 11.8 / 12.3, 12.3 / 14.8, 16.6 / 24.1, of 128 x 128 13.1 / 8.7, 14.6 / 10.3,
// 15.2 / 12.2, 15.5 / 13.5, 17.4 / 17.9, 23.1 / 27.3; inverse with the update of 96 x 64 11.8 / 9.9, 12.1 / 11.6,
// 12.3 / 12.6, 12.6 / 13.0, 13.4 / 14.7, 17.7 / 25.0, of 96 x 96 15.5 / 10.5, 15.9 / 13.7, 16.5 / 14.9, 16.8 / 17.2,
// 18.1 / 20.7, 22.4 / 29.3, of 128 x 128 23.3 / 9.7, 24.0 / 12.6, 25.1 / 20.3, 25.6 / 22.3, 26.4 / 26.3, 34.9 / 43.1.
bool lx_plane_pays(int H, int W, int64_t planes, bool inverse) {
  if (!inverse) return H * W <= 9216 || planes >= (W < 128 ? 96 : 256);
  return H * W <= 6144 || planes >= (W < 128 || H < 96 ? 160 : 256);
}

// The reverse sums a world's gradient scalars in an order that its route fixes, and a world's gradients do not
// depend on the batch it is in: the route goes by the world's size alone.  Large planes of worlds of 64 planes up,
// but not 128-point rows by 96 or more (LDS leaves two workgroups per CU, and 96 rows are a round and a half).
// Measured as above, four steps and their reverse: 96 x 96 210 / 164, 242 / 220, 254 / 260, 261 / 280, 327 / 404,
// 534 / 712; 128 x 96 236 / 160, 276 / 231, 287 / 287, 298 / 312, 398 / 518, 747 / 880; 128 x 128 327 / 161, 368 / 268,
// 380 / 315, 398 / 361, 544 / 611, 1082 / 1075.
bool lx_plane_pays_reverse(int D, int H, int W) { return H * W <= 6144 || (D >= 64 && !(W >= 128 && H >= 96)); }

int lx_plane_fwd(int H, int W, const float* A, float2* S, int64_t planes, hipStream_t st) {
  PlaneTables tb;
  if (int rc = plane_tables_of(H, W, st, &tb)) return rc;
  int rc = LX_OK;
  by_plane(H, W, [&](auto h, auto w) {
    constexpr int HH = decltype(h)::value, WW = decltype(w)::value;
    constexpr size_t lds = plane_lds(HH, WW);
    if ((rc = allow_lds(plane_fwd_kernel<HH, WW>, lds))) return;
    hipLaunchKernelGGL((plane_fwd_kernel<HH, WW>), dim3(unsigned(planes)), dim3(plane_threads(HH, WW)), lds, st, A, S,
                       tb);
    rc = launched("plane forward");
  });
  return rc;
}

int lx_plane_inv(const RowArgs& a, int D, int H, int W, int64_t images, hipStream_t st) {
  PlaneTables tb;
  if (int rc = plane_tables_of(H, W, st, &tb)) return rc;
  const int64_t B = images / a.C;
  const bool one = a.C == 1 && a.K == 1;
  PlaneInv p;
  p.U = a.U; p.pot = a.pot; p.pot_stride = int64_t(H) * W;
  p.A = a.A; p.A_out = a.A_out; p.field = a.field; p.gf = a.gf; p.w = a.w; p.dt = a.dt;
  p.gf_bs = a.gf_bs; p.w_bs = a.w_bs; p.dt_bs = a.dt_bs;
  p.D = D; p.kind = a.gfk[0]; p.state_fn = a.state_fn; p.average = a.average; p.update = one && a.update; p.sel = a.sel;
  p.dt_val = a.dt_val; p.fin = a.fin; p.fin_blocks = 0;
  if (!one && !p.pot) {  // the potentials over their planes' spectra, which each workgroup has read
    p.pot = reinterpret_cast<float*>(const_cast<float2*>(a.U));
    p.pot_stride = int64_t(H) * (W / 2 + 1) * 2;
  }
  const int64_t nout = (a.fin.g_gf ? (a.fin.gf_bs ? a.fin.B : 1) * 2 : 0) +
                       (a.fin.g_w ? (a.fin.w_bs ? a.fin.B : 1) : 0) + (a.fin.g_dt ? (a.fin.dt_bs ? a.fin.B : 1) : 0);
  int rc = LX_OK;
  by_plane(H, W, [&](auto h, auto w) {
    constexpr int HH = decltype(h)::value, WW = decltype(w)::value, NT = plane_threads(HH, WW);
    constexpr size_t lds = plane_lds(HH, WW);
    if (a.fin.blocks) p.fin_blocks = int((nout + NT / 64 - 1) / (NT / 64));
    if ((rc = allow_lds(plane_inv_kernel<HH, WW>, lds))) return;
    hipLaunchKernelGGL((plane_inv_kernel<HH, WW>), dim3(unsigned(B * a.K * D) + unsigned(p.fin_blocks)), dim3(NT), lds,
                       st, p, tb);
    rc = launched("plane inverse");
  });
  if (rc || one || !a.update) return rc;
  Points q;
  q.pot = p.pot; q.pot_stride = p.pot_stride; q.A = a.A; q.A_out = a.A_out; q.field = a.field;
  q.gf = a.gf; q.w = a.w; q.dt = a.dt; q.gf_bs = a.gf_bs; q.w_bs = a.w_bs; q.dt_bs = a.dt_bs;
  q.kinds = q.cins = 0;
  for (int k = 0; k < a.K; ++k) {
    q.kinds |= uint64_t(a.gfk[k] & 15) << (4 * k);
    q.cins |= uint64_t(a.cin[k] & 15) << (4 * k);
  }
  q.images = images; q.D = D; q.cells = H * W; q.C = a.C; q.K = a.K;
  q.state_fn = a.state_fn; q.average = a.average; q.sel = a.sel;
  q.want_all = a.pot != nullptr; q.dt_val = a.dt_val;
  const int64_t items = int64_t(D) * H * W / 4;
  hipLaunchKernelGGL(points_kernel, dim3(unsigned((items + 255) / 256), unsigned(std::min(images, kGridY))),
                     dim3(256), 0, st, q);
  return launched("points");
}

int lx_shared_conv(const LineArgs& a, int L, int64_t images, hipStream_t st, int* taken) {
  *taken = 0;
  if (a.mode != 0 || a.dspec || a.kquad || a.k_bstride != 0 || a.C != 1 || a.K != 1 || images < 2) return LX_OK;
  SharedConv c;
  c.lines = a.A * a.WH; c.st = int(a.st);
  // lines of an image are contiguous where the convolution axis is the outermost of three
  if (a.A < 2 || a.a_stride != a.WH || images > kGridY) return LX_OK;
  const int64_t waves = images * c.lines * lx_row_tpr(L) / 64;
  // worlds per group: as many as leave about three waves per SIMD (16 worlds of 96^3: 1, 2, 3, 4, 8 worlds
  // 38.7, 33.8, 32.1, 35.3, 46.1 us)
  const int64_t NB = std::min<int64_t>(8, waves / 3000);
  if (NB < 2) return LX_OK;
  LxPassTables tb;
  if (int rc = lx_pass_tables(L, st, &tb)) return rc;
  c.S = a.S; c.U = a.U; c.Kh = a.Kh; c.tw = tb.tw; c.twl = tb.twl; c.FA = a.FA; c.img_elems = a.img_elems;
  c.B = int(images); c.NB = int(NB); c.csign = a.conjk ? -1.f : 1.f;
  const bool ok = by_side(L, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    const int per = 256 / row_tpr(LL);
    hipLaunchKernelGGL((shared_conv_kernel<LL>), dim3(unsigned((c.lines + per - 1) / per), unsigned((images + NB - 1) / NB)),
                       dim3(256), 0, st, c);
  });
  if (!ok) return LX_OK;
  *taken = 1;
  return launched("conv (shared spectrum)");
}

int lx_plane_adj(const LxPlaneAdj& c, int D, int H, int W, int64_t B, bool bridge, hipStream_t st) {
  PlaneTables tb;
  if (int rc = plane_tables_of(H, W, st, &tb)) return rc;
  PlaneAdj a;
  a.X = c.X; a.U = c.U; a.lam = c.lam; a.A = c.A; a.part = c.part; a.gf = c.gf; a.w = c.w; a.dt = c.dt;
  a.gf_bs = c.gf_bs; a.w_bs = c.w_bs; a.dt_bs = c.dt_bs;
  a.D = D; a.kind = c.kind; a.average = c.average; a.accumulate = c.accumulate;
  a.mode = c.state_fn == LX_STATE_V2 ? 2 : (c.state_fn == LX_STATE_V1 && !c.ste ? 1 : 0);
  int rc = LX_OK;
  by_plane(H, W, [&](auto h, auto w) {
    constexpr int HH = decltype(h)::value, WW = decltype(w)::value;
    constexpr size_t lds = plane_lds(HH, WW);
    if ((rc = allow_lds(bridge ? plane_adj_kernel<HH, WW, true> : plane_adj_kernel<HH, WW, false>, lds))) return;
    const dim3 grid{unsigned(B * D)}, block(plane_threads(HH, WW));
    if (bridge) hipLaunchKernelGGL((plane_adj_kernel<HH, WW, true>), grid, block, lds, st, a, tb);
    else hipLaunchKernelGGL((plane_adj_kernel<HH, WW, false>), grid, block, lds, st, a, tb);
    rc = launched("plane reverse");
  });
  return rc;
}
