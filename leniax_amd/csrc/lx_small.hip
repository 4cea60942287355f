// The passes of a few worlds.  With a world or a few in flight a pass has fewer waves than the chip has
// SIMDs and its time is a chain of waits: arguments, parameters, rows, twiddles, one after the other, each
// most of a microsecond when another XCD wrote it, and then the kernels of a channel in turn.  These
// variants (the same arithmetic in the same order as lx_fft.hip's, bit for bit)
//  * give every kernel a lane group of its own, also where that repeats a channel's forward line transform;
//  * take compact arguments, all loaded at once (an argument block of several cache lines, read where it
//    is needed, costs a wait per line), and issue every load, twiddles and parameters included, before
//    the first transform waits;
//  * use workgroups of one wave (lines) or one row pair's kernels (rows), spread over the CUs.
#include <stdint.h>
#include <algorithm>

#include "lx_pass.h"

namespace {

// A lane group's transform with the lane's twiddles in registers (LDS exchange) or from the table.
template <int L, bool STRIDED = false>
struct GroupFft {
  using LC = Lanes<L>;
  static constexpr int TPR = LC::TPR, P = LC::P;
  float2 w[LC::XL ? P : 1];
  const float2* table;
  LX_DEV void load(const float2* tw, const float2* twl, int t) {
    table = tw;
    if constexpr (LC::XL) {
      const float4* row = reinterpret_cast<const float4*>(twl + t * twl_row(P));
#pragma unroll
      for (int k = 0; k < P; k += 2) {
        const float4 v = row[k / 2];
        w[k] = make_float2(v.x, v.y);
        w[k + 1] = make_float2(v.z, v.w);
      }
    }
  }
  template <bool INV>
  LX_DEV void run(float2* x, int t, int lane, float2* xch) const {
    if constexpr (LC::XL) {
      fft_xlds_mul<P, TPR, INV>(x, t, [&](float2* y) {
#pragma unroll
        for (int k = 1; k < P; ++k) y[k] = INV ? cmulc(y[k], w[k]) : cmul(y[k], w[k]);
      }, xch);
    } else if constexpr (STRIDED) {
      fft_strided<P, TPR, INV>(x, t, lane, table);
    } else {
      fft_lanes<P, TPR, INV>(x, t, lane, table);
    }
  }
};

// An argument the compiler must hold in scalar registers here: pinned together at a kernel's start, they
// arrive in one round of loads.
template <typename T>
LX_DEV void pin(T v) {
  __asm__ volatile("" ::"s"(v));
}

struct SmallConv {
  const float2* S;
  float2* U;
  const float2* Kh;
  const float2* tw;
  const float2* twl;
  float2* FA;  // spectra to keep (one channel and kernel)
  int64_t k_bstride, k_elems, img_elems;
  uint64_t cins;  // 4 bits per kernel: the channel it reads
  int total, per_img, WH, a_stride, st, C, K;  // total, per_img: lines of the K images of all worlds, of one
  float csign;                                 // -1: multiply by conj(K)
  const int32_t* list;                         // LIST
  const int32_t* nlive;
  // GRAD: dspec[b][k] += X_k conj(FAin[b][channel of k]) (C_fa channels, 4 bits per kernel)
  const float2* FAin;
  float2* dspec;
  uint64_t fa_cins;
  int C_fa;
};

// One wave of a few worlds' convolution pass: lane group = (kernel, line).  GRAD: with the kernel-spectrum
// gradient of a reverse step, its operands loaded before the transform as well.
template <int L, bool LIST, bool KQ, bool GRAD = false>
__global__ __launch_bounds__(64) void small_conv_kernel(SmallConv a) {
  using LC = Lanes<L>;
  constexpr int TPR = LC::TPR, P = LC::P, NG = 64 / TPR;
  using SG = Strided<TPR>;
  __shared__ __align__(16) float2 xch_all[LC::XL ? NG * strided_scratch<L, TPR>() : 2];
  pin(a.S); pin(a.U); pin(a.Kh); pin(a.tw); pin(a.twl); pin(a.FA); pin(a.k_bstride); pin(a.k_elems); pin(a.img_elems);
  pin(a.cins); pin(a.total); pin(a.per_img); pin(a.WH); pin(a.a_stride); pin(a.st); pin(a.C); pin(a.K); pin(a.csign);
  if constexpr (GRAD) {
    pin(a.FAin); pin(a.dspec); pin(a.fa_cins); pin(a.C_fa);
  }
  const int lane = threadIdx.x, t = SG::point(lane);
  float2* xch = xch_all + (LC::XL ? SG::line(lane) * strided_scratch<L, TPR>() : 0);
  const int lid = int(blockIdx.x) * NG + SG::line(lane);
  int total = a.total;
  if constexpr (LIST) {
    total *= *a.nlive;  // total: of one slot's world
    if (int(blockIdx.x) * NG >= total) return;
  }
  const bool live = lid < total;
  const int img = live ? lid / a.per_img : 0;  // image of U
  const int rem = live ? lid - img * a.per_img : 0;
  const int aa = rem / a.WH;
  const int off = aa * a.a_stride + (rem - aa * a.WH);
  const int b = img / a.K, k = img - b * a.K;
  const int cin = int(a.cins >> (4 * k)) & 15;
  const int64_t bw = LIST ? a.list[b] : b;
  const int st = a.st;
  const float2* src = a.S + int64_t(b * a.C + cin) * a.img_elems + off;
  const int64_t kb = bw * a.k_bstride + int64_t(k) * a.k_elems + off;
  float2 x[P], kv[P];
#pragma unroll
  for (int m = 0; m < P; ++m) x[m] = src[(TPR * m + t) * st];
  GroupFft<L, true> fft;
  fft.load(a.tw, a.twl, t);
  if constexpr (KQ) {
    const float* kq = reinterpret_cast<const float*>(a.Kh) + kb;
#pragma unroll
    for (int e = 0; e < P; ++e) {
      const int f = freq_of<L>(t, e);
      kv[e] = make_float2(kq[(f <= L / 2 ? f : L - f) * st], 0.f);
    }
  } else {
    const float2* kk = a.Kh + kb;
#pragma unroll
    for (int e = 0; e < P; ++e) kv[e] = kk[freq_of<L>(t, e) * st];
  }
  float2 fv[GRAD ? P : 1], dv[GRAD ? P : 1];
  float2* ds = nullptr;
  if constexpr (GRAD) {
    const float2* fa = a.FAin + int64_t(b * a.C_fa + (int(a.fa_cins >> (4 * k)) & 15)) * a.img_elems + off;
    ds = a.dspec + int64_t(img) * a.img_elems + off;
#pragma unroll
    for (int e = 0; e < P; ++e) {
      fv[e] = fa[freq_of<L>(t, e) * st];
      dv[e] = ds[freq_of<L>(t, e) * st];
    }
  }
  __builtin_amdgcn_sched_barrier(0);  // every load is issued here
  fft.template run<false>(x, t, lane, xch);
  if (a.FA && live) {
    float2* fa = a.FA + int64_t(img) * a.img_elems + off;
#pragma unroll
    for (int e = 0; e < P; ++e) fa[freq_of<L>(t, e) * st] = x[e];
  }
#pragma unroll
  for (int e = 0; e < P; ++e) {
    if constexpr (GRAD) {
      if (live) ds[freq_of<L>(t, e) * st] = cadd(dv[e], cmulc(x[e], fv[e]));
    }
    x[e] = cmul(x[e], make_float2(kv[e].x, a.csign * kv[e].y));
  }
  wave_lds_fence();
  fft.template run<true>(x, t, lane, xch);
  float2* dst = a.U + int64_t(img) * a.img_elems + off;
  if (live) {
#pragma unroll
    for (int m = 0; m < P; ++m) dst[(TPR * m + t) * st] = x[m];
  }
}

constexpr int kSmallItems = 4;  // four-point items of a thread: 4 channels of 512 points

struct SmallRows {
  const float2* U;
  const float* A;
  float* A_out;
  float* field;
  float* pot;
  const float* gf;
  const float* w;
  const float* dt;
  const float2* tw;
  const float2* twl;
  uint64_t kinds, cins;  // 4 bits per kernel: its growth function, the channel it reads
  int gf_bs, w_bs, dt_bs;
  float dt_val;
  int npairs, half_rows, C, K, RP;  // npairs: row pairs of all worlds (LIST: of one slot's)
  int state_fn, average, update, sel, fin_blocks;
  LxAdjFinish fin;
  // statistics, LIST
  float* part;
  const char* carry;
  int carry_bytes;
  int ndim, d0, d1;
  RunView rv;
  float* cells_hist;
  int64_t hist_B;
};

// g for four points of one kernel
template <int KIND>
LX_DEV void grow4(float4& u, const float4& par) {
  u.x = growth_pre<KIND>(par.x, par.y, par.z, par.w, u.x);
  u.y = growth_pre<KIND>(par.x, par.y, par.z, par.w, u.y);
  u.z = growth_pre<KIND>(par.x, par.y, par.z, par.w, u.z);
  u.w = growth_pre<KIND>(par.x, par.y, par.z, par.w, u.w);
}

// A few worlds' inverse row pass.  A workgroup holds RP row pairs of worlds.  First K lane groups per pair
// transform one kernel's two rows each and leave the potentials in LDS; after the barrier all 256 threads
// take four neighbouring points each: the potential's store, the kernels' growth summed in order, the
// update (16-byte loads and stores).  With statistics the points' state and field go through LDS to the
// lanes that sum the pair's record in the order of the pass for many worlds.
template <int W, bool STATS, bool LIST>
__global__ __launch_bounds__(256) void small_rows_kernel(SmallRows a) {
  using LC = Lanes<W>;
  constexpr int TPR = LC::TPR, P = LC::P, WH = W / 2 + 1, GRS = TPR * LC::XRS, NI = (WH + TPR - 1) / TPR;
  constexpr int Q = W / 4, IT = kSmallItems;  // quads of a row; items of a thread
  extern __shared__ __align__(16) float lds[];
  pin(a.U); pin(a.A); pin(a.A_out); pin(a.field); pin(a.pot); pin(a.gf); pin(a.w); pin(a.dt); pin(a.tw); pin(a.twl);
  pin(a.kinds); pin(a.cins); pin(a.gf_bs); pin(a.w_bs); pin(a.dt_bs); pin(a.dt_val); pin(a.npairs); pin(a.half_rows); pin(a.C);
  pin(a.K); pin(a.RP); pin(a.state_fn); pin(a.average); pin(a.update); pin(a.sel); pin(a.fin_blocks);
  const int tid = threadIdx.x, lane = tid & 63, t = tid % TPR, gi = tid / TPR;
  const int C = a.C, K = a.K, RP = a.RP;
  if constexpr (!STATS && !LIST) {
    const int first = int(gridDim.x) - a.fin_blocks;
    if (int(blockIdx.x) >= first) {
      const int64_t i = int64_t(int(blockIdx.x) - first) * 4 + (tid >> 6);
      if (i < lx_adj_finish_outputs(a.fin)) lx_adj_finish_wave(a.fin, i);
      return;
    }
  }
  const int groups = RP * K, rows = a.half_rows * 2, wp0 = int(blockIdx.x) * RP;
  int npairs = a.npairs;
  if constexpr (LIST) {
    npairs *= *a.rv.nlive;
    if (wp0 >= npairs) return;
  }
  float4* par = reinterpret_cast<float4*>(lds);               // [RP][K] growth parameters
  float2* xch_all = reinterpret_cast<float2*>(par + groups);  // [RP][K] exchange rows, then potentials
  float* wl = reinterpret_cast<float*>(xch_all + groups * GRS);  // [RP][C][K]
  float* counts = wl + RP * C * K;                               // [RP][K]
  float* vg = counts + ((groups + RP * C * K + 3) & ~3) - RP * C * K;  // STATS: [RP][C][2 rows][state, field][W]
  // the world (LIST: slot) and first row of the block's pair q (pairs past the last: the first world's)
  // (a single world, and below a single pair, take no division: its 30 instructions at one wave's issue rate
  // stood before the loads several times.  With the taken kernels' bits below, for one world: 13.8 -> 12.2 us
  // with statistics at 256^2, 3 channels, 6 kernels, 9.6 -> 7.9 at 128^2, 3 channels, 15 kernels)
  auto world = [&](int q, int64_t& r2) {
    const int wp = wp0 + q;
    int b = 0;
    if (npairs > a.half_rows) b = wp < npairs ? wp / a.half_rows : 0;
    r2 = wp < npairs ? (wp - b * a.half_rows) * 2 : 0;
    return b;
  };
  auto pair_of = [&](int i, int per) { return RP > 1 ? i / per : 0; };
  auto params_of = [&](int b) { return LIST ? int64_t(a.rv.list[b]) : int64_t(b); };
  // ---- every load first: the groups' rows and twiddles, parameters, the state of the thread's points
  const bool mine = gi < groups;
  const int gp = mine ? pair_of(gi, K) : 0, gk = mine ? gi - gp * K : 0;
  float2 p0[NI], p1[NI];
  GroupFft<W> fft;
  if (mine) {
    int64_t r2;
    const int b = world(gp, r2);
    const float2* u0 = a.U + (int64_t(b * K + gk) * rows + r2) * WH;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int col = min(t + TPR * i, WH - 1);
      p0[i] = u0[col];
      p1[i] = u0[WH + col];
    }
    fft.load(a.tw, a.twl, t);
  }
  float wreg = 0.f, gm = 0.f, gs = 1.f;
  if (a.update && !a.sel) {
    if (tid < RP * C * K) {
      const int q = pair_of(tid, C * K);
      int64_t r2;
      wreg = a.w[params_of(world(q, r2)) * a.w_bs + (tid - q * C * K)];
    }
    if (tid < groups) {
      const int q = pair_of(tid, K);
      int64_t r2;
      const float* g = a.gf + params_of(world(q, r2)) * a.gf_bs + 2 * (tid - q * K);
      gm = g[0];
      gs = g[1];
    }
  }
  const int items = RP * C * 2 * Q;
  float4 v[IT];
  float dtw[IT];
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int item = tid + 256 * it;
    dtw[it] = 1.f;
    if (a.update && item < items) {
      const int pc = item / (2 * Q), q = pair_of(pc, C), c = pc - q * C;
      int64_t r2;
      const int b = world(q, r2);
      const int64_t bw = params_of(b);
      const int64_t in_world = (int64_t(c) * rows + r2 + (item / Q & 1)) * W + item % Q * 4;
      const float* src = LIST ? run_state(a.rv, bw, false) + in_world : a.A + int64_t(b) * C * rows * W + in_world;
      v[it] = *reinterpret_cast<const float4*>(src);
      if (!a.sel) dtw[it] = a.dt ? a.dt[bw * a.dt_bs] : a.dt_val;
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // ---- transforms
  if (mine) {
    float2* xch = xch_all + gi * GRS;
    // the pair's rows, repacked as one complex row: Z[k] = A[k] + i B[k], A[k] = conj(A[W-k]) above W/2
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      const int col = t + TPR * i;
      if (col < WH) {
        xch[col] = p0[i];
        xch[WH + col] = p1[i];
      }
    }
    wave_lds_fence();
    float2 x[P];
#pragma unroll
    for (int e = 0; e < P; ++e) {
      const int f = freq_of<W>(t, e);
      const bool mirror = f >= W / 2;
      const float sg = mirror ? -1.f : 1.f;
      const int col = mirror ? W - f : f;
      const float2 ya = xch[col], yb = xch[WH + col];
      float2 z = make_float2(fmaf(-sg, yb.y, ya.x), fmaf(sg, ya.y, yb.x));
      if (f == 0 || f == W / 2) z = make_float2(ya.x, yb.x);
      x[e] = z;
    }
    wave_lds_fence();
    fft.template run<true>(x, t, lane, xch);
    wave_lds_fence();
    const float inv_n = 1.f / float(int64_t(rows) * W);
    float* u = reinterpret_cast<float*>(xch);  // the two rows of potentials
    float nU = 0.f;
#pragma unroll
    for (int m = 0; m < P; ++m) {
      const float U0 = x[m].x * inv_n, U1 = x[m].y * inv_n;
      u[TPR * m + t] = U0;
      u[W + TPR * m + t] = U1;
      if (STATS) nU += (U0 > LX_EPS ? 1.f : 0.f) + (U1 > LX_EPS ? 1.f : 0.f);
    }
    if constexpr (STATS) {  // counts of cells: exact in float32 whatever the order
#pragma unroll
      for (int off = TPR / 2; off >= 1; off >>= 1) nU += __shfl_xor(nU, off, 64);
      if (t == 0) counts[gi] = nU;
    }
  }
  if (a.update && !a.sel) {
    if (tid < RP * C * K) wl[tid] = wreg;
    if (tid < groups) par[tid] = make_float4(gm, gs, 1.f / gs, 1.f / (9.f * (gs * gs)));
  }
  __syncthreads();
  const float* pots = reinterpret_cast<const float*>(xch_all);
  // ---- the potentials
  if (a.pot) {
    for (int item = tid; item < groups * 2 * Q; item += 256) {
      const int pk = item / (2 * Q), q = pair_of(pk, K), k = pk - q * K, r = item / Q & 1, col = item % Q * 4;
      if (wp0 + q >= npairs) continue;
      int64_t r2;
      const int b = world(q, r2);
      int64_t img = int64_t(b) * K + k;
      if constexpr (LIST) {
        const int64_t bw = a.rv.list[b];
        img = (int64_t(a.rv.carry[bw].t) * a.hist_B + bw) * K + k;
      }
      *reinterpret_cast<float4*>(a.pot + (img * rows + r2 + r) * W + col) =
          *reinterpret_cast<const float4*>(pots + pk * (2 * GRS) + r * W + col);
    }
  }
  if (!a.update) return;
  // ---- growth, weighted sum, update
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int item = tid + 256 * it;
    if (item >= items) break;
    const int pc = item / (2 * Q), q = pair_of(pc, C), c = pc - q * C, r = item / Q & 1, col = item % Q * 4;
    if (wp0 + q >= npairs) continue;
    const float* w = wl + pc * K;
    float4 G = make_float4(0.f, 0.f, 0.f, 0.f);
    float den = 0.f;
    // the kernels with a weight here, and in channel 0 those that no channel takes (they count, times 0, where
    // their potential is wanted): the weights' LDS reads overlap, where a test per kernel waited for each
    uint32_t take = 0;
    if (a.sel) {
      for (int k = 0; k < K; ++k) take |= uint32_t((int(a.cins >> (4 * k)) & 15) == c) << k;
    } else {
#pragma unroll 4
      for (int k = 0; k < K; ++k) take |= uint32_t(w[k] != 0.f) << k;
      if (c == 0 && (STATS || a.pot)) {
        uint32_t any = take;
        for (int cc = 1; cc < C; ++cc)
#pragma unroll 4
          for (int k = 0; k < K; ++k) any |= uint32_t(w[cc * K + k] != 0.f) << k;
        take |= ~any & ((1u << K) - 1u);
      }
    }
    for (; take; take &= take - 1) {
      const int k = __builtin_ctz(take);
      const float wk = a.sel ? 1.f : w[k];
      den = add_nc(den, wk);
      float4 g = *reinterpret_cast<const float4*>(pots + (q * K + k) * (2 * GRS) + r * W + col);
      if (!a.sel) {
        const float4 pk = par[q * K + k];
        switch (int(a.kinds >> (4 * k)) & 15) {
          case LX_GF_POLY_QUAD4: grow4<LX_GF_POLY_QUAD4>(g, pk); break;
          case LX_GF_GAUSSIAN: grow4<LX_GF_GAUSSIAN>(g, pk); break;
          case LX_GF_GAUSSIAN_TARGET: grow4<LX_GF_GAUSSIAN_TARGET>(g, pk); break;
          case LX_GF_STEP: grow4<LX_GF_STEP>(g, pk); break;
          case LX_GF_STAIRCASE: grow4<LX_GF_STAIRCASE>(g, pk); break;
          case LX_GF_TRIANGLE: grow4<LX_GF_TRIANGLE>(g, pk); break;
          default: break;
        }
      }
      G.x = add_nc(G.x, mul_nc(wk, g.x));
      G.y = add_nc(G.y, mul_nc(wk, g.y));
      G.z = add_nc(G.z, mul_nc(wk, g.z));
      G.w = add_nc(G.w, mul_nc(wk, g.w));
    }
    if (a.average) G = make_float4(G.x / den, G.y / den, G.z / den, G.w / den);
    int64_t r2;
    const int b = world(q, r2);
    const int64_t in_world = (int64_t(c) * rows + r2 + r) * W + col;
    float* out;
    float* fld = a.field;
    if constexpr (LIST) {
      const int64_t bw = a.rv.list[b];
      out = run_state(a.rv, bw, true) + in_world;
      const int64_t h = (int64_t(a.rv.carry[bw].t) * a.hist_B + bw) * a.rv.world_elems + in_world;
      if (fld) fld += h;
      if (a.cells_hist) *reinterpret_cast<float4*>(a.cells_hist + h) = v[it];
    } else {
      const int64_t o = int64_t(b) * C * rows * W + in_world;
      out = a.A_out + o;
      if (fld) fld += o;
    }
    if (fld) *reinterpret_cast<float4*>(fld) = G;
    if constexpr (STATS) {
      *reinterpret_cast<float4*>(vg + ((pc * 2 + r) * 2) * W + col) = v[it];
      *reinterpret_cast<float4*>(vg + ((pc * 2 + r) * 2 + 1) * W + col) = G;
    }
    *reinterpret_cast<float4*>(out) =
        make_float4(step_value(a.state_fn, v[it].x, G.x, dtw[it]), step_value(a.state_fn, v[it].y, G.y, dtw[it]),
                    step_value(a.state_fn, v[it].z, G.z, dtw[it]), step_value(a.state_fn, v[it].w, G.w, dtw[it]));
  }
  // ---- the pairs' records
  if constexpr (STATS) {
    __syncthreads();
    for (int pc = gi; pc < RP * C; pc += 256 / TPR) {
      const int q = pair_of(pc, C), c = pc - q * C;
      if (wp0 + q >= npairs) continue;
      int64_t r2;
      const int b = world(q, r2);
      int sh[3];
      pair_shift(LIST ? a.rv.carry[a.rv.list[b]] : *pair_carry(a.carry, a.carry_bytes, b), a.ndim, a.d0, a.d1, W, sh);
      const float* x = vg + pc * 4 * W;
      PairSums sums;
#pragma unroll
      for (int m = 0; m < P; ++m) {
        const int col = TPR * m + t;
        int zc = col - sh[2];
        zc += zc < 0 ? W : 0;
        sums.add(x[col], x[2 * W + col], x[W + col], x[3 * W + col], float(zc - W / 2));
      }
      float n = 0.f;
      if (c == 0 && t == 0)
#pragma unroll 4
        for (int k = 0; k < K; ++k) n += counts[q * K + k];
      pair_record<TPR>(sums, n, sh, r2, a.ndim, a.d0, a.d1, t,
                       a.part + (int64_t(b * C + c) * a.half_rows + (r2 >> 1)) * LX_PAIR_REC);
    }
  }
}

// LDS floats of small_rows_kernel for RP pairs
template <int W>
size_t small_rows_lds(int RP, int C, int K, bool stats) {
  using LC = Lanes<W>;
  const size_t g = size_t(RP) * K;
  return g * 4 + g * LC::TPR * LC::XRS * 2 + ((g + size_t(RP) * C * K + 3) & ~size_t(3)) +
         (stats ? size_t(RP) * C * 4 * W : 0);
}

int launched(const char* what) {
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? LX_OK : lx_fail(LX_EDEVICE, "%s launch: %s", what, hipGetErrorString(e));
}

template <typename F>
int by_length(int L, F&& f) {
  switch (L) {
    case 16: return f(IntC<16>{});
    case 32: return f(IntC<32>{});
    case 48: return f(IntC<48>{});
    case 64: return f(IntC<64>{});
    case 96: return f(IntC<96>{});
    case 128: return f(IntC<128>{});
    case 192: return f(IntC<192>{});
    case 256: return f(IntC<256>{});
    case 384: return f(IntC<384>{});
    case 512: return f(IntC<512>{});
    default: return lx_fail(LX_ENOTSUP, "transform length %d", L);
  }
}

// Waves up to which a pass counts as a few worlds': at most two per SIMD (4 SIMDs x 256 CUs).  The chip has
// idle issue slots for the repeated transforms and the barriers up to a number that falls with the points a
// lane holds and grows with the kernels per channel, which the general passes take in turn; measured (general
// time / these, kernels spread over the channels) at 150 to 2000 waves of the general pass:
//   inverse rows, 256 points: one kernel a channel 1.3 at 600, 0.95 at 1000; two 1.2 at 1000, 1.1 at 1500; five
//     1.4 at 1000, 1.1 at 2000; 128 and 96 alike; 48 and 32 points above 1.1 throughout; 192: 1.0, 1.2 and 1.8
//     at 1000 (one, two, five); 384: 1.1, 1.7, 2.7 at 300 and 0.7, 0.9, 1.3 at 1000
//   convolution, 256 points: one kernel a channel 1.1 at 300 waves of its own, 0.9 at 600; two 1.2 at 1100;
//     five 1.5 at 1450; 128: 1.06 at 600, 0.92 at 1000; 64 and fewer above 1.05 to 1500; 512: 1.04 at 300, 0.9 at
//     600.
constexpr int64_t kSmallWaves = 2048;

int64_t small_conv_waves(int L, int C, int K) {
  const int tpr = lx_row_tpr(L);
  const int64_t one = tpr == 4 ? 2048 : tpr == 8 ? (L / tpr <= 16 ? 1024 : 512) : 384;
  return std::min(kSmallWaves, one * std::max(C, K) / C);
}

// of the general pass, whose channels' waves count.  With statistics half, and less of the shortest rows: the
// records are the work of a few lanes at the end of a workgroup (64 points, two kernels a channel, 1000 waves:
// 18.7 against 14.9 us; 96 points, one, 700 waves: 11.5 against 9.2).
int64_t small_rows_waves(int W, int C, int K, bool stats) {
  const int tpr = lx_row_tpr(W), each = std::min(C, K);
  const int64_t one = W <= 48 && !stats ? 2048 : W / tpr <= 16 ? 768 : tpr == 8 ? 512 : 256;
  return std::min(kSmallWaves, one * (each + K) / (2 * each)) / (stats ? 2 : 1);
}

}  // namespace

int lx_small_conv(const LineArgs& a, int L, int64_t lines, bool list, hipStream_t st, int* taken) {
  *taken = 0;
  // spectra to keep are the single kernel's group's to write
  if (a.mode != 0 || (a.FA && !(a.C == 1 && a.K == 1)) || (a.dspec && (a.FA || a.kquad || list))) return LX_OK;
  const int64_t groups = lines / a.C * a.K, per = 64 / lx_row_tpr(L);
  if ((groups + per - 1) / per > small_conv_waves(L, a.C, a.K)) return LX_OK;
  LxPassTables tb;
  if (int rc = lx_pass_tables(L, st, &tb)) return rc;
  SmallConv c;
  c.S = a.S; c.U = a.U; c.Kh = a.Kh; c.tw = tb.tw; c.twl = tb.twl; c.FA = a.FA;
  c.k_bstride = a.k_bstride; c.k_elems = a.k_elems; c.img_elems = a.img_elems;
  c.cins = c.fa_cins = 0;
  for (int k = 0; k < a.K; ++k) {
    c.cins |= uint64_t(a.cin[k] & 15) << (4 * k);
    c.fa_cins |= uint64_t(a.acc_cin[k] & 15) << (4 * k);
  }
  c.FAin = a.FAin; c.dspec = a.dspec; c.C_fa = a.C_fa;
  c.total = int(a.nlines / a.C * a.K); c.per_img = a.A * a.WH; c.WH = a.WH; c.a_stride = int(a.a_stride); c.st = int(a.st);
  c.C = a.C; c.K = a.K; c.csign = a.conjk ? -1.f : 1.f; c.list = a.list; c.nlive = a.nlive;
  *taken = 1;
  const dim3 grid(unsigned((groups + per - 1) / per));
  return by_length(L, [&](auto l) {
    constexpr int LL = decltype(l)::value;
    if (a.dspec) hipLaunchKernelGGL((small_conv_kernel<LL, false, false, true>), grid, dim3(64), 0, st, c);
    else if (list && a.kquad) hipLaunchKernelGGL((small_conv_kernel<LL, true, true>), grid, dim3(64), 0, st, c);
    else if (list) hipLaunchKernelGGL((small_conv_kernel<LL, true, false>), grid, dim3(64), 0, st, c);
    else if (a.kquad) hipLaunchKernelGGL((small_conv_kernel<LL, false, true>), grid, dim3(64), 0, st, c);
    else hipLaunchKernelGGL((small_conv_kernel<LL, false, false>), grid, dim3(64), 0, st, c);
    return launched("conv (few worlds)");
  });
}

int lx_small_rows(const RowArgs& a, int W, int64_t images, bool list, hipStream_t st, int* taken) {
  *taken = 0;
  const int tpr = lx_row_tpr(W), K = a.K, C = a.C;
  const int64_t pairs = images / C * (a.rows / 2);
  if (pairs * std::min(C, K) * tpr > small_rows_waves(W, C, K, a.part != nullptr) * 64) return LX_OK;
  if (std::max({a.gf_bs, a.w_bs, a.dt_bs}) > INT32_MAX) return LX_OK;
  // 16-byte accesses: states, fields and potentials start on 16 bytes (rows are multiples of 4 floats)
  const auto wide = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (!wide(a.A) || !wide(a.A_out) || !wide(a.field) || !wide(a.pot) || !wide(a.cells_hist) ||
      (list && !(wide(a.rv.X0) && wide(a.rv.X1))))
    return LX_OK;
  // row pairs per workgroup: one item per thread where a pair has fewer than 256 (C W / 2), two where the
  // grid has workgroups to spare, at most 256 lanes of transforms
  const int RP = std::max(1, std::min((pairs > 1024 ? 1024 : 512) / (C * W), 256 / (K * tpr)));
  SmallRows r;
  r.U = a.U; r.A = a.A; r.A_out = a.A_out; r.field = a.field; r.pot = a.pot; r.gf = a.gf; r.w = a.w; r.dt = a.dt;
  r.kinds = r.cins = 0;
  for (int k = 0; k < K; ++k) {
    r.kinds |= uint64_t(a.gfk[k] & 15) << (4 * k);
    r.cins |= uint64_t(a.cin[k] & 15) << (4 * k);
  }
  r.gf_bs = int(a.gf_bs); r.w_bs = int(a.w_bs); r.dt_bs = int(a.dt_bs); r.dt_val = a.dt_val;
  r.npairs = int(a.npairs / C); r.half_rows = int(a.rows / 2); r.C = C; r.K = K; r.RP = RP;
  r.state_fn = a.state_fn; r.average = a.average; r.update = a.update; r.sel = a.sel;
  r.fin = a.fin; r.fin_blocks = 0;
  r.part = a.part; r.carry = a.carry; r.carry_bytes = a.carry_bytes; r.ndim = a.ndim; r.d0 = a.d0; r.d1 = a.d1; r.rv = a.rv;
  r.cells_hist = a.cells_hist; r.hist_B = a.hist_B;
  if (a.fin.blocks) {  // one wave per gradient element
    const int64_t nout = (a.fin.g_gf ? (a.fin.gf_bs ? a.fin.B : 1) * 2 : 0) +
                         (a.fin.g_w ? (a.fin.w_bs ? a.fin.B : 1) : 0) + (a.fin.g_dt ? (a.fin.dt_bs ? a.fin.B : 1) : 0);
    r.fin_blocks = int((nout + 3) / 4);
  }
  return by_length(W, [&](auto w) {
    constexpr int WW = decltype(w)::value;
    const size_t lds = small_rows_lds<WW>(RP, C, K, a.part != nullptr) * sizeof(float);
    if (lds > 65536) return int(LX_OK);
    LxPassTables tb;
    if (int rc = lx_pass_tables(WW, st, &tb)) return rc;
    r.tw = tb.tw; r.twl = tb.twl;
    *taken = 1;
    const dim3 grid(unsigned((pairs + RP - 1) / RP) + unsigned(r.fin_blocks));
    if (a.part) {
      if (list) hipLaunchKernelGGL((small_rows_kernel<WW, true, true>), grid, dim3(256), lds, st, r);
      else hipLaunchKernelGGL((small_rows_kernel<WW, true, false>), grid, dim3(256), lds, st, r);
    } else {
      hipLaunchKernelGGL((small_rows_kernel<WW, false, false>), grid, dim3(256), lds, st, r);
    }
    return launched("rows (few worlds)");
  });
}
