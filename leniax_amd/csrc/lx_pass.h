// What the kernels of the multi-pass step share (lx_fft.hip: the passes; lx_small.hip: their variants for a
// few worlds): how a transform is spread over lanes, the arguments of the passes, the tables.
#pragma once
#include <type_traits>

#include "lx_internal.h"

namespace lx_pass {

// lanes per transform of the row passes: 8 from 96 points up (96 = 8 lanes x 12 points through
// the DPP network rather than 4 x 24 through LDS: half the registers of rows_inv, 3 waves per
// SIMD instead of 2)
constexpr int row_tpr(int L) { return L <= 64 ? 4 : (L <= 192 ? 8 : 16); }
// lanes per transform of the line passes: as the rows, except the plain forward and inverse
// passes (modes 1 and 2) at 96 points, which take 4 x 24 through LDS, as the columns of the plane
// kernels do (a step's bits are then the same either way).  The strided groups below bound both
// forms by memory: 16 worlds of 96^3 22.3 and 23.4 us forward and inverse (101 and 113 VGPRs)
// against 21.7 and 22.1 on 8 lanes (59 and 65); the convolution pass takes 114 VGPRs on 8 lanes, 173 on 4
constexpr int line_tpr(int L, int mode) { return L == 96 && mode != 0 ? 4 : row_tpr(L); }

template <int L, int T = row_tpr(L)>
struct Lanes {
  static constexpr int TPR = T;
  static constexpr int P = L / TPR;                                // points per lane
  static constexpr bool XL = P % TPR == 0;                         // cross-lane step through LDS
  static constexpr int XRS = xch_row(P);                           // group scratch row stride
  static constexpr int XCH = 256 * XRS;                            // scratch of a 256-thread block
  static_assert(TPR == 4 || TPR == 8 || TPR == 16, "lane groups of 4, 8 or 16");
  static_assert(TPR * XRS >= L + 2, "a group's scratch holds one transform plus two");
};

template <int V>
using IntC = std::integral_constant<int, V>;

// Frequency held by register e of lane t after a forward group transform: with the LDS
// exchange e = j TPR + k2 holds (J t + j) + P k2; with the DPP network e holds e + P bitrev(t).
template <int L, int T = row_tpr(L)>
LX_DEV int freq_of(int t, int e) {
  using LC = Lanes<L, T>;
  if constexpr (LC::XL) {
    constexpr int J = LC::P / LC::TPR;
    return J * t + e / LC::TPR + LC::P * (e % LC::TPR);
  } else {
    return e + LC::P * bitrev_n(t, LC::TPR);
  }
}

// Lane groups of the line passes.  Neighbouring lines are neighbouring complex elements of a half-spectrum
// row, and the texture unit takes a wave's addresses four neighbouring lanes at a time: four lanes of one
// group (rows far apart) cost it four requests of 8 bytes, four lanes of four groups one of 32.  So lane l
// of a wave holds point t = l / G of line l % G, G = 64 / T lines per wave.  (With a group's lanes side by
// side the passes ran at one request per clock and CU, whatever their bytes: 16 worlds of 96^3, 7.2 M
// elements read and written, 25 us = 56 k requests per CU.  Strided: the convolution along D of 8 worlds of
// 96^3 29.5 -> 19.4 us.)
template <int T>
struct Strided {
  static constexpr int G = 64 / T;  // lines of a wave
  static LX_DEV int point(int lane) { return lane / G; }
  static LX_DEV int line(int lane) { return lane % G; }
};
// Exchange scratch of a strided group (complex): its rows padded so that the 16-byte accesses of 16
// consecutive lanes (16 / G points of G lines) lie in different banks.
template <int L, int T>
constexpr int strided_scratch() {
  return T * xch_row(L / T) + (T == 4 ? 2 : T == 8 ? 20 : 8);
}

// p + sgn v over the lanes D apart (p the partner's value; sgn +1 in the lower lane, -1 in the upper):
// 16 and 32 apart through the row and half swaps, which leave the lower lane's value in one register of
// both lanes and the upper's in the other.
template <int D>
LX_DEV float strided_pair(float v, float sgn, int lane) {
  if constexpr (D == 4 || D == 8) {
    return fmaf(sgn, v, xor_fetch<D>(v, lane));
  } else {
    const unsigned u = __builtin_bit_cast(unsigned, v);
    const auto r = D == 16 ? __builtin_amdgcn_permlane16_swap(u, u, false, false)
                           : __builtin_amdgcn_permlane32_swap(u, u, false, false);
    return fmaf(sgn, __builtin_bit_cast(float, unsigned(r[1])), __builtin_bit_cast(float, unsigned(r[0])));
  }
}

// lane_stage (lx_device.h) over strided groups: the same arithmetic
template <int P, int T, int L, bool INV, int H>
LX_DEV void strided_stage(float2* x, int t, int lane, const float2* tw) {
  using LT = LaneTwiddle<P, T, INV, H>;
  const float sgn = (t & H) != 0 ? -1.f : 1.f;
  const float2 w = LT::get(t, tw);
#pragma unroll
  for (int k = 0; k < P; ++k) {
    const float2 o = LT::ANY && LT::FIRST ? cmul(x[k], w) : x[k];
    const float2 v =
        make_float2(strided_pair<H * (64 / T)>(o.x, sgn, lane), strided_pair<H * (64 / T)>(o.y, sgn, lane));
    x[k] = LT::ANY && !LT::FIRST ? cmul(v, w) : v;
  }
}
template <int P, int T, int L, bool INV, int H>
LX_DEV void strided_network(float2* x, int t, int lane, const float2* tw) {
  if constexpr (INV ? H < T : H >= 1) {
    strided_stage<P, T, L, INV, H>(x, t, lane, tw);
    strided_network<P, T, L, INV, (INV ? H * 2 : H / 2)>(x, t, lane, tw);
  }
}
// fft_lanes over strided groups
template <int P, int T, bool INV>
LX_DEV void fft_strided(float2* x, int t, int lane, const float2* tw) {
  if constexpr (!INV) {
    fft_reg<P, false>(x);
    int j = 0;
#pragma unroll
    for (int k = 1; k < P; ++k) {
      j += t;
      x[k] = cmul(x[k], tw[j]);
    }
    strided_network<P, T, T * P, false, T / 2>(x, t, lane, tw);
  } else {
    strided_network<P, T, T * P, true, 1>(x, t, lane, tw);
    int j = 0;
#pragma unroll
    for (int k = 1; k < P; ++k) {
      j += t;
      x[k] = cmulc(x[k], tw[j]);
    }
    fft_reg<P, true>(x);
  }
}

LX_DEV void wave_lds_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); }

// ---------------------------------------------------------------- batched-run indirection
// The kernels of lx_run's multi-pass path (LIST = true) step the worlds of a live list: slot s of
// the list holds world list[s], slots >= *nlive are empty.  The per-step temporaries (spectra S,
// U, the row-pair records) are indexed by slot; what persists (the state, carry, parameters,
// spectra, statistics) by world.  World b's state after t of its steps lives in X0 (t even) or X1
// (t odd), t = carry[b].t: worlds advance in lockstep inside a step but start at different steps.
struct RunView {
  const int32_t* list;
  const int32_t* nlive;
  const lx_carry* carry;
  float* X0;
  float* X1;
  int64_t world_elems;  // C * cells floats per world
};

// the state buffer holding world b's current state
LX_DEV float* run_state(const RunView& v, int64_t b, bool next) {
  const bool odd = ((v.carry[b].t & 1) != 0) != next;
  return (odd ? v.X1 : v.X0) + b * v.world_elems;
}

// ---------------------------------------------------------------- pass arguments
struct LineArgs {
  const float2* S;
  float2* U;
  const float2* Kh;
  int64_t k_bstride;
  int64_t nlines;      // images * A * WH
  int WH, A;
  int64_t a_stride, st, img_elems;
  int C, K;            // images per world (channels) and kernels (mode 0)
  int cin[LX_MAX_K];   // mode 0: kernel k reads channel cin[k]
  int mode;            // 0: conv, 1: forward in place, 2: inverse S -> U
  int conjk;           // mode 0: multiply by conj(K) (adjoint of the potential)
  // mode 0: Kh holds real quadrants (float [world][K][L/2 + 1][WH], 2-D): the spectrum of kernel
  // k at frequency f of a line is the real value at row min(f, L - f); k_elems: the elements (float2,
  // or float for quadrants) of one kernel's spectrum
  int kquad;
  int64_t k_elems;
  // mode 0, optional: the forward spectra of the input images, FA [img][half]
  float2* FA;
  // mode 0, optional: dspec[b][k] += X_k * conj(FAin[b][acc_cin[k]]) (kernel-spectrum gradient)
  const float2* FAin;
  float2* dspec;
  int C_fa;
  int acc_cin[LX_MAX_K];
  // batched run (LIST kernels): nlines is the lines of one slot's slot_imgs images; the spectra
  // of a slot's lines are those of world list[slot]
  const int32_t* list;
  const int32_t* nlive;
  int xcd;  // blocks in XCD-contiguous order (xcd_block) or in launch order
};

inline LineArgs line_args() {
  LineArgs a;
  a.S = nullptr; a.U = nullptr; a.Kh = nullptr; a.k_bstride = 0; a.nlines = 0;
  a.WH = 0; a.A = 1; a.a_stride = 0; a.st = 0; a.img_elems = 0; a.C = 1; a.K = 0;
  for (int k = 0; k < LX_MAX_K; ++k) { a.cin[k] = -1; a.acc_cin[k] = 0; }
  a.mode = 0; a.conjk = 0; a.kquad = 0; a.k_elems = 0; a.FA = nullptr; a.FAin = nullptr; a.dspec = nullptr; a.C_fa = 1;
  a.list = nullptr; a.nlive = nullptr; a.xcd = 1;
  return a;
}

struct RowArgs {
  const float2* U;
  const float* A;
  float* A_out;
  float* field;
  float* pot;
  const float* gf;
  int64_t gf_bs;
  const float* w;
  int64_t w_bs;
  const float* dt;  // per world, or NULL: dt_val
  int64_t dt_bs;
  float dt_val;
  int64_t npairs;  // images * rows / 2
  int64_t rows;    // rows per image
  int C, K;
  int gfk[LX_MAX_K];
  int state_fn, average;
  int update;      // 0: potential only
  // selection mode: weight of kernel k in channel c is (cin[k] == c), growth is the identity and the
  // update is A_out = A + G (no gf / w / dt reads).  Used for the potential alone, the adjoint of the
  // potential (lambda += correlations) and the inverse real FFT.
  int sel;
  int cin[LX_MAX_K];
  // statistics mode: the step's world sums of leniax/statistics.py:35-126 over each row pair's
  // input state, field and potential, LX_PAIR_REC floats per pair at part[pair index] (sA, sG,
  // nA, nG, nU, sAy[3], sGy[3], sAyy[3]), in the re-centred coordinates of the carried shift
  float* part;
  const char* carry;  // world b's lx_carry at carry + b carry_bytes
  int carry_bytes;
  int ndim, d0, d1;  // rows = d0 d1 (d0 = 1 for 2-D worlds)
  // batched run (LIST kernels): npairs is the pairs of one slot; state from / to rv's buffers, the
  // carry is rv.carry; with hist_B > 0, field and pot (and cells_hist, when set) are the run's
  // histories [max_steps][hist_B][C or K][dims], written at the world's step
  RunView rv;
  float* cells_hist;
  int64_t hist_B;
  // the reverse step's gradient scalars, summed by fin.blocks workgroups after the row pairs' (not in
  // the statistics or LIST kernels)
  LxAdjFinish fin;
};

// ---------------------------------------------------------------- the update and the statistics of a row pair
// leniax's state functions (leniax/core.py:245-319), each operation rounded as leniax's
LX_DEV float step_value(int state_fn, float v, float g, float dt) {
  if (state_fn == LX_STATE_V2) return add_nc(mul_nc(v, sub_nc(1.f, dt)), mul_nc(dt, g));
  float n = add_nc(v, mul_nc(dt, g));
  if (state_fn == LX_STATE_V1) n = n < 0.f ? 0.f : (n > 1.f ? 1.f : n);
  return n;
}

// A lane's part of a row pair's world sums: per row sums of A, A z, A z^2, G+, G+ z (z the re-centred
// column) and counts.
struct PairSums {
  float sAr0 = 0.f, sAr1 = 0.f, sAz = 0.f, sAzz = 0.f, sGr0 = 0.f, sGr1 = 0.f, sGz = 0.f, nA = 0.f, nG = 0.f;
  LX_DEV void add(float v0, float v1, float g0, float g1, float cz) {
    const float gp0 = g0 != g0 ? g0 : fmaxf(g0, 0.f), gp1 = g1 != g1 ? g1 : fmaxf(g1, 0.f);
    sAr0 += v0;
    sAr1 += v1;
    const float vs = v0 + v1, gs2 = gp0 + gp1;
    sAz = fmaf(vs, cz, sAz);
    sAzz = fmaf(vs * cz, cz, sAzz);
    sGr0 += gp0;
    sGr1 += gp1;
    sGz = fmaf(gs2, cz, sGz);
    nA += (v0 > LX_EPS ? 1.f : 0.f) + (v1 > LX_EPS ? 1.f : 0.f);
    nG += (gp0 > LX_EPS ? 1.f : 0.f) + (gp1 > LX_EPS ? 1.f : 0.f);
  }
};

LX_DEV const lx_carry* pair_carry(const char* carry, int bytes, int64_t b) {
  return reinterpret_cast<const lx_carry*>(carry + b * bytes);
}

// the carried shift reduced into [0, size) along (d0, d1, W)
LX_DEV void pair_shift(const lx_carry& cc, int ndim, int d0, int d1, int W, int (&sh)[3]) {
  auto modp = [](int v, int m) { v %= m; return v < 0 ? v + m : v; };
  sh[0] = ndim == 3 ? modp(cc.shift[0], d0) : 0;
  sh[1] = modp(cc.shift[ndim - 2], d1);
  sh[2] = modp(cc.shift[ndim - 1], W);
}

// The pair's record (rows r2, r2 + 1): the lanes' sums added over the TPR lanes of the group (a
// butterfly: every lane ends with the same sums), stored by lane t as fields t, t + TPR, ...
template <int TPR>
LX_DEV void pair_record(const PairSums& s, float nU, const int (&sh)[3], int64_t r2, int ndim, int d0, int d1, int t,
                        float* dst) {
  // re-centred row coordinates of the pair's two rows: (x, y) in 3-D, y in 2-D
  float cx[2], cy[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = int(r2) + i;
    int x = row / d1, y = row - (row / d1) * d1;
    x -= sh[0]; x += x < 0 ? d0 : 0;
    y -= sh[1]; y += y < 0 ? d1 : 0;
    cx[i] = float(x - d0 / 2);
    cy[i] = float(y - d1 / 2);
  }
  const bool d3 = ndim == 3;
  float rec[LX_PAIR_REC];
  rec[0] = s.sAr0 + s.sAr1;
  rec[1] = s.sGr0 + s.sGr1;
  rec[2] = s.nA;
  rec[3] = s.nG;
  rec[4] = nU;
  const float ay = fmaf(s.sAr0, cy[0], s.sAr1 * cy[1]), ayy = fmaf(s.sAr0 * cy[0], cy[0], s.sAr1 * cy[1] * cy[1]);
  const float gy = fmaf(s.sGr0, cy[0], s.sGr1 * cy[1]);
  const float ax = fmaf(s.sAr0, cx[0], s.sAr1 * cx[1]), axx = fmaf(s.sAr0 * cx[0], cx[0], s.sAr1 * cx[1] * cx[1]);
  const float gx = fmaf(s.sGr0, cx[0], s.sGr1 * cx[1]);
  rec[5] = d3 ? ax : ay;     rec[6] = d3 ? ay : s.sAz;   rec[7] = d3 ? s.sAz : 0.f;
  rec[8] = d3 ? gx : gy;     rec[9] = d3 ? gy : s.sGz;   rec[10] = d3 ? s.sGz : 0.f;
  rec[11] = d3 ? axx : ayy;  rec[12] = d3 ? ayy : s.sAzz; rec[13] = d3 ? s.sAzz : 0.f;
  for (int i = 14; i < LX_PAIR_REC; ++i) rec[i] = 0.f;
#pragma unroll
  for (int off = TPR / 2; off >= 1; off >>= 1)
#pragma unroll
    for (int i = 0; i < 14; ++i) rec[i] += __shfl_xor(rec[i], off, 64);
#pragma unroll
  for (int e = 0; e < LX_PAIR_REC; ++e)
    if (e % TPR == t) dst[e] = rec[e];
}

}  // namespace lx_pass
using namespace lx_pass;

// Twiddle tables of length L on the current device (lx_fft.hip, built on first use, refused under a
// capture): exp(-2 pi i j / L), and the lane rows of row_tpr(L) lanes (twl_row(P) entries a row).
struct LxPassTables {
  const float2* tw;
  const float2* twl;
};
int lx_pass_tables(int L, hipStream_t st, LxPassTables* out);

// lx_small.hip: the passes of a few worlds.  Each returns LX_OK and sets *taken when its variant applies
// to the shape; with *taken = 0 nothing was launched and the pass is the caller's.
int lx_small_conv(const LineArgs& a, int L, int64_t lines, bool list, hipStream_t st, int* taken);
int lx_small_rows(const RowArgs& a, int W, int64_t images, bool list, hipStream_t st, int* taken);

// lx_plane.hip: the inner two axes of 3-D passes, one plane per workgroup (16-byte accesses: the caller's
// states, fields and potentials start on 16 bytes), and the convolution along the outer one for worlds
// that share a spectrum (*taken as above).
bool lx_plane_takes(int H, int W);
bool lx_plane_pays(int H, int W, int64_t planes, bool inverse);  // the planes are enough to fill the chip
bool lx_plane_pays_reverse(int D, int H, int W);
int lx_plane_fwd(int H, int W, const float* A, float2* S, int64_t planes, hipStream_t st);
int lx_plane_inv(const RowArgs& a, int D, int H, int W, int64_t images, hipStream_t st);
struct LxPlaneAdj {
  float2* X;
  const float* U;
  float* lam;
  const float* A;
  float* part;
  const float* gf;
  const float* w;
  const float* dt;
  int64_t gf_bs, w_bs, dt_bs;
  int kind, state_fn, ste, average, accumulate;
};
int lx_plane_adj(const LxPlaneAdj& c, int D, int H, int W, int64_t B, bool bridge, hipStream_t st);
int lx_shared_conv(const LineArgs& a, int L, int64_t images, hipStream_t st, int* taken);
