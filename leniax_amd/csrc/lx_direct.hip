// Direct-convolution potential (leniax/core.py:105-146 get_potential): the depthwise
// cross-correlation of the wrap-padded state with small real kernels, as
// jax.lax.conv_general_dilated(..., 'VALID', feature_group_count=C) computes it, with the
// padding of leniax/helpers.py:465-481 (before = size // 2 on every axis).
//
//   U[b][k][y][x] = sum_{i<kh, j<kw} A[b][cin k][(y + i - ph) mod H][(x + j - pw) mod W] * kern[k][i][j]
//
// The potential and its reverse are sums of products over a sliding window: contractions of the
// staged image with a Toeplitz matrix of the taps, taken on the matrix cores in float32
// (v_mfma_f32_4x4x1: 16 independent 4 x 4 outer products, 512 flop in about 9 cycles; the vector
// unit does as many in FMAs of registers, 2.2 cycles each, and half with a scalar operand, 4.1, as a
// tap is; what the matrix form saves are the operands: one LDS read of a lane feeds 16 products).
// Kernels of at most 5 columns stay on the vector unit.  Any world size; kernels up to 64 x 64.
#include <algorithm>
#include <type_traits>

#include "lx_internal.h"

namespace {

constexpr int MAXK = 64, TX = 64;  // largest kernel side; output columns of a workgroup
typedef float f4v __attribute__((ext_vector_type(4)));

// LDS row stride of at least `need` floats: 16 or 48 mod 64, so that the four rows of four 16-byte
// pieces that 16 lanes read at once lie in different banks
__host__ __device__ inline int bank_stride(int need) { return (need - 16 + 31) / 32 * 32 + 16; }

LX_DEV bool not_finite(float v) { return !(fabsf(v) <= 3.402823466e38f); }

// Stage rows [y0 - qh, y0 - qh + trows) x columns [x0 - qw, x0 - qw + tcols) of an H x W
// image, wrapped, into tile[trows][stride]: each thread keeps one column (one modulo per thread,
// not per element) and walks rows nsplit apart.  tcols <= 256.  Returns whether this thread met a
// value that is not finite.
LX_DEV bool stage_tile(float* tile, const float* img, int H, int W, int y0, int x0, int qh, int qw, int trows,
                       int tcols, int stride) {
  const int nsplit = 256 / tcols;
  const int t = threadIdx.x;
  bool odd = false;
  if (t < nsplit * tcols) {
    const int c = t % tcols, r0 = t / tcols;
    int gx = (x0 + c - qw) % W;
    gx += gx < 0 ? W : 0;
    int gy = (y0 + r0 - qh) % H;
    gy += gy < 0 ? H : 0;
    // 16 rows per round: the loads are all issued before the first LDS write waits on them.
    // The row advances by nsplit, i.e. by step = nsplit mod H < H, so one conditional
    // subtraction keeps gy in [0, H) for any world height.
    constexpr int BATCH = 16;
    const int step = nsplit % H;
    for (int rb = r0; rb < trows; rb += BATCH * nsplit) {
      float v[BATCH];
#pragma unroll
      for (int u = 0; u < BATCH; ++u) {
        v[u] = rb + u * nsplit < trows ? img[int64_t(gy) * W + gx] : 0.f;
        gy += step;
        gy -= gy >= H ? H : 0;
      }
#pragma unroll
      for (int u = 0; u < BATCH; ++u) {
        if (rb + u * nsplit < trows) tile[(rb + u * nsplit) * stride + c] = v[u];
        odd |= not_finite(v[u]);
      }
    }
  }
  return odd;
}

struct DirectArgs {
  const float* A;
  const float* kern;
  int H, W, C, K, kh, kw, ph, pw;
  int vec;  // rows of U (or dA) take 16-byte stores
  int cin[LX_MAX_K];
};

// Columns of the input that the 4 outputs of a lane's block read, in quads: taps 0..kw-1 of 4 shifts
__host__ __device__ inline int tap_quads(int kw) { return (kw + 3 + 3) / 4; }
// tap row stride: >= 4 quads + 3, 4 mod 8 (the four tap rows 4 apart that a wave reads: different banks)
__host__ __device__ inline int tap_stride(int kw) { return (4 * tap_quads(kw) + 3 + 3) / 8 * 8 + 4; }
__host__ __device__ inline int direct_stride(int kw) { return bank_stride(TX - 4 + 4 * tap_quads(kw)); }
size_t direct_lds(int R, int kh, int kw) {
  return (size_t(16 * R + kh - 1) * direct_stride(kw) + size_t(kh + 1) * tap_stride(kw)) * sizeof(float);
}

// The potential of kernels at most 5 columns wide: a workgroup stages 16 rows x 64 columns with their halo, a
// thread computes four neighbouring outputs from an 8-wide window of each row and uniform taps.  The matrix
// form pays for its zero-padded tap rows and the extra quad there: 128 worlds of 128^2, 1, 3 and 5 taps a side,
// us of the matrix form against these: 9.9 / 6.5, 12.0 / 7.1, 13.3 / 8.4; one world of 64^2 1 us less each.
constexpr int kNarrow = 5, kNarrowStride = TX + 8;

template <int KW>
__global__ __launch_bounds__(256) void direct_narrow_kernel(DirectArgs a, const float* in, float* out) {
  extern __shared__ __align__(16) float tile[];  // (16 + kh - 1) rows
  const int x0 = blockIdx.x * TX, y0 = blockIdx.y * 16;
  const int64_t b = blockIdx.z / a.K;
  const int k = int(blockIdx.z - b * a.K);
  stage_tile(tile, in + (b * a.C + a.cin[k]) * int64_t(a.H) * a.W, a.H, a.W, y0, x0, a.ph, a.pw, 16 + a.kh - 1, TX + 4,
             kNarrowStride);
  __syncthreads();
  const int y = y0 + threadIdx.x / (TX / 4), x = threadIdx.x % (TX / 4) * 4;
  const float* row = tile + (y - y0) * kNarrowStride + x;
  const float* kk = a.kern + int64_t(k) * a.kh * KW;
  f4v acc = {0.f, 0.f, 0.f, 0.f};
  for (int i = 0; i < a.kh; ++i, row += kNarrowStride, kk += KW) {
    const float4 lo = *reinterpret_cast<const float4*>(row), hi = *reinterpret_cast<const float4*>(row + 4);
    const float w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
    for (int j = 0; j < KW; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(kk[j], w[e + j], acc[e]);
  }
  if (y >= a.H || x0 + x >= a.W) return;
  float* dst = out + (int64_t(blockIdx.z) * a.H + y) * a.W + x0 + x;
  if (a.vec) {
    *reinterpret_cast<f4v*>(dst) = acc;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (x0 + x + e < a.W) dst[e] = acc[e];
  }
}

// The potential (ADJ: the state side of its reverse, dA[b][c] = sum over the kernels k fed by c of the
// correlation of dU[b][k] with the flipped kernel, wrap-padded with kh - 1 - ph before).  A workgroup
// computes 16 R rows x 64 columns of one image, a wave 4 R x 64: in lane 4 b + n, accumulator g holds
// the outputs of row 4 g + n at columns 4 b .. 4 b + 3.  For input row s of the wave's window and
// column jj of a block's, the instruction takes the lane's input value (row n + s, column 4 b + jj)
// times the four taps k[s - 4 g][jj - m], m < 4 (zero outside the kernel): one 16-byte LDS read feeds
// 4 R instructions, and one register holds the taps of 4 columns and R accumulators, broadcast by
// block, so 7 quads of columns take 28 tap columns for a 25-tap row (1.12x the products).  Each output
// adds its products in the order of i, then j.  A tile that holds a value that is not finite is summed
// product by product, so that none meets a zero beside the kernel.
// Measured, 128 worlds of 128^2, 25 x 25 taps, R = 2: potential 60 -> 41 us (64 TFLOP/s of the taps; 45 beside
// the gradients' kernels), state side 94 -> 42 us (the vector units' window kernel before took its flipped taps one by one); 12 us of
// it stage the tiles, the instructions themselves need 25.  Groups of equal size rather than of four quads with
// a partly empty last one: 47 -> 41 us there, 72 -> 57 at 33 taps a side, 149 -> 122 at 48.
template <int R, bool ADJ>
__global__ __launch_bounds__(256) void direct_mfma_kernel(DirectArgs a, const float* in, float* out) {
  extern __shared__ __align__(16) float lds[];
  const int S = direct_stride(a.kw), TS = tap_stride(a.kw), Q = tap_quads(a.kw), rows = 16 * R + a.kh - 1;
  float* tile = lds;
  float* taps = lds + rows * S;
  const int x0 = blockIdx.x * TX, y0 = blockIdx.y * 16 * R;
  const int nout = ADJ ? a.C : a.K;
  const int64_t b = blockIdx.z / nout;
  const int o = int(blockIdx.z - b * nout);  // the kernel, or (ADJ) the channel
  const int lane = threadIdx.x & 63, wy = (threadIdx.x >> 6) * 4 * R;
  const int n = lane & 3, blk = lane >> 2;
  const bool busy = y0 + wy < a.H;  // the wave has rows of the image
  f4v acc[R];
#pragma unroll
  for (int g = 0; g < R; ++g) acc[g] = f4v{0.f, 0.f, 0.f, 0.f};
  for (int k = ADJ ? 0 : o; k < (ADJ ? a.K : o + 1); ++k) {
    if (ADJ && a.cin[k] != o) continue;
    const int64_t img = ADJ ? b * a.K + k : b * a.C + a.cin[k];
    const int qh = ADJ ? a.kh - 1 - a.ph : a.ph, qw = ADJ ? a.kw - 1 - a.pw : a.pw;
    __syncthreads();  // the previous kernel's tile is consumed
    const bool odd = stage_tile(tile, in + img * a.H * a.W, a.H, a.W, y0, x0, qh, qw, rows, TX - 4 + 4 * Q, S);
    const float* kk = a.kern + int64_t(k) * a.kh * a.kw;
    for (int e = threadIdx.x; e < (a.kh + 1) * TS; e += 256) {
      const int i = e / TS, j = e - i * TS - 3;
      const bool in_row = i < a.kh && j >= 0 && j < a.kw;
      taps[e] = !in_row ? 0.f : ADJ ? kk[(a.kh - 1 - i) * a.kw + a.kw - 1 - j] : kk[i * a.kw + j];
    }
    const bool slow = __syncthreads_or(odd);
    if (!busy) continue;
    if (!slow) {
      // lane 16 g + 4 e + m of the tap register: k[s - 4 g][4 q + e - m]
      const int tg = lane >> 4;
      const float* tcol = taps + ((lane >> 2) & 3) - n + 3;
      const float* col = tile + (wy + n) * S + 4 * blk;
      const int last = a.kh - 1 + 4 * (R - 1);
      // the quads in groups of at most 4 and as equal as can be (`more` groups of each + 1, then groups of each):
      // a group's reads are in flight together, then its instructions
      const int groups = (Q + 3) / 4, each = Q / groups, more = Q - groups * each;
      auto rows_of = [&](auto each_c) {
        constexpr int EACH = decltype(each_c)::value;
        for (int s = 0; s <= last; ++s) {
          const int ti = unsigned(s - 4 * tg) < unsigned(a.kh) ? s - 4 * tg : a.kh;  // row kh holds zeros
          const float* trow = tcol + ti * TS;
          const float* irow = col + s * S;
          auto group = [&](auto n_c) {
            constexpr int N = decltype(n_c)::value;
            float4 v[N];
            float t[N];
#pragma unroll
            for (int u = 0; u < N; ++u) {
              v[u] = *reinterpret_cast<const float4*>(irow + 4 * u);
              t[u] = trow[4 * u];
            }
            irow += 4 * N;
            trow += 4 * N;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < N; ++u) {
              auto column = [&](auto e_c, float x) {
                constexpr int E = decltype(e_c)::value;
                acc[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(t[u], x, acc[0], 4, E, 0);
                if constexpr (R > 1) acc[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(t[u], x, acc[1], 4, 4 + E, 0);
              };
              column(std::integral_constant<int, 0>{}, v[u].x);
              column(std::integral_constant<int, 1>{}, v[u].y);
              column(std::integral_constant<int, 2>{}, v[u].z);
              column(std::integral_constant<int, 3>{}, v[u].w);
            }
          };
          if constexpr (EACH < 4)
            for (int g = 0; g < more; ++g) group(std::integral_constant<int, EACH + 1>{});
          for (int g = more; g < groups; ++g) group(std::integral_constant<int, EACH>{});
        }
      };
      switch (each) {
        case 4: rows_of(std::integral_constant<int, 4>{}); break;
        case 3: rows_of(std::integral_constant<int, 3>{}); break;
        case 2: rows_of(std::integral_constant<int, 2>{}); break;
        default: rows_of(std::integral_constant<int, 1>{}); break;
      }
    } else {
      for (int i = 0; i < a.kh; ++i)
        for (int j = 0; j < a.kw; ++j) {
          const float t = taps[i * TS + j + 3];
          const float* v = tile + (wy + n + i) * S + 4 * blk + j;
#pragma unroll
          for (int g = 0; g < R; ++g)
#pragma unroll
            for (int m = 0; m < 4; ++m) acc[g][m] = fmaf(t, v[4 * g * S + m], acc[g][m]);
        }
    }
  }
  const int x = x0 + 4 * blk;
  if (!busy || x >= a.W) return;
#pragma unroll
  for (int g = 0; g < R; ++g) {
    const int y = y0 + wy + 4 * g + n;
    if (y >= a.H) continue;
    float* dst = out + (int64_t(blockIdx.z) * a.H + y) * a.W + x;
    if (a.vec) {
      *reinterpret_cast<f4v*>(dst) = acc[g];
    } else {
#pragma unroll
      for (int m = 0; m < 4; ++m)
        if (x + m < a.W) dst[m] = acc[g][m];
    }
  }
}

// The launch for `images` output images: R = 2 halves the LDS reads per instruction (with groups of four quads 52
// against 64 us at the size above; R = 4 measured 58, its tiles leave two workgroups per CU); R = 1 where R = 2
// would leave CUs with fewer than two workgroups (512).  R = 2's tile takes up to 75 KB of LDS (64 taps a side:
// still two workgroups per CU); with R = 1 beyond 64 KB the same 128 worlds took 389 us for 64 x 64 taps, 182 now.
template <bool ADJ>
int launch_direct(DirectArgs a, int64_t images, const float* in, float* out, hipStream_t st) {
  a.vec = a.W % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0;
  auto grid = [&](int R) {
    return dim3(unsigned((a.W + TX - 1) / TX), unsigned((a.H + 16 * R - 1) / (16 * R)), unsigned(images));
  };
  if constexpr (!ADJ) {
    auto narrow = [&](auto kw_c) {
      constexpr int KW = decltype(kw_c)::value;
      hipLaunchKernelGGL((direct_narrow_kernel<KW>), grid(1), dim3(256),
                         size_t(16 + a.kh - 1) * kNarrowStride * sizeof(float), st, a, in, out);
      return LX_OK;
    };
    static_assert(kNarrow == 5, "one case per width");
    switch (a.kw) {
      case 1: return narrow(std::integral_constant<int, 1>{});
      case 2: return narrow(std::integral_constant<int, 2>{});
      case 3: return narrow(std::integral_constant<int, 3>{});
      case 4: return narrow(std::integral_constant<int, 4>{});
      case 5: return narrow(std::integral_constant<int, 5>{});
      default: break;
    }
  }
  auto go = [&](auto r_c) {
    constexpr int R = decltype(r_c)::value;
    const size_t lds = direct_lds(R, a.kh, a.kw);
    if (lds > 65536 &&
        hipFuncSetAttribute(reinterpret_cast<const void*>(direct_mfma_kernel<R, ADJ>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)) != hipSuccess)
      return lx_fail(LX_EDEVICE, "direct potential: %zu bytes of LDS refused", lds);
    hipLaunchKernelGGL((direct_mfma_kernel<R, ADJ>), grid(R), dim3(256), lds, st, a, in, out);
    return int(LX_OK);
  };
  const dim3 two = grid(2);
  if (int64_t(two.x) * two.y * two.z >= 512) return go(std::integral_constant<int, 2>{});
  return go(std::integral_constant<int, 1>{});
}

// Reverse of the direct potential, kernel side: dK[k][i][j] = sum over worlds and cells of
// dU[b][k][y][x] A[b][cin k][(y + i - ph) mod H][(x + j - pw) mod W] (grid: kh * kw x K; one block
// per tap, so the sum needs no atomics and is deterministic).
__global__ __launch_bounds__(256) void direct_kgrad_kernel(DirectArgs a, int64_t B, const float* dU, float* dK) {
  const int tap = blockIdx.x;
  const int i = tap / a.kw, j = tap - i * a.kw;
  const int k = blockIdx.y;
  const int64_t n = int64_t(a.H) * a.W;
  float acc = 0.f;
  for (int64_t b = 0; b < B; ++b) {
    const float* G = dU + (b * a.K + k) * n;
    const float* A = a.A + (b * a.C + a.cin[k]) * n;
    for (int64_t p = threadIdx.x; p < n; p += 256) {
      const int y = int(p / a.W), x = int(p - int64_t(y) * a.W);
      int gy = (y + i - a.ph) % a.H;
      gy += gy < 0 ? a.H : 0;
      int gx = (x + j - a.pw) % a.W;
      gx += gx < 0 ? a.W : 0;
      acc = fmaf(G[p], A[int64_t(gy) * a.W + gx], acc);
    }
  }
  __shared__ float red[4];
  const float s = wave_sum(acc);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) dK[(int64_t(k) * a.kh + i) * a.kw + j] = red[0] + red[1] + red[2] + red[3];
}

// The kernel side on the matrix cores, for callers with a workspace.  With i = 4 ib + n and
// j = 4 jb + m, dK[i][j] = sum over cells of dU[y][x - m] A[y + 4 ib + n - ph][x + 4 jb - pw] (both
// images are periodic, so the sum over x may start at any shift): for each cell (y, x) a 4 x 4 outer
// product per (ib, jb), which is one v_mfma_f32_4x4x1 for 16 (ib, jb) pairs.  Lane 4 s + n of a set
// holds its pair's n-th row of A, four cells per 16-byte LDS read; the dU operand is the same for
// every pair, so one register holds 16 cells' (lane 4 p + m: dU[y][x + p - m]) and the instruction
// broadcasts block p of it.  A block takes tiles of kGY x kGX cells in turn (waves take rows), adds
// its waves' sums in order and stores one row of partial sums; direct_kgrad_sum_kernel adds the rows
// in a fixed order, so the gradient is deterministic.  In the matrix form every LDS value feeds 4
// multiply-adds of its lane and the pass is bound by LDS reads and MFMA issue (the one-block-per-tap
// kernel above re-reads both images for every tap with a division and two remainders per product).
// Measured, 128 worlds of 128^2 with a 25 x 25 kernel: 3457 -> 59 + 5 us (2.6 GFLOP of taps: 41 TFLOP/s),
// error against 64 bits 1.6e-6 -> 4.7e-7 (shorter chains of additions).
// Few worlds take other chains, so that no size is summed less accurately than by one block per tap, whose
// threads add every 256th cell: up to 2^17 cells a row's cells go into four sums of their own (a lane's chain is
// 16 + 2 + 4 additions of a tile instead of 256; two worlds of 167 x 82, 25 taps a side: 2.2e-7 -> 1.3e-7, one block
// per tap 1.4e-7; 7% of the time there, 25% for many worlds, whose waves are fewer by its 135 VGPRs), and up to 6144
// cells with up to 1200 taps one block per tap is the faster too (one world of 64^2, 5, 25 and 33 taps a side: 7.9,
// 10 and 13.5 against 11.6, 16.9 and 17.3 us).
constexpr int kGY = 16, kGX = 64, kGridRows = 1024, kGSets = 4;

__host__ __device__ inline int kgrad_stride(int kw) { return bank_stride(kGX + ((kw + 3) & ~3)); }
__host__ __device__ inline int kgrad_rows(int kh) { return kGY - 1 + ((kh + 3) & ~3); }
constexpr int kGDU = kGX + 4;  // dU tile row: 3 columns before, one spare

// NS: sets of 16 (ib, jb) pairs per block; blockIdx.y = k * groups + group of NS sets.  FINE: a row's cells in four
// chains of additions that start anew, for few cells (kgrad_fine)
template <int NS, bool FINE>
__global__ __launch_bounds__(256) void direct_kgrad_mfma_kernel(DirectArgs a, int64_t B, const float* dU, float* part,
                                                                int groups, int tx, int64_t ntiles) {
  extern __shared__ __align__(16) float lds[];
  const int S = kgrad_stride(a.kw), R = kgrad_rows(a.kh);
  float* tA = lds;          // [R][S]
  float* tG = lds + R * S;  // [kGY][kGDU]
  const int k = blockIdx.y / groups, set0 = (blockIdx.y - k * groups) * NS;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nj = (a.kw + 3) / 4, nb = nj * ((a.kh + 3) / 4);
  int off[NS];  // the lane's first A value of each set (pairs past the last read pair 0, unused)
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    int blk = (set0 + s) * 16 + (lane >> 2);
    if (blk >= nb) blk = 0;
    const int ib = blk / nj, jb = blk - ib * nj;
    off[s] = (4 * ib + (lane & 3)) * S + 4 * jb;
  }
  f4v acc[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) acc[s] = f4v{0.f, 0.f, 0.f, 0.f};
  const int64_t n = int64_t(a.H) * a.W;
  const int ty = (a.H + kGY - 1) / kGY;
  for (int64_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
    const int64_t b = tile / (int64_t(tx) * ty);
    const int rem = int(tile - b * tx * ty);
    const int y0 = (rem / tx) * kGY, x0 = (rem % tx) * kGX;
    __syncthreads();  // the previous tile is consumed
    const bool odd = stage_tile(tA, a.A + (b * a.C + a.cin[k]) * n, a.H, a.W, y0, x0, a.ph, a.pw, R,
                                kGX + 4 * nj, S);
    stage_tile(tG, dU + (b * a.K + k) * n, a.H, a.W, y0, x0, 0, 3, kGY, kGDU, kGDU);
    const bool slow = __syncthreads_or(odd);
    const int rows = min(kGY, a.H - y0), cols = min(kGX, a.W - x0);
    if (!slow) {
      for (int r = wave; r < rows; r += 4) {
        f4v part[FINE ? NS : 1][4];  // FINE: sums of every fourth cell of the row
        if constexpr (FINE)
#pragma unroll
          for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[s][e] = f4v{0.f, 0.f, 0.f, 0.f};
        for (int xg = 0; xg < cols; xg += 16) {
          const int p = lane >> 2;
          // cells past the image's last column count nothing
          const float g = xg + p < cols ? tG[r * kGDU + xg + p - (lane & 3) + 3] : 0.f;
          const float* row = tA + r * S + xg;
          auto quad = [&](auto q_c) {
            constexpr int Q = decltype(q_c)::value;
            float4 v[NS];
#pragma unroll
            for (int s = 0; s < NS; ++s) v[s] = *reinterpret_cast<const float4*>(row + off[s] + 4 * Q);
            auto cell = [&](auto e_c, auto of) {
              constexpr int E = decltype(e_c)::value;
#pragma unroll
              for (int s = 0; s < NS; ++s) {
                f4v& sum = FINE ? part[FINE ? s : 0][E] : acc[s];
                sum = __builtin_amdgcn_mfma_f32_4x4x1f32(g, of(v[s]), sum, 4, 4 * Q + E, 0);
              }
            };
            cell(std::integral_constant<int, 0>{}, [](const float4& w) { return w.x; });
            cell(std::integral_constant<int, 1>{}, [](const float4& w) { return w.y; });
            cell(std::integral_constant<int, 2>{}, [](const float4& w) { return w.z; });
            cell(std::integral_constant<int, 3>{}, [](const float4& w) { return w.w; });
          };
          quad(std::integral_constant<int, 0>{});
          quad(std::integral_constant<int, 1>{});
          quad(std::integral_constant<int, 2>{});
          quad(std::integral_constant<int, 3>{});
        }
        if constexpr (FINE)
#pragma unroll
          for (int s = 0; s < NS; ++s) acc[s] += (part[s][0] + part[s][1]) + (part[s][2] + part[s][3]);
      }
    } else {
      // a state that is not finite: product by product, so that none is taken with the zero of a
      // cell past the last column
      for (int r = wave; r < rows; r += 4)
        for (int x = 0; x < cols; ++x)
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            const float v = tA[r * S + x + off[s]];
#pragma unroll
            for (int m = 0; m < 4; ++m) acc[s][m] = fmaf(tG[r * kGDU + x - m + 3], v, acc[s][m]);
          }
    }
  }
  // the waves' sums in order, then the block's row of partial sums
  __syncthreads();
  float* red = lds;  // [4][NS][64][4] floats
#pragma unroll
  for (int s = 0; s < NS; ++s)
    *reinterpret_cast<f4v*>(red + ((wave * NS + s) * 64 + lane) * 4) = acc[s];
  __syncthreads();
  float* dst = part + (int64_t(blockIdx.x) * a.K + k) * a.kh * a.kw;
  for (int e = threadIdx.x; e < NS * 256; e += 256) {
    const int s = e >> 8, l = (e >> 2) & 63, m = e & 3;
    const int blk = (set0 + s) * 16 + (l >> 2);
    const int ib = blk / nj, jb = blk - ib * nj;
    const int i = 4 * ib + (l & 3), j = 4 * jb + m;
    if (blk < nb && i < a.kh && j < a.kw) {
      float v = 0.f;
#pragma unroll
      for (int w = 0; w < 4; ++w) v += red[(w * NS * 64) * 4 + e];
      dst[i * a.kw + j] = v;
    }
  }
}

// dK[tap] = sum of the partial rows: 32 taps per block, 32 threads per tap take every 32nd row (8 loads
// in flight), then their sums are added in order
__global__ __launch_bounds__(1024) void direct_kgrad_sum_kernel(const float* part, int rows, int taps, float* dK) {
  __shared__ float red[32][32];
  const int t = threadIdx.x & 31, sl = threadIdx.x >> 5;
  const int tap = blockIdx.x * 32 + t;
  float acc = 0.f;
  if (tap < taps) {
#pragma unroll 8
    for (int r = sl; r < rows; r += 32) acc += part[int64_t(r) * taps + tap];
  }
  red[sl][t] = acc;
  __syncthreads();
  if (sl == 0 && tap < taps) {
#pragma unroll
    for (int i = 1; i < 32; ++i) acc += red[i][t];
    dK[tap] = acc;
  }
}

int kgrad_tiles_x(int W) { return (W + kGX - 1) / kGX; }
int64_t kgrad_tiles(const lx_rule* r, int64_t B) {
  return B * kgrad_tiles_x(r->dims[1]) * ((r->dims[0] + kGY - 1) / kGY);
}
bool kgrad_fine(const lx_rule* r, int64_t B) { return B * r->dims[0] * r->dims[1] <= (1 << 17); }
bool kgrad_by_tap(const lx_rule* r, int64_t B, int kh, int kw) {
  return B * r->dims[0] * r->dims[1] <= 6144 && r->K * kh * kw <= 1200;
}
// blocks of NS = kgrad_ns(sets) sets per kernel and rows of partial sums: enough blocks to fill 256 CUs
// a few times over, no more than tiles; at most kGridRows x 16 kGSets taps x 16 B of partial sums
int kgrad_sets(int kh, int kw) { return (((kh + 3) / 4) * ((kw + 3) / 4) + 15) / 16; }
int kgrad_ns(int sets) { return sets < 3 ? sets : kGSets; }
int64_t kgrad_part_rows(const lx_rule* r, int64_t B, int kh, int kw) {
  const int sets = kgrad_sets(kh, kw), per = r->K * ((sets + kgrad_ns(sets) - 1) / kgrad_ns(sets));
  return std::min<int64_t>(kgrad_tiles(r, B), (kGridRows + per - 1) / per);
}

DirectArgs direct_args(const lx_rule* rule, const float* A, const float* kern, int kh, int kw) {
  DirectArgs a;
  a.A = A; a.kern = kern; a.vec = 0;
  a.H = rule->dims[0]; a.W = rule->dims[1]; a.C = rule->C; a.K = rule->K;
  a.kh = kh; a.kw = kw; a.ph = kh / 2; a.pw = kw / 2;
  for (int k = 0; k < LX_MAX_K; ++k) a.cin[k] = k < rule->K ? rule->cin[k] : 0;
  return a;
}

}  // namespace

namespace {

// the reverse of the direct potential; work: lx_potential_direct_adjoint_size bytes, or NULL (the
// kernel side then takes one block per tap)
int direct_adjoint(const char* fn, const lx_rule* rule, const float* state_d, int64_t B, const float* kern_d,
                   int32_t kh, int32_t kw, const float* dpot_d, float* dstate_d, float* dkern_d, float* work,
                   hipStream_t st) {
  int rc = lx_check_rule(rule);
  if (rc) return rc;
  if (rule->ndim != 2) return lx_fail(LX_ENOTSUP, "%s: 2-D worlds only", fn);
  if (kh < 1 || kw < 1 || kh > MAXK || kw > MAXK) return lx_fail(LX_ENOTSUP, "kernel %dx%d (1..%d)", kh, kw, MAXK);
  if (B < 0) return lx_fail(LX_EINVAL, "B < 0");
  if (B == 0) return LX_OK;
  if (!kern_d || !dpot_d || (!dstate_d && !dkern_d) || (dkern_d && !state_d)) return lx_fail(LX_EINVAL, "NULL pointer");
  if (B * rule->C > 65535) return lx_fail(LX_ENOTSUP, "%s: B * C > 65535", fn);
  const DirectArgs a = direct_args(rule, state_d, kern_d, kh, kw);
  if (dstate_d) {
    if ((rc = launch_direct<true>(a, B * rule->C, dpot_d, dstate_d, st))) return rc;
  }
  if (dkern_d && work && !kgrad_by_tap(rule, B, kh, kw)) {
    const int64_t rows = kgrad_part_rows(rule, B, kh, kw);
    const int sets = kgrad_sets(kh, kw);
    auto go = [&](auto ns_c) {
      constexpr int NS = decltype(ns_c)::value;
      const int groups = (sets + NS - 1) / NS;
      const size_t tiles = size_t(kgrad_rows(kh)) * kgrad_stride(kw) + size_t(kGY) * kGDU;
      const size_t lds = std::max(tiles, size_t(4) * NS * 256) * sizeof(float);
      const dim3 grid{unsigned(rows), unsigned(rule->K * groups)};
      const int tx = kgrad_tiles_x(a.W);
      const int64_t ntiles = kgrad_tiles(rule, B);
      if (kgrad_fine(rule, B))
        hipLaunchKernelGGL((direct_kgrad_mfma_kernel<NS, true>), grid, dim3(256), lds, st, a, B, dpot_d, work, groups,
                           tx, ntiles);
      else
        hipLaunchKernelGGL((direct_kgrad_mfma_kernel<NS, false>), grid, dim3(256), lds, st, a, B, dpot_d, work, groups,
                           tx, ntiles);
    };
    switch (kgrad_ns(sets)) {
      case 1: go(std::integral_constant<int, 1>{}); break;
      case 2: go(std::integral_constant<int, 2>{}); break;
      default: go(std::integral_constant<int, kGSets>{}); break;
    }
    const int taps = rule->K * kh * kw;
    hipLaunchKernelGGL(direct_kgrad_sum_kernel, dim3(unsigned((taps + 31) / 32)), dim3(1024), 0, st, work, int(rows),
                       taps, dkern_d);
  } else if (dkern_d) {
    hipLaunchKernelGGL(direct_kgrad_kernel, dim3(unsigned(kh * kw), unsigned(rule->K)), dim3(256), 0, st, a, B,
                       dpot_d, dkern_d);
  }
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? LX_OK : lx_fail(LX_EDEVICE, "direct adjoint launch: %s", hipGetErrorString(e));
}

}  // namespace

extern "C" int lx_potential_direct_adjoint(const lx_rule* rule, const float* state_d, int64_t B,
                                           const float* kern_d, int32_t kh, int32_t kw, const float* dpot_d,
                                           float* dstate_d, float* dkern_d, void* stream) {
  return direct_adjoint("lx_potential_direct_adjoint", rule, state_d, B, kern_d, kh, kw, dpot_d, dstate_d, dkern_d,
                        nullptr, (hipStream_t)stream);
}

extern "C" int lx_potential_direct_adjoint_size(const lx_rule* rule, int64_t B, int32_t kh, int32_t kw,
                                                size_t* bytes) {
  int rc = lx_check_rule(rule);
  if (rc) return rc;
  if (rule->ndim != 2) return lx_fail(LX_ENOTSUP, "lx_potential_direct_adjoint_size: 2-D worlds only");
  if (kh < 1 || kw < 1 || kh > MAXK || kw > MAXK) return lx_fail(LX_ENOTSUP, "kernel %dx%d (1..%d)", kh, kw, MAXK);
  if (B < 0 || !bytes) return lx_fail(LX_EINVAL, "B < 0 or NULL pointer");
  *bytes = size_t(kgrad_part_rows(rule, B, kh, kw)) * rule->K * kh * kw * sizeof(float);
  return LX_OK;
}

extern "C" int lx_potential_direct_adjoint_work(const lx_rule* rule, const float* state_d, int64_t B,
                                                const float* kern_d, int32_t kh, int32_t kw, const float* dpot_d,
                                                float* dstate_d, float* dkern_d, void* work_d, void* stream) {
  if (B > 0 && dkern_d && !work_d) return lx_fail(LX_EINVAL, "lx_potential_direct_adjoint_work: NULL workspace");
  return direct_adjoint("lx_potential_direct_adjoint_work", rule, state_d, B, kern_d, kh, kw, dpot_d, dstate_d,
                        dkern_d, static_cast<float*>(work_d), (hipStream_t)stream);
}

extern "C" int lx_potential_direct(const lx_rule* rule, const float* state_d, int64_t B, const float* kern_d,
                                   int32_t kh, int32_t kw, float* potential_d, void* stream) {
  int rc = lx_check_rule(rule);
  if (rc) return rc;
  if (rule->ndim != 2) return lx_fail(LX_ENOTSUP, "lx_potential_direct: 2-D worlds only");
  if (kh < 1 || kw < 1 || kh > MAXK || kw > MAXK) return lx_fail(LX_ENOTSUP, "kernel %dx%d (1..%d)", kh, kw, MAXK);
  if (B < 0) return lx_fail(LX_EINVAL, "B < 0");
  if (B == 0) return LX_OK;
  if (!state_d || !kern_d || !potential_d) return lx_fail(LX_EINVAL, "NULL pointer");
  if (B * rule->K > 65535) return lx_fail(LX_ENOTSUP, "lx_potential_direct: B * K > 65535");
  const DirectArgs a = direct_args(rule, state_d, kern_d, kh, kw);
  if ((rc = launch_direct<false>(a, B * rule->K, state_d, potential_d, (hipStream_t)stream))) return rc;
  hipError_t e = hipGetLastError();
  return e == hipSuccess ? LX_OK : lx_fail(LX_EDEVICE, "direct potential launch: %s", hipGetErrorString(e));
}
