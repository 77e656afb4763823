// Batched Stockham FFTs on the oversampled grid, fused with deconvolution,
// zero-padding / cropping and the SENSE coil expand / conjugate combine.
//
// Replaces the FFT, deapodisation, pad and crop stages inside cufinufft's
// Plan.execute (operators/interfaces/cufinufft.py:127-133), the SENSE
// broadcast multiply (cufinufft.py:497) and the coil-combine kernel
// (operators/gpu_utils.py:12-24, operators/toeplitz.py:299-321).
//
// Layout: the fine grid of transform t is grid[t][nf0][nf1][nf2] (C order,
// axis 2 contiguous; 2D / 1D grids use leading axes of size 1).  Image index
// i along an axis of size M is frequency k = i - M/2 and lives at fine-grid
// position (k mod nf).  Every pass works in place on whole lines held in LDS:
// a workgroup owns L lines (L adjacent columns for the strided axes, so
// global accesses are L*8-byte contiguous segments), loads only the positions
// that are non-zero (pruned input), runs all Stockham passes in LDS and
// stores only the positions later stages read (pruned output).

#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "addressing.h"
#include "internal.h"

namespace hn {
namespace {


__device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ __forceinline__ float2 cscale(float2 a, float s) { return make_float2(a.x * s, a.y * s); }
// a * (S i)
template <int S>
__device__ __forceinline__ float2 mul_si(float2 a) {
  return S > 0 ? make_float2(-a.y, a.x) : make_float2(a.y, -a.x);
}

// y_k = sum_j v_j exp(S 2 pi i j k / R)
template <int S>
__device__ __forceinline__ void dft2(float2* v) {
  const float2 t = v[0];
  v[0] = cadd(t, v[1]);
  v[1] = csub(t, v[1]);
}

template <int S>
__device__ __forceinline__ void dft4(float2& v0, float2& v1, float2& v2, float2& v3) {
  const float2 a0 = cadd(v0, v2), a1 = csub(v0, v2), a2 = cadd(v1, v3);
  const float2 a3 = mul_si<S>(csub(v1, v3));
  v0 = cadd(a0, a2);
  v2 = csub(a0, a2);
  v1 = cadd(a1, a3);
  v3 = csub(a1, a3);
}

template <int S>
__device__ __forceinline__ void dft4(float2* v) {
  dft4<S>(v[0], v[1], v[2], v[3]);
}

template <int S>
__device__ __forceinline__ void dft8(float2* v) {
  float2 e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
  float2 o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
  dft4<S>(e0, e1, e2, e3);
  dft4<S>(o0, o1, o2, o3);
  const float h = 0.70710678118654752f;
  const float2 w1 = cscale(cadd(o1, mul_si<S>(o1)), h);   // W8^1 o1
  const float2 w2 = mul_si<S>(o2);                        // W8^2 o2
  const float2 w3 = cscale(csub(mul_si<S>(o3), o3), h);   // W8^3 o3
  v[0] = cadd(e0, o0);
  v[4] = csub(e0, o0);
  v[1] = cadd(e1, w1);
  v[5] = csub(e1, w1);
  v[2] = cadd(e2, w2);
  v[6] = csub(e2, w2);
  v[3] = cadd(e3, w3);
  v[7] = csub(e3, w3);
}

template <int S>
__device__ __forceinline__ void dft3(float2* v) {
  const float c = 0.86602540378443865f;
  const float2 t = cadd(v[1], v[2]);
  const float2 s = cscale(mul_si<S>(csub(v[1], v[2])), c);
  const float2 m = make_float2(v[0].x - 0.5f * t.x, v[0].y - 0.5f * t.y);
  v[0] = cadd(v[0], t);
  v[1] = cadd(m, s);
  v[2] = csub(m, s);
}

template <int S>
__device__ __forceinline__ void dft5(float2* v) {
  const float c1 = 0.30901699437494742f, c2 = -0.80901699437494742f;
  const float s1 = 0.95105651629515357f, s2 = 0.58778525229247313f;
  const float2 a1 = cadd(v[1], v[4]), b1 = csub(v[1], v[4]);
  const float2 a2 = cadd(v[2], v[3]), b2 = csub(v[2], v[3]);
  const float2 x0 = v[0];
  const float2 p1 = make_float2(x0.x + c1 * a1.x + c2 * a2.x, x0.y + c1 * a1.y + c2 * a2.y);
  const float2 p2 = make_float2(x0.x + c2 * a1.x + c1 * a2.x, x0.y + c2 * a1.y + c1 * a2.y);
  const float2 q1 = mul_si<S>(make_float2(s1 * b1.x + s2 * b2.x, s1 * b1.y + s2 * b2.y));
  const float2 q2 = mul_si<S>(make_float2(s2 * b1.x - s1 * b2.x, s2 * b1.y - s1 * b2.y));
  v[0] = make_float2(x0.x + a1.x + a2.x, x0.y + a1.y + a2.y);
  v[1] = cadd(p1, q1);
  v[4] = csub(p1, q1);
  v[2] = cadd(p2, q2);
  v[3] = csub(p2, q2);
}

// 6 = 2 x 3 by the prime-factor mapping (no inner twiddles): inputs
// (3 n1 + 2 n2) mod 6 go through two 3-point DFTs over n2, then 2-point
// DFTs over n1, and (k1, k2) lands at (3 k1 + 4 k2) mod 6
template <int S>
__device__ __forceinline__ void dft6(float2* v) {
  float2 a[3] = {v[0], v[2], v[4]};
  float2 b[3] = {v[3], v[5], v[1]};
  dft3<S>(a);
  dft3<S>(b);
  v[0] = cadd(a[0], b[0]);
  v[3] = csub(a[0], b[0]);
  v[4] = cadd(a[1], b[1]);
  v[1] = csub(a[1], b[1]);
  v[2] = cadd(a[2], b[2]);
  v[5] = csub(a[2], b[2]);
}

// 10 = 2 x 5 by the same mapping: inputs (5 n1 + 2 n2) mod 10, two 5-point
// DFTs over n2, 2-point DFTs over n1, outputs at (5 k1 + 6 k2) mod 10
template <int S>
__device__ __forceinline__ void dft10(float2* v) {
  float2 a[5] = {v[0], v[2], v[4], v[6], v[8]};
  float2 b[5] = {v[5], v[7], v[9], v[1], v[3]};
  dft5<S>(a);
  dft5<S>(b);
  v[0] = cadd(a[0], b[0]);
  v[5] = csub(a[0], b[0]);
  v[6] = cadd(a[1], b[1]);
  v[1] = csub(a[1], b[1]);
  v[2] = cadd(a[2], b[2]);
  v[7] = csub(a[2], b[2]);
  v[8] = cadd(a[3], b[3]);
  v[3] = csub(a[3], b[3]);
  v[4] = cadd(a[4], b[4]);
  v[9] = csub(a[4], b[4]);
}

template <int R, int S>
__device__ __forceinline__ void dftR(float2* v) {
  if constexpr (R == 2) dft2<S>(v);
  if constexpr (R == 3) dft3<S>(v);
  if constexpr (R == 4) dft4<S>(v);
  if constexpr (R == 5) dft5<S>(v);
  if constexpr (R == 6) dft6<S>(v);
  if constexpr (R == 8) dft8<S>(v);
  if constexpr (R == 10) dft10<S>(v);
}

// One Stockham radix-R pass over L interleaved lines of length n held in LDS
// at buf[pos * LP + line].  Every thread first reads all its butterflies into
// registers, then (after a barrier) writes the results: a single LDS buffer.
template <int R, int S, int EPT, int NT = kThreads>
__device__ __forceinline__ void stockham_pass(float2* buf, int n, int lgL, int LP, int Ns,
                                              uint32_t ns_magic, const float2* tw) {
  constexpr int MAXB = (EPT + R - 1) / R;
  const int L = 1 << lgL;
  // uniform (scalar) quantities; every LDS address below is one 24-bit
  // multiply per butterfly plus uniform strides per radix leg
  const int nr = n / R;
  const int nbf = nr << lgL;
  const int tstep = n / (Ns * R);
  const int in_stride = nr * LP;
  const int out_stride = Ns * LP;
  const int NsR = Ns * R;
  float2 v[MAXB][R];
#pragma unroll
  for (int i = 0; i < MAXB; ++i) {
    const int b = threadIdx.x + i * NT;
    if (b < nbf) {
      const int l = b & (L - 1), j = b >> lgL;
      const int a0 = __mul24(j, LP) + l;
#pragma unroll
      for (int r = 0; r < R; ++r) v[i][r] = buf[a0 + r * in_stride];
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MAXB; ++i) {
    const int b = threadIdx.x + i * NT;
    if (b < nbf) {
      const int l = b & (L - 1), j = b >> lgL;
      // q = j / Ns by multiply-high (exact for j < 2^16); Ns = 1 in the first pass
      const int q = Ns == 1 ? j : (int)__umulhi((uint32_t)j, ns_magic);
      const int k = j - __mul24(q, Ns);
      if (Ns > 1) {  // the first pass has unit twiddles
        const int kt = __mul24(k, tstep);
#pragma unroll
        for (int r = 1; r < R; ++r) {
          float2 w = tw[r * kt];
          if (S > 0) w.y = -w.y;
          v[i][r] = cmul(v[i][r], w);
        }
      }
      dftR<R, S>(v[i]);
      const int o0 = __mul24(__mul24(q, NsR) + k, LP) + l;
#pragma unroll
      for (int r = 0; r < R; ++r) buf[o0 + r * out_stride] = v[i][r];
    }
  }
  __syncthreads();
}

// The same Stockham pass with the line length N, the lines 2^LGL and the
// pass's Ns known at compile time: strides fold into the LDS instruction
// offsets, j / Ns is a shift for the power-of-two Ns of an 8 * 8 * R plan,
// and the butterfly-range test disappears when NT divides the butterflies.
template <int R, int S, int EPT, int NT, int N, int LGL, int NS>
__device__ __forceinline__ void stockham_pass_ct(float2* buf, const float2* tw) {
  constexpr int MAXB = (EPT + R - 1) / R;
  constexpr int L = 1 << LGL, LP = L + 1;
  constexpr int nr = N / R;
  constexpr int nbf = nr << LGL;
  constexpr int tstep = N / (NS * R);
  constexpr int in_stride = nr * LP;
  constexpr int out_stride = NS * LP;
  constexpr int NsR = NS * R;
  static_assert(nbf <= MAXB * NT, "butterflies exceed the threads' slots");
  float2 v[MAXB][R];
#pragma unroll
  for (int i = 0; i < MAXB; ++i) {
    const int b = threadIdx.x + i * NT;
    if (nbf % NT == 0 || b < nbf) {
      const int l = b & (L - 1), j = b >> LGL;
      const int a0 = j * LP + l;
#pragma unroll
      for (int r = 0; r < R; ++r) v[i][r] = buf[a0 + r * in_stride];
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < MAXB; ++i) {
    const int b = threadIdx.x + i * NT;
    if (nbf % NT == 0 || b < nbf) {
      const int l = b & (L - 1), j = b >> LGL;
      const int q = j / NS;
      const int k = j - q * NS;
      if constexpr (NS > 1) {  // the first pass has unit twiddles
        const int kt = k * tstep;
#pragma unroll
        for (int r = 1; r < R; ++r) {
          float2 w = tw[r * kt];
          if (S > 0) w.y = -w.y;
          v[i][r] = cmul(v[i][r], w);
        }
      }
      dftR<R, S>(v[i]);
      const int o0 = (q * NsR + k) * LP + l;
#pragma unroll
      for (int r = 0; r < R; ++r) buf[o0 + r * out_stride] = v[i][r];
    }
  }
  __syncthreads();
}

// The p-th radix of the plan of an n-point line: 8s, then at most one each of
// 4, 6, 10 and 2, then 3s and 5s (0 past the end) -- the rule of the host's axis
// set-up, so that a compile-time plan can be checked against the runtime one
__host__ __device__ constexpr int plan_radix(int n, int p) {
  int rad[16] = {};
  int k = 0, m = n;
  while (m % 8 == 0 && k < 16) { rad[k++] = 8; m /= 8; }
  if (m % 4 == 0) { rad[k++] = 4; m /= 4; }
  if (m % 6 == 0) { rad[k++] = 6; m /= 6; }
  if (m % 10 == 0) { rad[k++] = 10; m /= 10; }
  if (m % 2 == 0) { rad[k++] = 2; m /= 2; }
  while (m % 3 == 0 && k < 16) { rad[k++] = 3; m /= 3; }
  while (m % 5 == 0 && k < 16) { rad[k++] = 5; m /= 5; }
  return p < k ? rad[p] : 0;
}

__host__ __device__ constexpr int plan_ns(int n, int p) {
  int ns = 1;
  for (int i = 0; i < p; ++i) ns *= plan_radix(n, i);
  return ns;
}

template <int S, int EPT, int NT, int N, int LGL, int P>
__device__ __forceinline__ void fft_lines_ct_from(float2* buf, const float2* twl) {
  constexpr int R = plan_radix(N, P);
  if constexpr (R != 0) {
    stockham_pass_ct<R, S, EPT, NT, N, LGL, plan_ns(N, P)>(buf, twl);
    fft_lines_ct_from<S, EPT, NT, N, LGL, P + 1>(buf, twl);
  }
}

// All passes of N-point lines on 2^LGL lines, every size fixed at compile time
template <int S, int EPT, int NT, int N, int LGL>
__device__ __forceinline__ void fft_lines_ct(float2* buf, const float2* twl) {
  fft_lines_ct_from<S, EPT, NT, N, LGL, 0>(buf, twl);
}

// FIX of a kernel whose lines take a runtime plan with a radix-10 pass
constexpr int kTen = -1;

// All passes of the FFT of the L lines in buf; twl is the twiddle table
// staged in LDS by stage_twiddles (visible after the caller's barrier).
// TEN: plans with a radix-10 pass.  Its ten values and their temporaries cost
// every kernel that holds the case up to 12 VGPRs, whatever its own plan (the
// adjoint last-axis pass of 300 and 360 points ran at 2 waves per SIMD instead
// of 3: 150^3, 4 coils 226 us against 163), so only plans that have one take
// these instances (400 points, 200^3, 4 coils: axis-0 pass 838 us against 930
// with 2 and 5 apart).
template <int S, int EPT, int NT = kThreads, bool TEN = false>
__device__ void fft_lines(float2* buf, const float2* twl, const FFTAxis& ax, int lgL, int LP) {
  int Ns = 1;
  for (int p = 0; p < ax.nrad; ++p) {
    const int R = ax.rad[p];
    const uint32_t mg = ax.ns_magic[p];
    switch (R) {
      case 2: stockham_pass<2, S, EPT, NT>(buf, ax.n, lgL, LP, Ns, mg, twl); break;
      case 3: stockham_pass<3, S, EPT, NT>(buf, ax.n, lgL, LP, Ns, mg, twl); break;
      case 4: stockham_pass<4, S, EPT, NT>(buf, ax.n, lgL, LP, Ns, mg, twl); break;
      case 5: stockham_pass<5, S, EPT, NT>(buf, ax.n, lgL, LP, Ns, mg, twl); break;
      case 6: stockham_pass<6, S, EPT, NT>(buf, ax.n, lgL, LP, Ns, mg, twl); break;
      case 10:
        if constexpr (TEN) stockham_pass<10, S, EPT, NT>(buf, ax.n, lgL, LP, Ns, mg, twl);
        break;
      default: stockham_pass<8, S, EPT, NT>(buf, ax.n, lgL, LP, Ns, mg, twl); break;
    }
    Ns *= R;
  }
}

// twiddles go after the n * LP data elements of the dynamic LDS buffer
template <int NT = kThreads>
__device__ __forceinline__ float2* stage_twiddles(float2* buf, const FFTAxis& ax, int LP) {
  float2* twl = buf + ax.n * LP;
  for (int i = threadIdx.x; i < ax.n; i += NT) twl[i] = ax.tw[i];
  return twl;
}

__device__ __forceinline__ int kept_pos(int i, int M, int nf) {
  int p = i - M / 2;
  return p < 0 ? p + nf : p;
}

// ---------------------------------------------------------------------------
// fastest axis, fused with the image side
// ---------------------------------------------------------------------------
struct RowsArgs {
  const float2* img;
  float2* img_out;
  const float2* smaps;
  int C, t0, T;
  int conj_smaps;  // forward: multiply by conj(smap) instead of smap
  int smaps_all;   // smaps hold one map per transform ([B][C]) instead of [C]
  // optional second factor cmap[L][N]: transforms are ordered [B][C][L] and
  // transform tt also multiplies by cmap[tt % L] (off-resonance interpolators)
  const float2* cmap;
  int L;
  float2* grid;
  int64_t gstride;
  int M0, M1, M2;
  int nf0, nf1, nf2;
  const float* dec0;
  const float* dec1;
  const float* dec2;
  float scale;
  FFTAxis ax;
  int lgL;
  int lgQ;  // adjoint: 2^lgQ transforms of an image side by side in a workgroup
};

// image rows -> deconvolve * scale (* smap) -> pad -> FFT -> grid rows
template <int S, int EPT, int FIX = 0, int FLGL = 0>
__global__ __launch_bounds__(kThreads) void k_rows_fwd(RowsArgs a) {
  extern __shared__ float2 buf[];
  // FIX > 0: FIX-point rows, 2^FLGL per workgroup, passes fixed at compile time
  if constexpr (FIX > 0) a.lgL = FLGL;
  const int L = 1 << a.lgL, LP = L + 1;
  const float2* twl = stage_twiddles(buf, a.ax, LP);
  const int rows = a.M0 * a.M1;
  // transforms fastest in the remapped order: the workgroups that read one
  // block of image rows (all coils of an image) run together on one XCD, so
  // the image comes from HBM once rather than once per coil (192^3, 16
  // coils: 0.809 -> 0.788 ms)
  const BlockIdx3 bi = remapped_block();
  const int lin = bi.x + (int)gridDim.x * bi.y;
  const int t = lin % (int)gridDim.y;
  const int r0 = (lin / (int)gridDim.y) * L;
  const int tt = a.t0 + t;
  const int64_t N = (int64_t)rows * a.M2;
  const int n = a.nf2;
  // line-major thread mapping: thread (l, x0) handles positions x0 + j * TPL
  // of row r0 + l (n <= TPL * EPT), so it keeps one row base and one scale
  const int TPL = kThreads >> a.lgL;
  const int l = threadIdx.x / TPL, x0 = threadIdx.x - l * TPL;
  const int r = r0 + l;
  const bool rok = r < rows;
  const int i0 = rok ? r / a.M1 : 0, i1 = rok ? r - i0 * a.M1 : 0;
  const int per_img = (a.smaps ? a.C : 1) * a.L;  // transforms of one image
  const int rl = rok ? r : 0;  // lanes past the last row read row 0 and drop it
  const float2* src = a.img + (int64_t)(tt / per_img) * N + (int64_t)rl * a.M2;
  const float2* sm =
      a.smaps ? a.smaps + (int64_t)(a.smaps_all ? tt : (tt / a.L) % a.C) * N + (int64_t)rl * a.M2
              : nullptr;
  const float2* cm = a.cmap ? a.cmap + (int64_t)(tt % a.L) * N + (int64_t)rl * a.M2 : nullptr;
  const float rs = rok ? a.dec0[i0] * a.dec1[i1] * a.scale : 0.f;
  const int M2 = a.M2, h2 = M2 / 2;

  // loads first, then the arithmetic and LDS stores
  float2 v[EPT], sv[EPT];
  if constexpr (FIX > 0) {
    // all in flight together: no branch and no arithmetic on a loaded value
    // between them (positions past the row end read its last element and
    // are dropped).  The lengths fixed at compile time have the registers
    // for it within the workgroups per CU their LDS allows.
#pragma unroll
    for (int j = 0; j < EPT; ++j) v[j] = src[min(x0 + j * TPL, M2 - 1)];
    if (sm) {
#pragma unroll
      for (int j = 0; j < EPT; ++j) sv[j] = sm[min(x0 + j * TPL, M2 - 1)];
    } else {
#pragma unroll
      for (int j = 0; j < EPT; ++j) sv[j] = make_float2(1.f, 0.f);
    }
    if (cm) {
#pragma unroll
      for (int j = 0; j < EPT; ++j) v[j] = cmul(v[j], cm[min(x0 + j * TPL, M2 - 1)]);
    }
#pragma unroll
    for (int j = 0; j < EPT; ++j)
      if (!rok) v[j] = make_float2(0.f, 0.f);
  } else {
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int x = x0 + j * TPL;
      v[j] = make_float2(0.f, 0.f);
      sv[j] = make_float2(1.f, 0.f);
      if (rok && x < M2) {
        v[j] = src[x];
        if (sm) sv[j] = sm[x];
        if (cm) v[j] = cmul(v[j], cm[x]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int x = x0 + j * TPL;
    if (x < M2) {
      float2 s2 = sv[j];
      if (a.conj_smaps) s2.y = -s2.y;
      const float2 w = cscale(cmul(v[j], s2), rs * a.dec2[x]);
      buf[(x < h2 ? x - h2 + n : x - h2) * LP + l] = w;
    }
  }
  const int gap0 = M2 - h2, gap = n - M2;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int e = x0 + j * TPL;
    if (e < gap) buf[(gap0 + e) * LP + l] = make_float2(0.f, 0.f);
  }
  __syncthreads();
  if constexpr (FIX > 0)
    fft_lines_ct<S, EPT, kThreads, FIX, FLGL>(buf, twl);
  else
    fft_lines<S, EPT, kThreads, FIX == kTen>(buf, twl, a.ax, a.lgL, LP);
  if (!rok) return;
  float2* g = a.grid + (int64_t)t * a.gstride +
              ((int64_t)kept_pos(i0, a.M0, a.nf0) * a.nf1 + kept_pos(i1, a.M1, a.nf1)) * n;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int x = x0 + j * TPL;
    if (x < n) g[x] = buf[x * LP + l];
  }
}

// grid rows -> FFT -> crop -> deconvolve * scale (* conj smap, summed over the
// chunk's coils of one batch) -> image rows
//
// A workgroup's 2^lgL lines are 2^(lgL - lgQ) image rows of 2^lgQ transforms
// each: with many rows a workgroup walks the coils of its rows one by one
// (lgQ = 0), with few rows (2D images) that serial walk on a few workgroups
// is all there is to see -- 32 workgroups for 256 rows, each waiting for one
// coil's loads, FFT and maps after the other -- so the coils go side by side
// and their sums meet in LDS at the end, in coil order.  Measured with
// lgQ = 0 against the rule of rows_adj(): 256^2, 8 coils 47.6 -> 10.3 us,
// 16 coils 89 -> 17; 320^2, 32 coils 233 -> 71 (before its fixed plan); 192^2, 12 frames of 8 coils
// 43 -> 29.
// SIDE: lgQ > 0 (a walk one by one keeps its transform in scalar registers:
// 1024 stacked planes, one transform each, 120 us against 155 without the
// distinction).
template <int S, int EPT, bool SIDE, int FIX = 0, int FLGL = 0>
__global__ __launch_bounds__(kThreads) void k_rows_adj(RowsArgs a) {
  extern __shared__ float2 buf[];
  const int lgQ = SIDE ? a.lgQ : 0;
  // FIX > 0: FIX-point rows, 2^FLGL per workgroup, passes fixed at compile time
  if constexpr (FIX > 0) a.lgL = FLGL;
  const int L = 1 << a.lgL, LP = L + 1;
  const int lgR = a.lgL - lgQ, R = 1 << lgR, Q = 1 << lgQ;
  const float2* twl = stage_twiddles(buf, a.ax, LP);
  const int rows = a.M0 * a.M1;
  const BlockIdx3 bi = remapped_block();
  const int r0 = bi.x * R;
  const int n = a.nf2;
  const int64_t N = (int64_t)rows * a.M2;
  // one output image per image present in the chunk, the sum of its
  // per_img consecutive transforms (coils and / or interpolators)
  const int per_img = (a.smaps ? a.C : 1) * a.L;
  const int out_img = a.t0 / per_img + bi.y;
  const int tb = max(a.t0, out_img * per_img);
  const int te = min(a.t0 + a.T, (out_img + 1) * per_img);
  const bool add_existing = tb % per_img != 0;
  // line-major thread mapping: thread (l, x0) handles positions x0 + j * TPL
  // of line l (row l / Q, transform l % Q of the Q), so it keeps one row base
  // across the coil loop
  const int TPL = kThreads >> a.lgL;  // threads per line (n <= TPL * EPT)
  const int l = threadIdx.x / TPL, x0 = threadIdx.x - l * TPL;
  const int q = SIDE ? l & (Q - 1) : 0;
  const int r = r0 + (l >> lgQ);
  const bool rok = r < rows;
  int64_t grow = 0;
  if (rok) {
    const int i0 = r / a.M1, i1 = r - i0 * a.M1;
    grow = ((int64_t)kept_pos(i0, a.M0, a.nf0) * a.nf1 + kept_pos(i1, a.M1, a.nf1)) * n;
  }
  // sum of the line's transforms, cropped, in LDS after the line data and
  // twiddles; each entry is only touched by the thread that owns it
  float2* acc0 = buf + (size_t)n * (LP + 1);
  float2* accl = acc0 + (size_t)l * a.M2;

  for (int tg = tb; tg < te; tg += Q) {
    const int tt = SIDE ? min(tg + q, te - 1) : tg;
    const bool tok = rok && (!SIDE || tg + q < te);
    const float2* g = a.grid + (int64_t)(tt - a.t0) * a.gstride + grow;
    {
      float2 v[EPT];
#pragma unroll
      for (int j = 0; j < EPT; ++j) {
        const int x = x0 + j * TPL;
        v[j] = (tok && x < n) ? g[x] : make_float2(0.f, 0.f);
      }
#pragma unroll
      for (int j = 0; j < EPT; ++j) {
        const int x = x0 + j * TPL;
        if (x < n) buf[x * LP + l] = v[j];
      }
    }
    __syncthreads();
    // the FFT's addressing is the same for every coil; hiding the line
    // geometry from the optimiser keeps it from hoisting all of it out of the
    // coil loop into registers
    if constexpr (FIX > 0) {
      fft_lines_ct<S, EPT, kThreads, FIX, FLGL>(buf, twl);
    } else {
      int lg = a.lgL, lp = LP;
      asm volatile("" : "+s"(lg), "+s"(lp));
      fft_lines<S, EPT, kThreads, FIX == kTen>(buf, twl, a.ax, lg, lp);
    }
    const int rl = rok ? r : 0;  // lanes past the last row read row 0's maps and drop them
    const float2* sm =
        a.smaps ? a.smaps + (int64_t)(a.smaps_all ? tt : (tt / a.L) % a.C) * N + (int64_t)rl * a.M2
                : nullptr;
    const float2* cm = a.cmap ? a.cmap + (int64_t)(tt % a.L) * N + (int64_t)rl * a.M2 : nullptr;
    // the coil's map values, all loads in flight together (compile-time
    // lengths; the others load each where it is used)
    float2 sv[EPT];
    if constexpr (FIX > 0) {
      if (sm) {
#pragma unroll
        for (int j = 0; j < EPT; ++j) sv[j] = sm[min(x0 + j * TPL, a.M2 - 1)];
      }
    }
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int x = x0 + j * TPL;
      if (x < a.M2) {
        float2 v = make_float2(0.f, 0.f);
        if (tok) {
          v = buf[kept_pos(x, a.M2, n) * LP + l];
          if (sm) {
            float2 s2 = FIX > 0 ? sv[j] : sm[x];
            v = cmul(v, make_float2(s2.x, -s2.y));
          }
          if (cm) {
            float2 cv = cm[x];
            cv.y = -cv.y;
            v = cmul(v, cv);
          }
        }
        accl[x] = (tg == tb) ? v : cadd(accl[x], v);
      }
    }
    __syncthreads();
  }
  // thread (row, x1) sums the Q lines of its row in transform order
  const int TPR = kThreads >> lgR;
  const int ro = threadIdx.x / TPR, x1 = threadIdx.x - ro * TPR;
  const int rr = r0 + ro;
  if (rr >= rows) return;
  const int i0 = rr / a.M1, i1 = rr - i0 * a.M1;
  const float rs = a.dec0[i0] * a.dec1[i1] * a.scale;
  const float2* accr = acc0 + (size_t)(ro << lgQ) * a.M2;
  float2* dst = a.img_out + (int64_t)out_img * N + (int64_t)rr * a.M2;
  for (int x = x1; x < a.M2; x += TPR) {
    float2 v = accr[x];
    for (int k = 1; k < Q; ++k) v = cadd(v, accr[(size_t)k * a.M2 + x]);
    v = cscale(v, rs * a.dec2[x]);
    if (add_existing) v = cadd(v, dst[x]);
    dst[x] = v;
  }
}

// ---------------------------------------------------------------------------
// stacked 2.5D: the Cartesian z axis (the image's last, contiguous axis)
// ---------------------------------------------------------------------------

// Direct DFT of the L lines of n elements in buf (any n): each output is a
// sum over the whole line with twiddle index (j k) mod n advanced by k.
template <int S, int EPT>
__device__ void dft_lines_direct(float2* buf, const float2* twl, int n, int lgL, int LP) {
  const int L = 1 << lgL, E = kThreads >> lgL;
  const int l = threadIdx.x & (L - 1), e0 = threadIdx.x >> lgL;
  float2 out[EPT];
#pragma unroll
  for (int q = 0; q < EPT; ++q) {
    const int k = e0 + q * E;
    float2 acc = make_float2(0.f, 0.f);
    if (k < n) {
      int t = 0;
      for (int j = 0; j < n; ++j) {
        float2 w = twl[t];
        if (S > 0) w.y = -w.y;
        const float2 v = buf[j * LP + l];
        acc.x += v.x * w.x - v.y * w.y;
        acc.y += v.x * w.y + v.y * w.x;
        t += k;
        if (t >= n) t -= n;
      }
    }
    out[q] = acc;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < EPT; ++q) {
    const int k = e0 + q * E;
    if (k < n) buf[k * LP + l] = out[q];
  }
  __syncthreads();
}

template <int S, int EPT, bool TEN>
__device__ __forceinline__ void fft_lines_any(float2* buf, const float2* twl, const FFTAxis& ax,
                                              int lgL, int LP) {
  if (ax.direct)
    dft_lines_direct<S, EPT>(buf, twl, ax.n, lgL, LP);
  else
    fft_lines<S, EPT, kThreads, TEN>(buf, twl, ax, lgL, LP);
}

struct StackArgs {
  const float2* img;
  const float2* smaps;
  float2* planes;         // forward output
  const float2* planes_in;  // adjoint input
  float2* img_out;
  const int32_t* z_index;
  const int32_t* z_plane;
  int C, t0, T;
  int NZ;
  int64_t rows;
  float scale;
  FFTAxis ax;
  int lgL;
};

// rows r0 .. r0 + L of transform t: (smap *) image rows -> centred DFT along
// z -> the NZ sampled positions, written plane-major (L adjacent rows of a
// plane are one contiguous run)
template <int EPT, bool TEN>
__global__ __launch_bounds__(kThreads) void k_stack_fwd(StackArgs a) {
  extern __shared__ float2 buf[];
  const int L = 1 << a.lgL, LP = L + 1;
  const float2* twl = stage_twiddles(buf, a.ax, LP);
  const int Z = a.ax.n, h = Z / 2;
  const int64_t r0 = (int64_t)blockIdx.x * L;
  const int t = blockIdx.y, tt = a.t0 + t;
  // line-major loads: thread (l, x0) holds positions x0 + j * TPL of row r0 + l
  const int TPL = kThreads >> a.lgL;
  {
    const int l = threadIdx.x / TPL, x0 = threadIdx.x - l * TPL;
    const int64_t r = r0 + l;
    const bool rok = r < a.rows;
    const int64_t N = a.rows * Z;
    const float2* src = a.img + (int64_t)(a.smaps ? tt / a.C : tt) * N + r * Z;
    const float2* sm = a.smaps ? a.smaps + (int64_t)(tt % a.C) * N + r * Z : nullptr;
    float2 v[EPT], sv[EPT];
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int x = x0 + j * TPL;
      v[j] = make_float2(0.f, 0.f);
      sv[j] = make_float2(1.f, 0.f);
      if (rok && x < Z) {
        v[j] = src[x];
        if (sm) sv[j] = sm[x];
      }
    }
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int x = x0 + j * TPL;
      // centred input: position x sits at (x - Z/2) mod Z of the DFT line
      if (x < Z) buf[(x < h ? x - h + Z : x - h) * LP + l] = cmul(v[j], sv[j]);
    }
  }
  __syncthreads();
  fft_lines_any<-1, EPT, TEN>(buf, twl, a.ax, a.lgL, LP);
  // plane-major stores: thread (l, i0) writes planes i0 + q * (kThreads / L)
  const int l = threadIdx.x & (L - 1), i0 = threadIdx.x >> a.lgL;
  const int64_t r = r0 + l;
  if (r >= a.rows) return;
  float2* dst = a.planes + (int64_t)t * a.NZ * a.rows + r;
  for (int i = i0; i < a.NZ; i += TPL) {
    const int k = a.z_index[i];  // centred output k is DFT index (k - Z/2) mod Z
    dst[(int64_t)i * a.rows] = cscale(buf[(k < h ? k - h + Z : k - h) * LP + l], a.scale);
  }
}

// rows r0 .. r0 + L of the output image(s) of block y: per transform of the
// chunk, zero-filled z line from the planes -> centred inverse DFT -> conj
// smap, summed over the transforms of one image in registers
template <int EPT, bool TEN>
__global__ __launch_bounds__(kThreads) void k_stack_adj(StackArgs a) {
  extern __shared__ float2 buf[];
  const int L = 1 << a.lgL, LP = L + 1;
  const float2* twl = stage_twiddles(buf, a.ax, LP);
  const int Z = a.ax.n, h = Z / 2;
  const int64_t r0 = (int64_t)blockIdx.x * L;
  int tb, te, out_img;
  if (a.smaps) {
    const int b = a.t0 / a.C + blockIdx.y;
    out_img = b;
    tb = max(a.t0, b * a.C);
    te = min(a.t0 + a.T, (b + 1) * a.C);
  } else {
    out_img = a.t0 + blockIdx.y;
    tb = out_img;
    te = out_img + 1;
  }
  const bool add_existing = a.smaps && (tb % a.C != 0);
  const int TPL = kThreads >> a.lgL;
  const int lq = threadIdx.x & (L - 1), q0 = threadIdx.x >> a.lgL;  // gather mapping
  const int lr = threadIdx.x / TPL, x0 = threadIdx.x - lr * TPL;    // row mapping
  const int64_t rq = r0 + lq, rr = r0 + lr;
  const int64_t N = a.rows * Z;
  float2 acc[EPT];
#pragma unroll
  for (int j = 0; j < EPT; ++j) acc[j] = make_float2(0.f, 0.f);
  for (int tt = tb; tt < te; ++tt) {
    const float2* pl = a.planes_in + (int64_t)(tt - a.t0) * a.NZ * a.rows + rq;
    // DFT position j holds centred position (j + Z/2) mod Z
    for (int j = q0; j < Z; j += TPL) {
      const int k = j + h < Z ? j + h : j + h - Z;
      const int i = a.z_plane[k];
      buf[j * LP + lq] = (i >= 0 && rq < a.rows) ? pl[(int64_t)i * a.rows] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    fft_lines_any<1, EPT, TEN>(buf, twl, a.ax, a.lgL, LP);
    const float2* sm = a.smaps ? a.smaps + (int64_t)(tt % a.C) * N + rr * Z : nullptr;
#pragma unroll
    for (int j = 0; j < EPT; ++j) {
      const int x = x0 + j * TPL;
      if (x < Z && rr < a.rows) {
        float2 v = cscale(buf[(x < h ? x - h + Z : x - h) * LP + lr], a.scale);
        if (sm) {
          float2 sv = sm[x];
          sv.y = -sv.y;
          v = cmul(v, sv);
        }
        acc[j] = cadd(acc[j], v);
      }
    }
    __syncthreads();
  }
  if (rr >= a.rows) return;
  float2* dst = a.img_out + (int64_t)out_img * N + rr * Z;
#pragma unroll
  for (int j = 0; j < EPT; ++j) {
    const int x = x0 + j * TPL;
    if (x < Z) dst[x] = add_existing ? cadd(acc[j], dst[x]) : acc[j];
  }
}

// ---------------------------------------------------------------------------
// strided axes (0 and 1), in place
// ---------------------------------------------------------------------------
struct StridedArgs {
  float2* data;
  int64_t tstride;
  int n;
  int64_t lstride;
  int nouter, outer_M, outer_nf;  // outer_M > 0: outer index i maps to kept_pos
  int64_t ostride;
  int nx;
  int in_M, out_M;  // 0: full line, > 0: kept positions only
  FFTAxis ax;
  int lgL;
  const float2* K;  // CONV: spectrum (one grid) applied between the FFTs
  // tiles along the axis whose cells the points' footprints touch, one mask
  // per (outer tile, column tile) (line_mask); the other positions of the
  // full side of the pass (its output forward, its input backward) are
  // neither stored nor loaded.  null: all positions count
  const uint64_t* lmask;
  int otile_sh, tile_sh, ctile_sh;  // log2 of the tile along the outer axis, the line, the columns
  int mrow;        // masks per outer tile (0: the outer axis does not select)
  int zero_empty;  // store zeros for a line without any touched tile (else skip it)
};

// A cell at a uniform base plus a per-thread byte offset.  The offset is
// hidden from the optimiser at each access: seen as one value it is widened
// to 64 bits once, far from the accesses, which then no longer take the form
// with a scalar base and a 32-bit offset but a vector address of their own
__device__ __forceinline__ float2 load_at(const char* base, uint32_t off) {
  asm("" : "+v"(off));
  return *reinterpret_cast<const float2*>(base + off);
}
__device__ __forceinline__ void store_at(char* base, uint32_t off, float2 v) {
  asm("" : "+v"(off));
  *reinterpret_cast<float2*>(base + off) = v;
}

// In-place FFT of L adjacent lines along a strided axis.  CONV: forward FFT,
// multiply by the spectrum K, inverse FFT, all in LDS (the middle of the
// Toeplitz convolution, one grid round trip instead of three).
//
// Memory and vector arithmetic bound the pass about equally, so it gains by
// moving less and by addressing for free:
// - positions outside the tiles that footprints touch (lmask) are neither
//   loaded nor stored, lines without any are skipped;
// - a wave holds 64 / L consecutive positions per slot.  Tiles are at least
//   that long and aligned (see build_line_masks), so whether a slot counts,
//   and on which side of the wrap of a kept half it lies, is one scalar
//   branch per wave, and every address is a scalar base plus a 32-bit offset
//   per thread; loads are buffer loads bounded by the lines' end;
// - the twiddles are staged behind the lines' loads: before them, they cost
//   every workgroup a memory latency of its own.
// 192^3, 16 coils, 3D radial (a ball): both forward passes 3.60 -> 3.22 ms,
// both backward ones 3.43 -> 2.98 (2.90 and 2.78 with the kept halves' loop at
// the end rolled); nothing to skip: 256^3 Toeplitz grids, 8 coils, 0.84 ->
// 0.80 ms, 320^2, 32 coils 116 -> 116 us.
// HUGE: lines of 4 GiB or more, whose cells need 64-bit offsets.
template <int S, bool CONV, int EPT, int NT, bool HUGE, int FIX = 0, int FLGL = 0>
__global__ __launch_bounds__(NT) void k_fft_strided(StridedArgs a) {
  extern __shared__ float2 buf[];
  // FIX > 0: FIX-point lines, 2^FLGL per workgroup, passes fixed at compile time
  if constexpr (FIX > 0) {
    a.lgL = FLGL;
    a.n = FIX;
  }
  const int L = 1 << a.lgL, LP = L + 1;
  const BlockIdx3 bi = remapped_block();
  const int x0 = bi.x * L;
  const int oi = bi.y;
  const int t = bi.z;
  const int opos = a.outer_M ? kept_pos(oi, a.outer_M, a.outer_nf) : oi;
  // the touched tiles of these lines (uniform: the L columns share a tile)
  uint64_t tm0 = ~(uint64_t)0, tm1 = ~(uint64_t)0;
  bool empty = false;
  static_assert(kMaskWords == 2, "two words");
  if constexpr (!CONV) {
    if (a.lmask) {
      const uint64_t* lm =
          a.lmask + kMaskWords * ((int64_t)a.mrow * (opos >> a.otile_sh) + (x0 >> a.ctile_sh));
      tm0 = lm[0];
      tm1 = lm[1];
      empty = (tm0 | tm1) == 0;
      if (empty && !a.zero_empty) return;
    }
  }
  // thread -> (line l, positions e0 + i*E, i < EPT); n <= EPT * E
  const int E = NT >> a.lgL;
  const int PW = 64 >> a.lgL;  // positions of a wave's slot
  const int l = threadIdx.x & (L - 1), e0 = threadIdx.x >> a.lgL;
  const int wpos = __builtin_amdgcn_readfirstlane(e0);
  const bool lok = x0 + l < a.nx;
  const int n = a.n;
  const int64_t ls8 = a.lstride * (int64_t)sizeof(float2);
  const int64_t line0 = (int64_t)t * a.tstride + (int64_t)opos * a.ostride + x0;
  char* lines = reinterpret_cast<char*>(a.data + line0);                // uniform
  const int cols = min(L, a.nx - x0);
  const int lc = min(l, cols - 1);  // lanes past the last column repeat it and store nothing
  const uint32_t v0 = strided_thread_offset(e0, a.lstride, lc);         // per thread
  const int hin = a.in_M / 2, hout = a.out_M / 2;
  // slot i of the full side counts
  auto full = [&](int i) {
    const int w0 = wpos + i * E;
    if constexpr (CONV) return w0 < n;
    const int tt = w0 >> a.tile_sh;
    return w0 < n && (((tt & 64 ? tm1 : tm0) >> (tt & 63)) & 1);
  };
  const bool whole = FIX > 0 && EPT * (NT >> FLGL) == FIX;  // no slot passes the line's end

  // kept positions: e of the M kept ones sits at e - h (+ n if e < h).  Where
  // M and h are multiples of PW a wave's slot is kept, and wraps, as one
  const int q0 = e0 * LP + l;
  const int64_t step8 = (int64_t)E * ls8;

  // all of a thread's loads are issued before the first LDS store, so they
  // overlap instead of paying one memory latency each.  One code path and no
  // per-thread branch: alternatives for a register would wait for each
  // other's loads.  A wave's slot that holds the last position is loaded as
  // one: its lanes past it load another cell of their lines, or nothing past
  // the lines' end, and drop it.  (Bounded by the buffer's length the pass
  // costs less than with each lane's offset clamped: over unbounded loads,
  // 0.5 against 0.8% of the 128^3 Toeplitz call, 0.1 against 0.3% of the
  // 192^3, 16-coil adjoint.)
  float2 v[EPT];
  const int nin = a.in_M ? a.in_M : n;
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      lines, (short)0, (int)strided_line_bytes(n, a.lstride, cols), kBufferWord3);
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const int w0 = wpos + i * E, e = e0 + i * E;
    v[i] = make_float2(0.f, 0.f);
    if (a.in_M ? w0 < a.in_M : full(i)) {
      if constexpr (HUGE) {
        const int el = min(e, nin - 1);
        v[i] = *reinterpret_cast<const float2*>(
            lines + (el - hin + (el < hin ? n : 0)) * ls8 + (int64_t)lc * 8);
      } else {
        v[i] = __builtin_bit_cast(
            float2, __builtin_amdgcn_raw_buffer_load_b64(
                        rs,
                        (int)strided_cell_offset(v0, strided_slot_offset(i, E, hin, a.lstride), e,
                                                 hin, (uint32_t)(n * ls8)),
                        0, 0));
      }
    }
  }
  // (the twiddles' round trip overlaps the lines')
  const float2* twl = stage_twiddles<NT>(buf, a.ax, LP);
  if (a.in_M) {
    if ((a.in_M | hin) % PW == 0) {
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        const int w0 = wpos + i * E;
        if (w0 < a.in_M) buf[q0 + (i * E - hin + (w0 < hin ? n : 0)) * LP] = v[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < EPT; ++i) {
        const int e = e0 + i * E;
        if (e < a.in_M) buf[(e - hin + (e < hin ? n : 0)) * LP + l] = v[i];
      }
    }
    // zero the positions between the kept halves
    const int gap0 = a.in_M - hin, gap = n - a.in_M;
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (e0 + i * E < gap) buf[q0 + (gap0 + i * E) * LP] = make_float2(0.f, 0.f);
  } else {
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (whole || e0 + i * E < n) buf[q0 + i * E * LP] = v[i];
  }
  __syncthreads();
  if (!empty) {  // (uniform; the lines of an empty one are zero either way)
    if constexpr (FIX > 0)
      fft_lines_ct<S, EPT, NT, FIX, FLGL>(buf, twl);
    else
      fft_lines<S, EPT, NT, FIX == kTen>(buf, twl, a.ax, a.lgL, LP);
  }
  if constexpr (CONV) {
    const char* kl = reinterpret_cast<const char*>(a.K + (int64_t)opos * a.ostride + x0);
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      v[i] = make_float2(0.f, 0.f);
      if (whole || e0 + i * E < n)
        v[i] = load_at(kl + i * step8, v0);
    }
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (whole || e0 + i * E < n) buf[q0 + i * E * LP] = cmul(buf[q0 + i * E * LP], v[i]);
    __syncthreads();
    if constexpr (FIX > 0)
      fft_lines_ct<-S, EPT, NT, FIX, FLGL>(buf, twl);
    else
      fft_lines<-S, EPT, NT, FIX == kTen>(buf, twl, a.ax, a.lgL, LP);
  }
  if (!lok) return;
  if (!a.out_M) {
    char* p = lines;
#pragma unroll
    for (int i = 0; i < EPT; ++i, p += step8)
      if (full(i) && (whole || e0 + i * E < n))
        store_at(p, v0, buf[q0 + i * E * LP]);
  } else if ((a.out_M | hout) % PW == 0) {
    char* p = lines - hout * ls8;
#pragma unroll
    for (int i = 0; i < EPT; ++i, p += step8) {
      const int w0 = wpos + i * E;
      if (w0 < a.out_M)
        store_at(p + (w0 < hout ? n * ls8 : 0), v0,
                 buf[q0 + (i * E - hout + (w0 < hout ? n : 0)) * LP]);
    }
  } else {
    // A kept half that is no multiple of a wave's positions.  A loop, not
    // unrolled: a dozen copies of it cost the other forms their place in the
    // instruction cache (192^3, 16 coils, which never come here: axis-0 pass
    // 1.99 -> 1.85 ms forward, 1.89 -> 1.77 adjoint).  32-bit offsets where the
    // length is not fixed (150^3, 4 coils, axis 0: 437 us with 64, 418); in the
    // fixed-length kernels they changed the other forms for the worse (1.85 ->
    // 2.02), and 64 bits cost them nothing here (126^3: 153 us either way).
#pragma unroll 1
    for (int e = e0; e < a.out_M; e += E) {
      const int pos = e - hout + (e < hout ? n : 0);
      if constexpr (HUGE || FIX > 0)
        *reinterpret_cast<float2*>(lines + (int64_t)pos * ls8 + 8 * l) = buf[pos * LP + l];
      else
        store_at(lines, strided_thread_offset(pos, a.lstride, lc), buf[pos * LP + l]);
    }
  }
}

int lg2(int x) {
  int l = 0;
  while ((1 << l) < x) ++l;
  return l;
}

size_t fft_lds(const FFTAxis& ax, int L) { return sizeof(float2) * (size_t)ax.n * (L + 2); }
size_t fft_lds(const FFTAxis& ax) { return fft_lds(ax, ax.L); }

// the axis has n points and its runtime radix plan is the compile-time one
// of fft_lines_ct
bool fixed_plan(const FFTAxis& ax, int n) {
  if (ax.n != n || ax.direct) return false;
  int p = 0;
  for (; p < ax.nrad; ++p)
    if (ax.rad[p] != plan_radix(n, p)) return false;
  return plan_radix(n, p) == 0;
}

// the axis's runtime plan has a radix-10 pass
bool has_ten(const FFTAxis& ax) {
  return std::find(ax.rad, ax.rad + ax.nrad, 10) != ax.rad + ax.nrad;
}

// complex elements per thread for L lines of n elements: the smallest of 4,
// 8, 12, 16 with n * L <= EPT * nt (fewer registers, more resident waves for
// the shorter lines)
int ept_of(int n, int L, int nt = kThreads) {
  const int need = (n * L + nt - 1) / nt;
  return need <= 4 ? 4 : need <= 8 ? 8 : need <= 12 ? 12 : 16;
}

#define HN_EPT_SWITCH(ept, ...)             \
  switch (ept) {                            \
    case 4: { constexpr int EE = 4; __VA_ARGS__ } break;   \
    case 8: { constexpr int EE = 8; __VA_ARGS__ } break;   \
    case 12: { constexpr int EE = 12; __VA_ARGS__ } break; \
    default: { constexpr int EE = 16; __VA_ARGS__ } break; \
  }

}  // namespace

// k_rows_adj also keeps the coil sum of its L cropped lines in LDS
size_t rows_adj_lds(const FFTAxis& ax, int64_t m2) {
  return fft_lds(ax) + sizeof(float2) * (size_t)m2 * ax.L;
}

namespace {

template <int EPT, int NT, int FIX = 0, int FLGL = 0>
void launch_strided(bool conv, int sign, dim3 grd, size_t lds, hipStream_t s,
                    const StridedArgs& a) {
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grd, dim3(NT), lds, s, a); };
  // 4 GiB lines have more than 64 positions and are never few: no quarter of
  // the lines per workgroup, more than 4 elements per thread
  if constexpr (EPT > 4) {
    if (!strided_fits_32(a.n, a.lstride, a.nx)) {
      if (conv && sign < 0) go(k_fft_strided<-1, true, EPT, NT, true, FIX, FLGL>);
      else if (conv) go(k_fft_strided<1, true, EPT, NT, true, FIX, FLGL>);
      else if (sign < 0) go(k_fft_strided<-1, false, EPT, NT, true, FIX, FLGL>);
      else go(k_fft_strided<1, false, EPT, NT, true, FIX, FLGL>);
      return;
    }
  }
  if (conv && sign < 0) go(k_fft_strided<-1, true, EPT, NT, false, FIX, FLGL>);
  else if (conv) go(k_fft_strided<1, true, EPT, NT, false, FIX, FLGL>);
  else if (sign < 0) go(k_fft_strided<-1, false, EPT, NT, false, FIX, FLGL>);
  else go(k_fft_strided<1, false, EPT, NT, false, FIX, FLGL>);
}

int strided(const hipnufft_plan_s* p, int axis, int T, int in_M, int out_M, int outer_M,
            int sign, int stage, const float2* K = nullptr) {
  const FFTAxis& ax = p->fft[axis];
  StridedArgs a{};
  a.data = p->grid;
  a.tstride = grid_size(p);
  a.n = (int)p->nf[axis];
  a.nx = (int)p->nf[2];
  a.in_M = in_M;
  a.out_M = out_M;
  a.ax = ax;
  if (axis == 1) {
    a.lstride = p->nf[2];
    a.ostride = p->nf[1] * p->nf[2];
    a.outer_nf = (int)p->nf[0];
  } else {
    a.lstride = p->nf[1] * p->nf[2];
    a.ostride = p->nf[2];
    a.outer_nf = (int)p->nf[1];
  }
  a.outer_M = outer_M;
  a.nouter = outer_M ? outer_M : a.outer_nf;
  a.K = K;
  if (p->prune && !K) {
    // axis 0: masks per (tile of axis 1, tile of axis 2); axis 1: per tile of
    // axis 2.  Backward, the last-axis pass reads every kept position that
    // the axis-1 pass leaves, so that one stores zeros for empty lines
    a.lmask = p->line_mask + (axis == 0 ? 0 : (int64_t)kMaskWords * p->nt[1] * p->nt[2]);
    a.mrow = axis == 0 ? p->nt[2] : 0;
    a.otile_sh = lg2(p->tile[1]);
    a.tile_sh = lg2(p->tile[axis]);
    a.ctile_sh = lg2(p->tile[2]);
    a.zero_empty = axis == 1 && out_M != 0;
  }
  const int L = lines_of(ax.L, (int64_t)a.nx * a.nouter * T, a.lmask ? 64 / p->tile[axis] : 1);
  a.lgL = lg2(L);
  const dim3 grd((unsigned)((a.nx + L - 1) / L), (unsigned)a.nouter, (unsigned)T);
  StageScope timer(p, stage);
  const size_t lds = fft_lds(ax, L);
  // strided axes may hold up to 2 * kMaxElemsFFT elements (16 lines of up to
  // 512): those run 512-thread workgroups
// compile-time plans: points, log2 lines, threads, elements per thread
#define HN_STRIDED_FIXED(NN, LG, NTT, EPTT)                                   \
  if (L == 1 << LG && fixed_plan(ax, NN)) {                                     \
    launch_strided<EPTT, NTT, NN, LG>(K != nullptr, sign, grd, lds, p->stream, a); \
    HN_LAUNCH_CHECK();                                                          \
    return 0;                                                                   \
  }
  HN_STRIDED_FIXED(384, 4, 2 * kThreads, 12)
  HN_STRIDED_FIXED(384, 2, 2 * kThreads, 3)
  HN_STRIDED_FIXED(256, 4, kThreads, 16)
  HN_STRIDED_FIXED(256, 2, kThreads, 4)
  HN_STRIDED_FIXED(512, 3, kThreads, 16)
  HN_STRIDED_FIXED(512, 1, kThreads, 4)
  HN_STRIDED_FIXED(768, 3, 2 * kThreads, 12)
  HN_STRIDED_FIXED(768, 1, 2 * kThreads, 3)
  HN_STRIDED_FIXED(640, 3, 2 * kThreads, 10)
  HN_STRIDED_FIXED(640, 1, 2 * kThreads, 3)
  HN_STRIDED_FIXED(320, 4, 2 * kThreads, 10)
  HN_STRIDED_FIXED(192, 4, kThreads, 12)
  HN_STRIDED_FIXED(128, 4, kThreads, 8)
#undef HN_STRIDED_FIXED
  const bool ten = has_ten(ax);
  if (ax.n * L > kMaxElemsFFT) {
    // (more than 8 elements per thread)
    auto go = [&](auto ept) {
      constexpr int EE = decltype(ept)::value, NT2 = 2 * kThreads;
      if (ten) launch_strided<EE, NT2, kTen>(K != nullptr, sign, grd, lds, p->stream, a);
      else launch_strided<EE, NT2>(K != nullptr, sign, grd, lds, p->stream, a);
    };
    if (ept_of(ax.n, L, 2 * kThreads) <= 12) go(std::integral_constant<int, 12>{});
    else go(std::integral_constant<int, 16>{});
  } else {
    HN_EPT_SWITCH(ept_of(ax.n, L), {
      if (ten) launch_strided<EE, kThreads, kTen>(K != nullptr, sign, grd, lds, p->stream, a);
      else launch_strided<EE, kThreads>(K != nullptr, sign, grd, lds, p->stream, a);
    });
  }
  HN_LAUNCH_CHECK();
  return 0;
}

RowsArgs rows_args(const hipnufft_plan_s* p) {
  RowsArgs a{};
  a.grid = p->grid;
  a.gstride = grid_size(p);
  a.M0 = (int)p->N[0];
  a.M1 = (int)p->N[1];
  a.M2 = (int)p->N[2];
  a.nf0 = (int)p->nf[0];
  a.nf1 = (int)p->nf[1];
  a.nf2 = (int)p->nf[2];
  a.dec0 = p->dec[0];
  a.dec1 = p->dec[1];
  a.dec2 = p->dec[2];
  a.ax = p->fft[2];
  a.lgL = lg2(p->fft[2].L);
  a.L = 1;
  return a;
}

}  // namespace

int64_t grid_size(const hipnufft_plan_s* p) { return p->nf[0] * p->nf[1] * p->nf[2]; }

namespace {

// grid[t][i] *= K[i] for the T grids of a chunk (the Toeplitz spectrum)
__global__ __launch_bounds__(kThreads) void k_mul_spectrum(float2* grid, const float2* K, int64_t G) {
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= G) return;
  float2* g = grid + (int64_t)blockIdx.y * G;
  g[i] = cmul(g[i], K[i]);
}

}  // namespace

int mul_spectrum(const hipnufft_plan_s* p, const float2* K, int T) {
  const int64_t G = grid_size(p);
  if (T <= 0 || G <= 0) return 0;
  const dim3 grd((unsigned)((G + kThreads - 1) / kThreads), (unsigned)T);
  hipLaunchKernelGGL(k_mul_spectrum, grd, dim3(kThreads), 0, p->stream, p->grid, K, G);
  HN_LAUNCH_CHECK();
  return 0;
}

namespace {

// the row kernels with compile-time plans (points, log2 lines, elements per
// thread), else the runtime plan (640 points, of 320^2 with 32 coils:
// forward rows 37 -> 27 us, adjoint rows 70 -> 41, each column pass 58 -> 36)
#define HN_ROWS_FIXED(NN, LG, EPTT)         \
  if (L == 1 << LG && fixed_plan(ax, NN)) { \
    HN_ROWS(EPTT, NN, LG);                  \
  } else
#define HN_ROWS_SWITCH                                                    \
  HN_ROWS_FIXED(384, 3, 12)                                               \
  HN_ROWS_FIXED(384, 1, 3)                                                \
  HN_ROWS_FIXED(256, 4, 16)                                               \
  HN_ROWS_FIXED(256, 2, 4)                                                \
  HN_ROWS_FIXED(512, 3, 16)                                               \
  HN_ROWS_FIXED(512, 1, 4)                                                \
  HN_ROWS_FIXED(768, 2, 12)                                               \
  HN_ROWS_FIXED(768, 0, 3)                                                \
  HN_ROWS_FIXED(640, 2, 10)                                               \
  HN_ROWS_FIXED(640, 0, 3)                                                \
  HN_ROWS_FIXED(320, 3, 10)                                               \
  HN_ROWS_FIXED(192, 4, 12)                                               \
  HN_ROWS_FIXED(128, 4, 8)                                                \
  if (has_ten(ax)) {                                                      \
    HN_EPT_SWITCH(ept_of(ax.n, L), { HN_ROWS(EE, kTen); });               \
  } else {                                                                \
    HN_EPT_SWITCH(ept_of(ax.n, L), { HN_ROWS(EE); });                     \
  }

int rows_fwd(const hipnufft_plan_s* p, const float2* img, const float2* smaps, int C, int t0, int T,
             float scale, int sign, int conj_smaps, int smaps_all, const float2* cmap = nullptr,
             int nmaps = 1) {
  RowsArgs a = rows_args(p);
  a.conj_smaps = conj_smaps;
  a.smaps_all = smaps_all;
  a.cmap = cmap;
  a.L = nmaps;
  a.img = img;
  a.smaps = smaps;
  a.C = C;
  a.t0 = t0;
  a.T = T;
  a.scale = scale;
  const int rows = a.M0 * a.M1;
  const FFTAxis& ax = p->fft[2];
  const int L = lines_of(ax.L, (int64_t)rows * T);
  a.lgL = lg2(L);
  const dim3 grd((unsigned)((rows + L - 1) / L), (unsigned)T);
  const size_t lds = fft_lds(ax, L);
  StageScope timer(p, kStageRowsFwd);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grd, dim3(kThreads), lds, p->stream, a);
  };
#define HN_ROWS(...)                            \
  if (sign < 0) go(k_rows_fwd<-1, __VA_ARGS__>); \
  else go(k_rows_fwd<1, __VA_ARGS__>)
  HN_ROWS_SWITCH
#undef HN_ROWS
  HN_LAUNCH_CHECK();
  return 0;
}

int rows_adj(const hipnufft_plan_s* p, float2* img, const float2* smaps, int C, int t0, int T,
             float scale, int sign, int smaps_all, const float2* cmap = nullptr, int nmaps = 1) {
  RowsArgs a = rows_args(p);
  a.img_out = img;
  a.smaps = smaps;
  a.smaps_all = smaps_all;
  a.cmap = cmap;
  a.L = nmaps;
  a.C = C;
  a.t0 = t0;
  a.T = T;
  a.scale = scale;
  const int rows = a.M0 * a.M1;
  const FFTAxis& ax = p->fft[2];
  const int per_img = (smaps ? C : 1) * nmaps;
  const int nimg = (t0 + T - 1) / per_img - t0 / per_img + 1;
  const int L = lines_of(ax.L, (int64_t)rows * std::min(T, per_img * nimg));
  a.lgL = lg2(L);
  // transforms of an image side by side while the rows alone give fewer than
  // two workgroups per CU (each then walks fewer coils)
  while ((1 << a.lgQ) < L && (1 << a.lgQ) < std::min(per_img, T) &&
         (int64_t)((rows * (int64_t)(1 << a.lgQ) + L - 1) / L) * nimg < 512)
    ++a.lgQ;
  const int R = L >> a.lgQ;
  const dim3 grd((unsigned)((rows + R - 1) / R), (unsigned)nimg);
  const size_t lds = fft_lds(ax, L) + sizeof(float2) * (size_t)a.M2 * L;
  StageScope timer(p, kStageRowsAdj);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grd, dim3(kThreads), lds, p->stream, a);
  };
#define HN_ROWS(EPTT, ...)                                                  \
  if (sign < 0 && a.lgQ) go(k_rows_adj<-1, EPTT, true, ##__VA_ARGS__>);       \
  else if (sign < 0) go(k_rows_adj<-1, EPTT, false, ##__VA_ARGS__>);          \
  else if (a.lgQ) go(k_rows_adj<1, EPTT, true, ##__VA_ARGS__>);               \
  else go(k_rows_adj<1, EPTT, false, ##__VA_ARGS__>)
  HN_ROWS_SWITCH
#undef HN_ROWS
  HN_LAUNCH_CHECK();
  return 0;
}

}  // namespace

int fwd_to_grid(const hipnufft_plan_s* p, const float2* img, const float2* smaps, int C, int t0,
                int T, float scale, int sign, int conj_smaps, int smaps_all, const float2* cmap,
                int L) {
  if (T <= 0) return 0;
  int rc = rows_fwd(p, img, smaps, C, t0, T, scale, sign, conj_smaps, smaps_all, cmap, L);
  if (rc) return rc;
  if (p->ndim >= 2 &&
      (rc = strided(p, 1, T, (int)p->N[1], 0, (int)p->N[0], sign, kStageColsFwd)))
    return rc;
  if (p->ndim == 3 && (rc = strided(p, 0, T, (int)p->N[0], 0, 0, sign, kStageSlabsFwd)))
    return rc;
  return 0;
}

int grid_to_img(const hipnufft_plan_s* p, float2* img, const float2* smaps, int C, int t0, int T,
                float scale, int sign, int smaps_all, const float2* cmap, int L) {
  if (T <= 0) return 0;
  int rc;
  if (p->ndim == 3 && (rc = strided(p, 0, T, 0, (int)p->N[0], 0, sign, kStageSlabsAdj)))
    return rc;
  if (p->ndim >= 2 &&
      (rc = strided(p, 1, T, 0, (int)p->N[1], (int)p->N[0], sign, kStageColsAdj)))
    return rc;
  return rows_adj(p, img, smaps, C, t0, T, scale, sign, smaps_all, cmap, L);
}

int gram_chain(const hipnufft_plan_s* p, const float2* img, const float2* smaps, float2* out,
               const float2* K, int C, int t0, int T) {
  if (T <= 0) return 0;
  int rc;
  if (p->ndim == 1) {  // the only FFT axis is the contiguous one: unfused
    if ((rc = fwd_to_grid(p, img, smaps, C, t0, T, 1.0f, -1))) return rc;
    if ((rc = mul_spectrum(p, K, T))) return rc;
    return grid_to_img(p, out, smaps, C, t0, T, 1.0f, 1);
  }
  if ((rc = rows_fwd(p, img, smaps, C, t0, T, 1.0f, -1, 0, 0))) return rc;
  if (p->ndim == 3) {
    if ((rc = strided(p, 1, T, (int)p->N[1], 0, (int)p->N[0], -1, kStageColsFwd))) return rc;
    // axis 0: forward FFT, spectrum, inverse FFT in one pass
    if ((rc = strided(p, 0, T, (int)p->N[0], (int)p->N[0], 0, -1, kStageSlabsFwd, K))) return rc;
    if ((rc = strided(p, 1, T, 0, (int)p->N[1], (int)p->N[0], 1, kStageColsAdj))) return rc;
  } else {
    if ((rc = strided(p, 1, T, (int)p->N[1], (int)p->N[1], (int)p->N[0], -1, kStageColsFwd, K)))
      return rc;
  }
  return rows_adj(p, out, smaps, C, t0, T, 1.0f, 1, 0);
}

int stack_fwd(const StackGeom& g, const float2* img, const float2* smaps, int C, int t0, int T,
              float scale, float2* planes, hipStream_t s) {
  if (T <= 0 || g.rows <= 0) return 0;
  StackArgs a{};
  a.img = img;
  a.smaps = smaps;
  a.planes = planes;
  a.z_index = g.z_index;
  a.C = C;
  a.t0 = t0;
  a.T = T;
  a.NZ = g.NZ;
  a.rows = g.rows;
  a.scale = scale;
  a.ax = g.ax;
  a.lgL = lg2(g.ax.L);
  const dim3 grd((unsigned)((g.rows + g.ax.L - 1) / g.ax.L), (unsigned)T);
  HN_EPT_SWITCH(ept_of(g.ax.n, g.ax.L), {
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grd, dim3(kThreads), fft_lds(g.ax), s, a);
    };
    if (has_ten(g.ax)) go(k_stack_fwd<EE, true>);
    else go(k_stack_fwd<EE, false>);
  });
  HN_LAUNCH_CHECK();
  return 0;
}

int stack_adj(const StackGeom& g, const float2* planes, const float2* smaps, int C, int t0, int T,
              float scale, float2* img, hipStream_t s) {
  if (T <= 0 || g.rows <= 0) return 0;
  StackArgs a{};
  a.planes_in = planes;
  a.smaps = smaps;
  a.img_out = img;
  a.z_plane = g.z_plane;
  a.C = C;
  a.t0 = t0;
  a.T = T;
  a.NZ = g.NZ;
  a.rows = g.rows;
  a.scale = scale;
  a.ax = g.ax;
  a.lgL = lg2(g.ax.L);
  const int nimg = smaps ? ((t0 + T - 1) / C - t0 / C + 1) : T;
  const dim3 grd((unsigned)((g.rows + g.ax.L - 1) / g.ax.L), (unsigned)nimg);
  HN_EPT_SWITCH(ept_of(g.ax.n, g.ax.L), {
    auto go = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, grd, dim3(kThreads), fft_lds(g.ax), s, a);
    };
    if (has_ten(g.ax)) go(k_stack_adj<EE, true>);
    else go(k_stack_adj<EE, false>);
  });
  HN_LAUNCH_CHECK();
  return 0;
}

}  // namespace hn
