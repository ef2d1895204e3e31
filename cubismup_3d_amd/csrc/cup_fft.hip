// cup_fft.hip -- hand-written 3-D real-to-complex FFT for the periodic Poisson solve.
//
// Spectral layout ("packed half spectrum"): complex S[z][y][kx], kx in [0, Nx/2). The
// x transform is real-to-complex; its kx = 0 and kx = Nx/2 outputs are both real and are
// packed into slot 0 as (X[0], X[Nx/2]). The y and z transforms then act on Nx/2 complex
// columns. Slot 0 carries A + iB with A, B the kx = 0 and kx = Nx/2 planes; because the
// grid-consistent Poisson symbol is real, even, and equal at kx = 0 and kx = Nx/2
// (cos(4 pi k/N) = 1 at both), dividing the packed column by the kx = 0 symbol solves both
// planes at once.
//
// Passes (each one HBM read + write of S; x FFTs run in LDS, radix 8/4/2 Stockham; y and z
// FFTs of 64 to 256 points in registers with one LDS transpose, others as the x FFTs):
//   x-forward : 8 rows (one block row of a z plane) per workgroup, two real rows packed
//               into one complex FFT; the source is either a real block-layout field or,
//               fused, the central divergence of the advected velocity (PressureRHS).
//   y         : TK consecutive kx columns x all y of one z plane per workgroup.
//   z         : TK columns x all z of one y row; fused: forward, spectral division, inverse.
//   x-inverse : 8 rows per workgroup, complex-to-real, written into a block-layout field.
// Unnormalized in both directions like FFTW's r2c/c2r; the 1/N^3 and h factors live in the
// division (PoissonSolverPeriodic.cpp:23-35).
//
// Compiled in two halves, for the build's time: the FP64 forms by cup_fft_f64.hip, which includes this
// file, everything else here.
#include "cup_internal.h"
#include "cup_forcing_dev.h"

#include <algorithm>
#include <cmath>
#include <new>
#include <type_traits>
#include <vector>

namespace cup {

template <typename T>
__device__ __forceinline__ C2<T> cmul(C2<T> a, C2<T> b)
{
  return C2<T>{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T>
__device__ __forceinline__ C2<T> cadd(C2<T> a, C2<T> b) { return C2<T>{a.x + b.x, a.y + b.y}; }
template <typename T>
__device__ __forceinline__ C2<T> csub(C2<T> a, C2<T> b) { return C2<T>{a.x - b.x, a.y - b.y}; }
// a * e^{DIR i pi/2}: DIR=-1 -> -i a, DIR=+1 -> +i a
template <int DIR, typename T>
__device__ __forceinline__ C2<T> rot90(C2<T> a)
{
  return DIR < 0 ? C2<T>{a.y, -a.x} : C2<T>{-a.y, a.x};
}

template <int DIR, typename T>
__device__ __forceinline__ void dft2(C2<T>* v)
{
  const C2<T> a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}

template <int DIR, typename T>
__device__ __forceinline__ void dft4(C2<T>& v0, C2<T>& v1, C2<T>& v2, C2<T>& v3)
{
  const C2<T> t0 = cadd(v0, v2), t1 = csub(v0, v2), t2 = cadd(v1, v3), t3 = rot90<DIR>(csub(v1, v3));
  v0 = cadd(t0, t2);
  v2 = csub(t0, t2);
  v1 = cadd(t1, t3);
  v3 = csub(t1, t3);
}

template <int DIR, typename T>
__device__ __forceinline__ void dft8(C2<T>* v)
{
  C2<T> e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
  C2<T> o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
  dft4<DIR>(e0, e1, e2, e3);
  dft4<DIR>(o0, o1, o2, o3);
  const T c = (T)0.70710678118654752440;
  // W^k, W = e^{DIR 2 pi i / 8}
  const C2<T> w1o = cmul(o1, C2<T>{c, (T)DIR * c});
  const C2<T> w2o = rot90<DIR>(o2);
  const C2<T> w3o = cmul(o3, C2<T>{-c, (T)DIR * c});
  v[0] = cadd(e0, o0);
  v[4] = csub(e0, o0);
  v[1] = cadd(e1, w1o);
  v[5] = csub(e1, w1o);
  v[2] = cadd(e2, w2o);
  v[6] = csub(e2, w2o);
  v[3] = cadd(e3, w3o);
  v[7] = csub(e3, w3o);
}

// 16-point DFT in registers, natural order in and out: radix 4 x 4 with n = q + 4p,
// k = r + 4s, X[r + 4s] = sum_q W16^{qr} W4^{qs} sum_p v[q + 4p] W4^{pr}, W16 = e^{DIR 2 pi i/16}.
template <int DIR, typename T>
__device__ __forceinline__ void dft16(C2<T>* v)
{
  C2<T> b[4][4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    b[q][0] = v[q];
    b[q][1] = v[q + 4];
    b[q][2] = v[q + 8];
    b[q][3] = v[q + 12];
    dft4<DIR>(b[q][0], b[q][1], b[q][2], b[q][3]);
  }
  const T c1 = (T)0.92387953251128675613, s1 = (T)0.38268343236508977173, h = (T)0.70710678118654752440;
  const T d = (T)DIR;
  // W16^m for m = q r: 1, 2, 3, 4 (a quarter turn), 6, 9
  b[1][1] = cmul(b[1][1], C2<T>{c1, d * s1});
  b[1][2] = cmul(b[1][2], C2<T>{h, d * h});
  b[1][3] = cmul(b[1][3], C2<T>{s1, d * c1});
  b[2][1] = cmul(b[2][1], C2<T>{h, d * h});
  b[2][2] = rot90<DIR>(b[2][2]);
  b[2][3] = cmul(b[2][3], C2<T>{-h, d * h});
  b[3][1] = cmul(b[3][1], C2<T>{s1, d * c1});
  b[3][2] = cmul(b[3][2], C2<T>{-h, d * h});
  b[3][3] = cmul(b[3][3], C2<T>{-c1, -d * s1});
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    dft4<DIR>(b[0][r], b[1][r], b[2][r], b[3][r]);
    v[r] = b[0][r];
    v[r + 4] = b[1][r];
    v[r + 8] = b[2][r];
    v[r + 12] = b[3][r];
  }
}

// 3- and 5-point DFTs, W = e^{DIR 2 pi i / R}: X_q = sum_r v_r W^{q r}. The conjugate pairs
// W^r + W^{-r} and W^r - W^{-r} are formed once (for R = 5 with c_m = cos(2 pi m/5),
// s_m = DIR sin(2 pi m/5)).
template <int DIR, typename T>
__device__ __forceinline__ void dft3(C2<T>* v)
{
  const T s = (T)DIR * (T)0.86602540378443864676;  // sin(2 pi/3)
  const C2<T> a = v[0], t1 = cadd(v[1], v[2]), t3 = csub(v[1], v[2]);
  const C2<T> m = C2<T>{a.x - (T)0.5 * t1.x, a.y - (T)0.5 * t1.y};
  const C2<T> n = C2<T>{-s * t3.y, s * t3.x};  // i s (v1 - v2)
  v[0] = cadd(a, t1);
  v[1] = cadd(m, n);
  v[2] = csub(m, n);
}

template <int DIR, typename T>
__device__ __forceinline__ void dft5(C2<T>* v)
{
  const T c1 = (T)0.30901699437494742410, c2 = (T)-0.80901699437494742410;
  const T s1 = (T)DIR * (T)0.95105651629515357212, s2 = (T)DIR * (T)0.58778525229247312917;
  const C2<T> a = v[0];
  const C2<T> t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]), t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
  const C2<T> m1 = C2<T>{a.x + c1 * t1.x + c2 * t2.x, a.y + c1 * t1.y + c2 * t2.y};
  const C2<T> m2 = C2<T>{a.x + c2 * t1.x + c1 * t2.x, a.y + c2 * t1.y + c1 * t2.y};
  // i (s1 t3 + s2 t4) and i (s2 t3 - s1 t4)
  const C2<T> n1 = C2<T>{-(s1 * t3.y + s2 * t4.y), s1 * t3.x + s2 * t4.x};
  const C2<T> n2 = C2<T>{-(s2 * t3.y - s1 * t4.y), s2 * t3.x - s1 * t4.x};
  v[0] = cadd(a, cadd(t1, t2));
  v[1] = cadd(m1, n1);
  v[4] = csub(m1, n1);
  v[2] = cadd(m2, n2);
  v[3] = csub(m2, n2);
}

template <int R, int DIR, typename T>
__device__ __forceinline__ void dftR(C2<T>* v)
{
  if constexpr (R == 16) dft16<DIR>(v);
  else if constexpr (R == 8) dft8<DIR>(v);
  else if constexpr (R == 4) dft4<DIR>(v[0], v[1], v[2], v[3]);
  else if constexpr (R == 5) dft5<DIR>(v);
  else if constexpr (R == 3) dft3<DIR>(v);
  else dft2<DIR>(v);
}

constexpr int ilog2(int n) { return n <= 1 ? 0 : 1 + ilog2(n / 2); }

// One Stockham stage (radix R, Ns = product of the earlier radices) over NFFT transforms
// of length N held in LDS at buf[f + n*NFFT] (columns interleaved: the thread map
// f-fastest is conflict free). tw[t] = e^{-2 pi i t/N}.
template <int N, int NFFT, int R, int Ns, int DIR, typename T>
__device__ __forceinline__ void fft_stage(C2<T>* buf, const C2<T>* __restrict__ tw)
{
  constexpr int NB = NFFT * (N / R);
  constexpr int IT = (NB + NT - 1) / NT;
  C2<T> v[IT][R];
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int t = threadIdx.x + it * NT;
    if (NB % NT == 0 || t < NB) {
      const int f = t % NFFT, j = t / NFFT, k = j % Ns;
#pragma unroll
      for (int r = 0; r < R; ++r) v[it][r] = buf[f + (j + r * (N / R)) * NFFT];
      if (Ns > 1) {
#pragma unroll
        for (int r = 1; r < R; ++r) {
          C2<T> w = tw[r * k * (N / (Ns * R))];
          if (DIR > 0) w.y = -w.y;
          v[it][r] = cmul(v[it][r], w);
        }
      }
      dftR<R, DIR>(v[it]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int t = threadIdx.x + it * NT;
    if (NB % NT == 0 || t < NB) {
      const int f = t % NFFT, j = t / NFFT, k = j % Ns;
      const int base = (j / Ns) * Ns * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) buf[f + (base + r * Ns) * NFFT] = v[it][r];
    }
  }
  __syncthreads();
}

template <int N, int NFFT, int Ns, int DIR, typename T>
__device__ __forceinline__ void fft_stages(C2<T>* buf, const C2<T>* __restrict__ tw)
{
  if constexpr (Ns < N) {
    constexpr int rem = N / Ns;
    constexpr int R = rem >= 8 ? 8 : rem;
    fft_stage<N, NFFT, R, Ns, DIR>(buf, tw);
    fft_stages<N, NFFT, Ns * R, DIR>(buf, tw);
  }
}

// NFFT complex transforms of length N in LDS, in place; caller synchronizes before.
template <int N, int NFFT, int DIR, typename T>
__device__ __forceinline__ void lds_fft(C2<T>* buf, const C2<T>* __restrict__ tw)
{
  fft_stages<N, NFFT, 1, DIR>(buf, tw);
}

// The same Stockham stages for a length known at run time (the sizes that are not powers of
// two: N = 8 x blocks with factors 2, 3 and 5, up to FFT_MAX_N), radices from the plan.
// A stage's butterflies are held in registers across the barrier, as in fft_stage: at most
// ITM = ceil(NFFT M / (R NT)) per thread for lengths up to M, predicated on the actual count.
template <int R, int NFFT, int DIR, int M, typename T>
__device__ __forceinline__ void fft_stage_rt(C2<T>* buf, const C2<T>* __restrict__ tw, int n, int Ns)
{
  constexpr int ITM = (NFFT * M / R + NT - 1) / NT;
  const int NB = NFFT * (n / R), m = n / R, st = n / (Ns * R);
  C2<T> v[ITM][R];
#pragma unroll
  for (int it = 0; it < ITM; ++it) {
    const int t = threadIdx.x + it * NT;
    if (t < NB) {
      const int f = t % NFFT, j = t / NFFT, k = j % Ns;
#pragma unroll
      for (int r = 0; r < R; ++r) v[it][r] = buf[f + (j + r * m) * NFFT];
#pragma unroll
      for (int r = 1; r < R; ++r) {
        C2<T> w = tw[r * k * st];
        if (DIR > 0) w.y = -w.y;
        v[it][r] = cmul(v[it][r], w);
      }
      dftR<R, DIR>(v[it]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < ITM; ++it) {
    const int t = threadIdx.x + it * NT;
    if (t < NB) {
      const int f = t % NFFT, j = t / NFFT, k = j % Ns;
      const int base = (j / Ns) * Ns * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) buf[f + (base + r * Ns) * NFFT] = v[it][r];
    }
  }
  __syncthreads();
}

template <int NFFT, int DIR, int M, typename T>
__device__ __forceinline__ void lds_fft_rt(C2<T>* buf, const C2<T>* __restrict__ tw, const FftPlan& p)
{
  int Ns = 1;
  for (int s = 0; s < p.ns; ++s) {
    const int R = p.r[s];
    if (R == 8) fft_stage_rt<8, NFFT, DIR, M>(buf, tw, p.n, Ns);
    else if (R == 4) fft_stage_rt<4, NFFT, DIR, M>(buf, tw, p.n, Ns);
    else if (R == 2) fft_stage_rt<2, NFFT, DIR, M>(buf, tw, p.n, Ns);
    else if (R == 3) fft_stage_rt<3, NFFT, DIR, M>(buf, tw, p.n, Ns);
    else fft_stage_rt<5, NFFT, DIR, M>(buf, tw, p.n, Ns);
    Ns *= R;
  }
}

// The LDS tile of a pass: a static array of COUNT elements, or for COUNT == 0 (a length known
// at run time) the dynamic shared memory the launch sizes.
template <typename T, int COUNT>
__device__ __forceinline__ C2<T>* lds_tile()
{
  if constexpr (COUNT > 0) {
    __shared__ __align__(32) C2<T> tile[COUNT > 0 ? COUNT : 1];
    return tile;
  } else {
    extern __shared__ __align__(32) unsigned char dyn_lds[];
    return reinterpret_cast<C2<T>*>(dyn_lds);
  }
}

// A short run-time length's twiddles, copied behind the tile while the first loads are under way: every
// stage then reads them from LDS, not through the cache (the caller synchronizes before the first use).
// 20.2 -> 18.5 us for the x pass of 160 x 96 x 120 in FP32. Above 256 the tile alone may be 64 KB.
template <typename T>
__device__ __forceinline__ const C2<T>* lds_twiddles(C2<T>* behind, const C2<T>* __restrict__ tw, int n)
{
  for (int i = threadIdx.x; i < n; i += blockDim.x) behind[i] = tw[i];
  return behind;
}

// --------------------------------------------------------------------- x passes

// N: the row length, or for a length known at run time 0 (up to FFT_MAX_N) or X_SHORT (up to 256,
// whose butterflies take half the registers, so twice the workgroups share a CU: forward and inverse
// pass in FP32 18.5 and 12.7 us on 160 x 96 x 120 with the larger bound, 14.0 and 8.5 so; 7.8 and 6.0
// to 6.4 and 5.1 on 48^3, 53 and 35 to 35 and 20 on 192^3; FP64 18.1 and 11.8 to 15.1 and 7.8 on 96^3).
constexpr int X_SHORT = -256;
constexpr int x_max(int N) { return N < 0 ? -N : FFT_MAX_N; }
constexpr int XROWS = 8;         // rows per workgroup = one block row of a z plane
constexpr int XFFT = XROWS / 2;  // complex FFTs per workgroup (two real rows each)

// XSRC_PAD: a field of half the cells per axis, zero beyond it (the free-space solve).
enum XSrc { XSRC_FIELD = 0, XSRC_DIV = 1, XSRC_PAD = 2 };

// Up to three fields that one launch transforms (one per grid z): a pass over a single field of a
// small grid leaves CUs idle (128^3 FP32: three forward transforms 59 us one by one, 37 together).
template <typename T>
struct Three {
  T* p[3];
};

// Reduce-scatter steps over lanes that differ in bit 5, 4 or 0: of the pair (a, b), the lanes
// with the bit clear get a's sum over both, the others b's. The first two are one register swap
// between halves or rows of 16 (no LDS traffic, unlike a general shuffle).
__device__ __forceinline__ float scatter_step32(float a, float b)
{
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float scatter_step16(float a, float b)
{
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float swap_lane1(float v)  // the value of lane ^ 1
{
  return __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), 0xB1, 0xf, 0xf, true));
}
__device__ __forceinline__ double join64(unsigned lo, unsigned hi) { return __hiloint2double((int)hi, (int)lo); }
__device__ __forceinline__ double scatter_step32(double a, double b)
{
  const auto l = __builtin_amdgcn_permlane32_swap(__double2loint(a), __double2loint(b), false, false);
  const auto h = __builtin_amdgcn_permlane32_swap(__double2hiint(a), __double2hiint(b), false, false);
  return join64(l[0], h[0]) + join64(l[1], h[1]);
}
__device__ __forceinline__ double scatter_step16(double a, double b)
{
  const auto l = __builtin_amdgcn_permlane16_swap(__double2loint(a), __double2loint(b), false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(__double2hiint(a), __double2hiint(b), false, false);
  return join64(l[0], h[0]) + join64(l[1], h[1]);
}
__device__ __forceinline__ double swap_lane1(double v)
{
  return join64(__builtin_amdgcn_mov_dpp(__double2loint(v), 0xB1, 0xf, 0xf, true),
                __builtin_amdgcn_mov_dpp(__double2hiint(v), 0xB1, 0xf, 0xf, true));
}
template <typename T>
__device__ __forceinline__ T scatter_step1(T a, T b, bool odd)
{
  const T keep = odd ? b : a, send = odd ? a : b;
  return keep + swap_lane1(send);
}

// Real rows -> packed half spectrum. grid = (Ny/8, Nz).
// FORCE (fused linear forcing): the same pass also forms, per grid row, the x-DFT at
// kx = 0, 1, 2 of each advected velocity component and sum |u*|^2: 16 values per row
// (component q's kx = 0, then re/im of kx = 1, 2 at 5q..5q+4; |u*|^2 at 15), written to
// rowbuf[(z*Ny + y)*16 + slot]. The divergence already loads v on row y+1 and w on plane
// z+1, so the workgroup of row (y, z) takes u of (y, z), v of (y+1, z) and w of (y, z+1);
// every row of every component is summed by exactly one workgroup.
// Each thread's cells lie in one row; the 8 lanes of a row in a wave (bits 0, 4 and 5) reduce
// their 16 sums by halving, each ending with two of them (14 exchanges in registers, where summing
// every value over every lane took 48 shuffles through the LDS pipe: the pass
// took 66 us at 256^3 FP32 and 24 at 128^3 FP64, now 61 and 19), and the 4
// waves' sums meet in LDS.
template <typename T, int N, int SRC, bool FORCE>
__global__ __launch_bounds__(NT) void k_fft_x_fwd(const T* __restrict__ src0, const T* __restrict__ src1,
                                                  const T* __restrict__ src2, Three<C2<T>> spec,
                                                  const C2<T>* __restrict__ tw, GridArgs g,
                                                  const DevScalars* __restrict__ sc, const int* __restrict__ ob_slot,
                                                  const T* __restrict__ ob_rhs, double* __restrict__ rowbuf,
                                                  FftPlan pl)
{
  const int n = N > 0 ? N : pl.n;
  C2<T>* buf = lds_tile<T, (N > 0 ? N : 0) * XFFT>();
  constexpr int NA = 1 + 2 * LOW_KX;  // row DFT values per component: kx=0 (real), kx=1..: re, im
  static_assert(LOW_KX == 2, "the row DFT below evaluates kx = 1, 2");
  static_assert(3 * NA + 1 == 16, "16 row values");
  __shared__ double rowacc[FORCE ? NT / 64 : 1][FORCE ? XROWS : 1][FORCE ? 3 * NA + 1 : 1];
  const int by = blockIdx.x, z = blockIdx.y;
  const int bz = z >> 3, iz = z & 7;
  C2<T>* __restrict__ S = spec.p[blockIdx.z];
  const T* __restrict__ field = blockIdx.z == 0 ? src0 : (blockIdx.z == 1 ? src1 : src2);
  T fac = 0;
  if (SRC == XSRC_DIV) fac = (T)(0.5 * g.h * g.h / sc->dt);
  T* rb = (T*)buf;
  const C2<T>* twl = N < 0 ? lds_twiddles(buf + n * XFFT, tw, n) : tw;
  T acc[FORCE ? 3 * NA + 1 : 1];
  if (FORCE)
#pragma unroll
    for (int q = 0; q < 3 * NA + 1; ++q) acc[q] = 0;
  // Each thread takes quads of 4 x-adjacent cells (half a block row): q -> bx = q/16,
  // iy = (q/2)%8, x0 = 8 bx + 4 (q%2), with 16-byte loads of u, of v at y +- 1, of w at
  // z +- 1, and single loads of u across the quad's two x ends.
  using V4 = typename Vec4<T>::type;
  for (int q4 = threadIdx.x; q4 < n * XROWS / 4; q4 += NT) {
    const int bx = q4 >> 4, iy = (q4 >> 1) & 7, half = q4 & 1, ix0 = 4 * half;
    const int x0 = bx * BS + ix0;
    const int b = bx + g.nbx * (by + g.nby * bz);
    const size_t o = (size_t)b * BS3 + (iz * BS + iy) * BS + ix0;
    T val[4];
    if (SRC == XSRC_FIELD) {
      const V4 a = *reinterpret_cast<const V4*>(field + o);
      val[0] = a.x; val[1] = a.y; val[2] = a.z; val[3] = a.w;
    } else if (SRC == XSRC_PAD) {
      V4 a = {0, 0, 0, 0};
      if (2 * bx < g.nbx)
        a = *reinterpret_cast<const V4*>(field + (size_t)(bx + (g.nbx >> 1) * (by + (g.nby >> 1) * bz)) * BS3 +
                                         (iz * BS + iy) * BS + ix0);
      val[0] = a.x; val[1] = a.y; val[2] = a.z; val[3] = a.w;
    } else {
      const int slot = ob_slot ? ob_slot[b] : -1;
      // neighbour offsets inside the block, or into the periodic neighbour block
      const long sx = BS3, sy = (long)g.nbx * BS3, sz = (long)g.nbx * g.nby * BS3;
      const long on = iy < 7 ? BS : (by + 1 < g.nby ? sy : sy - (long)g.nby * sy) - 7 * BS;
      const long os = iy > 0 ? -BS : (by > 0 ? -sy : (long)(g.nby - 1) * sy) + 7 * BS;
      const long ob = iz < 7 ? BS * BS : (bz + 1 < g.nbz ? sz : sz - (long)g.nbz * sz) - 7 * BS * BS;
      const long of = iz > 0 ? -BS * BS : (bz > 0 ? -sz : (long)(g.nbz - 1) * sz) + 7 * BS * BS;
      // u west of x0 and east of x0 + 3
      const long ow = half ? -1 : (bx > 0 ? -sx : (long)(g.nbx - 1) * sx) + 7;
      const long oe = half ? 3 + (bx + 1 < g.nbx ? sx : sx - (long)g.nbx * sx) - 7 : 4;
      const V4 uc = *reinterpret_cast<const V4*>(src0 + o);
      const T uu[6] = {src0[o + ow], uc.x, uc.y, uc.z, uc.w, src0[o + oe]};
      const V4 vn = *reinterpret_cast<const V4*>(src1 + o + on), wb = *reinterpret_cast<const V4*>(src2 + o + ob);
      const T vN[4] = {vn.x, vn.y, vn.z, vn.w}, wB[4] = {wb.x, wb.y, wb.z, wb.w};
      if (slot >= 0) {
        const V4 r = *reinterpret_cast<const V4*>(ob_rhs + (size_t)slot * BS3 + (iz * BS + iy) * BS + ix0);
        val[0] = r.x; val[1] = r.y; val[2] = r.z; val[3] = r.w;
      } else {
        const V4 vs = *reinterpret_cast<const V4*>(src1 + o + os), wf = *reinterpret_cast<const V4*>(src2 + o + of);
        const T vS[4] = {vs.x, vs.y, vs.z, vs.w}, wF[4] = {wf.x, wf.y, wf.z, wf.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) val[k] = fac * (uu[k + 2] - uu[k] + vN[k] - vS[k] + wB[k] - wF[k]);
      }
      if (FORCE) {
        // u of this row, v of row y+1, w of plane z+1 (see above)
        const T* cv = vN;
        const T* cw = wB;
        // e^{-2 pi i x/Nx} at x0, rotated by the table's first entries for x0 + 1..3
        const C2<T> e0 = tw[x0];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          C2<T> e1 = e0;
          if (k > 0) {
            const C2<T> r = tw[k];
            e1 = C2<T>{e0.x * r.x - e0.y * r.y, e0.x * r.y + e0.y * r.x};
          }
          const C2<T> e2 = {e1.x * e1.x - e1.y * e1.y, 2 * e1.x * e1.y};  // e^{-4 pi i x/Nx}
          const T cu[3] = {uu[k + 1], cv[k], cw[k]};
          acc[3 * NA] += cu[0] * cu[0] + cu[1] * cu[1] + cu[2] * cu[2];
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            acc[q * NA] += cu[q];
            acc[q * NA + 1] += cu[q] * e1.x;
            acc[q * NA + 2] += cu[q] * e1.y;
            acc[q * NA + 3] += cu[q] * e2.x;
            acc[q * NA + 4] += cu[q] * e2.y;
          }
        }
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) rb[2 * ((x0 + k) * XFFT + (iy >> 1)) + (iy & 1)] = val[k];
  }
  if constexpr (FORCE) {
    // rows: lanes with the same iy = (lane >> 1) & 7 differ in bits 0 (half) and 4-5 (bx)
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, iy = (lane >> 1) & 7;
    const bool odd = lane & 1;
    T a8[8], a4[4];
#pragma unroll
    for (int q = 0; q < 8; ++q) a8[q] = scatter_step32(acc[q], acc[q + 8]);
#pragma unroll
    for (int q = 0; q < 4; ++q) a4[q] = scatter_step16(a8[q], a8[q + 4]);
    const int q0 = 8 * (lane >> 5) + 4 * ((lane >> 4) & 1) + 2 * (lane & 1);
    rowacc[wv][iy][q0] = (double)scatter_step1(a4[0], a4[2], odd);
    rowacc[wv][iy][q0 + 1] = (double)scatter_step1(a4[1], a4[3], odd);
  }
  __syncthreads();
  if constexpr (FORCE) if (threadIdx.x < XROWS * (3 * NA + 1)) {
    // the rows' sums over the 4 waves, in wave order, to the row each component belongs to
    const int r = threadIdx.x >> 4, q = threadIdx.x & 15;
    const double v = rowacc[0][r][q] + rowacc[1][r][q] + rowacc[2][r][q] + rowacc[3][r][q];
    const int y = by * BS + r;
    const int yy = (q >= NA && q < 2 * NA) ? (y + 1 < g.Ny ? y + 1 : 0) : y;
    const int zz = (q >= 2 * NA && q < 3 * NA) ? (z + 1 < g.Nz ? z + 1 : 0) : z;
    rowbuf[((size_t)zz * g.Ny + yy) * 16 + q] = v;
  }
  if constexpr (N > 0) lds_fft<N, XFFT, -1>(buf, tw);
  else lds_fft_rt<XFFT, -1, x_max(N)>(buf, twl, pl);
  // Separate the two real transforms of each complex FFT and pack kx = N/2 into slot 0.
  for (int t = threadIdx.x; t < XROWS * (n / 2); t += NT) {
    const int row = t / (n / 2), k = t % (n / 2);
    const int q = row >> 1, odd = row & 1;
    const C2<T> Z = buf[k * XFFT + q];
    C2<T> out;
    if (k == 0) {
      const C2<T> Zn = buf[(n / 2) * XFFT + q];
      out = odd ? C2<T>{Z.y, Zn.y} : C2<T>{Z.x, Zn.x};
    } else {
      const C2<T> Zm = buf[(n - k) * XFFT + q];
      // Xa = (Z + conj Zm)/2 ; Xb = -i (Z - conj Zm)/2
      out = odd ? C2<T>{(T)0.5 * (Z.y + Zm.y), (T)0.5 * (Zm.x - Z.x)}
                : C2<T>{(T)0.5 * (Z.x + Zm.x), (T)0.5 * (Z.y - Zm.y)};
    }
    const int y = by * BS + row;
    S[((size_t)z * g.Ny + y) * (n / 2) + k] = out;
  }
}

// Packed half spectrum -> real rows of a block-layout field. grid = (Ny/8, Nz).
// XF: also write each block's x faces (ix = 0 and 7) to xf[(b*2 + side)*64 + iz*8 + iy], so that
// the gradient reads them as 64 contiguous values instead of one value per 32-byte sector.
// PAD: the inverse of XSRC_PAD, the field's own half of each row.
template <typename T, int N, bool XF = false, bool PAD = false>
__global__ __launch_bounds__(NT) void k_fft_x_inv(Three<C2<T>> spec, Three<T> fields,
                                                  const C2<T>* __restrict__ tw, GridArgs g, FftPlan pl,
                                                  T* __restrict__ xf = nullptr)
{
  const int n = N > 0 ? N : pl.n;
  C2<T>* buf = lds_tile<T, (N > 0 ? N : 0) * XFFT>();
  const int by = blockIdx.x, z = blockIdx.y;
  const int bz = z >> 3, iz = z & 7;
  const C2<T>* __restrict__ S = spec.p[blockIdx.z];
  T* __restrict__ dst = fields.p[blockIdx.z];
  const C2<T>* twl = N < 0 ? lds_twiddles(buf + n * XFFT, tw, n) : tw;
  for (int t = threadIdx.x; t < XFFT * (n / 2); t += NT) {
    const int q = t / (n / 2), k = t % (n / 2);
    const int ya = by * BS + 2 * q;
    const C2<T> A = S[((size_t)z * g.Ny + ya) * (n / 2) + k];
    const C2<T> B = S[((size_t)z * g.Ny + ya + 1) * (n / 2) + k];
    if (k == 0) {
      buf[0 * XFFT + q] = C2<T>{A.x, B.x};
      buf[(n / 2) * XFFT + q] = C2<T>{A.y, B.y};
    } else {
      buf[k * XFFT + q] = C2<T>{A.x - B.y, A.y + B.x};
      buf[(n - k) * XFFT + q] = C2<T>{A.x + B.y, B.x - A.y};
    }
  }
  __syncthreads();
  if constexpr (N > 0) lds_fft<N, XFFT, +1>(buf, tw);
  else lds_fft_rt<XFFT, +1, x_max(N)>(buf, twl, pl);
  const T* rb = (const T*)buf;
  for (int t = threadIdx.x; t < (PAD ? n / 2 : n) * XROWS; t += NT) {
    const int bx = t >> 6, iy = (t >> 3) & 7, ix = t & 7;
    const int x = bx * BS + ix;
    const int b = PAD ? bx + (g.nbx >> 1) * (by + (g.nby >> 1) * bz) : bx + g.nbx * (by + g.nby * bz);
    // streamed past the caches: the gradient pass reads p with its own halo order
    const T v = rb[2 * (x * XFFT + (iy >> 1)) + (iy & 1)];
    __builtin_nontemporal_store(v, &dst[(size_t)b * BS3 + (iz * BS + iy) * BS + ix]);
    if (XF && (ix == 0 || ix == BS - 1)) xf[((size_t)b * 2 + (ix != 0)) * 64 + iz * BS + iy] = v;
  }
}

// ------------------------------------------------------------------ y / z passes

enum ZMode { ZM_FWD = 0, ZM_INV = 1, ZM_POISSON = 2 };

// Column passes of the lengths without a register four-step form below: 512 and 1024 (N > 0, radices
// known at compile time) and every length that is not a power of two, or below 64 (N = 0, the plan's
// radices). M bounds the length. A workgroup of BT threads takes TK columns, at most 16 elements per
// thread, in Stockham stages whose butterflies a thread holds in registers: the first stage reads its
// inputs j + r n/R from global memory, the last writes its outputs (the same indices) there, and
// only the stages between exchange through LDS. The z pass's division happens on the last forward
// stage's registers, which are also the inputs of the first inverse stage when the inverse takes the
// radices in reverse order. Against a tile staged in LDS at both ends this halves the LDS traffic:
// on 512^3 FP32 (1 GiB of traffic) a y pass went from 325 to 215 us, the rate of a large copy, and the
// z pass from 614 to 370; on 160 x 96 x 120 from 20 to 8 and from 28 to 15 us.
template <typename T, int M>
struct ColTile {
  // 16 columns (8 for 1024) in FP32, 64 KiB of LDS at most: 128-byte segments, or 64 at 1024
  static constexpr int TK = sizeof(T) == 4 ? (M <= 512 ? 16 : 8) : (M <= 256 ? 16 : (M <= 512 ? 8 : 4));
  static constexpr int BT = TK * M / 16;
  static constexpr int E = 16;  // elements per thread
};

// k = j % Ns for j < 2^20 and Ns <= 1024 (rNs = 1/Ns rounded): the quotient's estimate is below the
// next integer by at least 1/(2 Ns), more than the product's rounding.
__device__ __forceinline__ int mod_ns(int j, int Ns, float rNs) { return j - Ns * (int)(((float)j + 0.5f) * rNs); }

// The forcing's factor times h^2/dt, 0 where it does not force (called by whole waves).
__device__ __forceinline__ double forcing_gg(const ForcingArgs& fa, const LowModes& lm)
{
  double tke, tke_low;
  const double fac = forcing_factor(fa, lm.n, tke, tke_low);
  return fac > 0 ? fac * fa.h * fa.h / fa.sc->dt : 0.0;
}

template <typename T, int N, int M>
struct ColStages {
  using CT = ColTile<T, M>;
  static constexpr int TK = CT::TK, BT = CT::BT;
  C2<T>* S;
  C2<T>* buf;
  const C2<T>* tw;
  size_t base, stride;  // element e of column f is S[base + f + e stride]
  bool inv;             // an inverse transform: the forward one with the real and imaginary parts swapped
  int n, nc;            // length, live columns
  int kx0, ky, Ny;      // the z pass's symbol and forcing modes
  double norm;
  const double *cx, *cy, *cz;
  const LowModes* lmp;  // null: no forcing
  ForcingArgs fa;
  double gg;            // the forcing's factor times h^2/dt (0: none)

  __device__ __forceinline__ C2<T> load(int f, int e) const
  {
    const C2<T> a = f < nc ? S[base + f + e * stride] : C2<T>{0, 0};
    return inv ? C2<T>{a.y, a.x} : a;
  }

  // the spectral division of the outputs kz = j + r n/R of column kx0 + f, after the forcing's modes
  template <int R>
  __device__ __forceinline__ void divide(C2<T> (&v)[R], int f, int j) const
  {
    const int m = n / R;
    if (lmp && kx0 == 0) {
      const LowModes& lm = *lmp;
      for (int e = 0; e < lm.npos; ++e) {
        const int slot = lm.pos[e][0], kye = lm.pos[e][1], kz = lm.pos[e][2], mc = lm.pos[e][3];
        if (kye != ky || slot != f) continue;
        const C2<double> cm = forcing_rhs_mode(fa, lm, mc >> 1, gg);
        const double ci = (mc & 1) ? -cm.y : cm.y;
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (kz == j + r * m) {
            v[r].x = (T)((double)v[r].x + cm.x);
            v[r].y = (T)((double)v[r].y + ci);
          }
      }
    }
    // PoissonSolverPeriodic::_solve's grid-consistent branch (PoissonSolverPeriodic.cpp:23-61):
    // norm/(2D-6), D = cos(4 pi kx/Nx) + cos(4 pi ky/Ny) + cos(4 pi kz/Nz), in FP64; the modes with
    // every index in {0, N/2} are zeroed (kx slot 0 carries kx = 0 and Nx/2)
    const int kx = kx0 + f;
    const double dxy = f < nc ? cx[kx] + cy[ky] : 0.0;
    const bool zxy = kx == 0 && (ky == 0 || 2 * ky == Ny);
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int kz = j + r * m;
      const double D = dxy + cz[kz];
      double fac = norm / (2 * D - 6);
      const bool zero = zxy && (kz == 0 || 2 * kz == n);
      if (zero) fac = 0;
      v[r].x = (T)((double)v[r].x * fac);
      v[r].y = (T)((double)v[r].y * fac);
      if (zero) v[r] = C2<T>{0, 0};
    }
  }

  // One stage of radix R after Ns = the product of the earlier radices. FIRST and LAST: it reads
  // from and writes to global memory. MID: the forward transform's last stage, the division and the
  // inverse transform's first stage, after which the parts are swapped.
  template <int R, bool FIRST, bool LAST, bool MID>
  __device__ __forceinline__ void stage(int Ns)
  {
    constexpr int IT = (CT::E + R - 1) / R;
    const int m = n / R, NB = TK * m, st = n / (Ns * R);
    const float rNs = 1.0f / (float)Ns;
    C2<T> v[IT][R];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int t = threadIdx.x + it * BT;
      if (t >= NB) continue;
      const int f = t % TK, j = t / TK;
      if (FIRST) {
#pragma unroll
        for (int r = 0; r < R; ++r) v[it][r] = load(f, j + r * m);
      } else {
        const int k = N > 0 ? j % Ns : mod_ns(j, Ns, rNs);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          v[it][r] = buf[f + (j + r * m) * TK];
          if (r) v[it][r] = cmul(v[it][r], tw[r * k * st]);
        }
      }
      dftR<R, -1>(v[it]);
      if (MID) {
        divide<R>(v[it], f, j);
#pragma unroll
        for (int r = 0; r < R; ++r) v[it][r] = C2<T>{v[it][r].y, v[it][r].x};
        dftR<R, -1>(v[it]);
      }
    }
    if (!FIRST && !LAST) __syncthreads();  // the stage's reads are done
    const bool swap = LAST && (MID || inv);
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int t = threadIdx.x + it * BT;
      if (t >= NB) continue;
      const int f = t % TK, j = t / TK;
      if (LAST) {
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (f < nc) S[base + f + (j + r * m) * stride] = swap ? C2<T>{v[it][r].y, v[it][r].x} : v[it][r];
      } else {
        // MID's outputs are those of the inverse's first stage: k = 0, from j R on
        const int k = MID || FIRST ? 0 : (N > 0 ? j % Ns : mod_ns(j, Ns, rNs));
        const int o = MID || FIRST ? j * R : (j - k) * R + k, step = MID ? 1 : Ns;
#pragma unroll
        for (int r = 0; r < R; ++r) buf[f + (o + r * step) * TK] = v[it][r];
      }
    }
    if (!LAST) __syncthreads();
  }

  template <bool LAST, bool MID>
  __device__ __forceinline__ void stage_rt(int R, int Ns)
  {
    if (R == 8) stage<8, false, LAST, MID>(Ns);
    else if (R == 4) stage<4, false, LAST, MID>(Ns);
    else if (R == 5) stage<5, false, LAST, MID>(Ns);
    else if (R == 3) stage<3, false, LAST, MID>(Ns);
    else stage<2, false, LAST, MID>(Ns);
  }

  // The plan's radices; the first is 8 (a length is 8 x blocks), and the only one at length 8.
  template <bool POISSON>
  __device__ __forceinline__ void run_rt(const FftPlan& pl)
  {
    const int last = pl.ns - 1;
    if (last == 0) {
      stage<8, true, true, POISSON>(1);
      return;
    }
    stage<8, true, false, false>(1);
    int Ns = 8;
    for (int s = 1; s < last; ++s) {
      stage_rt<false, false>(pl.r[s], Ns);
      Ns *= pl.r[s];
    }
    if constexpr (!POISSON) {
      stage_rt<true, false>(pl.r[last], Ns);
      return;
    }
    stage_rt<false, true>(pl.r[last], Ns);
    inv = true;
    Ns = pl.r[last];
    for (int s = last - 1; s > 0; --s) {
      stage_rt<false, false>(pl.r[s], Ns);
      Ns *= pl.r[s];
    }
    stage<8, false, true, false>(Ns);
  }

  // 512 = 8 8 8 and 1024 = 16 8 8: three stages each
  template <bool POISSON>
  __device__ __forceinline__ void run_ct()
  {
    constexpr int R0 = N / 64;
    stage<R0, true, false, false>(1);
    stage<8, false, false, false>(R0);
    if constexpr (!POISSON) {
      stage<8, false, true, false>(8 * R0);
    } else {
      stage<8, false, false, true>(8 * R0);
      inv = true;
      stage<8, false, false, false>(8);
      stage<R0, false, true, false>(64);
    }
  }
};

// Column FFT along y (axis 1) or z (axis 2). grid = (ceil(ncols/TK), other axis). POISSON (z only):
// forward transform, grid-consistent division and inverse transform.
template <typename T, int N, int M, bool POISSON>
__global__ __launch_bounds__((ColTile<T, M>::BT)) void k_fft_col(Three<C2<T>> S, const C2<T>* __restrict__ tw,
                                                               int ncols, int axis, int inv, int Ny, double norm,
                                                               const double* __restrict__ cx,
                                                               const double* __restrict__ cy,
                                                               const double* __restrict__ cz,
                                                               const LowModes* __restrict__ lmp, ForcingArgs fa,
                                                               FftPlan pl)
{
  using CS = ColStages<T, N, M>;
  C2<T>* buf = lds_tile<T, N * CS::TK>();
  const int kx0 = blockIdx.x * CS::TK, o = blockIdx.y;
  const size_t base = (axis == 1 ? (size_t)o * Ny : (size_t)o) * ncols + kx0;
  const size_t stride = axis == 1 ? (size_t)ncols : (size_t)Ny * ncols;
  const int n = N > 0 ? N : pl.n;
  CS cs{S.p[blockIdx.z], buf, tw, base, stride, inv != 0, n, min(CS::TK, ncols - kx0), kx0, o, Ny, norm,
        cx, cy, cz, lmp, fa, POISSON && lmp && kx0 == 0 ? forcing_gg(fa, *lmp) : 0.0};
  if constexpr (N > 0) cs.template run_ct<POISSON>();
  else cs.template run_rt<POISSON>(pl);
}

// ------------------------------------------- y / z passes, register four-step form
// N = 16 NTH (NTH = 4, 8, 16 threads per column), TK = NT/NTH columns per workgroup.
// Layout A: thread (f, j) holds v[m] = x[j + NTH m], m < 16. Layout B: thread (f, j) holds
// v[i NTH + k2] = X[k1 + 16 k2] for its RPT = 16/NTH rows k1 = j RPT + i. With
// W_N^{(j + NTH m)(k1 + 16 k2)} = W_N^{j k1} W_NTH^{j k2} W_16^{m k1}, a transform is a register
// DFT16 over m, the twiddle W_N^{j k1}, one LDS transpose, and register DFTs of length NTH
// over j (A -> B); B -> A runs the same steps in reverse order. Column f is the workgroup's
// f-th kx column; lanes run f fastest, so each global access covers 16 columns of a row.
template <typename T, int N>
struct ColReg {
  static constexpr bool ok = N >= 64 && N <= 256;
  static constexpr int NTH = ok ? N / 16 : 1, RPT = 16 / NTH, TK = NT / NTH;
  // LDS stride of one k1 row. Unpadded, the tile is 32 KiB (FP32), so five workgroups share
  // a CU; the transposes' writes are conflict free and their reads cost less than a lost slot.
  static constexpr int ROWP = NTH * TK;
};

template <int L, int DIR, typename T>
__device__ __forceinline__ void dftL(C2<T>* v)
{
  if constexpr (L == 16) dft16<DIR>(v);
  else if constexpr (L == 8) dft8<DIR>(v);
  else dft4<DIR>(v[0], v[1], v[2], v[3]);
}

// A -> B. The caller synchronizes before when buf was read since its last barrier.
template <typename T, int N, int DIR>
__device__ __forceinline__ void fft_a_to_b(C2<T> (&v)[16], C2<T>* buf, const C2<T>* __restrict__ tw, int f, int j)
{
  using CR = ColReg<T, N>;
  dft16<DIR>(v);
#pragma unroll
  for (int k1 = 1; k1 < 16; ++k1) {
    C2<T> w = tw[(j * k1) & (N - 1)];
    if (DIR > 0) w.y = -w.y;
    v[k1] = cmul(v[k1], w);
  }
#pragma unroll
  for (int k1 = 0; k1 < 16; ++k1) buf[k1 * CR::ROWP + j * CR::TK + f] = v[k1];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < CR::RPT; ++i)
#pragma unroll
    for (int jp = 0; jp < CR::NTH; ++jp) v[i * CR::NTH + jp] = buf[(j * CR::RPT + i) * CR::ROWP + jp * CR::TK + f];
#pragma unroll
  for (int i = 0; i < CR::RPT; ++i) dftL<CR::NTH, DIR>(v + i * CR::NTH);
}

// B -> A. The caller synchronizes before when buf was read since its last barrier.
template <typename T, int N, int DIR>
__device__ __forceinline__ void fft_b_to_a(C2<T> (&v)[16], C2<T>* buf, const C2<T>* __restrict__ tw, int f, int j)
{
  using CR = ColReg<T, N>;
#pragma unroll
  for (int i = 0; i < CR::RPT; ++i) {
    dftL<CR::NTH, DIR>(v + i * CR::NTH);
    const int k1 = j * CR::RPT + i;
#pragma unroll
    for (int jn = 1; jn < CR::NTH; ++jn) {
      C2<T> w = tw[(jn * k1) & (N - 1)];
      if (DIR > 0) w.y = -w.y;
      v[i * CR::NTH + jn] = cmul(v[i * CR::NTH + jn], w);
    }
#pragma unroll
    for (int jn = 0; jn < CR::NTH; ++jn) buf[k1 * CR::ROWP + jn * CR::TK + f] = v[i * CR::NTH + jn];
  }
  __syncthreads();
#pragma unroll
  for (int k1 = 0; k1 < 16; ++k1) v[k1] = buf[k1 * CR::ROWP + j * CR::TK + f];
  dft16<DIR>(v);
}

// The column pass of k_fft_col in the register form (same arguments and modes). EXTRA: the
// grid's first ex.ey rows are workgroups of the forcing's plane stage (1, beside the y forward
// pass) or row stage (2, beside the z pass), in the column tile's LDS.
template <typename T, int N, int AXIS, int MODE, bool FORCE = false, int EXTRA = 0>
__global__ __launch_bounds__(NT) void k_fft_colr(Three<C2<T>> spec, const C2<T>* __restrict__ tw, int ncols,
                                                 int Ny, int Nz, double norm, const double* __restrict__ cx,
                                                 const double* __restrict__ cy, const double* __restrict__ cz,
                                                 const LowModes* __restrict__ lmp, ForcingArgs fa, ColExtra ex)
{
  using CR = ColReg<T, N>;
  constexpr int TK = CR::TK, NTH = CR::NTH, RPT = CR::RPT;
  __shared__ __align__(16) C2<T> buf[16 * CR::ROWP];
  static_assert(EXTRA == 0 || (sizeof(buf) >= FORCING_PLANES_LDS && sizeof(buf) >= FORCING_ROWS_LDS),
                "the forcing stages fit the column tile's LDS");
  if constexpr (EXTRA != 0) {
    if ((int)blockIdx.y < ex.ey) {
      const int w = blockIdx.y * gridDim.x + blockIdx.x;  // uniform over the workgroup
      if (EXTRA == 1 && w < ex.nz * ex.parts)
        forcing_planes_wg<T>(ex.rowbuf, ex.plane, Ny, (const C2<T>*)ex.twy, w / ex.parts, w % ex.parts, ex.parts, buf);
      else if (EXTRA == 2 && w < ex.nz)
        forcing_rows_step<T>(lmp, fa, (const C2<T>*)ex.twy, (const C2<T>*)ex.twz, (T*)ex.rows, Ny, Nz, w, buf);
      return;
    }
  }
  C2<T>* __restrict__ S = spec.p[blockIdx.z];
  const int kx0 = blockIdx.x * TK, other = blockIdx.y - (EXTRA != 0 ? ex.ey : 0);
  const int f = threadIdx.x % TK, j = threadIdx.x / TK;
  const bool live = kx0 + f < ncols;
  // element n of column kx0 + f
  auto gi = [&](int n) -> size_t {
    return AXIS == 1 ? ((size_t)other * Ny + n) * ncols + kx0 + f : ((size_t)n * Ny + other) * ncols + kx0 + f;
  };
  C2<T> v[16];
  if (MODE == ZM_INV) {
#pragma unroll
    for (int i = 0; i < RPT; ++i)
#pragma unroll
      for (int k2 = 0; k2 < NTH; ++k2) v[i * NTH + k2] = live ? S[gi(j * RPT + i + 16 * k2)] : C2<T>{0, 0};
    fft_b_to_a<T, N, +1>(v, buf, tw, f, j);
    if (live)
#pragma unroll
      for (int m = 0; m < 16; ++m) S[gi(j + NTH * m)] = v[m];
    return;
  }
#pragma unroll
  for (int m = 0; m < 16; ++m) v[m] = live ? S[gi(j + NTH * m)] : C2<T>{0, 0};
  const double gg = FORCE && kx0 == 0 ? forcing_gg(fa, *lmp) : 0.0;  // while the columns arrive
  fft_a_to_b<T, N, -1>(v, buf, tw, f, j);
  if (FORCE && kx0 == 0) {
    // fused forcing: add the forcing's RHS modes (from the mode sums of k_forcing_reduce) to the
    // entries this thread holds (column f, k = k1 + 16 k2 with k1 / RPT = j)
    const LowModes& lm = *lmp;
    for (int e = 0; e < lm.npos; ++e) {
      const int slot = lm.pos[e][0], ky = lm.pos[e][1], kz = lm.pos[e][2], mc = lm.pos[e][3];
      if (ky != other || slot != f || (kz & 15) / RPT != j) continue;
      const int r = ((kz & 15) % RPT) * NTH + (kz >> 4);
      const C2<double> cm = forcing_rhs_mode(fa, lm, mc >> 1, gg);
      const double ci = (mc & 1) ? -cm.y : cm.y;
#pragma unroll
      for (int q = 0; q < 16; ++q)
        if (q == r) {
          v[q].x = (T)((double)v[q].x + cm.x);
          v[q].y = (T)((double)v[q].y + ci);
        }
    }
  }
  if (MODE == ZM_FWD) {
    if (live)
#pragma unroll
      for (int i = 0; i < RPT; ++i)
#pragma unroll
        for (int k2 = 0; k2 < NTH; ++k2) S[gi(j * RPT + i + 16 * k2)] = v[i * NTH + k2];
    return;
  }
  // ZM_POISSON (z): PoissonSolverPeriodic::_solve's grid-consistent branch
  // (PoissonSolverPeriodic.cpp:23-61), multiply by norm/(2D-6) in FP64 (also for FP32 fields:
  // an FP32 factor, even formed without cancellation as -norm/(4 sum sin^2), adds rounding to
  // the lowest modes that long FP32 trajectories and their adjoints amplify), zero the modes
  // with every index in {0, N/2}; then the inverse transform.
  {
    const int kx = kx0 + f, ky = other;
    const double dxy = live ? cx[kx] + cy[ky] : 0.0;
    const bool zxy = kx == 0 && (ky == 0 || 2 * ky == Ny);
#pragma unroll
    for (int i = 0; i < RPT; ++i)
#pragma unroll
      for (int k2 = 0; k2 < NTH; ++k2) {
        const int kz = j * RPT + i + 16 * k2;
        const double D = dxy + cz[kz];
        double fac = norm / (2 * D - 6);
        if (zxy && (kz == 0 || 2 * kz == N)) fac = 0;
        C2<T>& q = v[i * NTH + k2];
        q.x = (T)((double)q.x * fac);
        q.y = (T)((double)q.y * fac);
      }
  }
  __syncthreads();  // the forward transpose's reads of buf are done
  fft_b_to_a<T, N, +1>(v, buf, tw, f, j);
  if (live)
#pragma unroll
    for (int m = 0; m < 16; ++m) S[gi(j + NTH * m)] = v[m];
}

// ----------------------------------------------- y / z passes of the free-space solve

enum FreeMode { FC_FWD = 0, FC_INV = 1, FC_CONV = 2 };

// A transform's results, formed where this stands and not in the branches behind it: which product of
// a sum is rounded depends on the block that the compiler forms the sum in.
template <typename T>
__device__ __forceinline__ void hold(C2<T> (&v)[16])
{
#pragma unroll
  for (int q = 0; q < 16; ++q) asm volatile("" : "+v"(v[q].x), "+v"(v[q].y));
}

// Column passes on the padded grid of which only a part is needed: elements from nin on are zero,
// those from nout on are not wanted. FC_CONV (z) transforms forward, multiplies by the Green's
// function's spectrum (real, green, at the spectrum's indices) and transforms back. Slot 0 packs the
// kx = 0 and kx = Nx/2 planes as A + iB, for which the Green's function has two values, G0 = green and
// GN = green_n[kz][ky]: the product is a Z(k) + b conj Z(-k), a = (G0 + GN)/2, b = (G0 - GN)/2, so the
// slot's columns ky and -ky go together, TK/2 such pairs to each workgroup of the grid's last x index.
//
// The stages, their order and the packing are those of passes over whole columns and of a product of
// its own, so the result is theirs bit for bit. After the inflow correction the RHS's sum is rounding
// noise, and the solve returns it as most of the pressure's mean: another rounding of the solve changes
// the next step's noise, in FP32 by several times the solve's own error (3e-7 to 1e-5 of |p|).
struct FreeArgs {
  int ncols, axis, Ny, nin, nout;
  const double *green, *green_n;
};

// Thread (f, j) of a workgroup of TK columns: column f.
template <typename T, int TK, int MODE>
struct FreeCol {
  static constexpr int H = TK / 2;
  C2<T>* S;
  C2<T>* col;
  size_t stride;
  FreeArgs a;
  int n, f, row;
  bool pair, live, keep;

  // false: nothing to do for the workgroup
  __device__ __forceinline__ bool init(C2<T>* spec, const FreeArgs& args, int length)
  {
    a = args;
    S = spec;
    n = length;
    f = threadIdx.x % TK;
    const int o = blockIdx.y;
    pair = MODE == FC_CONV && blockIdx.x == gridDim.x - 1;
    if (pair && o * H > a.Ny / 2) return false;
    int kx = blockIdx.x * TK + f;
    row = o;
    live = keep = kx < a.ncols && !(MODE == FC_CONV && kx == 0);
    if (pair) {
      const int k = o * H + f % H, m = k == 0 ? 0 : a.Ny - k;
      kx = 0;
      live = k <= a.Ny / 2;
      row = f < H ? k : m;
      keep = live && (f < H || m != k);  // a column that is its own mirror is held twice
    }
    stride = a.axis == 1 ? (size_t)a.ncols : (size_t)a.Ny * a.ncols;
    col = S + (a.axis == 1 ? (size_t)row * a.Ny : (size_t)row) * a.ncols + kx;
    return true;
  }
  __device__ __forceinline__ C2<T> get(int e) const { return live && e < a.nin ? col[e * stride] : C2<T>{0, 0}; }
  __device__ __forceinline__ C2<T> times(const C2<T>& v, int e) const
  {
    const double gg = live ? a.green[(col - S) + e * stride] : 0.0;
    return C2<T>{(T)(v.x * gg), (T)(v.y * gg)};
  }
  // Element e of slot 0's column r with zm, element -e of the mirrored column. The pair takes the
  // Green's function at its lower index, and of each sum one product is rounded, in both elements the
  // same.
  __device__ __forceinline__ C2<T> times_pair(const C2<T>& z, const C2<T>& zm, int e, int r) const
  {
    const size_t i = (size_t)e * a.Ny + r, m = (size_t)(e == 0 ? 0 : n - e) * a.Ny + (r == 0 ? 0 : a.Ny - r);
    const size_t g = live ? min(i, m) : 0;
    const double g0 = a.green[g * a.ncols], gn = a.green_n[g];
    const double p = 0.5 * (g0 + gn), q = 0.5 * (g0 - gn), x = z.x, y = z.y, xm = zm.x, ym = zm.y;
    return C2<T>{(T)(i <= m ? fma(p, x, q * xm) : fma(q, xm, p * x)), (T)fma(p, y, -(q * ym))};
  }
  // the product of a tile buf[f + e*TK] of slot 0's columns, elements j, j + step, ..
  __device__ __forceinline__ void times_pairs(C2<T>* buf, int j, int step) const
  {
    if (f < H)
      for (int e = j; e < n; e += step) {
        const int me = e == 0 ? 0 : n - e;
        C2<T>&z = buf[f + e * TK], &zm = buf[f + H + me * TK];
        const C2<T> z0 = z, m0 = zm;
        z = times_pair(z0, m0, e, row);
        zm = times_pair(m0, z0, me, row == 0 ? 0 : a.Ny - row);
      }
  }
};

// Lengths L that are powers of two from 64 on: up to 256 in the register form, 512 and 1024 in LDS.
template <typename T, int L>
struct FreeTile {
  static constexpr int TK = L >= 512 ? 65536 / (L * (int)sizeof(C2<T>)) : 16 * NT / L;
};

template <typename T, int L, int MODE>
__global__ __launch_bounds__(NT) void k_free_col(C2<T>* __restrict__ S, const C2<T>* __restrict__ tw, FreeArgs a)
{
  constexpr bool REG = ColReg<T, L>::ok;
  constexpr int TK = FreeTile<T, L>::TK, NR = REG ? L : 64;
  using CR = ColReg<T, NR>;
  static_assert(!REG || CR::TK == TK, "both forms take as many columns");
  C2<T>* buf = lds_tile<T, L * TK>();
  FreeCol<T, TK, MODE> c;
  if (!c.init(S, a, L)) return;
  const int f = c.f, j = threadIdx.x / TK;
  if constexpr (REG) {
    constexpr int NTH = CR::NTH, RPT = CR::RPT;
    C2<T> v[16];
    if (MODE == FC_INV) {
#pragma unroll
      for (int i = 0; i < RPT; ++i)
#pragma unroll
        for (int k2 = 0; k2 < NTH; ++k2) v[i * NTH + k2] = c.get(j * RPT + i + 16 * k2);
    } else {
#pragma unroll
      for (int m = 0; m < 16; ++m) v[m] = c.get(j + NTH * m);
      fft_a_to_b<T, NR, -1>(v, buf, tw, f, j);
    }
    if (MODE == FC_FWD) {
      if (c.live)
#pragma unroll
        for (int i = 0; i < RPT; ++i)
#pragma unroll
          for (int k2 = 0; k2 < NTH; ++k2) c.col[(j * RPT + i + 16 * k2) * c.stride] = v[i * NTH + k2];
      return;
    }
    if (MODE == FC_CONV) {
      if (c.live) hold(v);
      else
#pragma unroll
        for (int q = 0; q < 16; ++q) v[q] = C2<T>{0, 0};
      __syncthreads();  // the forward transpose's reads of buf are done
      if (c.pair) {
#pragma unroll
        for (int i = 0; i < RPT; ++i)
#pragma unroll
          for (int k2 = 0; k2 < NTH; ++k2) buf[(j * RPT + i + 16 * k2) * TK + f] = v[i * NTH + k2];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < RPT; ++i)
#pragma unroll
          for (int k2 = 0; k2 < NTH; ++k2) {
            const int e = j * RPT + i + 16 * k2;
            v[i * NTH + k2] = c.times_pair(v[i * NTH + k2], buf[(e == 0 ? 0 : L - e) * TK + (f ^ (TK / 2))], e, c.row);
          }
        __syncthreads();
      } else {
#pragma unroll
        for (int i = 0; i < RPT; ++i)
#pragma unroll
          for (int k2 = 0; k2 < NTH; ++k2) v[i * NTH + k2] = c.times(v[i * NTH + k2], j * RPT + i + 16 * k2);
      }
    }
    fft_b_to_a<T, NR, +1>(v, buf, tw, f, j);
    if (c.keep) {
      hold(v);
#pragma unroll
      for (int m = 0; m < 16; ++m)
        if (j + NTH * m < a.nout) c.col[(j + NTH * m) * c.stride] = v[m];
    }
  } else {
    for (int e = j; e < L; e += NT / TK) buf[f + e * TK] = c.get(e);
    __syncthreads();
    if constexpr (MODE != FC_INV) lds_fft<L, TK, -1>(buf, tw);
    if (MODE == FC_CONV) {
      if (c.pair) c.times_pairs(buf, j, NT / TK);
      else
        for (int e = j; e < L; e += NT / TK) buf[f + e * TK] = c.times(buf[f + e * TK], e);
      __syncthreads();
    }
    if constexpr (MODE != FC_FWD) lds_fft<L, TK, +1>(buf, tw);
    for (int e = j; e < a.nout; e += NT / TK)
      if (c.keep) c.col[e * c.stride] = buf[f + e * TK];
  }
}

// Every other length, up to M, in ColTile's form: the first stage reads from global memory and the last
// writes there, and the product is taken on the last forward stage's registers (slot 0's in LDS).
// Staging whole columns in LDS took 133 us for a solve on 96^3 FP64 cells, this takes 100.
template <typename T, int M, int MODE>
struct FreeStages {
  using CT = ColTile<T, M>;
  static constexpr int TK = CT::TK, BT = CT::BT;
  FreeCol<T, TK, MODE> c;
  C2<T>* buf;
  const C2<T>* tw;

  template <int R, int DIR, bool FIRST, bool LAST>
  __device__ __forceinline__ void stage(int Ns)
  {
    constexpr int IT = (CT::E + R - 1) / R;
    constexpr bool MID = MODE == FC_CONV && DIR < 0 && LAST;  // the forward transform's end: into LDS
    constexpr bool STORE = LAST && !MID, LOAD = FIRST && !(MODE == FC_CONV && DIR > 0);
    const int m = c.n / R, NB = TK * m, st = c.n / (Ns * R), f = c.f;
    const float rNs = 1.0f / (float)Ns;
    C2<T> v[IT][R];
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int t = threadIdx.x + it * BT;
      if (t >= NB) continue;
      const int j = t / TK;
#pragma unroll
      for (int r = 0; r < R; ++r) v[it][r] = LOAD ? c.get(j + r * m) : buf[f + (j + r * m) * TK];
      if (!FIRST) {
        const int k = mod_ns(j, Ns, rNs);
#pragma unroll
        for (int r = 1; r < R; ++r) {
          C2<T> w = tw[r * k * st];
          if (DIR > 0) w.y = -w.y;
          v[it][r] = cmul(v[it][r], w);
        }
      }
      dftR<R, DIR>(v[it]);
#pragma unroll
      for (int r = 0; r < R; ++r) asm volatile("" : "+v"(v[it][r].x), "+v"(v[it][r].y));  // as hold()
      if (MID && !c.pair)
#pragma unroll
        for (int r = 0; r < R; ++r) v[it][r] = c.times(v[it][r], j + r * m);
    }
    if (!LOAD && !STORE) __syncthreads();  // the stage's reads are done
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int t = threadIdx.x + it * BT;
      if (t >= NB) continue;
      const int j = t / TK;
      if (STORE) {
        if (c.keep)
#pragma unroll
          for (int r = 0; r < R; ++r)
            if (j + r * m < c.a.nout) c.col[(j + r * m) * c.stride] = v[it][r];
      } else {
        const int k = FIRST ? 0 : mod_ns(j, Ns, rNs), o = FIRST ? j * R : (j - k) * R + k;
#pragma unroll
        for (int r = 0; r < R; ++r) buf[f + (o + r * Ns) * TK] = v[it][r];
      }
    }
    if (!STORE) __syncthreads();
  }

  template <int DIR, bool LAST>
  __device__ __forceinline__ void stage_rt(int R, int Ns)
  {
    if (R == 8) stage<8, DIR, false, LAST>(Ns);
    else if (R == 4) stage<4, DIR, false, LAST>(Ns);
    else if (R == 5) stage<5, DIR, false, LAST>(Ns);
    else if (R == 3) stage<3, DIR, false, LAST>(Ns);
    else stage<2, DIR, false, LAST>(Ns);
  }

  // the plan's radices: the first is 8, and there are two at least (a padded length is 16 x blocks)
  template <int DIR>
  __device__ __forceinline__ void transform(const FftPlan& pl)
  {
    stage<8, DIR, true, false>(1);
    int Ns = 8;
    for (int s = 1; s < pl.ns - 1; ++s) {
      stage_rt<DIR, false>(pl.r[s], Ns);
      Ns *= pl.r[s];
    }
    stage_rt<DIR, true>(pl.r[pl.ns - 1], Ns);
  }
};

template <typename T, int M, int MODE>
__global__ __launch_bounds__((ColTile<T, M>::BT)) void k_free_col_rt(C2<T>* __restrict__ S,
                                                                   const C2<T>* __restrict__ tw, FreeArgs a,
                                                                   FftPlan pl)
{
  using FS = FreeStages<T, M, MODE>;
  FS fs;
  fs.buf = lds_tile<T, 0>();
  fs.tw = tw;
  if (!fs.c.init(S, a, pl.n)) return;
  if constexpr (MODE != FC_INV) fs.template transform<-1>(pl);
  if (MODE == FC_CONV && fs.c.pair) {
    fs.c.times_pairs(fs.buf, threadIdx.x / FS::TK, FS::BT / FS::TK);
    __syncthreads();
  }
  if constexpr (MODE != FC_FWD) fs.template transform<+1>(pl);
}

// ------------------------------------------------------------------ dispatch

template <typename T, int N>
struct XPass {
  // dynamic LDS of the passes whose length is known at run time
  static size_t lds(const Ctx& c) { return N > 0 ? 0 : (size_t)c.N[0] * (N < 0 ? XFFT + 1 : XFFT) * sizeof(C2<T>); }
  static void fwd(Ctx& c, const T* s0, const T* s1, const T* s2, int src, bool force)
  {
    dim3 grid(c.N[1] / BS, c.N[2]);
    const int* slot = c.body.present && !c.plain_rhs ? c.ob_slot_all : nullptr;
    if (src == XSRC_FIELD)
      hipLaunchKernelGGL((k_fft_x_fwd<T, N, XSRC_FIELD, false>), grid, dim3(NT), lds(c), c.stream, s0, s1, s2,
                         Three<C2<T>>{(C2<T>*)c.spec}, (const C2<T>*)c.tw[0], c.grid(), c.sc, (const int*)nullptr,
                         (const T*)nullptr, (double*)nullptr, c.plan[0]);
    else if (force)
      hipLaunchKernelGGL((k_fft_x_fwd<T, N, XSRC_DIV, true>), grid, dim3(NT), lds(c), c.stream, s0, s1, s2, Three<C2<T>>{(C2<T>*)c.spec},
                         (const C2<T>*)c.tw[0], c.grid(), c.sc, slot, (const T*)c.ob_rhs_all, c.low_part, c.plan[0]);
    else
      hipLaunchKernelGGL((k_fft_x_fwd<T, N, XSRC_DIV, false>), grid, dim3(NT), lds(c), c.stream, s0, s1, s2,
                         Three<C2<T>>{(C2<T>*)c.spec}, (const C2<T>*)c.tw[0], c.grid(), c.sc, slot, (const T*)c.ob_rhs_all,
                         (double*)nullptr, c.plan[0]);
  }
  // nf fields to their spectra, and back
  static void fwd_to(Ctx& c, const Three<const T>& s, const Three<C2<T>>& spec, int nf)
  {
    dim3 grid(c.N[1] / BS, c.N[2], nf);
    hipLaunchKernelGGL((k_fft_x_fwd<T, N, XSRC_FIELD, false>), grid, dim3(NT), lds(c), c.stream, s.p[0], s.p[1], s.p[2],
                       spec, (const C2<T>*)c.tw[0], c.grid(), c.sc, (const int*)nullptr, (const T*)nullptr,
                       (double*)nullptr, c.plan[0]);
  }
  static void inv(Ctx& c, const Three<C2<T>>& spec, const Three<T>& dst, int nf, T* xf)
  {
    dim3 grid(c.N[1] / BS, c.N[2], nf);
    if (xf)
      hipLaunchKernelGGL((k_fft_x_inv<T, N, true>), grid, dim3(NT), lds(c), c.stream, spec, dst, (const C2<T>*)c.tw[0],
                         c.grid(), c.plan[0], xf);
    else
      hipLaunchKernelGGL((k_fft_x_inv<T, N>), grid, dim3(NT), lds(c), c.stream, spec, dst, (const C2<T>*)c.tw[0],
                         c.grid(), c.plan[0], (T*)nullptr);
  }
};

template <typename T, int N, int AXIS>
struct ColPass {
  // extra: 1 (y forward) or 2 (z pass with the forcing) runs the forcing's plane or row stage
  // beside the transforms; only the register form takes it (col_extra_ok)
  static void run(Ctx& c, const Three<C2<T>>& spec, int nf, int mode, double norm, bool force = false, int extra = 0)
  {
    if constexpr (ColReg<T, N>::ok) {
      constexpr int TK = ColReg<T, N>::TK;
      const int ncols = c.N[0] / 2;
      const int other = AXIS == 1 ? c.N[2] : c.N[1];
      const int gx = (ncols + TK - 1) / TK;
      ColExtra ex{};
      const ForcingArgs fa = c.forcing;
      if (extra) {
        ex = forcing_planes_extra(c);
        const int work = extra == 1 ? ex.nz * ex.parts : ex.nz;
        ex.ey = (work + gx - 1) / gx;
      }
      dim3 grid(gx, other + ex.ey, nf);
      const C2<T>* tw = (const C2<T>*)c.tw[AXIS];
      if (mode == ZM_FWD && extra == 1)
        hipLaunchKernelGGL((k_fft_colr<T, N, AXIS, ZM_FWD, false, 1>), grid, dim3(NT), 0, c.stream, spec, tw, ncols,
                           c.N[1], c.N[2], norm, c.cos4[0], c.cos4[1], c.cos4[2], c.low_dev, fa, ex);
      else if (mode == ZM_FWD)
        hipLaunchKernelGGL((k_fft_colr<T, N, AXIS, ZM_FWD>), grid, dim3(NT), 0, c.stream, spec, tw, ncols, c.N[1],
                           c.N[2], norm, c.cos4[0], c.cos4[1], c.cos4[2], c.low_dev, fa, ex);
      else if (mode == ZM_INV)
        hipLaunchKernelGGL((k_fft_colr<T, N, AXIS, ZM_INV>), grid, dim3(NT), 0, c.stream, spec, tw, ncols, c.N[1],
                           c.N[2], norm, c.cos4[0], c.cos4[1], c.cos4[2], c.low_dev, fa, ex);
      else if (AXIS == 2 && force && extra == 2)
        hipLaunchKernelGGL((k_fft_colr<T, N, 2, ZM_POISSON, true, 2>), grid, dim3(NT), 0, c.stream, spec, tw, ncols,
                           c.N[1], c.N[2], norm, c.cos4[0], c.cos4[1], c.cos4[2], c.low_dev, fa, ex);
      else if (AXIS == 2 && force)
        hipLaunchKernelGGL((k_fft_colr<T, N, 2, ZM_POISSON, true>), grid, dim3(NT), 0, c.stream, spec, tw, ncols,
                           c.N[1], c.N[2], norm, c.cos4[0], c.cos4[1], c.cos4[2], c.low_dev, fa, ex);
      else if (AXIS == 2)
        hipLaunchKernelGGL((k_fft_colr<T, N, 2, ZM_POISSON, false>), grid, dim3(NT), 0, c.stream, spec, tw, ncols,
                           c.N[1], c.N[2], norm, c.cos4[0], c.cos4[1], c.cos4[2], c.low_dev, fa, ex);
    } else if constexpr (N >= 512) {
      launch<N, N>(c, spec, nf, mode, norm, force);
    } else {
      const int n = c.N[AXIS];
      if (n <= 256) launch<0, 256>(c, spec, nf, mode, norm, force);
      else if (n <= 512) launch<0, 512>(c, spec, nf, mode, norm, force);
      else launch<0, FFT_MAX_N>(c, spec, nf, mode, norm, force);
    }
  }
  template <int NN, int M>
  static void launch(Ctx& c, const Three<C2<T>>& spec, int nf, int mode, double norm, bool force)
  {
    using CT = ColTile<T, M>;
    const int ncols = c.N[0] / 2;
    const dim3 grid((ncols + CT::TK - 1) / CT::TK, AXIS == 1 ? c.N[2] : c.N[1], nf), bt(CT::BT);
    const size_t lds = NN > 0 ? 0 : (size_t)c.N[AXIS] * CT::TK * sizeof(C2<T>);
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid, bt, lds, c.stream, spec, (const C2<T>*)c.tw[AXIS], ncols, AXIS,
                         mode == ZM_INV ? 1 : 0, c.N[1], norm, (const double*)c.cos4[0], (const double*)c.cos4[1],
                         (const double*)c.cos4[2], (const LowModes*)(force ? c.low_dev : nullptr),
                         c.forcing, c.plan[AXIS]);
    };
    if (mode == ZM_POISSON) go(k_fft_col<T, NN, M, true>);
    else go(k_fft_col<T, NN, M, false>);
  }
};

// The free-space solve's x passes on the padded grid: a field of the unpadded one and back.
template <typename T, int N>
struct GoXPad {
  static void go(Ctx& c, const T* src)
  {
    hipLaunchKernelGGL((k_fft_x_fwd<T, N, XSRC_PAD, false>), dim3(c.N[1] / 2 / BS, c.N[2] / 2), dim3(NT),
                       (XPass<T, N>::lds(c)), c.stream, src, src, src, Three<C2<T>>{(C2<T>*)c.spec},
                       (const C2<T>*)c.tw[0], c.grid(), c.sc, (const int*)nullptr, (const T*)nullptr,
                       (double*)nullptr, c.plan[0]);
  }
};
template <typename T, int N>
struct GoXUnpad {
  static void go(Ctx& c, T* dst)
  {
    hipLaunchKernelGGL((k_fft_x_inv<T, N, false, true>), dim3(c.N[1] / 2 / BS, c.N[2] / 2), dim3(NT),
                       (XPass<T, N>::lds(c)), c.stream, Three<C2<T>>{(C2<T>*)c.spec}, Three<T>{dst},
                       (const C2<T>*)c.tw[0], c.grid(), c.plan[0], (T*)nullptr);
  }
};
// A column pass of the free-space solve on the padded grid c, along axis 1 or 2.
template <typename T, int N>
struct GoFree {
  static void go(Ctx& c, int axis, int mode, int others, int nin, int nout)
  {
    const int ncols = c.N[0] / 2, n = c.N[axis];
    const double* G = (const double*)c.ghat;
    const FreeArgs a{ncols, axis, c.N[1], nin, nout, G, G + (mode == FC_CONV ? (size_t)ncols * c.N[1] * c.N[2] : 0)};
    auto grid = [&](int tk) { return dim3((ncols + tk - 1) / tk + (mode == FC_CONV ? 1 : 0), others); };
    if constexpr (N >= 64) {
      auto kern = mode == FC_FWD ? k_free_col<T, N, FC_FWD> : (mode == FC_INV ? k_free_col<T, N, FC_INV> : k_free_col<T, N, FC_CONV>);
      hipLaunchKernelGGL(kern, grid(FreeTile<T, N>::TK), dim3(NT), 0, c.stream, (C2<T>*)c.spec,
                         (const C2<T>*)c.tw[axis], a);
    } else {
      auto launch = [&](auto bound) {
        constexpr int M = decltype(bound)::value;
        using CT = ColTile<T, M>;
        auto kern = mode == FC_FWD ? k_free_col_rt<T, M, FC_FWD> : (mode == FC_INV ? k_free_col_rt<T, M, FC_INV> : k_free_col_rt<T, M, FC_CONV>);
        hipLaunchKernelGGL(kern, grid(CT::TK), dim3(CT::BT), (size_t)n * CT::TK * sizeof(C2<T>), c.stream,
                           (C2<T>*)c.spec, (const C2<T>*)c.tw[axis], a, c.plan[axis]);
      };
      if (n <= 256) launch(std::integral_constant<int, 256>{});
      else if (n <= 512) launch(std::integral_constant<int, 512>{});
      else launch(std::integral_constant<int, FFT_MAX_N>{});
    }
  }
};

// Runtime N -> template N.
template <template <typename, int> class F, typename T, typename... A>
static bool dispatch_n(int n, A&&... a)
{
  switch (n) {
    case 8: F<T, 8>::go(a...); return true;
    case 16: F<T, 16>::go(a...); return true;
    case 32: F<T, 32>::go(a...); return true;
    case 64: F<T, 64>::go(a...); return true;
    case 128: F<T, 128>::go(a...); return true;
    case 256: F<T, 256>::go(a...); return true;
    case 512: F<T, 512>::go(a...); return true;
    case 1024: F<T, 1024>::go(a...); return true;
    default: F<T, 0>::go(a...); return true;  // the plan's radices, fft_setup checked the length
  }
}

// The same for the x passes, whose run-time form has two bounds.
template <template <typename, int> class F, typename T, typename... A>
static bool dispatch_x(int n, A&&... a)
{
  if (n <= 256 && (n & (n - 1))) {
    F<T, X_SHORT>::go(a...);
    return true;
  }
  return dispatch_n<F, T>(n, a...);
}

template <typename T, int N>
struct GoXFwd {
  static void go(Ctx& c, const T* s0, const T* s1, const T* s2, int src, bool force)
  {
    XPass<T, N>::fwd(c, s0, s1, s2, src, force);
  }
};
template <typename T, int N>
struct GoXFwdTo {
  static void go(Ctx& c, const Three<const T>& s, const Three<C2<T>>& spec, int nf) { XPass<T, N>::fwd_to(c, s, spec, nf); }
};
template <typename T, int N>
struct GoXInv {
  static void go(Ctx& c, const Three<C2<T>>& spec, const Three<T>& dst, int nf, T* xf = nullptr)
  {
    XPass<T, N>::inv(c, spec, dst, nf, xf);
  }
};
template <typename T, int N>
struct GoY {
  static void go(Ctx& c, const Three<C2<T>>& spec, int nf, int mode, double norm)
  {
    ColPass<T, N, 1>::run(c, spec, nf, mode, norm);
  }
};
template <typename T, int N>
struct GoZ {
  static void go(Ctx& c, const Three<C2<T>>& spec, int nf, int mode, double norm)
  {
    ColPass<T, N, 2>::run(c, spec, nf, mode, norm);
  }
};
template <typename T, int N>
struct GoZF {
  static void go(Ctx& c, const Three<C2<T>>& spec, int mode, double norm)
  {
    ColPass<T, N, 2>::run(c, spec, 1, mode, norm, true);
  }
};
// the same passes with the forcing's plane stage (y forward) or row stage (z) beside them
template <typename T, int N>
struct GoYPlanes {
  static void go(Ctx& c, const Three<C2<T>>& spec, int mode, double norm)
  {
    ColPass<T, N, 1>::run(c, spec, 1, mode, norm, false, 1);
  }
};
template <typename T, int N>
struct GoZFRows {
  static void go(Ctx& c, const Three<C2<T>>& spec, int mode, double norm)
  {
    ColPass<T, N, 2>::run(c, spec, 1, mode, norm, true, 2);
  }
};

// The column lengths whose passes take the register form (ColReg::ok over dispatch_n's cases).
static bool col_extra_ok(int n) { return n == 64 || n == 128 || n == 256; }

static double poisson_norm(const Ctx& c)
{
  return 4.0 / ((double)c.N[0] * c.h * (double)c.N[1] * (double)c.N[2]);
}

template <typename T>
int poisson_fused_t(Ctx& c, bool force, double tke_target, double inj_rate, bool xface)
{
  const Three<C2<T>> S{(C2<T>*)c.spec};
  const double norm = poisson_norm(c);
  if (force) c.forcing = forcing_args(c, tke_target, inj_rate);
  stage_mark(c, ST_XFWD, false);
  dispatch_x<GoXFwd, T>(c.N[0], c, (const T*)c.f[c.ustar], (const T*)c.f[c.ustar + 1],
                        (const T*)c.f[c.ustar + 2], (int)XSRC_DIV, force);
  stage_mark(c, ST_XFWD, true);
  // With the register form of the column passes, the forcing's plane stage runs as extra
  // workgroups of the y forward pass and its row stage beside the z pass, leaving the mode sums
  // (k_forcing_reduce) the only kernel of the forcing between them. Otherwise the three stages
  // are small kernels in order (a second stream's fork and join cost more here).
  const bool extra = force && col_extra_ok(c.N[1]) && col_extra_ok(c.N[2]);
  if (force && !extra) {
    stage_mark(c, ST_FREDUCE, false);
    if (int rc = launch_forcing_reduce(c)) return rc;
    if (int rc = launch_forcing_rows(c)) return rc;
    stage_mark(c, ST_FREDUCE, true);
  }
  stage_mark(c, ST_YFWD, false);
  if (extra) dispatch_n<GoYPlanes, T>(c.N[1], c, S, (int)ZM_FWD, norm);
  else dispatch_n<GoY, T>(c.N[1], c, S, 1, (int)ZM_FWD, norm);
  stage_mark(c, ST_YFWD, true);
  if (extra) {
    stage_mark(c, ST_FREDUCE, false);
    if (int rc = launch_forcing_reduce(c, false)) return rc;
    stage_mark(c, ST_FREDUCE, true);
  }
  stage_mark(c, ST_ZPASS, false);
  if (extra) dispatch_n<GoZFRows, T>(c.N[2], c, S, (int)ZM_POISSON, norm);
  else if (force) dispatch_n<GoZF, T>(c.N[2], c, S, (int)ZM_POISSON, norm);
  else dispatch_n<GoZ, T>(c.N[2], c, S, 1, (int)ZM_POISSON, norm);
  stage_mark(c, ST_ZPASS, true);
  stage_mark(c, ST_YINV, false);
  dispatch_n<GoY, T>(c.N[1], c, S, 1, (int)ZM_INV, norm);
  stage_mark(c, ST_YINV, true);
  stage_mark(c, ST_XINV, false);
  dispatch_x<GoXInv, T>(c.N[0], c, S, Three<T>{(T*)c.f[CUP_P]}, 1, xface ? (T*)c.xface : (T*)nullptr);
  stage_mark(c, ST_XINV, true);
  c.xface_ok = xface;
  return check_hip(c, hipGetLastError(), "poisson_fused");
}

// The RHS stays in rbuf; the solution goes to p.
template <typename T>
int poisson_plain_t(Ctx& c)
{
  const Three<C2<T>> S{(C2<T>*)c.spec};
  const double norm = poisson_norm(c);
  dispatch_x<GoXFwdTo, T>(c.N[0], c, Three<const T>{(const T*)c.rbuf}, S, 1);
  dispatch_n<GoY, T>(c.N[1], c, S, 1, (int)ZM_FWD, norm);
  dispatch_n<GoZ, T>(c.N[2], c, S, 1, (int)ZM_POISSON, norm);
  dispatch_n<GoY, T>(c.N[1], c, S, 1, (int)ZM_INV, norm);
  dispatch_x<GoXInv, T>(c.N[0], c, S, Three<T>{(T*)c.f[CUP_P]}, 1);
  return check_hip(c, hipGetLastError(), "poisson_plain");
}

template <typename T>
int fwd_fields_t(Ctx& c, const void* const* real_blocks, void* const* spec, int nf)
{
  Three<const T> s{};
  Three<C2<T>> S{};
  for (int q = 0; q < nf; ++q) {
    s.p[q] = (const T*)real_blocks[q];
    S.p[q] = (C2<T>*)spec[q];
  }
  dispatch_x<GoXFwdTo, T>(c.N[0], c, s, S, nf);
  dispatch_n<GoY, T>(c.N[1], c, S, nf, (int)ZM_FWD, 0.0);
  dispatch_n<GoZ, T>(c.N[2], c, S, nf, (int)ZM_FWD, 0.0);
  return check_hip(c, hipGetLastError(), "fft_forward_fields");
}

template <typename T>
int inv_fields_t(Ctx& c, void* const* spec, void* const* real_blocks, int nf)
{
  Three<T> d{};
  Three<C2<T>> S{};
  for (int q = 0; q < nf; ++q) {
    d.p[q] = (T*)real_blocks[q];
    S.p[q] = (C2<T>*)spec[q];
  }
  dispatch_n<GoZ, T>(c.N[2], c, S, nf, (int)ZM_INV, 0.0);
  dispatch_n<GoY, T>(c.N[1], c, S, nf, (int)ZM_INV, 0.0);
  dispatch_x<GoXInv, T>(c.N[0], c, S, d, nf);
  return check_hip(c, hipGetLastError(), "fft_inverse_fields");
}

// ------------------------------------------------------- PoissonSolverMixed
// PoissonSolverMixed::solve (PoissonSolverMixed.cpp:66-103, _solve PoissonSolverMixed.h:27-80):
// FFTW r2r transforms per axis, R2HC / HC2R on periodic axes and REDFT10 / REDFT01 (DCT-II /
// DCT-III) on the others (PoissonSolverMixed.cpp:37-42), here as dense N x N matrices, a
// contraction over each line on the matrix cores; the coefficient (i, j, k) times
// norm / (denX_i + denY_j + denZ_k) in FP64, the first one zeroed.
//
// One workgroup transforms LN (16 or 32) lines of N cells: it stages them in LDS as X[j][line] and forms
// Y = M X in 16 x 16 tiles of the 16x16x4 matrix instruction (M's fragments from the cache, 16
// columns of j ahead; X's from LDS, two line groups per fragment of M), then stores each tile
// back over its lines. What bounds it is the latency of M's fragments in the cache, not the
// matrix units (2 us a pass at their rate) or the field's traffic: on 128 x 96 x 64 cells in FP64
// a pass takes 9 to 12 us, against 50 us with one thread per output walking its line, where every
// line read the whole matrix.
template <typename T>
struct MatTile;
template <>
struct MatTile<double> {
  typedef double acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc mma(double a, double b, acc c)
  {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // the tile row of a lane's v-th accumulator (its column is lane % 16)
  static __device__ __forceinline__ int row(int lane, int v) { return (lane >> 4) + 4 * v; }
};
template <>
struct MatTile<float> {
  typedef float acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc mma(float a, float b, acc c)
  {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int v) { return 4 * (lane >> 4) + v; }
};

constexpr int R2R_STAGE = 17;  // row pitch of a wave's 16 x 16 staging tile
// Row pitch of X: the four rows a fragment reads fall on distinct banks.
constexpr int r2r_pitch(int ln) { return ln == 16 ? 16 : ln + 16; }
// Threads: a wave for each 16 x 16 tile of 16 lines up to 128 cells (a launch of few workgroups lasts
// as long as a wave's tiles), four waves otherwise.
template <int LN>
constexpr int r2r_threads() { return LN == 16 ? 512 : NT; }
template <typename T, int LN, int AXIS>
inline size_t r2r_lds(int n)
{
  return ((size_t)n * r2r_pitch(LN) + (AXIS == 0 ? r2r_threads<LN>() / 64 * 16 * R2R_STAGE : 0)) * sizeof(T);
}

// src and dst may be the same field: a workgroup reads its lines before it writes them. dx, dy,
// dz: the symbol's terms when this pass (along z) also divides, else null.
template <typename T, int LN, int AXIS>
__global__ __launch_bounds__(r2r_threads<LN>()) void k_r2r_axis(const T* src, T* dst, const T* __restrict__ mt, GridArgs g,
                                                 double norm, const double* __restrict__ dx,
                                                 const double* __restrict__ dy, const double* __restrict__ dz)
{
  using MT = MatTile<T>;
  using V2 = typename Vec2<T>::type;
  using V4 = typename Vec4<T>::type;
  constexpr int BT = r2r_threads<LN>(), PX = r2r_pitch(LN), SUB = 64 / LN, NG = LN / 16, GI = NG > 1 ? 2 : 1;
  extern __shared__ __align__(32) unsigned char r2r_lds_buf[];
  T* X = reinterpret_cast<T*>(r2r_lds_buf);
  const int n = AXIS == 0 ? g.Nx : (AXIS == 1 ? g.Ny : g.Nz);
  const int sub = blockIdx.x % SUB, o = blockIdx.x / SUB;  // LN of the 64 lines through a row of blocks
  const int n1 = AXIS == 0 ? g.nby : g.nbx, o1 = o % n1, o2 = o / n1;
  auto block = [&](int q) -> size_t {  // the q-th block along the lines
    return AXIS == 0 ? q + (size_t)g.nbx * (o1 + (size_t)g.nby * o2)
                     : (AXIS == 1 ? o1 + (size_t)g.nbx * (q + (size_t)g.nby * o2)
                                  : o1 + (size_t)g.nbx * (o2 + (size_t)g.nby * q));
  };
  // Pairs of x-adjacent cells; line = (iz, iy) for x, (iz, ix) for y, (iy, ix) for z, the first
  // index from sub * LN/8 on. Each wave reads whole 64-byte sectors and writes runs of lines.
  #pragma unroll 4
  for (int r = threadIdx.x; r < n * LN / 2; r += BT) {
    const int q = r / (LN * 4), p = r % (LN * 4);
    int cell, j, line;
    if (AXIS == 0) {
      line = (p >> 6) * 16 + (p & 15);
      const int xp = (p >> 4) & 3;
      cell = (sub * LN + line) * BS + 2 * xp;
      j = q * BS + 2 * xp;
    } else if (AXIS == 1) {
      const int xp = p & 3, iz = (p >> 6) * 2 + ((p >> 2) & 1), iy = (p >> 3) & 7;
      line = iz * BS + 2 * xp;
      cell = ((sub * (LN / BS) + iz) * BS + iy) * BS + 2 * xp;
      j = q * BS + iy;
    } else {
      line = 2 * (p % (LN / 2));
      const int iz = p / (LN / 2);
      cell = iz * BS * BS + sub * LN + line;
      j = q * BS + iz;
    }
    const V2 v = *reinterpret_cast<const V2*>(src + block(q) * BS3 + cell);
    if (AXIS == 0) {
      X[j * PX + line] = v.x;
      X[(j + 1) * PX + line] = v.y;
    } else {
      *reinterpret_cast<V2*>(&X[j * PX + line]) = v;
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lc = lane & 15, lr = lane >> 4;
  const int items = (n + 15) / 16 * (NG / GI);
  for (int item = wv; item < items; item += BT / 64) {
    const int i0 = item / (NG / GI) * 16, g0 = item % (NG / GI) * GI;
    const int ai = min(i0 + lc, n - 1);  // the last tile's rows past n are not stored
    typename MT::acc acc[GI];
#pragma unroll
    for (int q = 0; q < GI; ++q) acc[q] = typename MT::acc{0, 0, 0, 0};
    // M's fragments, two groups of 16 columns ahead (n is a multiple of 8: the last group may be half
    // empty)
    T a[3][4];
    auto fetch = [&](T (&f)[4], int j0) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = j0 + 4 * q + lr;
        f[q] = j < n ? mt[(size_t)j * n + ai] : (T)0;
      }
    };
    fetch(a[0], 0);
    fetch(a[1], 16);
    for (int j0 = 0; j0 < n; j0 += 16) {
      fetch(a[2], j0 + 32);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int j = min(j0 + 4 * q + lr, n - 1);
#pragma unroll
        for (int k = 0; k < GI; ++k) acc[k] = MT::mma(a[0][q], X[j * PX + (g0 + k) * 16 + lc], acc[k]);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        a[0][q] = a[1][q];
        a[1][q] = a[2][q];
      }
    }
#pragma unroll
    for (int k = 0; k < GI; ++k) {
      const int line = (g0 + k) * 16 + lc;
      if (AXIS == 0) {
        // through the wave's staging tile, so that a line's cells leave as whole vectors
        T* st = X + (size_t)n * PX + wv * 16 * R2R_STAGE;
#pragma unroll
        for (int v = 0; v < 4; ++v) st[MT::row(lane, v) * R2R_STAGE + lc] = acc[k][v];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int sl = lane >> 2, i = 4 * (lane & 3);
        const V4 w = {st[i * R2R_STAGE + sl], st[(i + 1) * R2R_STAGE + sl], st[(i + 2) * R2R_STAGE + sl],
                      st[(i + 3) * R2R_STAGE + sl]};
        if (i0 + i < n)
          *reinterpret_cast<V4*>(dst + block((i0 + i) >> 3) * BS3 + (sub * LN + (g0 + k) * 16 + sl) * BS +
                                 ((i0 + i) & 7)) = w;
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = i0 + MT::row(lane, v);
          if (i >= n) continue;
          const int cell = AXIS == 1 ? ((sub * (LN / BS) + (line >> 3)) * BS + (i & 7)) * BS + (line & 7)
                                     : (i & 7) * BS * BS + sub * LN + line;
          T out = acc[k][v];
          if (AXIS == 2 && dx) {
            const int x = o1 * BS + (line & 7), y = o2 * BS + sub * (LN / BS) + (line >> 3);
            out = (x | y | i) ? (T)((double)out * (norm / (dx[x] + dy[y] + dz[i]))) : (T)0;
          }
          dst[block(i >> 3) * BS3 + cell] = out;
        }
      }
    }
  }
}

template <typename T>
static int mixed_setup(Ctx& c)
{
  const double tol = 0.01;  // PoissonSolverMixed.h:50
  for (int d = 0; d < 3; ++d) {
    if (c.mden[d]) continue;
    const int n = c.N[d];
    const bool per = c.bc[d] == CUP_BC_PERIODIC;
    std::vector<T> fw((size_t)n * n), bw((size_t)n * n);  // transposed: m[j][k] = M[k][j]
    for (int k = 0; k < n; ++k)
      for (int j = 0; j < n; ++j) {
        double f, b;
        if (per) {
          // R2HC (halfcomplex out: r_0..r_{n/2}, then i_{n/2-1}..i_1) and HC2R
          f = k <= n / 2 ? cos(2 * M_PI * (double)j * k / n) : -sin(2 * M_PI * (double)j * (n - k) / n);
          if (j == 0) b = 1;
          else if (2 * j == n) b = cos(M_PI * (double)k);
          else if (j < n / 2) b = 2 * cos(2 * M_PI * (double)j * k / n);
          else b = -2 * sin(2 * M_PI * (double)(n - j) * k / n);
        } else {
          f = 2 * cos(M_PI * (j + 0.5) * k / n);                      // REDFT10
          b = j == 0 ? 1 : 2 * cos(M_PI * (double)j * (k + 0.5) / n);  // REDFT01
        }
        fw[(size_t)j * n + k] = (T)f;
        bw[(size_t)j * n + k] = (T)b;
      }
    std::vector<double> den((size_t)n);
    const double wf = (per ? 2 : 1) * M_PI / n;
    for (int i = 0; i < n; ++i) {
      const int kk = per ? (i <= n / 2 ? i : n - i) : i;
      const double rk = (kk + (per ? 0.0 : 0.5)) * wf;
      den[i] = (1 - tol) * (cos(2 * wf * i) - 1) / 2 - tol * rk * rk;
    }
    for (int q = 0; q < 2; ++q) {
      if (check_hip(c, hipMalloc(&c.r2r[d][q], fw.size() * sizeof(T)), "hipMalloc r2r")) return CUP_E_NOMEM;
      hipMemcpy(c.r2r[d][q], q ? bw.data() : fw.data(), fw.size() * sizeof(T), hipMemcpyHostToDevice);
    }
    if (check_hip(c, hipMalloc(&c.mden[d], den.size() * sizeof(double)), "hipMalloc mixed symbol")) return CUP_E_NOMEM;
    hipMemcpy(c.mden[d], den.data(), den.size() * sizeof(double), hipMemcpyHostToDevice);
  }
  return CUP_OK;
}

// Lines per workgroup: 32 share each fragment of the matrix where the tile keeps two workgroups on a
// CU (64 KiB) and the launch has two for every CU, 16 otherwise. 16 / 32 lines, x, y and z pass: FP64
// 26.5 / 23.0, 24.4 / 23.4 and 28.5 / 26.8 us on 128^3, 14.0 / 17.8, 10.6 / 13.8 and 9.5 / 10.3 on
// 128 x 96 x 64; FP32 16.3 / 17.6, 16.0 / 18.3 and 20.1 / 19.2 on 128^3, 55.8 / 58.6, 63.5 / 60.5 and
// 68.3 / 67.8 on 192^3. 64 lines, where 64 KiB hold them, are slower (94, 90 and 109 there).
template <typename T, int AXIS>
static void r2r_pass(Ctx& c, const T* src, T* dst, int q, double norm, bool divide)
{
  const int n = c.N[AXIS], rows = (int)(c.ncell / (size_t)n / 64);
  auto go = [&](auto kern, int ln, size_t lds) {
    hipLaunchKernelGGL(kern, dim3(rows * (64 / ln)), dim3(ln == 16 ? r2r_threads<16>() : NT), lds, c.stream, src, dst, (const T*)c.r2r[AXIS][q],
                       c.grid(), norm, (const double*)(divide ? c.mden[0] : nullptr), (const double*)c.mden[1],
                       (const double*)c.mden[2]);
  };
  constexpr size_t cap = 64 * 1024;
  if (rows >= 256 && r2r_lds<T, 32, AXIS>(n) <= cap) go(k_r2r_axis<T, 32, AXIS>, 32, r2r_lds<T, 32, AXIS>(n));
  else go(k_r2r_axis<T, 16, AXIS>, 16, r2r_lds<T, 16, AXIS>(n));
}

// The RHS stays in rbuf; the transforms work in the spectrum's buffer and end in p.
template <typename T>
int poisson_mixed_t(Ctx& c)
{
  if (int rc = mixed_setup<T>(c)) return rc;
  T* a = (T*)c.spec;
  double norm = 1 / c.h;
  for (int d = 0; d < 3; ++d) norm *= (c.bc[d] == CUP_BC_PERIODIC ? 1.0 : 0.5) / c.N[d];
  r2r_pass<T, 0>(c, (const T*)c.rbuf, a, 0, norm, false);
  r2r_pass<T, 1>(c, a, a, 0, norm, false);
  r2r_pass<T, 2>(c, a, a, 0, norm, true);
  // The order of the inverse passes is free up to rounding. On the one box where it was measured
  // (dirichlet, wall, periodic, 128 x 96 x 64 in FP64, two steps) p is off by 2.5e-14 in the order
  // x, y, z and by 5.8e-14 in the order z, y, x.
  r2r_pass<T, 0>(c, a, a, 1, norm, false);
  r2r_pass<T, 1>(c, a, a, 1, norm, false);
  r2r_pass<T, 2>(c, a, (T*)c.f[CUP_P], 1, norm, false);
  return check_hip(c, hipGetLastError(), "poisson_mixed");
}

// ------------------------------------------------------ PoissonSolverUnbounded
// PoissonSolverUnbounded::solve (PoissonSolverUnbounded.cpp:126-157): Eastwood and
// Brownrigg's cyclic convolution of the zero-padded RHS with the free-space Green's function
// of the uniform mesh, -h^2/(4 pi r) (r in cells; r = 0: -0.1924173658 h^2, :216-218), times
// 1/h^3 (:50). The reference pads to 2N-1 points per axis; here the period is 2N (the FFT
// passes' lengths), with the Green's function mirrored about N: on the physical points the
// cyclic convolution of either period is the linear one (distances stay below N, and the
// entry at distance N never meets a non-zero RHS value), so the solution is the same. The
// padded grid is a periodic context of its own (2 bpd blocks per axis) that shares the
// parent's stream; its Green's function spectrum (real: the function is even) is computed
// once.

// The free-space Green's function on the padded grid (block layout), distances mirrored
// about N per axis, times 1/h^3: -1/(4 pi h r), r = 0: -0.1924173658/h.
template <typename T>
__global__ __launch_bounds__(NT) void k_green(T* __restrict__ G, GridArgs pg, double h)
{
  const int b = blockIdx.x;
  const int bx = b % pg.nbx, by = (b / pg.nbx) % pg.nby, bz = b / (pg.nbx * pg.nby);
  for (int c = threadIdx.x; c < BS3; c += NT) {
    const int X = bx * BS + (c & 7), Y = by * BS + ((c >> 3) & 7), Z = bz * BS + (c >> 6);
    const double xi = X <= pg.Nx / 2 ? X : pg.Nx - X, yi = Y <= pg.Ny / 2 ? Y : pg.Ny - Y,
                 zi = Z <= pg.Nz / 2 ? Z : pg.Nz - Z;
    const double r = sqrt(xi * xi + yi * yi + zi * zi);
    G[(size_t)b * BS3 + c] = (T)(r > 0 ? -1.0 / (4 * M_PI * h * r) : -0.1924173658 / h);
  }
}

// The Green's function's spectrum as the solve takes it: real (the function is even), times the
// normalization, in FP64; slot 0 of the packed spectrum holds its kx = 0 and kx = Nx/2 planes.
template <typename T>
__global__ void k_green_real(const C2<T>* __restrict__ S, double* __restrict__ G, double* __restrict__ GE, int ncols,
                             size_t n, double norm)
{
  for (size_t i = (size_t)blockIdx.x * NT + threadIdx.x; i < n; i += (size_t)gridDim.x * NT) {
    const C2<T> v = S[i];
    G[i] = (double)v.x * norm;
    if (i % ncols == 0) GE[i / ncols] = (double)v.y * norm;
  }
}

template <typename T>
static int unbounded_setup_t(Ctx& c)
{
  Ctx* p = new (std::nothrow) Ctx();
  if (!p) return set_error(c, CUP_E_NOMEM, "poisson_unbounded: out of host memory");
  c.unb = p;
  p->dev = c.dev;
  p->stream = c.stream;
  p->precision = c.precision;
  p->esz = c.esz;
  p->decomposition = CUP_PLAIN;
  for (int a = 0; a < 3; ++a) {
    p->bpd[a] = 2 * c.bpd[a];
    p->N[a] = 2 * c.N[a];
    p->extent[a] = 2 * c.extent[a];
  }
  p->nb = 8 * c.nb;
  p->ncell = 8 * c.ncell;
  p->h = c.h;
  p->maxextent = 2 * c.maxextent;
  p->sc = c.sc;
  if (int rc = fft_setup(*p)) return set_error(c, rc, "poisson_unbounded: " + p->err);
  const size_t nlines = (size_t)p->N[1] * p->N[2], ncols = p->N[0] / 2, nspec = ncols * nlines;
  // ghat: the kx = Nx/2 plane behind the others
  if (check_hip(c, hipMalloc(&p->spec, nspec * sizeof(C2<T>)), "hipMalloc unbounded spectrum") ||
      check_hip(c, hipMalloc(&p->rbuf, p->ncell * sizeof(T)), "hipMalloc unbounded kernel") ||
      check_hip(c, hipMalloc(&p->ghat, (nspec + nlines) * sizeof(double)), "hipMalloc unbounded kernel"))
    return CUP_E_NOMEM;
  hipLaunchKernelGGL((k_green<T>), dim3(p->nb), dim3(NT), 0, c.stream, (T*)p->rbuf, p->grid(), c.h);
  dispatch_x<GoXFwdTo, T>(p->N[0], *p, Three<const T>{(const T*)p->rbuf}, Three<C2<T>>{(C2<T>*)p->spec}, 1);
  dispatch_n<GoFree, T>(p->N[1], *p, 1, (int)FC_FWD, p->N[2], p->N[1], p->N[1]);
  dispatch_n<GoFree, T>(p->N[2], *p, 2, (int)FC_FWD, p->N[1], p->N[2], p->N[2]);
  hipLaunchKernelGGL((k_green_real<T>), dim3((unsigned)std::min<size_t>(65536, (nspec + NT - 1) / NT)), dim3(NT), 0,
                     c.stream, (const C2<T>*)p->spec, (double*)p->ghat, (double*)p->ghat + nspec, (int)ncols, nspec,
                     1.0 / ((double)p->N[0] * p->N[1] * p->N[2]));
  if (check_hip(c, hipGetLastError(), "unbounded kernel") ||
      check_hip(c, hipStreamSynchronize(c.stream), "synchronize"))
    return CUP_E_DEVICE;
  hipFree(p->rbuf);  // the Green's function itself is not needed again
  p->rbuf = nullptr;
  return CUP_OK;
}

// Only what the convolution needs: the RHS's rows forward along x (a quarter of the padded grid's
// rows), their planes along y (half), every column along z, forward, times the Green's function and
// back, the field's half of the planes along y and its quarter of the rows along x. Against padding
// the RHS, transforming the whole padded grid, multiplying and copying the solution out, a solve on
// 64^3 cells takes 39 us for 69 in FP64 and 30 for 58 in FP32, on 96^3 100 for 394 and 70 for 261.
template <typename T>
int poisson_unbounded_t(Ctx& c)
{
  if (!c.unb)
    if (int rc = unbounded_setup_t<T>(c)) {
      unbounded_free(c);
      return rc;
    }
  Ctx& p = *c.unb;
  p.stream = c.stream;
  dispatch_x<GoXPad, T>(p.N[0], p, (const T*)c.rbuf);
  dispatch_n<GoFree, T>(p.N[1], p, 1, (int)FC_FWD, c.N[2], c.N[1], p.N[1]);
  dispatch_n<GoFree, T>(p.N[2], p, 2, (int)FC_CONV, p.N[1], c.N[2], c.N[2]);
  dispatch_n<GoFree, T>(p.N[1], p, 1, (int)FC_INV, c.N[2], p.N[1], c.N[1]);
  dispatch_x<GoXUnpad, T>(p.N[0], p, (T*)c.f[CUP_P]);
  return check_hip(c, hipGetLastError(), "poisson_unbounded");
}

#ifdef CUP_FFT_F64
template int poisson_fused_t<double>(Ctx& c, bool force, double tke_target, double inj_rate, bool xface);
template int poisson_plain_t<double>(Ctx& c);
template int fwd_fields_t<double>(Ctx& c, const void* const* real_blocks, void* const* spec, int nf);
template int inv_fields_t<double>(Ctx& c, void* const* spec, void* const* real_blocks, int nf);
template int poisson_mixed_t<double>(Ctx& c);
template int poisson_unbounded_t<double>(Ctx& c);
#else
extern template int poisson_fused_t<double>(Ctx& c, bool force, double tke_target, double inj_rate, bool xface);
extern template int poisson_plain_t<double>(Ctx& c);
extern template int fwd_fields_t<double>(Ctx& c, const void* const* real_blocks, void* const* spec, int nf);
extern template int inv_fields_t<double>(Ctx& c, void* const* spec, void* const* real_blocks, int nf);
extern template int poisson_mixed_t<double>(Ctx& c);
extern template int poisson_unbounded_t<double>(Ctx& c);

int launch_poisson_fused(Ctx& c, bool force, double tke_target, double inj_rate, bool xface)
{
  c.xface_ok = false;
  if (force && !c.low_fused_ok) return set_error(c, CUP_E_INVALID, "fused forcing: low-mode set not supported");
  return c.precision == 4 ? poisson_fused_t<float>(c, force, tke_target, inj_rate, xface)
                          : poisson_fused_t<double>(c, force, tke_target, inj_rate, xface);
}

int launch_poisson_plain(Ctx& c)
{
  return c.precision == 4 ? poisson_plain_t<float>(c) : poisson_plain_t<double>(c);
}

int launch_fft_forward_fields(Ctx& c, const void* const* real_blocks, void* const* spec, int nf)
{
  return c.precision == 4 ? fwd_fields_t<float>(c, real_blocks, spec, nf)
                          : fwd_fields_t<double>(c, real_blocks, spec, nf);
}

int launch_fft_inverse_fields(Ctx& c, void* const* spec, void* const* real_blocks, int nf)
{
  return c.precision == 4 ? inv_fields_t<float>(c, spec, real_blocks, nf)
                          : inv_fields_t<double>(c, spec, real_blocks, nf);
}

int launch_poisson_mixed(Ctx& c)
{
  return c.precision == 4 ? poisson_mixed_t<float>(c) : poisson_mixed_t<double>(c);
}

void unbounded_free(Ctx& c)
{
  if (!c.unb) return;
  Ctx& p = *c.unb;
  void* bufs[] = {p.spec, p.rbuf, p.ghat, p.tw[0], p.tw[1], p.tw[2]};
  for (void* b : bufs)
    if (b) hipFree(b);
  for (auto* q : p.cos4)
    if (q) hipFree(q);
  delete c.unb;
  c.unb = nullptr;
}

int launch_poisson_unbounded(Ctx& c)
{
  if (2 * std::max(c.N[0], std::max(c.N[1], c.N[2])) > FFT_MAX_N)
    return set_error(c, CUP_E_INVALID, "poisson_unbounded: the padded grid needs at most 512 cells per axis");
  return c.precision == 4 ? poisson_unbounded_t<float>(c) : poisson_unbounded_t<double>(c);
}

// Twiddle tables e^{-2 pi i t/N} (t < N) per axis and the Poisson cosine tables, built in
// FP64 on the host.
int fft_setup(Ctx& c)
{
  for (int a = 0; a < 3; ++a) {
    const int n = c.N[a];
    // powers of two take the kernels specialised for their length; other lengths the
    // run-time radix plan (8, 4, 2, then 3 and 5), as FFTW plans any size
    // (PoissonSolverPeriodic.cpp:108-121)
    FftPlan& pl = c.plan[a];
    pl = FftPlan{};
    pl.n = n;
    int rem = n;
    for (int r : {8, 4, 2, 3, 5})
      while (rem % r == 0 && pl.ns < 16) {
        pl.r[pl.ns++] = r;
        rem /= r;
      }
    if (n < 8 || n > FFT_MAX_N || rem != 1)
      return set_error(c, CUP_E_INVALID,
                       "FFT sizes must be between 8 and 1024 cells per axis with no prime factor above 5");
    std::vector<double> tw(2 * (size_t)n), cs((size_t)n);
    for (int t = 0; t < n; ++t) {
      const double ang = 2.0 * M_PI * (double)t / (double)n;
      tw[2 * t] = cos(ang);
      tw[2 * t + 1] = -sin(ang);
      cs[t] = cos(4.0 * M_PI * (double)t / (double)n);
    }
    if (check_hip(c, hipMalloc(&c.tw[a], (size_t)n * 2 * c.esz), "hipMalloc twiddles")) return CUP_E_DEVICE;
    if (c.precision == 4) {
      std::vector<float> twf(2 * (size_t)n);
      for (size_t i = 0; i < twf.size(); ++i) twf[i] = (float)tw[i];
      hipMemcpy(c.tw[a], twf.data(), twf.size() * sizeof(float), hipMemcpyHostToDevice);
    } else {
      hipMemcpy(c.tw[a], tw.data(), tw.size() * sizeof(double), hipMemcpyHostToDevice);
    }
    if (check_hip(c, hipMalloc(&c.cos4[a], (size_t)n * sizeof(double)), "hipMalloc cos4")) return CUP_E_DEVICE;
    hipMemcpy(c.cos4[a], cs.data(), cs.size() * sizeof(double), hipMemcpyHostToDevice);
  }
  return CUP_OK;
}
#endif

}  // namespace cup
