// damp.hip -- FFT damping of the velocities (DAMPING = 1).
//
// damp_velocity (all_modules.f90:1802-1888) takes, per z plane, the
// unnormalised r2c transform of a velocity field, multiplies it by
// damping_rates(kx, ky) (INIT_DAMPING, initialize.f90:1276-1336; the rates
// carry the 1/(nx*ny) of the transform pair) and transforms back (c2r); the
// RHS subtracts the result (RHS.f90:166-172, 659-665).  Here a block takes one
// plane of one field through all of it in LDS (k_damp_plane), or, where a
// plane does not fit or its sides have other prime factors than 2, 3, 5 and 7,
// the nz planes of a field go through one batched hipFFT plan each way and the
// multiply is one kernel over the half spectra.  The stage kernel subtracts
// the three terms at the point after its boundary zeroing.
#include <hipfft/hipfft.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "sparc_dev.h"

namespace sparc {

// ---------------------------------------------------------------------------
// One plane in LDS
//
// Through the library a plane passes five launches (x and y transforms each
// way, the multiply) that read and write it ten times.  Here one block reads it
// once and writes the term once.  Three velocities, all planes, FP64: 48x48x96
// 39 -> 17 us, 64x96x100 61 -> 30, 100x100x100 136 -> 48, 128x128x64 65 -> 36,
// 128x96x100 81 -> 56 (100 KB, so one block a CU, and 300 blocks are two rounds
// of 256), 75x75x300 297 -> 67; FP32 128x96x100 67 -> 31, 128x128x128 78 -> 36.
// What bounds it: the first load, at the rate of HBM, then the LDS passes, each
// a round trip of the plane and the fetch of its instructions.
//
// Two rows r and r + ny/2 travel as the real and imaginary part of one complex
// line through the x transform, so LDS holds the plane's half spectrum (64x96
// FP64: 51 KB, three blocks a CU).  All transforms are in place, decimation in
// frequency on the way in and in time on the way back, so the spectrum stands
// in digit order and nothing is ever reordered: `places` tells where a
// frequency's column is and the rates are laid out in that order.  The last y
// pass of the way in and the first of the way back hold the same values:
// transform, multiply and transform back happen in registers.  The outer y
// passes hold both rows of a line where their radix is even, and split and join
// them.  The fewest passes win, up to radix 16 (128x96x100: radices up to 16 56
// us, up to 12 61, up to 8 67).  Lanes run over the lines and the line stride S
// is odd, so x passes are free of bank conflicts; y passes take the columns in
// the order in which they lie.
// ---------------------------------------------------------------------------
constexpr int DP_MAXPASS = 8;
constexpr size_t kLdsBytes = 160 * 1024;

template <typename T> struct alignas(2 * sizeof(T)) Cx {
  T x, y;
};
template <typename T> __device__ __forceinline__ Cx<T> operator+(Cx<T> a, Cx<T> b) { return {a.x + b.x, a.y + b.y}; }
template <typename T> __device__ __forceinline__ Cx<T> operator-(Cx<T> a, Cx<T> b) { return {a.x - b.x, a.y - b.y}; }
template <typename T> __device__ __forceinline__ Cx<T> operator*(T s, Cx<T> a) { return {s * a.x, s * a.y}; }
// a * w, or a * conj(w) on the way back
template <bool INV, typename T> __device__ __forceinline__ Cx<T> turn(Cx<T> a, Cx<T> w) {
  const T wy = INV ? -w.y : w.y;
  return {a.x * w.x - a.y * wy, a.x * wy + a.y * w.x};
}
// a * -i, or a * i on the way back
template <bool INV, typename T> __device__ __forceinline__ Cx<T> quarter(Cx<T> a) {
  return INV ? Cx<T>{-a.y, a.x} : Cx<T>{a.y, -a.x};
}

// cos and sin of 2 pi q / R, q <= (R - 1) / 2
template <int R> struct Roots;
template <> struct Roots<3> {
  static constexpr double c[2] = {1.0, -0.5}, s[2] = {0.0, 0.86602540378443864676};
};
template <> struct Roots<5> {
  static constexpr double c[3] = {1.0, 0.30901699437494742410, -0.80901699437494742410},
                          s[3] = {0.0, 0.95105651629515357212, 0.58778525229247312917};
};
template <> struct Roots<7> {
  static constexpr double c[4] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624},
                          s[4] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
};

// v = its transform of length R, unnormalised.  Odd R pair the terms r and
// R - r; 6, 10 and 12 split into coprime lengths, which leaves no twiddles.
template <int R, bool INV, typename T> __device__ __forceinline__ void dft(Cx<T> (&v)[R]) {
  if constexpr (R == 2) {
    const Cx<T> a = v[0] - v[1];
    v[0] = v[0] + v[1];
    v[1] = a;
  } else if constexpr (R == 4) {
    const Cx<T> a = v[0] + v[2], b = v[0] - v[2], c = v[1] + v[3], d = quarter<INV>(v[1] - v[3]);
    v[0] = a + c, v[1] = b + d, v[2] = a - c, v[3] = b - d;
  } else if constexpr (R == 8) {
    const T h = T(0.70710678118654752440);
    Cx<T> e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    dft<4, INV>(e);
    dft<4, INV>(o);
    const Cx<T> o1 = quarter<INV>(o[1]), o3 = quarter<INV>(o[3]);
    o[1] = h * (o[1] + o1);
    o[2] = quarter<INV>(o[2]);
    o[3] = h * (o3 - o[3]);
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = e[q] + o[q], v[q + 4] = e[q] - o[q];
  } else if constexpr (R == 16) {
    // x(4 a + b): transforms over a, the 16th roots, transforms over b
    const T h = T(0.70710678118654752440), c = T(0.92387953251128675613), n = T(0.38268343236508977173);
    const Cx<T> w[4][4] = {{}, {{}, {c, -n}, {h, -h}, {n, -c}}, {{}, {h, -h}, {0, -1}, {-h, -h}},
                           {{}, {n, -c}, {-h, -h}, {-c, n}}};
    Cx<T> t[4][4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
#pragma unroll
      for (int a = 0; a < 4; ++a) t[b][a] = v[4 * a + b];
      dft<4, INV>(t[b]);
#pragma unroll
      for (int k = 1; k < 4; ++k)
        if (b == 2 && k == 2) t[b][k] = quarter<INV>(t[b][k]);
        else if (b > 0) t[b][k] = turn<INV>(t[b][k], w[b][k]);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      Cx<T> y[4] = {t[0][k], t[1][k], t[2][k], t[3][k]};
      dft<4, INV>(y);
#pragma unroll
      for (int l = 0; l < 4; ++l) v[k + 4 * l] = y[l];
    }
  } else if constexpr (R % 2 == 0) {
    // term (B a + A b) mod R; result k has k mod A from a's, k mod B from b's
    constexpr int A = R % 4 == 0 ? 4 : 2, B = R / A;
    Cx<T> t[B][A];
#pragma unroll
    for (int b = 0; b < B; ++b) {
#pragma unroll
      for (int a = 0; a < A; ++a) t[b][a] = v[(B * a + A * b) % R];
      dft<A, INV>(t[b]);
    }
#pragma unroll
    for (int a = 0; a < A; ++a) {
      Cx<T> y[B];
#pragma unroll
      for (int b = 0; b < B; ++b) y[b] = t[b][a];
      dft<B, INV>(y);
#pragma unroll
      for (int k = a; k < R; k += A) v[k] = y[k % B];
    }
  } else {
    constexpr int H = (R - 1) / 2;
    Cx<T> a[H], b[H], sum = v[0];
    const Cx<T> v0 = v[0];
#pragma unroll
    for (int r = 1; r <= H; ++r) {
      a[r - 1] = v[r] + v[R - r];
      b[r - 1] = v[r] - v[R - r];
      sum = sum + a[r - 1];
    }
    v[0] = sum;
#pragma unroll
    for (int q = 1; q <= H; ++q) {
      Cx<T> A = v0, B = {T(0), T(0)};
#pragma unroll
      for (int r = 1; r <= H; ++r) {
        const int n = q * r % R, f = n > H ? R - n : n;
        A = A + T(Roots<R>::c[f]) * a[r - 1];
        B = B + T(n > H ? -Roots<R>::s[f] : Roots<R>::s[f]) * b[r - 1];
      }
      B = quarter<INV>(B);
      v[q] = A + B;
      v[R - q] = A - B;
    }
  }
}

struct DampShape {
  int nx, ny, nz;
  int mx;      // nx/2 + 1 columns of the half spectrum
  int pairs;   // (ny + 1) / 2: rows r and r + pairs are one line
  int S;       // line stride: nx + 2 (a pair's two spectra), made odd
  int npx, npy;
  int rx[DP_MAXPASS], ry[DP_MAXPASS];  // the passes' radices
  int ends;  // the outer y passes split and join the rows: their radix is even, so a butterfly holds r and r + pairs
  long fs;
};

// t / d for t, d < 2^16
struct Divide {
  uint32_t m;
  __device__ __forceinline__ explicit Divide(int d) : m(d > 1 ? 0xffffffffu / (uint32_t)d + 1u : 0u) {}
  __device__ __forceinline__ int operator()(int t) const { return m ? (int)__umulhi((uint32_t)t, m) : t; }
};

// A line's two rows: z, w = z(k), z(-k) to their spectra at k,
// a = (z + conj w) / 2 and b = (z - conj w) / 2i, and back: z = a + i b,
// w = conj a + i conj b.  Where k = -k (own) both are real, b stands past the
// line's values, and on the way back only the real parts count, as in any
// complex-to-real transform.
template <typename T> __device__ __forceinline__ void split_rows(Cx<T>& z, Cx<T>& w, bool own) {
  const Cx<T> a = {T(0.5) * (z.x + w.x), T(0.5) * (z.y - w.y)}, b = {T(0.5) * (z.y + w.y), T(0.5) * (w.x - z.x)};
  w = own ? Cx<T>{z.y, T(0)} : b;
  z = own ? Cx<T>{z.x, T(0)} : a;
}
template <typename T> __device__ __forceinline__ void join_rows(Cx<T>& a, Cx<T>& b, bool own) {
  const Cx<T> z = {a.x - b.y, a.y + b.x}, w = {a.x + b.y, b.x - a.y};
  a = own ? Cx<T>{a.x, b.x} : z;
  b = w;  // own: never read again
}

// One pass of radix R over all lines of length n along x, or along the columns
// (y), in blocks of R * m.  WAY: in, back, or the last pass of the way in and
// the first of the way back (m = 1, no twiddles) with the multiply between
// them; ends: see DampShape.  Lanes run over lines first, then butterflies.
// One code serves x and y and all lines: a block runs through some 70 KB of
// instructions once or twice otherwise, and what it waited for was their fetch
// (a second code with scalar indices for whole waves of lines, and x and y
// apart: 128x96x100 68 us, 100x100x100 60).
enum Way { IN, BACK, RATES };
template <int NT, int R, int WAY, typename T>
__device__ __forceinline__ void damp_pass(const DampShape& D, Cx<T>* __restrict__ L, const Cx<T>* __restrict__ tw,
                                          const ushort2* __restrict__ cols, const T* __restrict__ rates, int m, bool y,
                                          bool ends) {
  const int n = y ? D.ny : D.nx, nl = y ? D.mx : D.pairs, nb = n / R;
  const int step = nb / m;  // blocks; w_{R m} = w_n^step
  const int es = y ? D.S : 1, ms = m * es, half = y ? D.pairs : n;
  const Divide by_line(nl), by_m(m);
  for (int t = (int)threadIdx.x; t < nl * nb; t += NT) {
    const int b = by_line(t), line = t - b * nl, g = by_m(b), j = b - g * m, e0 = g * R * m + j;
    const ushort2 col = cols[y ? line : 0];
    const int ca = (y ? col.x : line * D.S) + e0 * es, cb = ca - col.x + col.y - D.pairs * D.S;
    auto at = [&](int r) { return (e0 + r * m < half ? ca : cb) + r * ms; };
    Cx<T> v[R];
#pragma unroll
    for (int r = 0; r < R; ++r) v[r] = L[at(r)];
    const bool own = col.y >= D.nx;
    if constexpr (WAY == RATES) {
      T w[R];
#pragma unroll
      for (int q = 0; q < R; ++q) w[q] = rates[(e0 + q) * nl + line];
      dft<R, false>(v);
#pragma unroll
      for (int q = 0; q < R; ++q) v[q] = w[q] * v[q];
      dft<R, true>(v);
    } else {
      const int js = j * step;
      if constexpr (WAY == IN && R % 2 == 0) {
        if (ends) {
#pragma unroll
          for (int r = 0; r < R / 2; ++r) split_rows(v[r], v[r + R / 2], own);
        }
      }
      if constexpr (WAY == IN) dft<R, false>(v);
#pragma unroll
      for (int q = 1; q < R; ++q) v[q] = turn<WAY == BACK>(v[q], tw[js * q]);
      if constexpr (WAY == BACK) dft<R, true>(v);
      if constexpr (WAY == BACK && R % 2 == 0) {
        if (ends) {
#pragma unroll
          for (int r = 0; r < R / 2; ++r) join_rows(v[r], v[r + R / 2], own);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) L[at(r)] = v[r];
  }
  __syncthreads();
}

template <int NT, int WAY, typename T>
__device__ __forceinline__ void damp_radix(const DampShape& D, int R, Cx<T>* L, const Cx<T>* tw, const ushort2* cols,
                                           const T* rates, int m, bool y, bool ends = false) {
  switch (R) {
    case 2: damp_pass<NT, 2, WAY>(D, L, tw, cols, rates, m, y, ends); break;
    case 3: damp_pass<NT, 3, WAY>(D, L, tw, cols, rates, m, y, ends); break;
    case 4: damp_pass<NT, 4, WAY>(D, L, tw, cols, rates, m, y, ends); break;
    case 5: damp_pass<NT, 5, WAY>(D, L, tw, cols, rates, m, y, ends); break;
    case 6: damp_pass<NT, 6, WAY>(D, L, tw, cols, rates, m, y, ends); break;
    case 7: damp_pass<NT, 7, WAY>(D, L, tw, cols, rates, m, y, ends); break;
    case 8: damp_pass<NT, 8, WAY>(D, L, tw, cols, rates, m, y, ends); break;
    case 10: damp_pass<NT, 10, WAY>(D, L, tw, cols, rates, m, y, ends); break;
    case 12: damp_pass<NT, 12, WAY>(D, L, tw, cols, rates, m, y, ends); break;
    default: damp_pass<NT, 16, WAY>(D, L, tw, cols, rates, m, y, ends); break;
  }
}

// Block b: plane b % nz of velocity b / nz.  roots: the nx roots, then the ny
// roots; LDS: the lines, the roots (once where nx = ny), the columns' places.
template <typename T, int NT>
__global__ __launch_bounds__(NT, 4) void k_damp_plane(const DampShape D, const T* __restrict__ u, T* __restrict__ term,
                                                      const Cx<T>* __restrict__ roots,
                                                      const ushort2* __restrict__ places,
                                                      const T* __restrict__ rates) {
  extern __shared__ double2 dp_lds[];
  Cx<T>* const L = (Cx<T>*)dp_lds;
  const int tid = (int)threadIdx.x, nx = D.nx, ny = D.ny, cells = D.pairs * nx, nr = nx == ny ? nx : nx + ny;
  Cx<T>* const twx = L + D.pairs * D.S;
  Cx<T>* const twy = nx == ny ? twx : twx + nx;
  ushort2* const cols = (ushort2*)(twy + ny);
  const int f = (int)blockIdx.x / D.nz, k = (int)blockIdx.x - f * D.nz;
  const long base = (long)f * D.fs + (long)k * nx * ny;
  const Divide by_nx(nx), by_pair(D.pairs);

  // rows r and r + pairs as one complex line; the row past an odd ny is zero
  constexpr int U = 6;
  for (int t0 = tid; t0 < cells; t0 += U * NT) {
    Cx<T> z[U];
#pragma unroll
    for (int c = 0; c < U; ++c) {
      const int t = t0 + c * NT, r = by_nx(t);
      z[c] = {T(0), T(0)};
      if (t < cells) {
        z[c].x = u[base + t];
        if (r + D.pairs < ny) z[c].y = u[base + cells + t];
      }
    }
#pragma unroll
    for (int c = 0; c < U; ++c) {
      const int t = t0 + c * NT, r = by_nx(t), x = t - r * nx;
      if (t < cells) L[r * D.S + x] = z[c];
    }
  }
  for (int t = tid; t < nr; t += NT) twx[t] = roots[t];
  for (int t = tid; t < D.mx; t += NT) cols[t] = places[t];
  __syncthreads();

  // f on the two values of every column in every line
  auto each_column = [&](auto f) {
    for (int t = tid; t < D.pairs * D.mx; t += NT) {
      const int q = by_pair(t), line = (t - q * D.pairs) * D.S;
      const ushort2 col = cols[q];
      Cx<T> a = L[line + col.x], b = L[line + col.y];
      f(a, b, col.y >= nx);
      L[line + col.x] = a;
      L[line + col.y] = b;
    }
    __syncthreads();
  };
  // the way in: the x passes, the rows apart, the y passes but one
  for (int p = 0, m = nx; p < D.npx + D.npy - 1; ++p) {
    const bool y = p >= D.npx;
    if (p == D.npx) {
      m = ny;
      if (!D.ends) each_column([](Cx<T>& z, Cx<T>& w, bool own) { split_rows(z, w, own); });
    }
    const int R = y ? D.ry[p - D.npx] : D.rx[p];
    m /= R;
    damp_radix<NT, IN>(D, R, L, y ? twy : twx, cols, rates, m, y, p == D.npx && D.ends);
  }
  if (D.npy == 1) each_column([](Cx<T>& z, Cx<T>& w, bool own) { split_rows(z, w, own); });
  damp_radix<NT, RATES>(D, D.ry[D.npy - 1], L, twy, cols, rates, 1, true);
  if (D.npy == 1) each_column([](Cx<T>& a, Cx<T>& b, bool own) { join_rows(a, b, own); });
  // and back
  for (int p = D.npx + D.npy - 2, m = D.npy > 1 ? D.ry[D.npy - 1] : 1; p >= 0; --p) {
    const bool y = p >= D.npx;
    const int R = y ? D.ry[p - D.npx] : D.rx[p];
    damp_radix<NT, BACK>(D, R, L, y ? twy : twx, cols, rates, m, y, p == D.npx && D.ends);
    m *= R;
    if (p == D.npx) {
      m = 1;
      if (!D.ends) each_column([](Cx<T>& a, Cx<T>& b, bool own) { join_rows(a, b, own); });
    }
  }
  for (int t = tid; t < cells; t += NT) {
    const int r = by_nx(t), x = t - r * nx;
    const Cx<T> z = L[r * D.S + x];
    term[base + t] = z.x;
    if (r + D.pairs < ny) term[base + cells + t] = z.y;
  }
}

struct DampPlan {
  bool plane = false;     // k_damp_plane
  DampShape shape{};
  size_t lds = 0;
  void* roots = nullptr;   // nx + ny complex roots
  void* places = nullptr;  // mx columns' places in a line
  hipfftHandle fwd = 0, inv = 0;
  bool f32 = false;
  int nx = 0, ny = 0, nz = 0;
  int nf = 1;             // fields per library transform: 3 or 1
  long fs = 0;
  void* spec = nullptr;   // half spectra of nf fields, (nx/2+1)*ny*nz complex each
  void* rates = nullptr;  // (nx/2+1)*ny, element type
  void* term = nullptr;   // 3 slabs of fs: the terms of vx, vy, vz
};

// w(kx, ky, k) *= rates(kx, ky); grid.y = plane
template <typename C, typename T>
__global__ __launch_bounds__(256) void k_damp_mul(C* __restrict__ w, const T* __restrict__ rates, int m) {
  const int q = blockIdx.x * 256 + threadIdx.x;
  if (q >= m) return;
  const long i = (long)blockIdx.y * m + q;
  const T r = rates[q];
  C v = w[i];
  v.x *= r;
  v.y *= r;
  w[i] = v;
}

static void library_free(DampPlan* d) {
  if (d->fwd) (void)hipfftDestroy(d->fwd);
  if (d->inv) (void)hipfftDestroy(d->inv);
  if (d->spec) (void)hipFree(d->spec);
  d->fwd = d->inv = 0;
  d->spec = nullptr;
}

void damp_destroy(DampPlan* d) {
  if (!d) return;
  library_free(d);
  if (d->roots) (void)hipFree(d->roots);
  if (d->places) (void)hipFree(d->places);
  if (d->rates) (void)hipFree(d->rates);
  if (d->term) (void)hipFree(d->term);
  delete d;
}

// The radices of a transform of length n: the fewest passes, then the smallest
// largest radix; 0 passes if n has other factors.
static int radices(int n, int (&r)[DP_MAXPASS], int cap = 16, int room = DP_MAXPASS) {
  if (n == 1 || room == 0) return 0;
  int best = 0;
  for (int q : {2, 3, 4, 5, 6, 7, 8, 10, 12, 16}) {
    if (q > cap || n % q != 0) continue;
    int rest[DP_MAXPASS];
    const int np = n == q ? 1 : 1 + radices(n / q, rest, q, room - 1);
    if ((n != q && np == 1) || (best && np >= best)) continue;
    best = np;
    r[0] = q;
    std::copy(rest, rest + np - 1, r + 1);
  }
  return best;
}

// Where frequency k of a line stands after the passes: its first digit counts
// blocks of n / r[0], and so on.
static int place_of(int k, int n, const int* r, int np) {
  int at = 0;
  for (int p = 0; p < np; ++p) {
    n /= r[p];
    at += k % r[p] * n;
    k /= r[p];
  }
  return at;
}

// The plane kernel's shape, if it can take the plane: LDS holds its half
// spectrum and its sides are products of 2, 3, 5 and 7.
static bool plane_shape(DampPlan* d) {
  DampShape& D = d->shape;
  D.nx = d->nx, D.ny = d->ny, D.nz = d->nz, D.fs = d->fs;
  D.mx = D.nx / 2 + 1;
  D.pairs = (D.ny + 1) / 2;
  D.S = (D.nx + 2) | 1;
  D.npx = radices(D.nx, D.rx);
  D.npy = radices(D.ny, D.ry);
  if (D.ny % 2 == 0 && D.npy > 1) std::swap(D.ry[0], *std::find_if(D.ry, D.ry + D.npy, [](int r) { return r % 2 == 0; }));
  D.ends = D.npy > 1 && D.ry[0] % 2 == 0;
  const size_t esz = d->f32 ? sizeof(float) : sizeof(double);
  d->lds = ((size_t)D.pairs * D.S + D.nx + (D.nx == D.ny ? 0 : D.ny)) * 2 * esz + sizeof(ushort2) * D.mx;
  return D.npx > 0 && D.npy > 0 && d->lds <= kLdsBytes;
}

// Threads of a block: 256 where five or more share a CU, which then fill its
// SIMDs together (60x60x200 FP64 29 us, 34 with 512), else 512 (64x64x64, four
// a CU, 18 us, 19 with 256; 128x96x100, one a CU, 56, 69 with 256; 1024 no
// faster there).
static int plane_threads(const DampPlan* d) { return 5 * d->lds <= kLdsBytes ? 256 : 512; }

template <typename T> using PlaneKernel = void (*)(const DampShape, const T*, T*, const Cx<T>*, const ushort2*, const T*);
template <typename T> static PlaneKernel<T> plane_kernel(const DampPlan* d) {
  return plane_threads(d) == 256 ? k_damp_plane<T, 256> : k_damp_plane<T, 512>;
}

template <typename T>
static bool plane_tables(DampPlan* d, const double* rates) {
  const DampShape& D = d->shape;
  std::vector<Cx<T>> w(D.nx + D.ny);
  for (int q = 0; q < D.nx + D.ny; ++q) {
    const int n = q < D.nx ? D.nx : D.ny, k = q < D.nx ? q : q - D.nx;
    const long double a = 2.0L * 3.14159265358979323846264338327950288L * k / n;
    w[q] = {(T)cosl(a), (T)-sinl(a)};
  }
  // the columns in the order in which they lie
  std::vector<int> kx(D.mx);
  for (int k = 0; k < D.mx; ++k) kx[k] = k;
  auto at = [&](int k) { return place_of(k, D.nx, D.rx, D.npx); };
  std::sort(kx.begin(), kx.end(), [&](int a, int b) { return at(a) < at(b); });
  std::vector<ushort2> cols(D.mx);
  for (int c = 0; c < D.mx; ++c) {
    const int k = kx[c], b = k == 0 ? D.nx : (2 * k == D.nx ? D.nx + 1 : at(D.nx - k));
    cols[c] = {(unsigned short)at(k), (unsigned short)b};
  }
  std::vector<T> rt((size_t)D.mx * D.ny);
  for (int ky = 0; ky < D.ny; ++ky) {
    const size_t row = (size_t)place_of(ky, D.ny, D.ry, D.npy) * D.mx;
    for (int c = 0; c < D.mx; ++c) rt[row + c] = (T)rates[(size_t)ky * D.mx + kx[c]];
  }
  auto put = [](void** p, const void* h, size_t n) {
    return hipMalloc(p, n) == hipSuccess && hipMemcpy(*p, h, n, hipMemcpyHostToDevice) == hipSuccess;
  };
  return put(&d->roots, w.data(), sizeof(Cx<T>) * w.size()) &&
         put(&d->places, cols.data(), sizeof(ushort2) * cols.size()) &&
         put(&d->rates, rt.data(), sizeof(T) * rt.size()) &&
         hipFuncSetAttribute((const void*)plane_kernel<T>(d), hipFuncAttributeMaxDynamicSharedMemorySize,
                             (int)kLdsBytes) == hipSuccess;
}

// The library's plans and the half spectra for nf fields at a time.
static bool library_plans(DampPlan* d, int nf, hipStream_t st) {
  // n, embeddings in C order (slowest first): a plane is ny rows of nx reals
  // or of nx/2+1 complex values; batch = the nz planes of each field
  const int nx = d->nx, ny = d->ny, mx = nx / 2 + 1, m = mx * ny;
  int n[2] = {ny, nx}, real_embed[2] = {ny, nx}, cplx_embed[2] = {ny, mx};
  const size_t esz = d->f32 ? sizeof(float) : sizeof(double);
  d->nf = nf;
  bool ok = hipMalloc(&d->spec, 2 * esz * m * d->nz * nf) == hipSuccess;
  ok = ok && hipfftPlanMany(&d->fwd, 2, n, real_embed, 1, nx * ny, cplx_embed, 1, m, d->f32 ? HIPFFT_R2C : HIPFFT_D2Z,
                            d->nz * nf) == HIPFFT_SUCCESS;
  ok = ok && hipfftPlanMany(&d->inv, 2, n, cplx_embed, 1, m, real_embed, 1, nx * ny, d->f32 ? HIPFFT_C2R : HIPFFT_Z2D,
                            d->nz * nf) == HIPFFT_SUCCESS;
  ok = ok && hipfftSetStream(d->fwd, st) == HIPFFT_SUCCESS && hipfftSetStream(d->inv, st) == HIPFFT_SUCCESS;
  if (!ok) {
    library_free(d);
    (void)hipGetLastError();
  }
  return ok;
}

// rates: (nx/2+1, ny) Fortran order = C (ny, nx/2+1), FP64 from the host.
// Returns nullptr on failure (and frees what it made).
DampPlan* damp_create(int nx, int ny, int nz, long fs, bool f32, const double* rates, hipStream_t st) {
  DampPlan* d = new DampPlan();
  d->f32 = f32;
  d->nx = nx;
  d->ny = ny;
  d->nz = nz;
  d->fs = fs;
  const int mx = nx / 2 + 1;
  const long m = (long)mx * ny;
  const size_t esz = f32 ? sizeof(float) : sizeof(double);
  if (plane_shape(d)) {
    d->plane = true;
    if (hipMalloc(&d->term, esz * 3 * fs) == hipSuccess &&
        (f32 ? plane_tables<float>(d, rates) : plane_tables<double>(d, rates)))
      return d;
    damp_destroy(d);
    return nullptr;
  }
  bool ok = hipMalloc(&d->rates, esz * m) == hipSuccess && hipMalloc(&d->term, esz * 3 * fs) == hipSuccess;
  if (ok) {
    if (f32) {
      std::vector<float> h(rates, rates + m);
      ok = hipMemcpy(d->rates, h.data(), esz * m, hipMemcpyHostToDevice) == hipSuccess;
    } else {
      ok = hipMemcpy(d->rates, rates, esz * m, hipMemcpyHostToDevice) == hipSuccess;
    }
  }
  // Three fields in one transform where the slabs are unpadded, within 65535 rows
  // of a launch and 2^31 values of a transform; one by one beyond, and where
  // there is no memory for three fields' spectra.
  const bool small = 3L * nz <= 65535 && 3L * fs < (1L << 31);
  ok = ok && ((fs == (long)nx * ny * nz && small && library_plans(d, 3, st)) || library_plans(d, 1, st));
  if (!ok) {
    damp_destroy(d);
    return nullptr;
  }
  return d;
}

const void* damp_term_slab(const DampPlan* d, int f) {
  return (const char*)d->term + (size_t)f * d->fs * (d->f32 ? sizeof(float) : sizeof(double));
}

// The terms of vx, vy, vz of the state buffer `u` (nv field slabs of fs).
// u stays unchanged (the r2c transforms are out of place).
template <typename T>
static hipError_t plane_terms(const DampPlan* d, const void* u, hipStream_t st) {
  hipLaunchKernelGGL(plane_kernel<T>(d), dim3((unsigned)(3 * d->nz)), dim3((unsigned)plane_threads(d)), d->lds, st,
                     d->shape, (const T*)u + (size_t)VX * d->fs, (T*)d->term, (const Cx<T>*)d->roots,
                     (const ushort2*)d->places, (const T*)d->rates);
  return hipGetLastError();
}
hipError_t damp_terms(DampPlan* d, const void* u, hipStream_t st) {
  if (d->plane) return d->f32 ? plane_terms<float>(d, u, st) : plane_terms<double>(d, u, st);
  const int mx = d->nx / 2 + 1;
  const int m = mx * d->ny;
  const size_t esz = d->f32 ? sizeof(float) : sizeof(double);
  dim3 grid((unsigned)((m + 255) / 256), (unsigned)(d->nz * d->nf));
  for (int f = 0; f < 3; f += d->nf) {
    const char* in = (const char*)u + (size_t)(VX + f) * d->fs * esz;
    char* out = (char*)d->term + (size_t)f * d->fs * esz;
    hipfftResult r;
    if (d->f32) {
      r = hipfftExecR2C(d->fwd, (hipfftReal*)in, (hipfftComplex*)d->spec);
      if (r != HIPFFT_SUCCESS) return hipErrorLaunchFailure;
      hipLaunchKernelGGL((k_damp_mul<float2, float>), grid, dim3(256), 0, st, (float2*)d->spec,
                         (const float*)d->rates, m);
      r = hipfftExecC2R(d->inv, (hipfftComplex*)d->spec, (hipfftReal*)out);
    } else {
      r = hipfftExecD2Z(d->fwd, (hipfftDoubleReal*)in, (hipfftDoubleComplex*)d->spec);
      if (r != HIPFFT_SUCCESS) return hipErrorLaunchFailure;
      hipLaunchKernelGGL((k_damp_mul<double2, double>), grid, dim3(256), 0, st, (double2*)d->spec,
                         (const double*)d->rates, m);
      r = hipfftExecZ2D(d->inv, (hipfftDoubleComplex*)d->spec, (hipfftDoubleReal*)out);
    }
    if (r != HIPFFT_SUCCESS) return hipErrorLaunchFailure;
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace sparc
