// openbc.hip — the open boundary of the field on the device (gtdgl/src/openbc.jl): δJ, the
// convolution with the lattice Green function by zero-padded FFTs, h_δ on the faces, and the
// clock that decides on which steps they run.
//
// The convolution is Hockney's: a padded size M >= 2n - 1 per axis (a product of 2, 3 and 5) and
// the Green function placed cyclically, so the first n outputs are the linear convolution, the
// same as the reference's 2n padding computes.  G is even along every axis, so its transform is
// real.  The padding is never stored: the x pass reads only the box and zero-extends, the z pass
// (forward, times Ĝ, inverse) keeps only the box's planes, the inverse passes write only the box.
#include "kernels.h"

namespace tdgl {

// ---------------------------------------------------------------- the clock (open_update!, :196-215)
__global__ void k_open_clock(int *ofl, int every) {
  if (threadIdx.x != 0) return;
  const int first = ofl[OF_COUNT] < 0;
  const int c = ofl[OF_COUNT] + 1;
  const int re = (c >= every || first) ? 1 : 0;
  ofl[OF_RECOMP] = re;
  ofl[OF_FIRST] = first;
  ofl[OF_COUNT] = re ? 0 : c;
}
hipError_t launch_open_clock(int *ofl, int every, hipStream_t s) {
  if (g_rec) return hipErrorNotSupported;
  TDGL_LAUNCH(k_open_clock, dim3(1), dim3(64), 0, s, ofl, every);
  return hipGetLastError();
}

// ---------------------------------------------------------------- δJ (_delta_current!, :143-160)
// δJ on the links of lattice c (blockIdx.y), compact (n1, n2, n3), zero on the face-normal links
__global__ void __launch_bounds__(256) k_open_dj(Geo g, OpenDJ a) {
  if (!a.ofl[OF_RECOMP]) return;
  const int c = blockIdx.y;
  const int n1 = a.n[c][0], n2 = a.n[c][1], n3 = a.n[c][2];
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n1 * n2 * n3) return;
  const int i = 1 + t % n1, j = 1 + (t / n1) % n2, k = 1 + t / (n1 * n2);
  const int Nx = g.Nx, Ny = g.Ny, Nz = g.Nz;
  const double *hx = a.h[0], *hy = a.h[1], *hz = a.h[2];
  const int sy = g.px, sz = g.px * g.py;
  double v = 0.0;
  if (c == 0) {
    if (k >= 2 && k <= Nz && j >= 2 && j <= Ny && i >= 2 && i <= Nx - 1) {
      const int q = g.at(i, j, k);
      v = a.k2 * ((hz[q] - hz[q - sy]) / a.dy - (hy[q] - hy[q - sz]) / a.dz) - a.HJp[0] * a.Jbar[(j - 1) + (Ny + 1) * (k - 1)];
    }
  } else if (c == 1) {
    if (k >= 2 && k <= Nz && j >= 2 && j <= Ny - 1 && i >= 2 && i <= Nx) {
      const int q = g.at(i, j, k);
      v = a.k2 * ((hx[q] - hx[q - sz]) / a.dz - (hz[q] - hz[q - 1]) / a.dx);
    }
  } else {
    if (k >= 2 && k <= Nz - 1 && j >= 2 && j <= Ny && i >= 2 && i <= Nx) {
      const int q = g.at(i, j, k);
      v = a.k2 * ((hy[q] - hy[q - 1]) / a.dx - (hx[q] - hx[q - sy]) / a.dy);
    }
  }
  a.dj[c][t] = v;
}
hipError_t launch_open_dj(const Geo &g, const OpenDJ &a, hipStream_t s) {
  if (g_rec) return hipErrorNotSupported;
  int m = 0;
  for (int c = 0; c < 3; ++c) m = std::max(m, a.n[c][0] * a.n[c][1] * a.n[c][2]);
  TDGL_LAUNCH(k_open_dj, dim3(cdiv(m, 256), 3), dim3(256), 0, s, g, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------- line FFTs
__device__ __forceinline__ cplx imul_s(cplx v, int s) { return s > 0 ? mk(-v.y, v.x) : mk(v.y, -v.x); }  // (s i) v

// the R-point DFT with exponent sign s, in place
template <int R>
__device__ __forceinline__ void dft_small(cplx (&v)[R], int s) {
  if constexpr (R == 2) {
    const cplx a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 4) {
    const cplx t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]), t2 = cadd(v[1], v[3]), t3 = imul_s(csub(v[1], v[3]), s);
    v[0] = cadd(t0, t2);
    v[1] = cadd(t1, t3);
    v[2] = csub(t0, t2);
    v[3] = csub(t1, t3);
  } else if constexpr (R == 3) {
    const double h3 = 0.86602540378443864676;  // √3/2
    const cplx t1 = cadd(v[1], v[2]), t2 = imul_s(rmul(h3, csub(v[1], v[2])), s);
    const cplx m = csub(v[0], rmul(0.5, t1));
    v[0] = cadd(v[0], t1);
    v[1] = cadd(m, t2);
    v[2] = csub(m, t2);
  } else {  // 5
    const double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;   // cos 2π/5, cos 4π/5
    const double s1 = 0.95105651629515357212, s2 = 0.58778525229247312917;    // sin 2π/5, sin 4π/5
    const cplx a1 = cadd(v[1], v[4]), b1 = csub(v[1], v[4]), a2 = cadd(v[2], v[3]), b2 = csub(v[2], v[3]);
    const cplx p1 = cadd(v[0], cadd(rmul(c1, a1), rmul(c2, a2)));
    const cplx p2 = cadd(v[0], cadd(rmul(c2, a1), rmul(c1, a2)));
    const cplx q1 = imul_s(cadd(rmul(s1, b1), rmul(s2, b2)), s);
    const cplx q2 = imul_s(csub(rmul(s2, b1), rmul(s1, b2)), s);
    v[0] = cadd(v[0], cadd(a1, a2));
    v[1] = cadd(p1, q1);
    v[4] = csub(p1, q1);
    v[2] = cadd(p2, q2);
    v[3] = csub(p2, q2);
  }
}

// The lines of a block lie interleaved in LDS, element e of line l at A[e LPB + l] with LPB a power of two:
// a thread keeps its line, consecutive lanes take consecutive lines of the same butterfly (no division by a
// length, no bank conflict, one twiddle for LPB lanes).
constexpr int FFT_T = 256;      // threads
constexpr int FFT_LDS = 2560;   // complex values of a block (40 KB: four blocks a CU)

// One Stockham autosort pass of radix R, in place: every butterfly of a thread is read into registers before any
// is written.  Butterfly j reads src[j + r M/R], twiddles r by ω^(r (j mod Ns) M/(Ns R)), writes
// dst[(j/Ns) Ns R + (j mod Ns) + r Ns].
template <int R>
__device__ __forceinline__ void fft_pass(cplx *A, int lg, int M, int Ns, const cplx *tw, int dir) {
  constexpr int IM = (FFT_LDS / R + FFT_T - 1) / FFT_T;
  const int MR = M / R, step = MR / Ns, items = MR << lg, l = threadIdx.x & ((1 << lg) - 1);
  const float inv = 1.0f / (float)Ns;
  cplx v[IM][R];
  int base[IM];
#pragma unroll
  for (int u = 0; u < IM; ++u) {
    const int item = (int)threadIdx.x + u * FFT_T;
    base[u] = -1;
    if (item < items) {
      const int j = item >> lg, q = (int)(((float)j + 0.5f) * inv), k = j - q * Ns;
#pragma unroll
      for (int r = 0; r < R; ++r) v[u][r] = A[((j + r * MR) << lg) + l];
      if (Ns > 1)
#pragma unroll
        for (int r = 1; r < R; ++r) {
          cplx w = tw[r * k * step];
          if (dir > 0) w.y = -w.y;
          v[u][r] = cmul(v[u][r], w);
        }
      dft_small<R>(v[u], dir);
      base[u] = q * Ns * R + k;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < IM; ++u)
    if (base[u] >= 0)
#pragma unroll
      for (int r = 0; r < R; ++r) A[((base[u] + r * Ns) << lg) + l] = v[u][r];
  __syncthreads();
}
__device__ void fft_lines(cplx *A, int lg, const FftAxis &ax, int dir) {
  int Ns = 1;
  for (int s = 0; s < ax.nrad; ++s) {
    const int R = ax.rad[s];
    if (R == 4)
      fft_pass<4>(A, lg, ax.M, Ns, ax.tw, dir);
    else if (R == 2)
      fft_pass<2>(A, lg, ax.M, Ns, ax.tw, dir);
    else if (R == 3)
      fft_pass<3>(A, lg, ax.M, Ns, ax.tw, dir);
    else
      fft_pass<5>(A, lg, ax.M, Ns, ax.tw, dir);
    Ns *= R;
  }
}

// The passes of up to three lattices in one launch (blockIdx.y).  Bound by the reads and writes of the lines,
// once a pass (1.35 GB a recomputation at 256 x 128 x 32, 0.28 ms at the rate of a copy), and by the passes'
// LDS traffic: 2.0 ms a recomputation with the radices known when compiled, in place, four blocks a CU; 9.7 ms
// with two buffers of 64 KB a block, the radix a runtime loop bound and the index divided by the line's length.
struct FftSet {
  FftPass p[3];
};
__global__ void __launch_bounds__(FFT_T, 4) k_fft(FftSet f, const int *gate) {
  if (gate && !*gate) return;
  const FftPass &p = f.p[blockIdx.y];
  extern __shared__ __align__(16) unsigned char fft_smem[];
  cplx *A = (cplx *)fft_smem;
  __shared__ long long lin[64], lout[64], lgh[64];  // where each line of the block starts
  const int M = p.ax.M, lg = p.lpb, LPB = 1 << lg;
  const int nlines = p.nl0 * p.nl1, L0 = blockIdx.x << lg, tid = threadIdx.x;
  if (L0 >= nlines) return;
  if (tid < LPB) {
    const int L = min(L0 + tid, nlines - 1), a = L % p.nl0, b = L / p.nl0;
    lin[tid] = (long long)a * p.in_l0 + (long long)b * p.in_l1;
    lout[tid] = (long long)a * p.out_l0 + (long long)b * p.out_l1;
    lgh[tid] = (long long)a * p.g_l0 + (long long)b * p.g_l1;
  }
  __syncthreads();
  const int tot = M << lg, nl = min(LPB, nlines - L0);
  const float invM = 1.0f / (float)M, invO = 1.0f / (float)p.nout;
  // load, zero beyond nin (clamped addresses, selected at the store), five in flight a thread
  for (int t0 = tid; t0 < tot; t0 += 5 * FFT_T) {
    cplx v[5];
    int to[5];
#pragma unroll
    for (int u = 0; u < 5; ++u) {
      const int t = min(t0 + u * FFT_T, tot - 1);
      const int l = p.lines_fast ? (t & (LPB - 1)) : (int)(((float)t + 0.5f) * invM), e = p.lines_fast ? (t >> lg) : t - l * M;
      const bool ok = e < p.nin;
      const long long idx = lin[l] + (long long)(ok ? e : 0) * p.in_s;
      v[u] = p.in_real ? mk(((const double *)p.in)[idx], 0.0) : ((const cplx *)p.in)[idx];
      to[u] = (e << lg) + l;
      if (!ok) v[u] = mk(0.0, 0.0);
    }
#pragma unroll
    for (int u = 0; u < 5; ++u)
      if (t0 + u * FFT_T < tot) A[to[u]] = v[u];
  }
  __syncthreads();
  fft_lines(A, lg, p.ax, p.dir);
  if (p.ghat) {
    // times Ĝ (real), then back (the z pass of a convolution)
    const int l = tid & (LPB - 1), le = FFT_T >> lg;
    const double *gl = p.ghat + lgh[l];
    for (int e0 = tid >> lg; e0 < M; e0 += 5 * le) {
      double g[5];
#pragma unroll
      for (int u = 0; u < 5; ++u) g[u] = gl[(long long)min(e0 + u * le, M - 1) * p.g_s];
#pragma unroll
      for (int u = 0; u < 5; ++u) {
        const int e = e0 + u * le;
        if (e < M) A[(e << lg) + l] = rmul(g[u], A[(e << lg) + l]);
      }
    }
    __syncthreads();
    fft_lines(A, lg, p.ax, -p.dir);
  }
  // store the first nout of every line
  for (int t = tid; t < (p.nout << lg); t += FFT_T) {
    const int l = p.lines_fast ? (t & (LPB - 1)) : (int)(((float)t + 0.5f) * invO), e = p.lines_fast ? (t >> lg) : t - l * p.nout;
    if (l >= nl) continue;
    const cplx v = A[(e << lg) + l];
    const long long idx = lout[l] + (long long)e * p.out_s;
    if (p.out_real)
      ((double *)p.out)[idx] = v.x * p.scale;
    else
      ((cplx *)p.out)[idx] = rmul(p.scale, v);
  }
}

// lines of a block, log2: the most (at most 64) whose elements fit FFT_LDS
static int fft_lg(int M) {
  int lg = 0;
  while (lg < 6 && (M << (lg + 1)) <= FFT_LDS) ++lg;
  return lg;
}

hipError_t launch_fft(const FftPass *p, int n, const int *gate, hipStream_t s) {
  if (g_rec) return hipErrorNotSupported;
  if (n < 1 || n > 3) return hipErrorInvalidValue;
  FftSet f{};
  int nb = 1;
  for (int q = 0; q < n; ++q) {
    f.p[q] = p[q];
    if (p[q].ax.M < 1 || p[q].ax.M > 2048 || p[q].nin < 1 || p[q].nin > p[q].ax.M || p[q].nout < 1 || p[q].nout > p[q].ax.M)
      return hipErrorInvalidValue;
    f.p[q].lpb = fft_lg(p[q].ax.M);
    nb = std::max(nb, cdiv(p[q].nl0 * p[q].nl1, 1 << f.p[q].lpb));
  }
  TDGL_LAUNCH(k_fft, dim3(nb, n), dim3(FFT_T), FFT_LDS * sizeof(cplx), s, f, gate);
  return hipGetLastError();
}

// ---------------------------------------------------------------- the padded Green function
// fac·G(d) at the padded index a (offset a for a <= M/2, a - M above: even, so Ĝ is real)
__device__ __forceinline__ double lgf_at(const OpenGreen &a, int i, int j, int k) {
  i = abs(i);
  j = abs(j);
  k = abs(k);
  const int R = a.R;
  if (i <= R && j <= R && k <= R) return a.lgf[i + (R + 1) * (j + (R + 1) * k)];
  const double r2 = (double)i * i + (double)j * j + (double)k * k, r = sqrt(r2);
  const double i4 = (double)i * i * i * i, j4 = (double)j * j * j * j, k4 = (double)k * k * k * k;
  return (1 + (5 * (i4 + j4 + k4) / (r2 * r2) - 3) / (8 * r2)) / (4 * 3.14159265358979323846 * r);
}
__global__ void __launch_bounds__(256) k_open_green(OpenGreen a) {
  const long long n = (long long)a.M[0] * a.M[1] * a.M[2];
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int x = (int)(t % a.M[0]), y = (int)((t / a.M[0]) % a.M[1]), z = (int)(t / ((long long)a.M[0] * a.M[1]));
  const int ox = x <= a.M[0] / 2 ? x : x - a.M[0], oy = y <= a.M[1] / 2 ? y : y - a.M[1], oz = z <= a.M[2] / 2 ? z : z - a.M[2];
  a.out[t] = a.fac * lgf_at(a, ox, oy, oz);
}
hipError_t launch_open_green(const OpenGreen &a, hipStream_t s) {
  const long long n = (long long)a.M[0] * a.M[1] * a.M[2];
  TDGL_LAUNCH(k_open_green, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
  return hipGetLastError();
}

// ---------------------------------------------------------------- h_δ on the faces (_face_field!, :175-188)
__global__ void __launch_bounds__(256) k_open_face(Geo g, OpenFace a) {
  if (!a.ofl[OF_RECOMP]) return;
  const int i = 1 + blockIdx.x * blockDim.x + threadIdx.x;
  const int j = 1 + blockIdx.y;
  const int k = 1 + blockIdx.z;
  const int Nx = g.Nx, Ny = g.Ny, Nz = g.Nz;
  if (i > Nx + 1) return;
  // θ_δ on lattice c at link (i, j, k), compact (n1, n2, n3)
  auto th = [&](int c, int ii, int jj, int kk) {
    return a.theta[c][(ii - 1) + a.n[c][0] * ((jj - 1) + a.n[c][1] * (kk - 1))];
  };
  const int q = g.at(i, j, k);
  // hz (Nx, Ny, Nz+1): faces j ∈ {1, Ny} and i ∈ {1, Nx}
  if (i <= Nx && j <= Ny && (j == 1 || j == Ny || i == 1 || i == Nx))
    a.hnew[2][q] = ((th(1, i + 1, j, k) - th(1, i, j, k)) - th(0, i, j + 1, k) + th(0, i, j, k)) / (a.dx * a.dy);
  // hx (Nx+1, Ny, Nz): faces j ∈ {1, Ny} and k ∈ {1, Nz}
  if (j <= Ny && k <= Nz && (j == 1 || j == Ny || k == 1 || k == Nz))
    a.hnew[0][q] = ((th(2, i, j + 1, k) - th(2, i, j, k)) - th(1, i, j, k + 1) + th(1, i, j, k)) / (a.dy * a.dz);
  // hy (Nx, Ny+1, Nz): faces k ∈ {1, Nz} and i ∈ {1, Nx}
  if (i <= Nx && k <= Nz && (k == 1 || k == Nz || i == 1 || i == Nx))
    a.hnew[1][q] = ((th(0, i, j, k + 1) - th(0, i, j, k)) - th(2, i + 1, j, k) + th(2, i, j, k)) / (a.dz * a.dx);
}
hipError_t launch_open_face(const Geo &g, const OpenFace &a, hipStream_t s) {
  if (g_rec) return hipErrorNotSupported;
  TDGL_LAUNCH(k_open_face, dim3(cdiv(g.Nx + 1, 64), g.Ny + 1, g.Nz + 1), dim3(64), 0, s, g, a);
  return hipGetLastError();
}

}  // namespace tdgl
