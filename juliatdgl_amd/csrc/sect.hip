// sect.hip — the insulating PCG, and the separable solve of large planes, sector by sector.
//
// The conductivity of the field solve is constant along x and mirror-symmetric in y and z (the bar and
// its padding, implicit.jl:126-140), so A = D + aK keeps three symmetries that the general PCG does not
// use: the x transform of the separable bases (V on nodes, U on edges) turns every x difference into a
// product with the mode's singular value, and the mirrors split the (y, z) plane of a mode into four
// parity sectors.  The solve is then 4 (Nx - 1) independent problems on quarter planes, each small
// enough for one workgroup's LDS and registers: k_sect_fwd takes the residual to the sectors, k_sect_cg
// runs the whole flexible CG of a sector in one launch, k_sect_inv takes the solution back.  The general
// iteration's six launches and 860 MB of HBM traffic (290 us on 256x128x32 cells, 20 to 24 a step; 50 us,
// launch-bound, on 96x48x24) become one launch a solve, whose iterations leave the CU only for the bases:
// a time step took 7.86 -> 1.42 ms on 256x128x32 cells, 458 -> 136 us on 96x48x24, 610 -> 160 us on 128x64x16 with
// KWT, 327 -> 78 us on 53x27x9 (with the open boundary's and the launches' own savings).
//
// A sector holds values on the half domain (the rest follows by parity): component c of mode mx at
// (j, k), j fastest, X (c = 0) then Y then Z.  With (py, pz) the parities of the sector's y and z wave
// numbers, a component is node-like (cosine) along an axis other than its own and edge-like (sine, the
// opposite parity) along its own.  A half axis of n nodes holds ceil(n/2) (even) or floor(n/2) (odd)
// nodes and ceil(n/2) - 1 or floor(n/2) edges; sums over a whole axis weigh each point by 2, a centre
// point by 1.  A difference across the centre takes the mirrored value (the ghosts of k_sect_cg).
#include "kernels.h"

namespace tdgl {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

__device__ __forceinline__ v4d ld4d(const double *p) {
  const v2d lo = *(const v2d *)p, hi = *(const v2d *)(p + 2);
  return v4d{lo.x, lo.y, hi.x, hi.y};
}
__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// ---------------------------------------------------------------------------- the x transforms
// Bound: 2 (Lx / 2) flop in FP64 per element on the matrix cores (the fold along x halves the dense
// product) against 16 B.  A block takes SX_J positions along y at one z and their mirror images, folds
// them into the four sectors and the two x parities in LDS and multiplies by the half-size x bases
// (padded to whole 16 x 16 tiles, read through L2); wave w owns the m tiles w, w + waves, ...  What it waits
// for is memory: the loads of the images (sixteen in flight a thread), of the bases (three groups ahead) and,
// on the way back, of θ and x (an image set together: one after the other behind the stores they took 31 us
// more).  Forward 72 us, back 109 us on 272 x 144 x 48 nodes (104 us each at first; 88 and 217 MB), 12 and 16 us on
// 100 x 52 x 28.  Four positions a block (half the LDS) took 92 to 102 and 116 to 131 us, 5 to 8 waves no less.
constexpr int SX_J = 8, SX_COLS = 4 * SX_J, SX_T = SX_COLS / 16;
constexpr int SX_WAVES = 10;

__device__ __forceinline__ int sx_stride(int qs) { return qs + 2; }  // LDS rows of 4 (mod 8) words

struct SxIdx {
  int c, k, j0;
};
// Blocks in contiguous runs of (j group, k, component) on each XCD (the hardware deals them to the eight in
// turn): neighbours along j share the lines of a sector's rows, which one L2 then merges
__device__ __forceinline__ SxIdx sx_idx(const SectX &p, int hw) {
  const int per = p.jg * p.kg, nb = 3 * per, x = hw & 7, bq = nb >> 3, br = nb & 7;
  const int b = (x < br ? x * (bq + 1) : br * (bq + 1) + (x - br) * bq) + (hw >> 3);
  SxIdx r;
  r.c = b / per;
  const int q = b - r.c * per;
  r.k = q / p.jg;
  r.j0 = (q - r.k * p.jg) * SX_J;
  return r;
}

__device__ __forceinline__ void sect_fwd_body(const SectX &p, int b) {
  extern __shared__ __align__(16) unsigned char sx_smem[];
  double *F = (double *)sx_smem;  // [x parity][column][i]
  const SxIdx ix = sx_idx(p, b);
  const int c = ix.c, k = ix.k, j0 = ix.j0, tid = threadIdx.x, nth = blockDim.x;
  const int L0 = p.L[c][0], L1 = p.L[c][1], L2 = p.L[c][2];
  const int hx = (L0 + 1) / 2, hy = (L1 + 1) / 2, hz = (L2 + 1) / 2;
  if (k >= hz || j0 >= hy) return;
  const int mt = (hx + 15) / 16, QS = 16 * mt, IS = sx_stride(QS);
  const View v = p.v[c];
  const double *base = (const double *)v.p;
  const int ks = L2 - 1 - k;
  // two items a thread at a time, their sixteen loads in flight together
  for (int t0 = tid; t0 < QS * SX_J; t0 += 2 * nth) {
    double a[2][2][4];
    bool ok[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = t0 + u * nth, i = t % QS, j = j0 + t / QS;
      ok[u] = t < QS * SX_J && i < hx && j < hy;
      const int ic = ok[u] ? i : 0, jc = ok[u] ? j : j0, is = L0 - 1 - ic, js = L1 - 1 - jc;
      const double *r00 = base + (size_t)v.s1 * jc + (size_t)v.s2 * k, *r10 = base + (size_t)v.s1 * js + (size_t)v.s2 * k;
      const double *r01 = base + (size_t)v.s1 * jc + (size_t)v.s2 * ks, *r11 = base + (size_t)v.s1 * js + (size_t)v.s2 * ks;
      a[u][0][0] = r00[ic], a[u][0][1] = r10[ic], a[u][0][2] = r01[ic], a[u][0][3] = r11[ic];
      a[u][1][0] = r00[is], a[u][1][1] = r10[is], a[u][1][2] = r01[is], a[u][1][3] = r11[is];
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int t = t0 + u * nth, i = t % QS, jj = t / QS;
      if (t >= QS * SX_J) continue;
      double s[2][4];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const double e0 = a[u][x][0] + a[u][x][1], o0 = a[u][x][0] - a[u][x][1], e1 = a[u][x][2] + a[u][x][3],
                     o1 = a[u][x][2] - a[u][x][3];
        s[x][0] = 0.25 * (e0 + e1);  // y even, z even
        s[x][1] = 0.25 * (e0 - e1);  // y even, z odd
        s[x][2] = 0.25 * (o0 + o1);  // y odd, z even
        s[x][3] = 0.25 * (o0 - o1);
      }
      const bool ci = L0 - 1 - i == i;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        F[(q * SX_J + jj) * IS + i] = !ok[u] ? 0.0 : (ci ? s[0][q] : s[0][q] + s[1][q]);
        F[(SX_COLS + q * SX_J + jj) * IS + i] = (!ok[u] || ci) ? 0.0 : s[0][q] - s[1][q];
      }
    }
  }
  __syncthreads();
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), nw = nth >> 6, l = tid & 63, lr = l & 15, lk = l >> 4;
  const int wx = c == 0 ? 1 : 0;
  for (int m = w; m < mt; m += nw)
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      v4d acc[SX_T];
#pragma unroll
      for (int t = 0; t < SX_T; ++t) acc[t] = v4d{0, 0, 0, 0};
      const double *A = p.B[wx][x] + (size_t)(16 * m + lr) * QS + 4 * lk;
      const double *B0 = F + (x * SX_COLS + lr) * IS + 4 * lk;
      // the bases come from L2: three groups ahead, an MFMA group takes 512 cycles of its SIMD
      v4d a = ld4d(A), an = ld4d(A + 16 * min(1, mt - 1)), a2 = ld4d(A + 16 * min(2, mt - 1));
      for (int g = 0; g < mt; ++g) {
        const v4d a3 = ld4d(A + 16 * min(g + 3, mt - 1));
        v4d b[SX_T];
#pragma unroll
        for (int t = 0; t < SX_T; ++t) b[t] = ld4d(B0 + 16 * t * IS + 16 * g);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int t = 0; t < SX_T; ++t) acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b[t][u], acc[t], 0, 0, 0);
        a = an;
        an = a2;
        a2 = a3;
      }
      // element r of lane l: mode 2 (16 m + 4 r + lk) + x of the column's sector and position
#pragma unroll
      for (int t = 0; t < SX_T; ++t) {
        const int col = 16 * t + lr, q = col / SX_J, j = j0 + col % SX_J;
        const int py = (q >> 1) ^ (c == 1 ? 1 : 0), pz = (q & 1) ^ (c == 2 ? 1 : 0), s = 2 * py + pz;
        const int ly = p.q.hy[c == 1 ? 1 : 0][py], lz = p.q.hz[c == 2 ? 1 : 0][pz];
        if (j >= ly || k >= lz) continue;
        double *o = p.S + p.q.off[s] + p.q.oc[c][s] + j + (size_t)ly * k;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int mode = 2 * (16 * m + 4 * r + lk) + x;
          if (mode < L0) o[(size_t)(mode + wx) * p.q.size[s]] = acc[t][r];
        }
      }
    }
}

// r to the sectors; block 0 also leaves ||r||² (the partials of the residual kernel) in SC_RR
__global__ void __launch_bounds__(64 * SX_WAVES, 5) k_sect_fwd(SectX p) {
  if (p.gate && !*p.gate) return;
  if (blockIdx.x == 0 && p.nparts > 0) {
    __shared__ double sh[SX_WAVES];
    const double *part = p.d.part + (size_t)PART_RR * 2 * MAX_PART;
    double s = 0.0;
    for (int e = threadIdx.x; e < p.nparts; e += blockDim.x) s += part[2 * e];
    s = wave_sum_d(s);
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
      double t = 0.0;
      for (int q = 0; q < (int)(blockDim.x >> 6); ++q) t += sh[q];
      p.d.sc[SC_RR] = t;
    }
  }
  sect_fwd_body(p, (int)blockIdx.x);
}

// Whether the sectors iterate: the source is not zero and the first residual is above the tolerance
__device__ __forceinline__ bool sect_active(const PcgDev &d) {
  const double tol = d.sc[SC_TOL] * d.sc[SC_NB];
  return d.fl[FL_NZ] && sqrt(d.sc[SC_RR]) > tol;
}

// The way back: out(i) = E + O and out(L - 1 - i) = E - O of the even and odd x modes, the four sectors
// summed with the signs of the mirror images.  The product is taken transposed (rows: sector r at
// position lk, columns: 16 consecutive i), so a lane holds the four sectors of its element and a store
// covers 16 consecutive doubles.  PCG: x += value, φ = θ + x, and the counts of the solve; with addth
// (the separable field) φ = θ + value.
template <bool PCG>
__device__ __forceinline__ void sect_inv_body(const SectX &p, int b, bool act) {
  extern __shared__ __align__(16) unsigned char sx_smem[];
  double *F = (double *)sx_smem;  // [x parity][16 t + 4 sector + j][u]
  const SxIdx ix = sx_idx(p, b);
  const int c = ix.c, k = ix.k, j0 = ix.j0, tid = threadIdx.x, nth = blockDim.x;
  const int L0 = p.L[c][0], L1 = p.L[c][1], L2 = p.L[c][2];
  const int hx = (L0 + 1) / 2, hy = (L1 + 1) / 2, hz = (L2 + 1) / 2;
  if (k >= hz || j0 >= hy) return;
  const int mt = (hx + 15) / 16, QS = 16 * mt, IS = sx_stride(QS);
  const int wx = c == 0 ? 1 : 0;
  if (act) {
    // a thread keeps its position and sector and steps through the modes (nth is a multiple of 32), eight loads
    // in flight
    const int jj = tid % SX_J, q = (tid / SX_J) % 4, j = j0 + jj, dm = nth / SX_COLS;
    const int py = (q >> 1) ^ (c == 1 ? 1 : 0), pz = (q & 1) ^ (c == 2 ? 1 : 0), s = 2 * py + pz;
    const int ly = p.q.hy[c == 1 ? 1 : 0][py], lz = p.q.hz[c == 2 ? 1 : 0][pz];
    const bool in = j < ly && k < lz;
    const size_t ms = (size_t)p.q.size[s];
    const double *src = p.S + p.q.off[s] + (size_t)wx * ms + p.q.oc[c][s] + (in ? (size_t)j + (size_t)ly * k : 0);
    double *dst = F + (16 * (jj >> 2) + 4 * q + (jj & 3)) * IS;
    for (int m0 = tid / SX_COLS; m0 < 2 * QS; m0 += 8 * dm) {
      double f[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) f[u] = src[(size_t)min(m0 + u * dm, L0 - 1) * ms];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const int mode = m0 + u * dm;
        if (mode < 2 * QS) dst[(mode & 1) * SX_COLS * IS + (mode >> 1)] = (in && mode < L0) ? f[u] : 0.0;
      }
    }
    __syncthreads();
  }
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), nw = nth >> 6, l = tid & 63, lr = l & 15, lk = l >> 4;
  const View vo = p.v[c], vt = p.th[c], vx = p.x[c];
  for (int m = w; m < mt; m += nw) {
    v4d acc[2][SX_T];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
      for (int t = 0; t < SX_T; ++t) acc[x][t] = v4d{0, 0, 0, 0};
    if (act)
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const double *B = p.B[wx][x] + (size_t)(16 * m + lr) * QS + 4 * lk;
        const double *A0 = F + (x * SX_COLS + lr) * IS + 4 * lk;
        v4d bb = ld4d(B), bn = ld4d(B + 16 * min(1, mt - 1)), b2 = ld4d(B + 16 * min(2, mt - 1));
        for (int g = 0; g < mt; ++g) {
          const v4d b3 = ld4d(B + 16 * min(g + 3, mt - 1));
          v4d a[SX_T];
#pragma unroll
          for (int t = 0; t < SX_T; ++t) a[t] = ld4d(A0 + 16 * t * IS + 16 * g);
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int t = 0; t < SX_T; ++t)
              acc[x][t] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[t][u], bb[u], acc[x][t], 0, 0, 0);
          bb = bn;
          bn = b2;
          b2 = b3;
        }
      }
    const int i = 16 * m + lr, is = L0 - 1 - i, ks = L2 - 1 - k;
    if (i >= hx) continue;
#pragma unroll
    for (int t = 0; t < SX_T; ++t) {
      const int j = j0 + 4 * t + lk, js = L1 - 1 - j;
      if (j >= hy) continue;
#pragma unroll
      for (int xi = 0; xi < 2; ++xi) {
        if (xi && is == i) continue;
        const int ii = xi ? is : i;
        // the operands of the four images together (a centre row's or plane's image is itself), then the stores
        double tv[4], xv[4];
#pragma unroll
        for (int im = 0; im < 4; ++im) {
          const int jj = (im & 1) ? js : j, kk = (im & 2) ? ks : k;
          tv[im] = ((const double *)vt.p)[(size_t)ii + (size_t)vt.s1 * jj + (size_t)vt.s2 * kk];
          xv[im] = PCG ? ((const double *)vx.p)[(size_t)ii + (size_t)vx.s1 * jj + (size_t)vx.s2 * kk] : 0.0;
        }
        double s[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) s[q] = xi ? acc[0][t][q] - acc[1][t][q] : acc[0][t][q] + acc[1][t][q];
        const double e = s[0] + s[2], o = s[0] - s[2], e1 = s[1] + s[3], o1 = s[1] - s[3];
        const double val[4] = {e + e1, o + o1, e - e1, o - o1};  // (j, k), (js, k), (j, ks), (js, ks)
#pragma unroll
        for (int im = 0; im < 4; ++im) {
          if (((im & 1) && js == j) || ((im & 2) && ks == k)) continue;
          const int jj = (im & 1) ? js : j, kk = (im & 2) ? ks : k;
          const size_t oo = (size_t)ii + (size_t)vo.s1 * jj + (size_t)vo.s2 * kk;
          if (PCG) {
            const double xn = xv[im] + val[im];
            if (act) ((double *)vx.p)[(size_t)ii + (size_t)vx.s1 * jj + (size_t)vx.s2 * kk] = xn;
            ((double *)vo.p)[oo] = tv[im] + xn;
          } else {
            ((double *)vo.p)[oo] = tv[im] + val[im];
          }
        }
      }
    }
  }
}

__global__ void __launch_bounds__(64 * SX_WAVES, 5) k_sect_inv(SectX p) {
  const bool act = sect_active(p.d);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    int *fl = p.d.fl;
    fl[FL_ITSUM] += fl[FL_IT];
    if (fl[FL_IT] > fl[FL_ITMAX]) fl[FL_ITMAX] = fl[FL_IT];
    const int cl = p.cls >= 0 && p.cls < PCG_NCLS ? p.cls : 0;
    if (fl[FL_IT] > fl[FL_ITMAXC + cl]) fl[FL_ITMAXC + cl] = fl[FL_IT];
  }
  sect_inv_body<true>(p, (int)blockIdx.x, act);
}

static int sx_tiles(const SectX &p) {
  int mt = 1;
  for (int c = 0; c < 3; ++c) mt = std::max(mt, cdiv(cdiv(p.L[c][0], 2), 16));
  return mt;
}
static size_t sx_lds(int mt) { return (size_t)2 * SX_COLS * (16 * mt + 2) * sizeof(double); }
constexpr size_t SECT_LDS_MAX = 160 * 1024;
bool sect_x_fits(const SectX &p) { return sx_lds(sx_tiles(p)) + 1024 <= SECT_LDS_MAX; }
static void sx_grid(SectX &p, int &blocks, int &threads, size_t &lds) {
  p.jg = p.kg = 1;
  for (int c = 0; c < 3; ++c) {
    p.jg = std::max(p.jg, cdiv(cdiv(p.L[c][1], 2), SX_J));
    p.kg = std::max(p.kg, cdiv(p.L[c][2], 2));
  }
  const int mt = sx_tiles(p);
  blocks = 3 * p.jg * p.kg;
  threads = 64 * std::min(SX_WAVES, std::max(4, mt));
  lds = sx_lds(mt);
}
int sect_x_blocks(const SectX &p0) {
  SectX p = p0;
  int nb, nt;
  size_t lds;
  sx_grid(p, nb, nt, lds);
  return nb;
}
hipError_t launch_sect_fwd(SectX p, hipStream_t s) {
  if (!sect_x_fits(p)) return hipErrorInvalidValue;
  int nb, nt;
  size_t lds;
  sx_grid(p, nb, nt, lds);
  if (g_rec) return (p.gate || p.nparts) ? hipErrorNotSupported : record(BK_SECTF, Geo{}, &p, sizeof p, nt, true, dim3(nb), lds);
  TDGL_LAUNCH(k_sect_fwd, dim3(nb), dim3(nt), lds, s, p);
  return hipGetLastError();
}
hipError_t launch_sect_inv(SectX p, hipStream_t s) {
  if (g_rec) return hipErrorNotSupported;
  if (!sect_x_fits(p)) return hipErrorInvalidValue;
  int nb, nt;
  size_t lds;
  sx_grid(p, nb, nt, lds);
  TDGL_LAUNCH(k_sect_inv, dim3(nb), dim3(nt), lds, s, p);
  return hipGetLastError();
}

__global__ void __launch_bounds__(64 * SX_WAVES, 5) k_sect_inv_sep(SectX p) { sect_inv_body<false>(p, (int)blockIdx.x, true); }
hipError_t launch_sect_inv_sep(SectX p, hipStream_t s) {
  if (!sect_x_fits(p)) return hipErrorInvalidValue;
  int nb, nt;
  size_t lds;
  sx_grid(p, nb, nt, lds);
  if (g_rec) return record(BK_SECTI, Geo{}, &p, sizeof p, nt, true, dim3(nb), lds);
  TDGL_LAUNCH(k_sect_inv_sep, dim3(nb), dim3(nt), lds, s, p);
  return hipGetLastError();
}
__global__ void __launch_bounds__(64 * SX_WAVES, 5) k_sect_fwd_b(BatchTab t) {
  const BatchIdx q = batch_idx(t);
  sect_fwd_body(((const SectX *)t.args)[q.r], q.b.x);
}
__global__ void __launch_bounds__(64 * SX_WAVES, 5) k_sect_inv_b(BatchTab t) {
  const BatchIdx q = batch_idx(t);
  sect_inv_body<false>(((const SectX *)t.args)[q.r], q.b.x, true);
}

// ---------------------------------------------------------------------------- the separable solve of a sector
// One block per sector and mode, in FP64 and in place: the y products (16 x 16 x 4 tiles, rows of T by the
// half-size basis, the basis from L2), the z products by component and 16 y modes a wave, (I + aK)^-1 by element
// over all threads, the inverse z and y products.  T's rows are the z columns of X, Z and Y as in k_sect_cg.
// Bound: the matrix products, 2 (Ly / 2) + 2 (Lz / 2) flop an element and direction.  With the z products, the
// projector and their inverse of 16 y modes in one wave's registers (five waves of eight at work, two FP64 divisions
// an element one behind the other) that part alone took 66 k of 155 k cycles.
// 257 x 129 x 33 nodes: fold, quarter planes, z pass and unfold took 363 us, the three launches here 237 (this one 140; three
// blocks a CU, the basis loads and products of their passes).
template <int ZT, int SM>
__device__ __forceinline__ void sect_sep_body(const SectSep &a, int b) {
  extern __shared__ __align__(16) unsigned char cg_smem[];
  const int tid = threadIdx.x, nth = blockDim.x, nw = nth >> 6;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, lr = l & 15, lk = l >> 4;
  const int s = b & 3, mx = b >> 2, py = s >> 1, pz = s & 1;
  const SectDims &q = a.q;
  const int n = q.size[s], ly = q.hy[0][py], le = q.hy[1][py], lz = q.hz[0][pz], lze = q.hz[1][pz];
  const int oY = q.oc[1][s], oZ = q.oc[2][s];
  const int yp = a.yp, ST = yp + 2, CY = lz + lze;
  const int mt = (ly + 15) / 16, nt1 = (CY + 15) / 16, nt2 = (lz + 15) / 16, ntile = mt * (nt1 + nt2);
  double *T = (double *)cg_smem;
  for (int t = tid; t < a.trows * ST; t += nth) T[t] = 0.0;
  const size_t base = (size_t)q.off[s] + (size_t)mx * n;
  const float iy = 1.0f / (float)ly, ie = 1.0f / (float)le;
  auto tat = [&](int e) {
    const int c = e < oY ? 0 : (e < oZ ? 1 : 2), f = e - (c == 0 ? 0 : (c == 1 ? oY : oZ)), row = c == 1 ? le : ly;
    const int k = (int)(((float)f + 0.5f) * (c == 1 ? ie : iy)), j = f - k * row;
    return (c == 0 ? k : (c == 1 ? CY + k : lz + k)) * ST + j;
  };
  __syncthreads();
  for (int e0 = tid; e0 < n; e0 += 4 * nth) {
    double v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = a.S[base + min(e0 + u * nth, n - 1)];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = e0 + u * nth;
      if (e < n) T[tat(e)] = (mx == 0 && e < oY) ? 0.0 : v[u];  // no edge mode of wave number 0
    }
  }
  __syncthreads();
  const float imt = 1.0f / (float)mt;
  auto ypass = [&](const double *BV, const double *BU) __attribute__((always_inline)) {
    v4d acc[SM];
#pragma unroll
    for (int t = 0; t < SM; ++t) {
      acc[t] = v4d{0, 0, 0, 0};
      const int tt = w + nw * t;
      if (tt < ntile) {
        const int nt = __builtin_amdgcn_readfirstlane((int)(((float)tt + 0.5f) * imt)), m = tt - nt * mt;
        const double *B = (nt < nt1 ? BV : BU) + (size_t)(16 * m + lr) * yp + 4 * lk;
        const double *A = T + ((nt < nt1 ? 16 * nt : CY + 16 * (nt - nt1)) + lr) * ST + 4 * lk;
        v4d bb = ld4d(B), bn = ld4d(B + 16 * min(1, mt - 1));
        for (int g = 0; g < mt; ++g) {
          const v4d b2 = ld4d(B + 16 * min(g + 2, mt - 1));
          const v4d av = ld4d(A + 16 * g);
#pragma unroll
          for (int u = 0; u < 4; ++u) acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u], bb[u], acc[t], 0, 0, 0);
          bb = bn;
          bn = b2;
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < SM; ++t) {
      const int tt = w + nw * t;
      if (tt < ntile) {
        const int nt = __builtin_amdgcn_readfirstlane((int)(((float)tt + 0.5f) * imt)), m = tt - nt * mt;
        const int row0 = nt < nt1 ? 16 * nt : CY + 16 * (nt - nt1), rows = nt < nt1 ? CY : CY + lz;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (row0 + lk + 4 * e < rows) T[(row0 + lk + 4 * e) * ST + 16 * m + lr] = acc[t][e];
      }
    }
    __syncthreads();
  };
  ypass(a.yb[py][0][0], a.yb[py][1][0]);
  // z forward and back, 16 y modes of a component a wave at a time, in place: the rows hold the z modes in between,
  // the edges' (none for wave number 0) from row 0 on
  const int sh = pz == 0 ? 1 : 0;
  auto zpass = [&](int back) __attribute__((always_inline)) {
    for (int o = w; o < 3 * mt; o += nw) {
      const int c = __builtin_amdgcn_readfirstlane((int)(((float)o + 0.5f) * imt)), m = o - c * mt;
      const int rows = c == 2 ? lze : lz, shi = c == 2 && back ? sh : 0, sho = c == 2 && !back ? sh : 0;
      double *Tq = T + (c == 0 ? 0 : (c == 1 ? CY : lz)) * ST + 16 * m + lr;
      const double *Z = a.zb[pz][c == 2][back] + (size_t)lr * a.zp + 4 * lk;
      v4d A[ZT][ZT], acc[ZT];
#pragma unroll
      for (int t = 0; t < ZT; ++t) {
        acc[t] = v4d{0, 0, 0, 0};
#pragma unroll
        for (int g = 0; g < ZT; ++g) A[t][g] = ld4d(Z + (size_t)16 * t * a.zp + 16 * g);
      }
#pragma unroll
      for (int g = 0; g < ZT; ++g) {
        double B[4];  // rows past the component's meet the zeros of the basis
#pragma unroll
        for (int u = 0; u < 4; ++u) B[u] = Tq[min(max(16 * g + 4 * lk + u - shi, 0), rows - 1) * ST];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int t = 0; t < ZT; ++t) acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(A[t][g][u], B[u], acc[t], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < ZT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int r = 16 * t + lk + 4 * e - sho;
          if (r >= 0 && r < rows) Tq[r * ST] = acc[t][e];
        }
    }
    __syncthreads();
  };
  zpass(0);
  {
    const double k1 = a.s[0][mx];
    const bool hx = mx > 0;
    for (int t = tid; t < ly * lz; t += nth) {
      // (I + aK)^{-1} = P_L + P_T / (1 + a |k|²) (implicit.jl:67-78); a component without the mode is zero
      const int r = (int)(((float)t + 0.5f) * iy), p = t - r * ly, my = 2 * p + py, mz = 2 * r + pz;
      const bool hy = my > 0, hz = mz > 0;
      const double k2 = a.s[1][my], k3 = a.s[2][mz], k2s = k1 * k1 + k2 * k2 + k3 * k3;
      double *X = T + r * ST + p, *Y = X + CY * ST, *Z = X + (lz - sh) * ST;
      const double x1 = hx ? *X : 0.0, y1 = hy ? *Y : 0.0, z1 = hz ? *Z : 0.0;
      double dd = 0.0, f = 1.0;
      if (k2s != 0) {
        dd = (k1 * x1 + k2 * y1 + k3 * z1) / k2s;
        f = 1.0 / (1.0 + a.a * k2s);
      }
      *X = hx ? k1 * dd + f * (x1 - k1 * dd) : 0.0;
      *Y = hy ? k2 * dd + f * (y1 - k2 * dd) : 0.0;
      if (hz) *Z = k3 * dd + f * (z1 - k3 * dd);
    }
  }
  __syncthreads();
  zpass(1);
  ypass(a.yb[py][0][1], a.yb[py][1][1]);
  for (int e = tid; e < n; e += nth) a.S[base + e] = T[tat(e)];
}
template <int ZT, int SM>
__global__ void __launch_bounds__(512, 4) k_sect_sep(SectSep a) {
  sect_sep_body<ZT, SM>(a, (int)blockIdx.x);
}
template <int ZT, int SM>
__global__ void __launch_bounds__(512, 4) k_sect_sep_b(BatchTab t) {
  const BatchIdx q = batch_idx(t);
  sect_sep_body<ZT, SM>(((const SectSep *)t.args)[q.r], q.b.x);
}
// z tiles, y tiles a wave (0: does not fit), LDS
static int sep_pick(SectSep &a, int &zt, size_t &lds) {
  const SectDims &q = a.q;
  int ntile = 0;
  a.trows = 0;
  zt = cdiv(q.hz[0][0], 16);
  for (int s = 0; s < 4; ++s) {
    const int py = s >> 1, pz = s & 1, lz = q.hz[0][pz], lze = q.hz[1][pz], CY = lz + lze;
    if (q.hy[0][py] < 1 || q.hy[1][py] < 1 || lz < 1 || lze < 1) return 0;
    ntile = std::max(ntile, cdiv(q.hy[0][py], 16) * (cdiv(CY, 16) + cdiv(lz, 16)));
    // the products read whole tiles of rows past the last component
    a.trows = std::max({a.trows, CY + 16 * cdiv(lz, 16), CY + 16 * zt, 16 * cdiv(CY, 16)});
  }
  const int sm = cdiv(ntile, 8);
  lds = (size_t)a.trows * (a.yp + 2) * sizeof(double);
  if (zt > 3 || sm > 8 || lds + 1024 > SECT_LDS_MAX) return 0;
  return sm <= 4 ? 4 : 8;
}
bool sect_sep_fits(const SectSep &a0) {
  SectSep a = a0;
  int zt;
  size_t lds;
  return sep_pick(a, zt, lds) > 0;
}
#define TDGL_SEP_ALL TDGL_SEP(1, 4) TDGL_SEP(2, 4) TDGL_SEP(3, 4) TDGL_SEP(1, 8) TDGL_SEP(2, 8) TDGL_SEP(3, 8)
hipError_t launch_sect_sep(SectSep a, hipStream_t s) {
  int zt;
  size_t lds;
  const int sm = sep_pick(a, zt, lds);
  if (!sm) return hipErrorInvalidValue;
  const dim3 grid(4 * a.q.nx);
  if (g_rec) return record(BK_SECTS, Geo{}, &a, sizeof a, 10 * zt + sm, true, grid, lds);
  switch (10 * zt + sm) {
#define TDGL_SEP(z, m) \
  case 10 * z + m: TDGL_LAUNCH((k_sect_sep<z, m>), grid, dim3(512), lds, s, a); break;
    TDGL_SEP_ALL
#undef TDGL_SEP
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}
hipError_t launch_sect_batch(int kind, int variant, size_t lds, const BatchTab &t, int blocks, hipStream_t s) {
  if (kind == BK_SECTF || kind == BK_SECTI) {
    if (variant < 64 || variant > 64 * SX_WAVES) return hipErrorInvalidValue;
    if (kind == BK_SECTF)
      TDGL_LAUNCH(k_sect_fwd_b, dim3(blocks), dim3(variant), lds, s, t);
    else
      TDGL_LAUNCH(k_sect_inv_b, dim3(blocks), dim3(variant), lds, s, t);
    return hipGetLastError();
  }
  switch (variant) {
#define TDGL_SEP(z, m) \
  case 10 * z + m: TDGL_LAUNCH((k_sect_sep_b<z, m>), dim3(blocks), dim3(512), lds, s, t); break;
    TDGL_SEP_ALL
#undef TDGL_SEP
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// ---------------------------------------------------------------------------- the CG of a sector
// One block per sector.  r, d, Q and z_old of a thread's elements (e = tid + threads i) stay in registers,
// the direction P in LDS (FP64, its stencil reads neighbours) with a ring of ghost places that follow the
// same recurrence with the mirrored z, so that every element's stencil is the same nine or eleven reads, and
// the preconditioner's work array T in LDS (Float32): rows are the sector's z columns (X's, then Z's, then
// Y's), j or the y mode along the row.
// The preconditioner multiplies every row by the half-size y basis (16 x 16 x 4 tiles, the basis from
// L2, its first groups asked for before the barrier), then each wave takes 16 y modes through the z transform,
// the projector and the inverse z transform in registers (a forward tile leaves in a lane the modes its inverse
// takes as operand), then the inverse y products.
// Bound: on 272 x 144 x 48 nodes the matrix products of an iteration are 11.8 k cycles of the 38 k it takes a
// block there (two share a CU), the rest the issue of the stencil's LDS reads, FP64 sums and what ten elements a
// thread spill past 128 registers; on small planes the issue of the instructions of two blocks and ten barriers an
// iteration, 7 to 13 k cycles.  Branches at every edge and d in global memory at first: 955 us on those nodes, 82 us
// on 100 x 52 x 28, 126 us on 83 x 49 x 21, 38 us on 57 x 31 x 13; with the ghosts 812, 54, 78 and 26; with
// the y tiles known when compiled (MT; 0: any) 762, 46, 65 and 22, and 75 to 63 on 132 x 68 x 20.
// The sums are FP64, in a fixed order: the same bits every time.
// Where it stops: a sector's share of (tight tol ||b||)² is half an equal share and half its share of
// the first residual, so the sectors' residuals together are below the tolerance, no sector iterates for
// the others and one that holds almost nothing stops at once.  What is left is spread over the sectors and
// not where the general iteration leaves it, and at the tolerance itself the fields came out up to nine
// times further from a solution to the rounding than that iteration's.  At a 16th they are nearer than by either
// of its preconditioner's paths (folds, full length) on all 27 runs measured: 2.3e-9 against 2.5e-9 and 7.1e-9 after
// six cycles of 96x48x24 cells, 8.3e-9 against 2.8e-8 and 7.3e-8 after one of 53x27x9, 8.7e-9 against 2.7e-8 and 1.3e-8
// (43x86x6), 6.9e-11 against 9.0e-10 and 8.7e-10 with KWT (128x64x16).  At an eighth three of them were further by up to
// twice (5.4e-9 on 96x48x24, 1.6e-8 on 43x86x6, 1.3e-8 against 1.0e-8 on 72x41x8); a 16th takes 4 to 8 % more
// iterations, a 24th another 3 %.
// the same value, which the compiler does not know to be: what is derived from it is formed where it is used
// and not kept in registers through the iterations
__device__ __forceinline__ int fresh(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// one step of a wave's sum through DPP: lanes outside the row mask or the row add 0
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xf, false);
  return v + __hiloint2double(hi, lo);
}
// the sum of a wave's values, in lane 63
__device__ __forceinline__ double wave_sum63(double v) {
  v = dpp_add<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
  v = dpp_add<0x112, 0xf>(v);
  v = dpp_add<0x114, 0xf>(v);
  v = dpp_add<0x118, 0xf>(v);
  v = dpp_add<0x142, 0xa>(v);  // row_bcast 15, 31
  return dpp_add<0x143, 0xc>(v);
}

// The y tiles a wave holds at once: one or two, or up to four, in one round; a plane with more goes in rounds of whole
// row groups (a tile reads and writes the rows of its own group only).  One instance of up to six tiles spilled 510 to
// 940 B a lane and was slower than the general iteration on some planes; a step with it, now and by the general
// iteration: 1265 / 444 / 1031 us (200x250x4 cells, buf 2), 1722 / 677 / 1587 (200x110x34), 1081 / 586 / 986 (8x640x5,
// rounds), 699 / 383 / 684 (16x60x88); 4244 / 1661 / 9309 us on 256x128x33 cells, buf 8.
constexpr int SECT_SM = 4;
template <int EPT, int ZT, int SM, int MT>
__global__ void __launch_bounds__(SECT_T, 4) k_sect_cg(SectCG a) {
  if (!sect_active(a.d)) return;
  extern __shared__ __align__(16) unsigned char cg_smem[];
  static_assert(SECT_T == 512, "eight waves");
  constexpr bool SMALL = EPT <= 4;  // few elements: what every iteration needs stays in registers
  __shared__ __align__(16) double red[4][8];
  __shared__ double pal[3 * DPAL_MAX];
  const int tid = threadIdx.x, nth = blockDim.x, nw = nth >> 6;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63, lr = l & 15, lk = l >> 4;
  const int s = blockIdx.x & 3, mx = blockIdx.x >> 2, py = s >> 1, pz = s & 1;
  const SectDims &q = a.q;
  const int n = q.size[s], ly = q.hy[0][py], le = q.hy[1][py], lz = q.hz[0][pz], lze = q.hz[1][pz];
  const int oY = q.oc[1][s], oZ = q.oc[2][s];
  double *P = (double *)cg_smem;
  float *T = (float *)(P + a.np);
  unsigned *G = (unsigned *)(T + a.trows * (a.yp + 4));
  const int yp = MT ? 16 * MT : a.yp, ST = (MT ? 16 * MT : a.yp) + 4, CY = lz + lze;
  const int mt = MT ? MT : (ly + 15) / 16, nt1 = (CY + 15) / 16, nt2 = (lz + 15) / 16, ntile = mt * (nt1 + nt2);
  // P: component c at pc[c] + (k + 1) RS + j + 1, a ring of ghost places around each
  const int RS = ly + 2, pY = (lz + 2) * RS, pZ = 2 * pY;
  auto pat = [&](int c, int j, int k) { return (c == 0 ? 0 : (c == 1 ? pY : pZ)) + (k + 1) * RS + j + 1; };
  auto tat = [&](int c, int j, int k) { return (c == 0 ? k : (c == 1 ? CY + k : lz + k)) * ST + j; };  // the place in T
  for (int t = tid; t < a.trows * ST; t += nth) T[t] = 0.0f;
  for (int t = tid; t < a.np; t += nth) P[t] = 0.0;
  if (tid < 3 * DPAL_MAX) pal[tid] = a.pal[tid];
  if (tid < 32) red[tid >> 3][tid & 7] = 0.0;
  float *kz = (float *)(G + a.ng);  // the z wave numbers of this parity
  for (int t = tid; t < lz; t += nth) kz[t] = 2 * t + pz < q.nz ? a.sfz[2 * t + pz] : 0.0f;
  const double sv = a.sx[mx], ca = a.ca;
  const double tolb = a.d.sc[SC_TOL] * a.d.sc[SC_NB];
  const size_t base = (size_t)q.off[s] + (size_t)mx * n;

  // The ghosts, place | source in T << 14 | sign << 28 (1 +, 2 -).  The difference across the boundary is zero
  // (the outer ring repeats the node, or is a zero edge); across the centre it is the mirrored node (even
  // count ± the last, odd count the one before the last) or edge (odd count - the last, even count the zero
  // centre).  A sign of 0 stays the zero that P was filled with.
  {
    const int yn = q.ny % 2 ? ly - 2 : ly - 1, zn = q.nz % 2 ? lz - 2 : lz - 1;
    const int sy = q.ny % 2 ? (py ? 0 : 1) : (py ? -1 : 1), sz = q.nz % 2 ? (pz ? 0 : 1) : (pz ? -1 : 1);
    const int ey = q.ny % 2 && !py ? -1 : 0, ez = q.nz % 2 && !pz ? -1 : 0;
    int at = 0;
    auto run = [&](int cnt, auto entry) {  // entry(i): component, source, place, sign
      for (int i = (tid + nth - at % nth) % nth; i < cnt; i += nth) entry(i);
      at += cnt;
    };
    int g0 = 0;
    auto put = [&](int i, int c, int j, int k, int js, int ks, int sg) {
      G[g0 + i] = (unsigned)pat(c, j, k) | ((unsigned)tat(c, sg ? js : 0, sg ? ks : 0) << 14) | (sg > 0 ? 1u << 28 : (sg < 0 ? 2u << 28 : 0u));
    };
    run(lz, [&](int k) { put(k, 0, -1, k, 0, k, 1); });
    g0 = at;
    run(lz, [&](int k) { put(k, 0, ly, k, yn, k, sy); });
    g0 = at;
    run(ly, [&](int j) { put(j, 0, j, -1, j, 0, 1); });
    g0 = at;
    run(ly, [&](int j) { put(j, 0, j, lz, j, zn, sz); });
    g0 = at;
    run(lz + 1, [&](int k) { put(k, 1, le, k, le - 1, k < lz ? k : zn, ey * (k < lz ? 1 : sz)); });
    g0 = at;
    run(le, [&](int j) { put(j, 1, j, -1, j, 0, 1); });
    g0 = at;
    run(le, [&](int j) { put(j, 1, j, lz, j, zn, sz); });
    g0 = at;
    run(lze, [&](int k) { put(k, 2, -1, k, 0, k, 1); });
    g0 = at;
    run(lze + 1, [&](int k) { put(k, 2, ly, k, yn, k < lze ? k : lze - 1, sy * (k < lze ? 1 : ez)); });
    g0 = at;
    run(ly, [&](int j) { put(j, 2, j, lze, j, lze - 1, ez); });
  }
  const int ng = 3 * (ly + lz) + 2 * (le + lze) + 2;

  // this thread's elements: place in P | place in T << 14 | log2 weight << 28 | component << 30, and D's codes
  unsigned id[EPT], code[(EPT + 7) / 8];
  double r[EPT], d[EPT];
  float zo[EPT];
  double rr = 0.0;
#pragma unroll
  for (int i = 0; i < (EPT + 7) / 8; ++i) code[i] = 0u;
#pragma unroll
  for (int i = 0; i < EPT; ++i) {
    const int e = tid + nth * i;
    id[i] = 0u;
    r[i] = d[i] = 0.0;
    zo[i] = 0.0f;
    if (e < n) {
      const int c = e < oY ? 0 : (e < oZ ? 1 : 2), f = e - (c == 0 ? 0 : (c == 1 ? oY : oZ)), row = c == 1 ? le : ly;
      const int k = f / row, j = f - k * row;
      const bool cy = c == 1 ? (q.ny % 2 == 0 && py && j == le - 1) : (q.ny % 2 == 1 && !py && j == ly - 1);
      const bool cz = c == 2 ? (q.nz % 2 == 0 && pz && k == lze - 1) : (q.nz % 2 == 1 && !pz && k == lz - 1);
      const unsigned wt = (cy ? 0u : 1u) + (cz ? 0u : 1u);
      code[i / 8] |= (unsigned)a.code[c][j + q.hy[c == 1][c == 1] * k] << (4 * (i % 8));
      id[i] = (unsigned)pat(c, j, k) | ((unsigned)tat(c, j, k) << 14) | (wt << 28) | ((unsigned)c << 30);
      if (!(c == 0 && mx == 0)) r[i] = a.R[base + e];
      rr += (double)(1u << wt) * (r[i] * r[i]);
    }
  }
  __syncthreads();  // T is zero
  auto sum_of = [&](int slot, double v) {
    v = wave_sum63(v);
    if (l == 63) red[slot][w] = v;
  };
  auto total = [&](int slot) {
    const double *p = red[slot];  // the waves that are not there hold 0
    return ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
  };
  auto put_r = [&] {
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (tid + nth * i < n) T[(id[i] >> 14) & 16383u] = (float)r[i];
  };
  auto weight = [&](unsigned v) { return (double)(1u << ((v >> 28) & 3u)); };
  sum_of(0, rr);
  put_r();
  __syncthreads();
  rr = total(0);
  const double thr = a.tight * a.tight * 0.5 * tolb * tolb * (a.share + rr / a.d.sc[SC_RR]);
  const float imt = 1.0f / (float)mt;
  // one pass of the y products over the rows of T: rows x basis, in place
  struct First {
    v4f a, b;  // the first tile's first two groups of the basis
  };
  // tile t of this wave in the round of row groups that starts at tile t0
  constexpr int SA = SM > SECT_SM ? SECT_SM : SM;  // accumulators a wave
  const int per = SM > SECT_SM ? mt * (SECT_SM * nw / mt) : ntile;
  auto tile = [&](int t0, int t, int &m, int &nt) __attribute__((always_inline)) {
    const int tt = t0 + w + nw * t;
    nt = MT ? tt / max(MT, 1) : __builtin_amdgcn_readfirstlane((int)(((float)tt + 0.5f) * imt));
    m = tt - nt * mt;
    return tt < (SM > SECT_SM ? min(t0 + per, ntile) : ntile);
  };
  auto first = [&](const float *BV, const float *BU) __attribute__((always_inline)) {
    First f{v4f{0, 0, 0, 0}, v4f{0, 0, 0, 0}};
    int m, nt;
    if (tile(0, 0, m, nt)) {
      const float *A = (nt < nt1 ? BV : BU) + 16 * m * yp + fresh(lr) * yp + 4 * lk;
      f.a = *(const v4f *)A;
      f.b = *(const v4f *)(A + 16 * min(1, mt - 1));
    }
    return f;
  };
  auto ypass = [&](const float *BV, const float *BU, const First f) __attribute__((always_inline)) {
    const int la = fresh(lr) * yp + 4 * lk, lb = fresh(lr) * ST + 4 * lk;
    int t0 = 0;
    do {
      v4f acc[SA];
#pragma unroll
      for (int t = 0; t < SA; ++t) {
        acc[t] = v4f{0, 0, 0, 0};
        int m, nt;
        if (tile(t0, t, m, nt)) {
          const float *A = (nt < nt1 ? BV : BU) + 16 * m * yp + la;
          const float *B = T + (nt < nt1 ? 16 * nt : CY + 16 * (nt - nt1)) * ST + lb;
          // the basis comes through L2: two groups of sixteen ahead
          const bool asked = t == 0 && (SM <= SECT_SM || t0 == 0);
          v4f av = asked ? f.a : *(const v4f *)A, an = asked ? f.b : *(const v4f *)(A + 16 * min(1, mt - 1));
#pragma unroll(MT ? MT : 1)
          for (int g = 0; g < mt; ++g) {
            const v4f aq = *(const v4f *)(A + 16 * min(g + 2, mt - 1));
            const v4f bv = *(const v4f *)(B + 16 * g);
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[u], bv[u], acc[t], 0, 0, 0);
            av = an;
            an = aq;
          }
        }
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < SA; ++t) {
        int m, nt;
        if (tile(t0, t, m, nt)) {
          const int col0 = nt < nt1 ? 16 * nt : CY + 16 * (nt - nt1);
          if (col0 + lr < (nt < nt1 ? CY : CY + lz)) *(v4f *)(T + col0 * ST + 16 * m + lb) = acc[t];
        }
      }
      t0 += per;
    } while (SM > SECT_SM && t0 < ntile);
    __syncthreads();
  };
  const float *const yf[2] = {a.yb[py][0][0], a.yb[py][1][0]}, *const yr[2] = {a.yb[py][0][1], a.yb[py][1][1]};
  First ff = first(yf[0], yf[1]), fr = ff;
  if (SMALL) fr = first(yr[0], yr[1]);
  // the z bases, fragment (t, g) of matrix: 0 V forward, 1 U forward, 2 V back, 3 U back
  constexpr bool ZREG = SMALL && ZT == 1;
  auto zfrag = [&](int which, int t, int g, int l) {
    return *(const v4f *)(a.zb[pz][which & 1][which >> 1] + (16 * t + (l & 15)) * a.zp + 16 * g + 4 * (l >> 4));
  };
  v4f zr[4] = {};
  if (ZREG)
#pragma unroll
    for (int i = 0; i < 4; ++i) zr[i] = zfrag(i, 0, 0, l);
  // the projector's factors, one tile a wave
  constexpr bool PREG = ZREG && EPT <= 2 && MT > 0 && MT <= 4;
  float pf[4] = {}, pk[4] = {}, pk2 = 0.0f;
  if (PREG) {
    const int my = 2 * (16 * w + lr) + py;
    const float k1 = a.sfx[mx], af = (float)a.a;
    pk2 = my < q.ny ? a.sfy[my] : 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int mz = 2 * (4 * lk + e) + pz;
      pk[e] = my < q.ny && mz < q.nz ? a.sfz[mz] : 0.0f;
      pf[e] = 1.0f / (1.0f + af * (k1 * k1 + pk2 * pk2 + pk[e] * pk[e]));
    }
  }
  double dreg[SMALL ? EPT : 1] = {};
  if (SMALL)
#pragma unroll
    for (int i = 0; i < (SMALL ? EPT : 1); ++i) dreg[i] = pal[DPAL_MAX * min(id[i] >> 30, 2u) + ((code[i / 8] >> (4 * (i % 8))) & 15u)];
  const unsigned gv = tid < ng ? G[tid] : 0u;  // the first ghost

  double rzold = 1.0;
  int it = 0;
  while (rr > thr && it < a.maxit) {
    // z = M⁻¹ r in Float32; T holds r
#pragma unroll
    for (int i = 0; i < EPT; ++i) id[i] = (unsigned)fresh((int)id[i]);
    ypass(yf[0], yf[1], ff);
    for (int m = w; m < mt; m += nw) {
      // 16 y modes: z forward, the projector, z back; k = 16 g + 4 lk + u of the rows (zero past them)
      const int lf = fresh(l), lr = lf & 15, lk = lf >> 4;
      const float *Tq = T + 16 * m + lr;
      v4f acc[3][ZT];
#pragma unroll
      for (int t = 0; t < ZT; ++t) acc[0][t] = acc[1][t] = acc[2][t] = v4f{0, 0, 0, 0};
#pragma unroll
      for (int g = 0; g < ZT; ++g) {
        // a component's rows at a time, the fragments of both node components once
        auto rows = [&](int row0, int cnt) {
          v4f B;
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const int k = 16 * g + 4 * lk + u;
            const float v = Tq[(row0 + min(k, cnt - 1)) * ST];
            B[u] = k < cnt ? v : 0.0f;
          }
          return B;
        };
        v4f A[ZT];
#pragma unroll
        for (int t = 0; t < ZT; ++t) A[t] = ZREG ? zr[0] : zfrag(0, t, g, lf);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const v4f B = rows(c == 0 ? 0 : (c == 1 ? CY : lz), c == 2 ? lze : lz);
          if (c == 2)
#pragma unroll
            for (int t = 0; t < ZT; ++t) A[t] = ZREG ? zr[1] : zfrag(1, t, g, lf);
#pragma unroll
          for (int t = 0; t < ZT; ++t)
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[c][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[t][u], B[u], acc[c][t], 0, 0, 0);
        }
        if (ZT > 1) __builtin_amdgcn_sched_barrier(0);  // the registers of one group at a time
      }
      {
        const int my = 2 * (16 * m + lr) + py;
        const float k1 = a.sfx[mx], k2 = PREG ? pk2 : (my < q.ny ? a.sfy[my] : 0.0f), af = (float)a.a;
        const bool live = my < q.ny, hx = mx > 0, hy = my > 0;
#pragma unroll
        for (int t = 0; t < ZT; ++t)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            // (I + aK)^{-1} = P_L + P_T / (1 + a |k|²) = (I + a k kᵀ) / (1 + a |k|²) (implicit.jl:67-78); a component
            // without the mode is zero
            const int mz = 2 * (16 * t + 4 * lk + e) + pz;
            const bool in = live && mz < q.nz;
            const float k3 = PREG ? pk[e] : (in ? kz[16 * t + 4 * lk + e] : 0.0f);
            const float f = PREG ? pf[e] : 1.0f / (1.0f + af * (k1 * k1 + k2 * k2 + k3 * k3));
            const float x1 = hx ? acc[0][t][e] : 0.0f, y1 = hy ? acc[1][t][e] : 0.0f, z1 = mz > 0 ? acc[2][t][e] : 0.0f;
            const float dd = af * (k1 * x1 + k2 * y1 + k3 * z1);
            acc[0][t][e] = hx ? f * (x1 + k1 * dd) : 0.0f;
            acc[1][t][e] = hy ? f * (y1 + k2 * dd) : 0.0f;
            acc[2][t][e] = mz > 0 ? f * (z1 + k3 * dd) : 0.0f;
            if (ZT > 1 && e % 2) __builtin_amdgcn_sched_barrier(0);
          }
      }
      __builtin_amdgcn_wave_barrier();  // the tile's columns are read: their rows take the result
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const int row0 = c == 0 ? 0 : (c == 1 ? CY : lz), rows = c == 2 ? lze : lz;
        float *To = T + row0 * ST + 16 * m + lr;
#pragma unroll
        for (int t = 0; t < ZT; ++t) {
          v4f o = v4f{0, 0, 0, 0};
#pragma unroll
          for (int g = 0; g < ZT; ++g) {
            const v4f A = ZREG ? zr[c == 2 ? 3 : 2] : zfrag(c == 2 ? 3 : 2, t, g, lf);
#pragma unroll
            for (int u = 0; u < 4; ++u) o = __builtin_amdgcn_mfma_f32_16x16x4f32(A[u], acc[c][g][u], o, 0, 0, 0);
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int k = 16 * t + 4 * lk + e;
            if (k < rows) To[k * ST] = o[e];
          }
        }
        if (ZT > 1) __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (!SMALL) fr = first(yr[0], yr[1]);
    __syncthreads();
    ypass(yr[0], yr[1], fr);
    // the dots and the direction
    float z[EPT];
    double rz = 0.0, rzo = 0.0;
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      z[i] = 0.0f;
      if (tid + nth * i < n) {
        z[i] = T[(id[i] >> 14) & 16383u];
        const double wr = weight(id[i]) * r[i];
        rz = fma(wr, (double)z[i], rz);
        rzo = fma(wr, (double)zo[i], rzo);
        zo[i] = z[i];
      }
    }
    sum_of(0, rz);
    sum_of(1, rzo);
    auto ghost_z = [&](unsigned v) { return (v >> 28) & 2u ? -(double)T[(v >> 14) & 16383u] : (double)T[(v >> 14) & 16383u]; };
    const double gz = ghost_z(gv), gp = P[gv & 16383u];
    double pold[SMALL ? EPT : 1];
    if (SMALL)
#pragma unroll
      for (int i = 0; i < (SMALL ? EPT : 1); ++i) pold[i] = P[id[i] & 16383u];
    __syncthreads();
    rz = total(0);
    const double beta = it > 0 ? (rz - total(1)) / rzold : 0.0;
    rzold = rz;
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (tid + nth * i < n) {
        double *p = P + (id[i] & 16383u);
        *p = fma(beta, SMALL ? pold[SMALL ? i : 0] : *p, (double)z[i]);
      }
    if (gv >> 28) P[gv & 16383u] = fma(beta, gp, gz);
    for (int g = tid + nth; g < ng; g += nth) {
      const unsigned v = G[g];
      double *p = P + (v & 16383u);
      if (v >> 28) *p = fma(beta, *p, ghost_z(v));
    }
    __syncthreads();
    // Q = (D + aK) P on the half domain: the ghosts make every place alike.  Edges along y and z: the same with
    // the directions swapped (da across the edge in the plane, db along it).
    double Q[EPT], pq = 0.0;
#pragma unroll
    for (int i = 0; i < EPT; ++i) {
      Q[i] = 0.0;
      if (tid + nth * i < n) {
        const unsigned v = (unsigned)fresh((int)id[i]), c = v >> 30;
        const double *A = P + (v & 16383u);
        const double p0 = A[0];
        double cur;
        if (c == 0) {
          const double *Y = A + pY, *Z = A + pZ;
          cur = fma(sv, Y[0] - Y[-1], (p0 - A[1]) + (p0 - A[-1])) + fma(sv, Z[0] - Z[-RS], (p0 - A[RS]) + (p0 - A[-RS]));
        } else {
          const int da = c == 1 ? RS : 1, db = c == 1 ? 1 : RS;
          const double *B = A + (c == 1 ? pY : -pY), *X = A - (c == 1 ? pY : pZ);
          cur = ((p0 - A[da]) + (p0 - A[-da])) + ((B[db] - B[0]) - (B[db - da] - B[-da])) + sv * fma(sv, p0, X[0] - X[db]);
        }
        Q[i] = fma(SMALL ? dreg[SMALL ? i : 0] : pal[DPAL_MAX * c + ((code[i / 8] >> (4 * (i % 8))) & 15u)], p0, ca * cur);
        pq = fma(weight(v) * p0, Q[i], pq);
      }
    }
    sum_of(2, pq);
    __syncthreads();
    const double al = rz / total(2);
    rr = 0.0;
#pragma unroll
    for (int i = 0; i < EPT; ++i)
      if (tid + nth * i < n) {
        d[i] = fma(al, P[id[i] & 16383u], d[i]);
        r[i] = fma(-al, Q[i], r[i]);
        rr = fma(weight(id[i]) * r[i], r[i], rr);
      }
    ++it;
    sum_of(3, rr);
    put_r();
    if (!SMALL) ff = first(yf[0], yf[1]);
    __syncthreads();
    rr = total(3);
  }
#pragma unroll
  for (int i = 0; i < EPT; ++i)
    if (tid + nth * i < n) a.X[base + tid + nth * i] = d[i];
  if (tid == 0) atomicMax(a.d.fl + FL_IT, it);
}

// The launch of the sectors' CG: threads, elements a thread, y tiles a wave.  8 waves a block, and EPT
// elements a thread of the sector's size; two blocks share a CU's LDS on the largest grids.
struct CgPick {
  bool ok;
  int threads, ept, zt, sm;
  size_t lds;
};
static CgPick cg_pick(const SectCG &a0, int &np, int &trows, int &ng) {
  CgPick k{};
  const SectDims &q = a0.q;
  int n = 0, ntile = 0, mtm = 0;
  np = trows = ng = 0;
  for (int s = 0; s < 4; ++s) {
    const int py = s >> 1, pz = s & 1, lz = q.hz[0][pz], lze = q.hz[1][pz], CY = lz + lze;
    if (q.hy[0][py] < 1 || q.hy[1][py] < 1 || lz < 1 || lze < 1) return k;
    if (q.hy[0][py] > 1023 || lz > 1023) return k;
    n = std::max(n, q.size[s]);
    const int mt = cdiv(q.hy[0][py], 16), nt = cdiv(CY, 16) + cdiv(lz, 16);
    ntile = std::max(ntile, mt * nt);
    mtm = std::max(mtm, mt);
    trows = std::max(trows, CY + 16 * cdiv(lz, 16));
    np = std::max(np, (2 * (lz + 2) + lze + 2) * (q.hy[0][py] + 2));
    ng = std::max(ng, 3 * (q.hy[0][py] + lz) + 2 * (q.hy[1][py] + lze) + 2);
  }
  np = (np + 1) / 2 * 2;
  k.zt = cdiv(q.hz[0][0], 16);
  const int epts[6] = {2, 4, 6, 8, 10, 11};
  for (int e : epts) {
    const int th = 64 * std::max(4, cdiv(n, 64 * e));
    if (th > SECT_T) continue;
    k.threads = th;
    k.ept = e;
    break;
  }
  if (!k.threads) return k;
  k.sm = cdiv(ntile, k.threads / 64);
  const size_t nT = (size_t)trows * (a0.yp + 4);
  k.lds = (size_t)np * sizeof(double) + nT * sizeof(float) + (size_t)ng * sizeof(unsigned) + (size_t)q.hz[0][0] * sizeof(float);
  // 14 bits hold a place in P and in T
  // a round of the y products takes whole row groups
  k.ok = k.zt <= 3 && k.sm <= 6 && mtm <= SECT_SM * (k.threads / 64) && np <= 16384 && nT <= 16384 && k.lds + 1024 <= SECT_LDS_MAX;
  return k;
}
bool sect_cg_fits(const SectCG &a) {
  int np, tr, ng;
  return cg_pick(a, np, tr, ng).ok;
}
hipError_t launch_sect_cg(SectCG a, hipStream_t s) {
  if (g_rec) return hipErrorNotSupported;
  const CgPick k = cg_pick(a, a.np, a.trows, a.ng);
  if (!k.ok) return hipErrorInvalidValue;
  const dim3 grid(4 * a.q.nx), blk(k.threads);
#define TDGL_CG(E, Z, M, T)                                              \
  if (k.ept == E && k.zt == Z && k.sm <= M && (T == 0 || a.yp == 16 * T)) { \
    TDGL_LAUNCH((k_sect_cg<E, Z, M, T>), grid, blk, k.lds, s, a);        \
    return hipGetLastError();                                            \
  }
  // the y tiles known when compiled, for sectors of one and two z tiles whose elements a thread go with that count on
  // planes up to twice as wide as deep or so; the others take the generic instance of their tiles a wave (of 5088 and
  // 5160 elements, 32 iterations: 964 us with, 1046 without)
  TDGL_CG(2, 1, 2, 1) TDGL_CG(2, 1, 2, 2) TDGL_CG(2, 1, 2, 3) TDGL_CG(2, 1, 2, 4) TDGL_CG(4, 1, 2, 2) TDGL_CG(4, 1, 2, 3)
  TDGL_CG(4, 1, 2, 4) TDGL_CG(4, 1, 2, 5) TDGL_CG(6, 1, 2, 3) TDGL_CG(6, 1, 2, 5)
  TDGL_CG(6, 1, 2, 4) TDGL_CG(2, 2, 2, 1) TDGL_CG(4, 2, 2, 2) TDGL_CG(6, 2, 2, 2) TDGL_CG(6, 2, 4, 3) TDGL_CG(8, 2, 4, 3)
  TDGL_CG(10, 2, 4, 4) TDGL_CG(10, 2, 4, 5)
#define TDGL_CG_Z(E, Z) TDGL_CG(E, Z, 2, 0) TDGL_CG(E, Z, 4, 0) TDGL_CG(E, Z, 6, 0)
#define TDGL_CG_E(E) TDGL_CG_Z(E, 1) TDGL_CG_Z(E, 2) TDGL_CG_Z(E, 3)
  TDGL_CG_E(2) TDGL_CG_E(4) TDGL_CG_E(6) TDGL_CG_E(8) TDGL_CG_E(10) TDGL_CG_E(11)
#undef TDGL_CG_E
#undef TDGL_CG_Z
#undef TDGL_CG
  return hipErrorInvalidValue;
}

}  // namespace tdgl
