// Grid kernels: scatter / product / gather / elementwise / reductions.
#include <algorithm>
#include <cmath>

#include "kernels.h"
#include "reduce.h"

namespace gmod {

constexpr int TPB = 256;
static inline unsigned nblocks(long n, int tpb = TPB, long cap = 1L << 20) {
  long b = (n + tpb - 1) / tpb;
  if (b > cap) b = cap;
  if (b < 1) b = 1;
  return (unsigned)b;
}

// ------------------------------------------------------------------ mesh
void Mesh::build(const int64_t* kmap, const int64_t* invk, long Nkall_, long Nk_, int Nx_, int Ny_,
                 int Nz_, int Nw_, hipStream_t s) {
  Nx = Nx_; Ny = Ny_; Nz = Nz_; Nw = Nw_; M = 2 * Nw_;
  Nkall = Nkall_; Nk = Nk_;
  if ((long)Nx * Ny * Nz != Nkall) throw Error("Nx*Ny*Nz != Nkall");
  std::vector<int> hirr(Nkall), hflag(Nkall), hsp(Nkall), hrev(Nkall), hirrsp(Nk, -1);
  kw_host.assign(Nk, 0.0);
  std::vector<char> seen(Nkall, 0);
  for (long i = 0; i < Nkall; ++i) {
    long x = kmap[3 * i], y = kmap[3 * i + 1], z = kmap[3 * i + 2];
    if (x < 0 || x >= Nx || y < 0 || y >= Ny || z < 0 || z >= Nz) throw Error("kmap entry outside the mesh");
    long sp_ = x + (long)Nx * (y + (long)Ny * z);
    if (seen[sp_]) throw Error("kmap is not a permutation of the mesh");
    seen[sp_] = 1;
    long k = invk[3 * i] - 1;
    if (k < 0 || k >= Nk) throw Error("invk(1,:) outside [1,Nk]");
    int f = (int)invk[3 * i + 1];
    if (f != 0 && f != 1) throw Error("invk(2,:) must be 0 or 1");
    hirr[i] = (int)k;
    hflag[i] = f;
    hsp[i] = (int)sp_;
    kw_host[k] += 1.0;
    if (f == 0 && hirrsp[k] < 0) hirrsp[k] = (int)sp_;
  }
  for (long z = 0; z < Nz; ++z)
    for (long y = 0; y < Ny; ++y)
      for (long x = 0; x < Nx; ++x) {
        long sp_ = x + Nx * (y + Ny * z);
        long rx = (Nx - x) % Nx, ry = (Ny - y) % Ny, rz = (Nz - z) % Nz;
        hrev[sp_] = (int)(rx + Nx * (ry + Ny * rz));
      }
  std::vector<int> hirr_s(Nkall), hflag_s(Nkall), hkgat_s(Nkall, -1);
  for (long i = 0; i < Nkall; ++i) {
    hirr_s[hsp[i]] = hirr[i];
    hflag_s[hsp[i]] = hflag[i];
  }
  complete = true;
  for (long k = 0; k < Nk; ++k) {
    if (hirrsp[k] >= 0) hkgat_s[hirrsp[k]] = (int)k;
    else complete = false;
  }
  irr.alloc(Nkall); flag.alloc(Nkall); sp.alloc(Nkall); rev.alloc(Nkall); irr_sp.alloc(Nk); kw.alloc(Nk);
  irr_s.alloc(Nkall); flag_s.alloc(Nkall); kgat_s.alloc(Nkall); kf_s.alloc(Nkall);
  irr_s.upload(hirr_s.data(), Nkall, s);
  flag_s.upload(hflag_s.data(), Nkall, s);
  std::vector<int> hkf_s(Nkall);
  for (long i = 0; i < Nkall; ++i) hkf_s[i] = (hirr_s[i] << 1) | (hflag_s[i] != 0 ? 1 : 0);
  kf_s.upload(hkf_s.data(), Nkall, s);
  kgat_s.upload(hkgat_s.data(), Nkall, s);
  kgat_host = hkgat_s;
  irr.upload(hirr.data(), Nkall, s);
  flag.upload(hflag.data(), Nkall, s);
  sp.upload(hsp.data(), Nkall, s);
  rev.upload(hrev.data(), Nkall, s);
  irr_sp.upload(hirrsp.data(), Nk, s);
  kw.upload(kw_host.data(), Nk, s);
  std::vector<int> hfull(Nkall), hnfull(Nkall);
  nfull_ok = true;
  for (long i = 0; i < Nkall; ++i) {
    hfull[hsp[i]] = (int)i;
    const long nf = invk[3 * i + 2] - 1;
    if (nf < 0 || nf >= Nkall) nfull_ok = false;
    hnfull[hsp[i]] = (nf < 0 || nf >= Nkall) ? 0 : (int)nf;
  }
  full_s.alloc(Nkall);
  nfull_s.alloc(Nkall);
  full_s.upload(hfull.data(), Nkall, s);
  nfull_s.upload(hnfull.data(), Nkall, s);
  GMOD_HIP(hipStreamSynchronize(s));
}

MeshDev mesh_dev(const Mesh& m) {
  MeshDev d{m.irr_s.p, m.flag_s.p, m.kgat_s.p, m.rev.p, m.kf_s.p, m.Nkall, m.Nk, m.Nw, m.M};
  d.full_s = m.full_s.p;
  d.nfull_s = m.nfull_s.p;
  return d;
}

template <typename R>
__global__ void k_mul_acc(cpx<R>* __restrict__ acc, const cpx<R>* __restrict__ A, const cpx<R>* __restrict__ B,
                          int first, long n) {
  for (long g = blockIdx.x * (long)blockDim.x + threadIdx.x; g < n; g += (long)gridDim.x * blockDim.x) {
    cpx<R> v = A[g] * B[g];
    acc[g] = first ? v : acc[g] + v;
  }
}

template <typename R>
void mul_acc(cpx<R>* acc, const cpx<R>* A, const cpx<R>* B, bool first, long n, hipStream_t s) {
  hipLaunchKernelGGL((k_mul_acc<R>), dim3(nblocks(n)), dim3(TPB), 0, s, acc, A, B, (int)first, n);
  GMOD_CHECK_LAUNCH();
}

// One thread per spatial point and chunk of L slots.  For band n with
// a = |e_n - mu|: E1(s) = exp(-a tau_s) falls by r = exp(-a dtau) per slot,
// E2(s) = exp(-a (beta - tau_s)) rises by 1/r; g0 = -(xi >= 0 ? E1 : E2) / d,
// g1 = (xi >= 0 ? E2 : E1) / d, d = 1 + exp(-beta a).  E2 is evaluated
// directly where its chunk start would underflow (deep bands, low T).
template <typename R, int NO>
__global__ void __launch_bounds__(256)
k_tau_ref(cpx<R>* ta, cpx<R>* tb, const double* __restrict__ eig, const zd* __restrict__ U, double mu, double mu2,
          int nv, double beta, double dtau, MeshDev m, int L) {
  const int a = blockIdx.y % NO, b = blockIdx.y / NO;
  ta += (long)blockIdx.y * m.Nkall * m.M;
  tb += (long)blockIdx.y * m.Nkall * m.M;
  const long nch = (m.M + L - 1) / L;
  const long tot = m.Nkall * nch;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < tot; e += (long)gridDim.x * blockDim.x) {
    const long sp = e % m.Nkall;
    const int s0 = (int)(e / m.Nkall) * L;
    const int s1 = s0 + L < m.M ? s0 + L : m.M;
    const long k = m.irr_s[sp];
    const bool rev = m.flag_s[sp] != 0;
    zd c[NO];
    double E1[NO][2], E2[NO][2], r[NO][2], ir[NO][2], id[NO][2], ad[NO][2];
    bool pos[NO][2], direct[NO][2];
#pragma unroll
    for (int n = 0; n < NO; ++n) {
      zd cn = U[a + NO * (n + (long)NO * k)] * conj(U[b + NO * (n + (long)NO * k)]);
      c[n] = rev ? conj(cn) : cn;
#pragma unroll
      for (int v = 0; v < 2; ++v) {
        const double xi = eig[n + (long)NO * k] - (v == 0 ? mu : mu2);
        const double aa = fabs(xi);
        pos[n][v] = xi >= 0.0;
        id[n][v] = 1.0 / (1.0 + exp(-beta * aa));
        ad[n][v] = aa * dtau;
        direct[n][v] = ad[n][v] * (double)(m.M - s0) > 600.0 || ad[n][v] > 300.0;
        E1[n][v] = exp(-ad[n][v] * (double)s0);
        E2[n][v] = direct[n][v] ? 0.0 : exp(-ad[n][v] * (double)(m.M - s0));
        r[n][v] = exp(-ad[n][v]);
        ir[n][v] = direct[n][v] ? 0.0 : exp(ad[n][v]);
      }
    }
    for (int s = s0; s < s1; ++s) {
      zd A(0, 0), B(0, 0);
#pragma unroll
      for (int n = 0; n < NO; ++n) {
#pragma unroll
        for (int v = 0; v < 2; ++v) {
          if (v >= nv) continue;
          const double e2 = direct[n][v] ? exp(-ad[n][v] * (double)(m.M - s)) : E2[n][v];
          const double g0 = -(pos[n][v] ? E1[n][v] : e2) * id[n][v];
          const double g1 = (pos[n][v] ? e2 : E1[n][v]) * id[n][v];
          const double sg = v == 0 ? 1.0 : -1.0;
          A += c[n] * (sg * g0);
          B += c[n] * (sg * g1);
          E1[n][v] *= r[n][v];
          E2[n][v] *= ir[n][v];
        }
      }
      ta[sp + m.Nkall * (long)s] = cpx<R>(A);
      tb[sp + m.Nkall * (long)s] = cpx<R>(B);
    }
  }
}

template <typename R>
void tau_ref_grids(cpx<R>* ta, cpx<R>* tb, const double* eig, const zd* uni, int No, double mu, double mu2, bool diff,
                   double beta, double dtau, const MeshDev& m, hipStream_t s) {
  const int L = 64;
  const long tot = m.Nkall * (long)((m.M + L - 1) / L);
  const int nv = diff ? 2 : 1;
  const dim3 g((unsigned)std::min<long>((tot + 255) / 256, 1L << 20), (unsigned)(No * No)), blk(256);
  switch (No) {
#define GMOD_TAU_CASE(NOV)                                                                                           \
  case NOV:                                                                                                          \
    hipLaunchKernelGGL((k_tau_ref<R, NOV>), g, blk, 0, s, ta, tb, eig, uni, mu, mu2, nv, beta, dtau, m, L); \
    break;
    GMOD_TAU_CASE(1) GMOD_TAU_CASE(2) GMOD_TAU_CASE(3) GMOD_TAU_CASE(4)
    GMOD_TAU_CASE(5) GMOD_TAU_CASE(6) GMOD_TAU_CASE(7) GMOD_TAU_CASE(8)
#undef GMOD_TAU_CASE
    default: throw Error("tau reference: Norb > 8 is not supported");
  }
  GMOD_CHECK_LAUNCH();
}

template void tau_ref_grids<float>(cpx<float>*, cpx<float>*, const double*, const zd*, int, double, double, bool,
                                   double, double, const MeshDev&, hipStream_t);
template void tau_ref_grids<double>(cpx<double>*, cpx<double>*, const double*, const zd*, int, double, double, bool,
                                    double, double, const MeshDev&, hipStream_t);

// ------------------------------------------------------------------ tail constants
// One work-group per density-matrix element, summed over the full zone in a
// fixed order.  Latency-bound (No^2 groups); it replaces a host loop of
// Nkall No^2 + Nk No^3 steps and a direct sawtooth sum of Nw x 2 Nw phases
// that kept the GPU idle in every iteration (1 orbital, 64x64 x 1024: 32.1 ms
// an iteration, now 2.4 ms; 32x32 x 256: 2.7 ms, now 0.9 ms).
__global__ void __launch_bounds__(256)
k_tail_density(zd* __restrict__ rb, const double* __restrict__ eig, const zd* __restrict__ U, int No, double mu,
               double beta, MeshDev m) {
  __shared__ double sr[256], si[256];
  const int a = blockIdx.x % No, b = blockIdx.x / No;
  zd acc(0, 0);
  for (long sp = threadIdx.x; sp < m.Nkall; sp += 256) {
    const int kf = m.kf_s[sp];
    const long k = kf >> 1;
    zd v(0, 0);
    for (int n = 0; n < No; ++n) {
      const double xi = eig[n + No * k] - mu, e = exp(-beta * fabs(xi));
      const double f = (xi >= 0 ? e : 1.0) / (1.0 + e);
      v += U[a + No * (n + No * k)] * conj(U[b + No * (n + No * k)]) * f;
    }
    acc += (kf & 1) ? conj(v) : v;
  }
  sr[threadIdx.x] = acc.re;
  si[threadIdx.x] = acc.im;
  __syncthreads();
  for (int o = 128; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) {
      sr[threadIdx.x] += sr[threadIdx.x + o];
      si[threadIdx.x] += si[threadIdx.x + o];
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) rb[blockIdx.x] = zd(sr[0] / (double)m.Nkall, si[0] / (double)m.Nkall);
}
void tail_density(zd* rb, const double* eig, const zd* uni, int No, double mu, double beta, const MeshDev& m,
                  hipStream_t s) {
  hipLaunchKernelGGL(k_tail_density, dim3((unsigned)(No * No)), dim3(256), 0, s, rb, eig, uni, No, mu, beta, m);
  GMOD_CHECK_LAUNCH();
}

__global__ void k_tail_jumps(zd* J, const zd* rb, const int* ol, int No, int Nchi) {
  for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < Nchi * Nchi; e += gridDim.x * blockDim.x) {
    const int l = e % Nchi, m = e / Nchi;
    const int a13 = ol[2 * l], b13 = ol[2 * m], a42 = ol[2 * m + 1], b42 = ol[2 * l + 1];
    zd v(0, 0);
    if (a13 == b13) v += rb[a42 + No * b42];
    if (a42 == b42) v -= rb[a13 + No * b13];
    J[e] = v;
  }
}
void tail_jumps(zd* J, const zd* rb, const int* ol, int No, int Nchi, hipStream_t s) {
  hipLaunchKernelGGL(k_tail_jumps, dim3(nblocks((long)Nchi * Nchi)), dim3(TPB), 0, s, J, rb, ol, No, Nchi);
  GMOD_CHECK_LAUNCH();
}

// sum_s e^{i x s} (1/2 - s/M) = -1 / (e^{i x} - 1) = 1/2 + (i/2) cot(x/2) for
// x = 2 pi j / M, j > 0, so the correction is -dtau/2 + (i dtau/2) (1/y - cot y)
// with y = pi j / M; the difference by its power series where it cancels
__global__ void k_sawtooth(zd* out, int Nw, double beta) {
  const double h = beta / (4.0 * (double)Nw);  // dtau / 2
  for (int j = blockIdx.x * blockDim.x + threadIdx.x; j < Nw; j += gridDim.x * blockDim.x) {
    const double y = 3.141592653589793238462643383279 * (double)j / (2.0 * (double)Nw), q = y * y;
    double d;
    if (y < 0.25)
      d = y * (1.0 / 3 + q * (1.0 / 45 + q * (2.0 / 945 + q * (1.0 / 4725 + q * (2.0 / 93555 + q * (1382.0 / 638512875))))));
    else
      d = 1.0 / y - cos(y) / sin(y);
    out[j] = zd(-h, h * d);
  }
}
void sawtooth(zd* sawc, int Nw, double temp, hipStream_t s) {
  hipLaunchKernelGGL(k_sawtooth, dim3(nblocks(Nw)), dim3(TPB), 0, s, sawc, Nw, 1.0 / temp);
  GMOD_CHECK_LAUNCH();
}

// ------------------------------------------------------------------ elementwise
__global__ void k_conj_copy(zd* dst, const zd* src, long n) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x)
    dst[e] = conj(src[e]);
}
void conj_copy(zd* dst, const zd* src, long n, hipStream_t s) {
  hipLaunchKernelGGL(k_conj_copy, dim3(nblocks(n)), dim3(TPB), 0, s, dst, src, n);
  GMOD_CHECK_LAUNCH();
}
__global__ void k_conj_copy_neg(zd* dst, const zd* src, long n) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    const zd v = src[e];
    dst[e] = zd(-v.re, v.im);
  }
}
void conj_copy(zd* dst, const zd* src, long n, double sign, hipStream_t s) {
  if (sign > 0) {
    conj_copy(dst, src, n, s);
    return;
  }
  hipLaunchKernelGGL(k_conj_copy_neg, dim3(nblocks(n)), dim3(TPB), 0, s, dst, src, n);
  GMOD_CHECK_LAUNCH();
}

// |Re| < eps -> Re = 0, then |Im| < eps -> Im = 0 (fchi.f90:499-500)
__global__ void k_threshold(zd* a, long n, double eps) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    zd v = a[e];
    if (fabs(v.re) < eps) v.re = 0.0;
    if (fabs(v.im) < eps) v.im = 0.0;
    a[e] = v;
  }
}
void threshold(zd* a, long n, double eps, hipStream_t s) {
  hipLaunchKernelGGL(k_threshold, dim3(nblocks(n)), dim3(TPB), 0, s, a, n, eps);
  GMOD_CHECK_LAUNCH();
}

__global__ void k_scale(zd* a, long n, double f) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x)
    a[e] = a[e] * f;
}
void scale(zd* a, long n, double f, hipStream_t s) {
  hipLaunchKernelGGL(k_scale, dim3(nblocks(n)), dim3(TPB), 0, s, a, n, f);
  GMOD_CHECK_LAUNCH();
}

__global__ void k_axpy(zd* y, const zd* x, zd al, long n) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x)
    y[e] = y[e] + al * x[e];
}
void axpy(zd* y, const zd* x, zd alpha, long n, hipStream_t s) {
  hipLaunchKernelGGL(k_axpy, dim3(nblocks(n)), dim3(TPB), 0, s, y, x, alpha, n);
  GMOD_CHECK_LAUNCH();
}

void copy(zd* dst, const zd* src, long n, hipStream_t s) {
  GMOD_HIP(hipMemcpyAsync(dst, src, n * sizeof(zd), hipMemcpyDeviceToDevice, s));
}

__global__ void k_threshold_copy(zd* dst, const zd* src, long n, double eps) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    zd v = src[e];
    if (fabs(v.re) < eps) v.re = 0.0;
    if (fabs(v.im) < eps) v.im = 0.0;
    dst[e] = v;
  }
}
void threshold_copy(zd* dst, const zd* src, long n, double eps, hipStream_t s) {
  hipLaunchKernelGGL(k_threshold_copy, dim3(nblocks(n)), dim3(TPB), 0, s, dst, src, n, eps);
  GMOD_CHECK_LAUNCH();
}

// dst(r, t) = src(-r, -t) on the full grid (t -> (M - t) mod M): an output
// row of x reads one input row in reverse order, so both sides coalesce
template <typename R>
__global__ void k_mirror_grid(cpx<R>* __restrict__ dst, const cpx<R>* __restrict__ src, int Nx, int Ny, int Nz,
                              int M) {
  const long S = (long)Nx * Ny * Nz, n = S * M;
  dst += (long)blockIdx.y * n;
  src += (long)blockIdx.y * n;
  for (long g = blockIdx.x * (long)blockDim.x + threadIdx.x; g < n; g += (long)gridDim.x * blockDim.x) {
    const long sp = g % S, t = g / S;
    const int x = (int)(sp % Nx), y = (int)((sp / Nx) % Ny), z = (int)(sp / ((long)Nx * Ny));
    const long rs = (x ? Nx - x : 0) + (long)Nx * ((y ? Ny - y : 0) + (long)Ny * (z ? Nz - z : 0));
    dst[g] = src[rs + S * (t ? M - t : 0)];
  }
}
template <typename R>
void mirror_grid(cpx<R>* dst, const cpx<R>* src, int Nx, int Ny, int Nz, int M, int n, hipStream_t s) {
  hipLaunchKernelGGL((k_mirror_grid<R>), dim3(nblocks((long)Nx * Ny * Nz * M), (unsigned)n), dim3(TPB), 0, s, dst, src,
                     Nx, Ny, Nz, M);
  GMOD_CHECK_LAUNCH();
}
template void mirror_grid<float>(cpx<float>*, const cpx<float>*, int, int, int, int, int, hipStream_t);
template void mirror_grid<double>(cpx<double>*, const cpx<double>*, int, int, int, int, int, hipStream_t);

// Streaming: every A grid is read once, the B grids (one per orbital pair)
// again for each output that uses them, from the cache when they fit it.
// One launch for all outputs; a launch per product wrote the running sum
// back and read it again each time (the 54 products of a 3-orbital gap step
// at 20x20x4 x 256: 290 us, now 107 us, 4.2 TB/s of grids counted once).
template <typename R>
__global__ void __launch_bounds__(TPB)
k_contract(cpx<R>* __restrict__ out, const cpx<R>* __restrict__ A, const cpx<R>* __restrict__ B,
           const int* __restrict__ off, const int* __restrict__ ta, const int* __restrict__ tb, long N, int add) {
  const int o = blockIdx.y, c0 = off[o], c1 = off[o + 1];
  for (long e = blockIdx.x * (long)TPB + threadIdx.x; e < N; e += (long)gridDim.x * TPB) {
    cpx<R> acc = add ? out[o * N + e] : A[ta[c0] * N + e] * B[tb[c0] * N + e];
    for (int c = add ? c0 : c0 + 1; c < c1; ++c) {
      const cpx<R> v = A[ta[c] * N + e] * B[tb[c] * N + e];
      acc = acc + v;
    }
    out[o * N + e] = acc;
  }
}
template <typename R>
void contract(cpx<R>* out, const cpx<R>* A, const cpx<R>* B, const int* off, const int* ta, const int* tb, int nout,
              long N, bool add, hipStream_t s) {
  hipLaunchKernelGGL((k_contract<R>), dim3(nblocks(N, TPB, 4096), (unsigned)nout), dim3(TPB), 0, s, out, A, B, off, ta,
                     tb, N, add ? 1 : 0);
  GMOD_CHECK_LAUNCH();
}

__global__ void k_partner_copies(zd* a, const int* tab, long NkNw) {
  const int src = tab[4 * blockIdx.y], dst = tab[4 * blockIdx.y + 1];
  if (dst < 0) return;
  const double sg = (tab[4 * blockIdx.y + 3] & 2) ? -1.0 : 1.0;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < NkNw; e += (long)gridDim.x * blockDim.x) {
    const zd v = a[NkNw * src + e];
    a[NkNw * dst + e] = zd(sg * v.re, -sg * v.im);
  }
}
void partner_copies(zd* a, const int* tab, int n, long NkNw, hipStream_t s) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_partner_copies, dim3(nblocks(NkNw, TPB, 1024), (unsigned)n), dim3(TPB), 0, s, a, tab, NkNw);
  GMOD_CHECK_LAUNCH();
}

__global__ void k_threshold_slice(zd* dst, const zd* src, long Nk, long NkNw, long nmat, double eps) {
  const long n = Nk * nmat;
  for (long g = blockIdx.x * (long)blockDim.x + threadIdx.x; g < n; g += (long)gridDim.x * blockDim.x) {
    const long k = g % Nk, e = g / Nk;
    zd v = src[k + NkNw * e];
    if (fabs(v.re) < eps) v.re = 0.0;
    if (fabs(v.im) < eps) v.im = 0.0;
    dst[g] = v;
  }
}
void threshold_slice(zd* dst, const zd* src, long Nk, long NkNw, long nmat, double eps, hipStream_t s) {
  const long n = Nk * nmat;
  hipLaunchKernelGGL(k_threshold_slice, dim3(nblocks(n)), dim3(TPB), 0, s, dst, src, Nk, NkNw, nmat, eps);
  GMOD_CHECK_LAUNCH();
}

__global__ void k_diff_to_f32(cpx<float>* dst, const zd* a, const zd* b, long n) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x)
    dst[e] = cpx<float>(a[e] - b[e]);
}
void diff_to_f32(cpx<float>* dst, const zd* a, const zd* b, long n, hipStream_t s) {
  hipLaunchKernelGGL(k_diff_to_f32, dim3(nblocks(n)), dim3(TPB), 0, s, dst, a, b, n);
  GMOD_CHECK_LAUNCH();
}

__global__ void k_lincomb(zd* y, const zd* a, double ca, const zd* b, double cb, long n) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x)
    y[e] = a[e] * ca + b[e] * cb;
}
void lincomb(zd* y, const zd* a, double ca, const zd* b, double cb, long n, hipStream_t s) {
  hipLaunchKernelGGL(k_lincomb, dim3(nblocks(n)), dim3(TPB), 0, s, y, a, ca, b, cb, n);
  GMOD_CHECK_LAUNCH();
}

// a <- a + b, b <- a - b (with the old a)
__global__ void k_sum_diff(zd* a, zd* b, long n) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    const zd x = a[e], y = b[e];
    a[e] = x + y;
    b[e] = x - y;
  }
}
void sum_diff(zd* a, zd* b, long n, hipStream_t s) {
  hipLaunchKernelGGL(k_sum_diff, dim3(nblocks(n)), dim3(TPB), 0, s, a, b, n);
  GMOD_CHECK_LAUNCH();
}

// ------------------------------------------------------------------ reductions
// One launch and one wait per result: latency-bound up to a few MB (the fields
// of the 4-orbital 16x16x8 x 256 mesh are 67 MB each, bound by their bytes).  The
// earlier form summed the 1024 partial results of a dot product in one thread
// of a second launch (90 us, a dependent load per term) and copied the sum
// back: 110 us on the device, now 15 with the wait.
static void wait(hipStream_t s) { GMOD_HIP(hipStreamSynchronize(s)); }

// The gap equation's norms and inner products are summed in one fixed order
// whatever the launch: element e belongs to work-group (e / 256) mod 1024, a
// work-group sums its threads by halves, the 1024 partial results are added in
// turn.  (A few Krylov steps or a slowly converging power iteration amplify a
// different rounding of these sums to the fourth digit of the gap.)
constexpr int ORD_BLOCKS = 1024;
static_assert(ORD_BLOCKS * 4 <= PIN_DOUBLES, "partial results of power_dots");
static int ord_blocks(long n) { return (int)std::max<long>(1, std::min<long>(ORD_BLOCKS, (n + RED_TPB - 1) / RED_TPB)); }

// sum over the work-group's 256 threads by halves, on thread 0
template <int W>
__device__ __forceinline__ void halves_sum(double (&v)[W], double* sh) {
#pragma unroll
  for (int c = 0; c < W; ++c) sh[c * RED_TPB + threadIdx.x] = v[c];
  __syncthreads();
  if (threadIdx.x < 128) {
#pragma unroll
    for (int c = 0; c < W; ++c) sh[c * RED_TPB + threadIdx.x] += sh[c * RED_TPB + threadIdx.x + 128];
  }
  __syncthreads();
  if (threadIdx.x < 64) {
#pragma unroll
    for (int c = 0; c < W; ++c) {
      double x = sh[c * RED_TPB + threadIdx.x] + sh[c * RED_TPB + threadIdx.x + 64];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) x += __shfl_down(x, o);
      v[c] = x;
    }
  }
  __syncthreads();
}

__global__ void __launch_bounds__(RED_TPB)
k_dot_w(const zd* __restrict__ u, const zd* __restrict__ v, const double* __restrict__ kw, long Nk, long n,
        double* part) {
  __shared__ double sh[2 * RED_TPB];
  double r[2] = {0, 0};
  for (long e = blockIdx.x * (long)RED_TPB + threadIdx.x; e < n; e += (long)ORD_BLOCKS * RED_TPB) {
    const zd p = conj(u[e]) * v[e];
    const double w = kw ? kw[e % Nk] : 1.0;
    r[0] += w * p.re;
    r[1] += w * p.im;
  }
  halves_sum<2>(r, sh);
  if (threadIdx.x == 0) { part[2 * blockIdx.x] = r[0]; part[2 * blockIdx.x + 1] = r[1]; }
}

zd dot_w(const zd* u, const zd* v, const double* kw, long Nk, long rest, hipStream_t s) {
  const long n = Nk * rest;
  const int nb = ord_blocks(n);
  const double* p = ctx().pin;
  hipLaunchKernelGGL(k_dot_w, dim3(nb), dim3(RED_TPB), 0, s, u, v, kw, Nk, n, ctx().pin);
  GMOD_CHECK_LAUNCH();
  wait(s);
  zd r(0, 0);
  for (int b = 0; b < nb; ++b) r += zd(p[2 * b], p[2 * b + 1]);
  return r;
}

// the sums of a power step: kw |nd|^2, Re kw conj(D) nd, kw |D|^2
__global__ void __launch_bounds__(RED_TPB)
k_power_dots(const zd* __restrict__ nd, const zd* __restrict__ D, const double* __restrict__ kw, long Nk, long n,
             double* part) {
  __shared__ double sh[3 * RED_TPB];
  double r[3] = {0, 0, 0};
  for (long e = blockIdx.x * (long)RED_TPB + threadIdx.x; e < n; e += (long)ORD_BLOCKS * RED_TPB) {
    const zd a = nd[e], d = D[e];
    const zd aa = conj(a) * a, da = conj(d) * a, dd = conj(d) * d;
    const double w = kw ? kw[e % Nk] : 1.0;
    r[0] += w * aa.re;
    r[1] += w * da.re;
    r[2] += w * dd.re;
  }
  halves_sum<3>(r, sh);
  if (threadIdx.x == 0)
    for (int c = 0; c < 3; ++c) part[3 * blockIdx.x + c] = r[c];
}
void power_dots(double out[3], const zd* nd, const zd* D, const double* kw, long Nk, long rest, hipStream_t s) {
  const int nb = ord_blocks(Nk * rest);
  const double* p = ctx().pin;
  hipLaunchKernelGGL(k_power_dots, dim3(nb), dim3(RED_TPB), 0, s, nd, D, kw, Nk, Nk * rest, ctx().pin);
  GMOD_CHECK_LAUNCH();
  wait(s);
  for (int c = 0; c < 3; ++c) {
    out[c] = 0.0;
    for (int b = 0; b < nb; ++b) out[c] += p[3 * b + c];
  }
}

// the nb partial results (re, im) added in turn, by threads 0 and 1 from LDS:
// s[0], s[1] (1024 dependent additions, 4 us)
__device__ __forceinline__ void turn_sum(double (&s)[2], const double* __restrict__ part, int nb, double* sh) {
  for (int i = threadIdx.x; i < 2 * nb; i += RED_TPB) sh[i] = part[i];
  __syncthreads();
  if (threadIdx.x < 2) {
    double t = 0.0;
    int b = 0;
    for (; b + 8 <= nb; b += 8) {
      double x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = sh[2 * (b + i) + threadIdx.x];
#pragma unroll
      for (int i = 0; i < 8; ++i) t += x[i];
    }
    for (; b < nb; ++b) t += sh[2 * b + threadIdx.x];
    s[0] = t;
  }
  __syncthreads();
  if (threadIdx.x < 2) sh[threadIdx.x] = s[0];
  __syncthreads();
  s[0] = sh[0];
  s[1] = sh[1];
  __syncthreads();
}

// One step of a modified Gram-Schmidt chain without a host wait: h = f times
// the sum of the previous launch's nb partial results (every work-group forms
// it), x -= h v, and the partial results of the next inner product,
// conj(vn) x (vn null: |x|^2), in pout.  v null: no update (the chain's
// start).  h goes to hout.
__global__ void __launch_bounds__(RED_TPB)
k_mgs(zd* __restrict__ x, const zd* __restrict__ v, const zd* __restrict__ vn, const double* __restrict__ kw, long Nk,
      long n, double f, const double* __restrict__ pin_, double* __restrict__ pout, double* hout) {
  __shared__ double sh[2 * ORD_BLOCKS];
  const int nb = gridDim.x;
  zd h(0, 0);
  if (v) {
    double t[2];
    turn_sum(t, pin_, nb, sh);
    h = zd(t[0] * f, t[1] * f);
    if (hout && blockIdx.x == 0 && threadIdx.x == 0) {
      hout[0] = h.re;
      hout[1] = h.im;
    }
    h = zd(0, 0) - h;
  }
  double r[2] = {0, 0};
  for (long e = blockIdx.x * (long)RED_TPB + threadIdx.x; e < n; e += (long)ORD_BLOCKS * RED_TPB) {
    zd a = x[e];
    if (v) {
      a = a + h * v[e];
      x[e] = a;
    }
    const zd p = conj(vn ? vn[e] : a) * a;
    const double w = kw ? kw[e % Nk] : 1.0;
    r[0] += w * p.re;
    r[1] += w * p.im;
  }
  halves_sum<2>(r, sh);
  if (threadIdx.x == 0) {
    pout[2 * blockIdx.x] = r[0];
    pout[2 * blockIdx.x + 1] = r[1];
  }
}

double gram_schmidt(zd* x, const std::vector<const zd*>& vs, zd* h, double f, const double* kw, long Nk, long rest,
                    hipStream_t s) {
  const long n = Nk * rest;
  Context& c = ctx();
  const int nb = ord_blocks(n), m = (int)vs.size();
  double* pnorm = c.pin;  // the last step's partial results go to the host, behind them the h
  double* hp = c.pin + 2 * ORD_BLOCKS;
  constexpr int ROOM = (PIN_DOUBLES - 2 * ORD_BLOCKS) / 2;
  double* part[2] = {c.red, c.red + 2 * ORD_BLOCKS};
  for (int i = -1; i < m; ++i) {
    const zd* vn = i + 1 < m ? vs[i + 1] : nullptr;
    hipLaunchKernelGGL(k_mgs, dim3(nb), dim3(RED_TPB), 0, s, x, i < 0 ? (const zd*)nullptr : vs[i], vn, kw, Nk, n, f,
                       (const double*)part[(i + 1) & 1], i + 1 < m ? part[i & 1] : pnorm,
                       i < 0 ? (double*)nullptr : hp + 2 * (i % ROOM));
    GMOD_CHECK_LAUNCH();
    if (i + 1 == m || i % ROOM == ROOM - 1) {
      wait(s);
      for (int j = i < 0 ? 0 : i - i % ROOM; j <= i; ++j) h[j] = zd(hp[2 * (j % ROOM)], hp[2 * (j % ROOM) + 1]);
    }
  }
  double t = 0.0;
  for (int b = 0; b < nb; ++b) t += pnorm[2 * b];
  return std::sqrt(f * t);
}

// sum conj(u) v_y of the nv vectors v + y stride (blockIdx.y = y)
__global__ void __launch_bounds__(RED_TPB)
k_dots(const zd* __restrict__ u, const zd* __restrict__ v, long stride, long n, double* part) {
  const zd* __restrict__ vy = v + (long)blockIdx.y * stride;
  double r[2] = {0, 0};
  for (long e = blockIdx.x * (long)RED_TPB + threadIdx.x; e < n; e += (long)gridDim.x * RED_TPB) {
    const zd p = conj(u[e]) * vy[e];
    r[0] += p.re;
    r[1] += p.im;
  }
  put_partial<RedSum, 2>(r, blockIdx.x, part + (long)blockIdx.y * 2 * gridDim.x);
}

void dots(zd* out, const zd* u, const zd* v, long stride, int nv, long n, hipStream_t s) {
  const double* p = ctx().pin;
  const int nb = red_blocks(n), room = PIN_DOUBLES / (2 * nb);
  for (int v0 = 0; v0 < nv; v0 += room) {
    const int m = std::min(room, nv - v0);
    hipLaunchKernelGGL(k_dots, dim3(nb, m), dim3(RED_TPB), 0, s, u, v + v0 * stride, stride, n, ctx().pin);
    GMOD_CHECK_LAUNCH();
    wait(s);
    for (int i = 0; i < m; ++i)
      out[v0 + i] = zd(sum_partials(p + 2 * nb * i, nb, 2, 0), sum_partials(p + 2 * nb * i, nb, 2, 1));
  }
}

// extremes: the partial results combined on the host; the error flag, when
// asked for, behind them
template <class Op>
static double host_extreme(int nb, const int* err, int* err_out) {
  const double* p = ctx().pin;
  double r = Op::id();
  for (int b = 0; b < nb; ++b) r = Op::op(r, p[b]);
  if (err) *err_out = (int)p[nb];
  return r;
}

__global__ void __launch_bounds__(RED_TPB)
k_max_rel(const zd* __restrict__ s0, const zd* __restrict__ sd, long n, double floor, double* part, const int* err) {
  double best[1] = {0.0};
  for (long e = blockIdx.x * (long)RED_TPB + threadIdx.x; e < n; e += (long)gridDim.x * RED_TPB) {
    const zd d = sd[e];
    const double ad = hypot(d.re, d.im);
    if (ad > floor) {
      const zd df = s0[e] - d;
      const double r = hypot(df.re, df.im) / ad;
      if (r > best[0]) best[0] = r;
    }
  }
  put_partial<RedMax, 1>(best, blockIdx.x, part);
  if (err && blockIdx.x == 0 && threadIdx.x == 0) part[gridDim.x] = (double)*err;
}
double max_rel_err(const zd* s0, const zd* sd, long n, double floor, hipStream_t s, const int* err, int* err_out) {
  const int nb = red_blocks(n);
  hipLaunchKernelGGL(k_max_rel, dim3(nb), dim3(RED_TPB), 0, s, s0, sd, n, floor, ctx().pin, err);
  GMOD_CHECK_LAUNCH();
  wait(s);
  return host_extreme<RedMax>(nb, err, err_out);
}

template <class Op>
__global__ void __launch_bounds__(RED_TPB)
k_extreme(const double* __restrict__ a, long stride, long n, double* part, const int* err) {
  double best[1] = {Op::id()};
  for (long e = blockIdx.x * (long)RED_TPB + threadIdx.x; e < n; e += (long)gridDim.x * RED_TPB)
    best[0] = Op::op(best[0], a[e * stride]);
  put_partial<Op, 1>(best, blockIdx.x, part);
  if (err && blockIdx.x == 0 && threadIdx.x == 0) part[gridDim.x] = (double)*err;
}
template <class Op>
static double extreme(const double* a, long stride, long n, hipStream_t s, const int* err, int* err_out) {
  const int nb = red_blocks(n);
  hipLaunchKernelGGL(k_extreme<Op>, dim3(nb), dim3(RED_TPB), 0, s, a, stride, n, ctx().pin, err);
  GMOD_CHECK_LAUNCH();
  wait(s);
  return host_extreme<Op>(nb, err, err_out);
}
double max_value(const double* a, long n, hipStream_t s, const int* err, int* err_out) {
  return extreme<RedMax>(a, 1, n, s, err, err_out);
}
double max_real(const zd* a, long n, hipStream_t s) {
  return extreme<RedMax>((const double*)a, 2, n, s, nullptr, nullptr);
}
double min_real(const zd* a, long n, hipStream_t s) {
  return extreme<RedMin>((const double*)a, 2, n, s, nullptr, nullptr);
}

// max |a - b| (b null: max |a|)
__global__ void __launch_bounds__(RED_TPB)
k_max_absdiff(const zd* __restrict__ a, const zd* __restrict__ b, long n, double* part) {
  double best[1] = {0.0};
  for (long e = blockIdx.x * (long)RED_TPB + threadIdx.x; e < n; e += (long)gridDim.x * RED_TPB) {
    const zd d = b ? a[e] - b[e] : a[e];
    const double r = hypot(d.re, d.im);
    if (r > best[0]) best[0] = r;
  }
  put_partial<RedMax, 1>(best, blockIdx.x, part);
}
double max_abs_diff(const zd* a, const zd* b, long n, hipStream_t s) {
  const int nb = red_blocks(n);
  hipLaunchKernelGGL(k_max_absdiff, dim3(nb), dim3(RED_TPB), 0, s, a, b, n, ctx().pin);
  GMOD_CHECK_LAUNCH();
  wait(s);
  return host_extreme<RedMax>(nb, nullptr, nullptr);
}

// y = sum_i c_i x_i over up to COMBINE vectors x + idx_i stride (add: onto y)
constexpr int COMBINE = 8;
struct CombineArgs {
  double c[COMBINE];
  long off[COMBINE];
  int n;
};
__global__ void k_combine(zd* __restrict__ y, const zd* __restrict__ x, CombineArgs a, int add, long n) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    zd r = add ? y[e] : zd(0, 0);
#pragma unroll
    for (int i = 0; i < COMBINE; ++i)
      if (i < a.n) r += x[a.off[i] + e] * a.c[i];
    y[e] = r;
  }
}
void combine(zd* y, const zd* x, long stride, const std::vector<int>& idx, const std::vector<double>& c, long n,
             hipStream_t s) {
  for (size_t i0 = 0; i0 < idx.size(); i0 += COMBINE) {
    CombineArgs a{};
    a.n = (int)std::min<size_t>(COMBINE, idx.size() - i0);
    for (int i = 0; i < a.n; ++i) {
      a.c[i] = c[i0 + i];
      a.off[i] = idx[i0 + i] * stride;
    }
    hipLaunchKernelGGL(k_combine, dim3(nblocks(n)), dim3(TPB), 0, s, y, x, a, i0 > 0 ? 1 : 0, n);
    GMOD_CHECK_LAUNCH();
  }
}

__global__ void k_scale_copy(zd* y, const zd* x, double f, long n) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x)
    y[e] = x[e] * f;
}
void scale_copy(zd* y, const zd* x, double f, long n, hipStream_t s) {
  hipLaunchKernelGGL(k_scale_copy, dim3(nblocks(n)), dim3(TPB), 0, s, y, x, f, n);
  GMOD_CHECK_LAUNCH();
}

// ------------------------------------------------------------------ Sigma reference-vertex term
// One thread per grid point: the No^2 increments Fd_ab in registers (read
// once), then every output's sum over its No^2 reference-vertex grids; the
// vertex grids are read once each, coalesced along the point index.
template <typename R, int NAB>
__global__ void __launch_bounds__(256)
k_sigma_ref_contract(cpx<R>* __restrict__ Y, cpx<R>* __restrict__ Gn, const cpx<R>* __restrict__ Fr,
                     const cpx<R>* __restrict__ Fd, const cpx<R>* __restrict__ FVr, const int* __restrict__ tab,
                     int nout, long N) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < N; e += (long)gridDim.x * blockDim.x) {
    cpx<R> fd[NAB];
#pragma unroll
    for (int ab = 0; ab < NAB; ++ab) {
      fd[ab] = Fd[ab * N + e];
      Gn[ab * N + e] = Fr[ab * N + e] + fd[ab];
    }
    for (int o = 0; o < nout; ++o) {
      const int* t = tab + o * NAB;
      cpx<R> acc(0, 0);
#pragma unroll
      for (int ab = 0; ab < NAB; ++ab) acc += FVr[(long)t[ab] * N + e] * fd[ab];
      Y[(long)o * N + e] = acc;
    }
  }
}

template <typename R>
void sigma_ref_contract(cpx<R>* Y, cpx<R>* Gn, const cpx<R>* Fr, const cpx<R>* Fd, const cpx<R>* FVr,
                        const int* tab, int nout, int No, long N, hipStream_t s) {
  const unsigned grid = (unsigned)std::min<long>((N + 255) / 256, 256L * 32);
  switch (No) {
    case 1: hipLaunchKernelGGL((k_sigma_ref_contract<R, 1>), dim3(grid), dim3(256), 0, s, Y, Gn, Fr, Fd, FVr, tab, nout, N); break;
    case 2: hipLaunchKernelGGL((k_sigma_ref_contract<R, 4>), dim3(grid), dim3(256), 0, s, Y, Gn, Fr, Fd, FVr, tab, nout, N); break;
    case 3: hipLaunchKernelGGL((k_sigma_ref_contract<R, 9>), dim3(grid), dim3(256), 0, s, Y, Gn, Fr, Fd, FVr, tab, nout, N); break;
    case 4: hipLaunchKernelGGL((k_sigma_ref_contract<R, 16>), dim3(grid), dim3(256), 0, s, Y, Gn, Fr, Fd, FVr, tab, nout, N); break;
    default: throw Error("sigma_ref_contract: Norb > 4");
  }
  GMOD_CHECK_LAUNCH();
}

// One thread per spatial point and a stride of slots: the reversed point of
// a thread is fixed, so its loads run along the grid (descending) as the
// direct ones do.  The orbital-pair grids stay in registers across outputs.
template <typename R, int NAB>
__global__ void __launch_bounds__(256)
k_sigma_inc_contract(cpx<R>* __restrict__ out, const cpx<R>* __restrict__ Fr, const cpx<R>* __restrict__ Fd,
                     const cpx<R>* __restrict__ FVr, const cpx<R>* __restrict__ DVt,
                     const cpx<R>* __restrict__ dhF, const cpx<R>* __restrict__ dhD, const int* __restrict__ tab,
                     int nout, unsigned S, unsigned M, const int* __restrict__ rev) {
  const unsigned sp = blockIdx.x * blockDim.x + threadIdx.x;
  if (sp >= S) return;
  const long N = (long)S * M;
  const unsigned rs = (unsigned)rev[sp];
  for (unsigned t = blockIdx.y; t < M; t += gridDim.y) {
    const long e = sp + (long)S * t, er = rs + (long)S * t;
    cpx<R> fd[NAB], gn[NAB];
#pragma unroll
    for (int ab = 0; ab < NAB; ++ab) {
      fd[ab] = Fd[ab * N + e];
      gn[ab] = Fr[ab * N + e] + fd[ab];
    }
    for (int o = 0; o < nout; ++o) {
      const int* tb = tab + 2 * o * NAB;
      cpx<R> acc(0, 0);
#pragma unroll
      for (int ab = 0; ab < NAB; ++ab) {
        const int ef = tb[2 * ab], ed = tb[2 * ab + 1];
        cpx<R> fv = FVr[(long)(ef >> 1) * N + ((ef & 1) ? er : e)];
        cpx<R> dv = DVt[(long)(ed >> 1) * N + ((ed & 1) ? er : e)];
        if (ef & 1) fv = conj(fv) + dhF[(long)(ef >> 1) * S + sp];
        if (ed & 1) dv = conj(dv) + dhD[(long)(ed >> 1) * S + sp];
        acc += fv * fd[ab] + dv * gn[ab];
      }
      out[(long)o * N + e] = acc;
    }
  }
}

template <typename R>
void sigma_inc_contract(cpx<R>* out, const cpx<R>* Fr, const cpx<R>* Fd, const cpx<R>* FVr, const cpx<R>* DVt,
                        const cpx<R>* dhF, const cpx<R>* dhD, const int* tab, int nout, int No, unsigned S,
                        unsigned M, const int* rev, hipStream_t s) {
  const unsigned gx = (S + 255) / 256;
  const unsigned gy = (unsigned)std::max<long>(1, std::min<long>(M, (256L * 32 + gx - 1) / gx));
  const dim3 g(gx, gy);
  switch (No) {
    case 1: hipLaunchKernelGGL((k_sigma_inc_contract<R, 1>), g, dim3(256), 0, s, out, Fr, Fd, FVr, DVt, dhF, dhD, tab, nout, S, M, rev); break;
    case 2: hipLaunchKernelGGL((k_sigma_inc_contract<R, 4>), g, dim3(256), 0, s, out, Fr, Fd, FVr, DVt, dhF, dhD, tab, nout, S, M, rev); break;
    case 3: hipLaunchKernelGGL((k_sigma_inc_contract<R, 9>), g, dim3(256), 0, s, out, Fr, Fd, FVr, DVt, dhF, dhD, tab, nout, S, M, rev); break;
    case 4: hipLaunchKernelGGL((k_sigma_inc_contract<R, 16>), g, dim3(256), 0, s, out, Fr, Fd, FVr, DVt, dhF, dhD, tab, nout, S, M, rev); break;
    default: throw Error("sigma_inc_contract: Norb > 4");
  }
  GMOD_CHECK_LAUNCH();
}

// ------------------------------------------------------------------ instantiations
#define INST(R) \
  template void mul_acc<R>(cpx<R>*, const cpx<R>*, const cpx<R>*, bool, long, hipStream_t); \
  template void contract<R>(cpx<R>*, const cpx<R>*, const cpx<R>*, const int*, const int*, const int*, int, long, \
                            bool, hipStream_t); \
  template void sigma_ref_contract<R>(cpx<R>*, cpx<R>*, const cpx<R>*, const cpx<R>*, const cpx<R>*, const int*, int, \
                                      int, long, hipStream_t); \
  template void sigma_inc_contract<R>(cpx<R>*, const cpx<R>*, const cpx<R>*, const cpx<R>*, const cpx<R>*, \
                                      const cpx<R>*, const cpx<R>*, const int*, int, int, unsigned, unsigned, const int*, \
                                      hipStream_t);
INST(double)
INST(float)

}  // namespace gmod
