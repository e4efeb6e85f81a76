// Matter power spectrum of the resident particles on the fine mesh
// (utilities/cicpower.f90:85-257 density, utilities/powerspectrum.f90:27-137
// estimator).
//
// Density: CIC of every particle on the nf^3 fine mesh.  cicpower puts the
// nodes at cell centres (pos-0.5) while the PM density has them at cell left
// edges; the two differ by a uniform half-cell shift, which changes only
// the phase of each Fourier mode, so |delta_k|^2 is the same.  delta =
// rho/mean - 1 and the forward transform is divided by nf^3
// (powerspectrum.f90:40-46).  Modes: the half space kx >= 0 with the
// conjugate duplicates on the kx = 0 and kx = nf/2 planes skipped as in
// powerspectrum.f90:63-66; signed frequencies mod(i+nyq-1,ng)-nyq; linear
// bins nint(|k|) with |k| in real(4) as the reference computes it;
// Delta^2 = |delta_k|^2 / sinc^4 * 4 pi |k|^3 with the CIC window
// sinc = prod_d sin(pi k_d/ng)/(pi k_d/ng).
#include "cube_internal.hpp"
#include <math.h>
#include <algorithm>
#include <mutex>
#include <vector>

#define PK_NT 256
#define PK_MAXBIN 2048

// One wavefront per (ky, kz) row, PK_U consecutive kx a lane and pass.  The
// window factors sin(x)/x come from a table in LDS (N/2+1 of them instead of
// three sines per mode), row and plane are uniform, and a lane adds its
// modes to the bin sums only where the bin changes: neighbouring modes share
// bins, and one atomic per mode met on the same addresses.  65 M modes
// (512^3 mesh) take 0.29 instead of 1.04 ms.
#define PK_U 4
template <typename T>
__global__ __launch_bounds__(PK_NT) void k_pk_bin(const cpx<T>* __restrict__ c, int N, double inv_norm, int nbin, double* bins) {
  extern __shared__ double win[];  // N/2+1 window factors, then 3 (nbin+1) bin sums
  const int H = N / 2 + 1, nyq = N / 2;
  double* const sb = win + H;
  for (int i = threadIdx.x; i < 3 * (nbin + 1); i += PK_NT) sb[i] = 0;
  for (int i = threadIdx.x; i < H; i += PK_NT) {
    const double x = M_PI * (double)i / (double)N;
    win[i] = i ? sin(x) / x : 1.0;
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int row = blockIdx.x * (PK_NT / 64) + wv; row < N * N; row += gridDim.x * (PK_NT / 64)) {
    const int ky = row % N, kz = row / N;
    const int qy = ky < nyq ? ky : ky - N, qz = kz < nyq ? kz : kz - N;
    // on the kx = 0 and nyq planes the conjugate duplicates are skipped
    const bool dup = ky > nyq || ((ky == 0 || ky == nyq) && kz > nyq);
    const int q2 = qy * qy + qz * qz;
    const double wy = win[abs(qy)], wz = win[abs(qz)];
    const cpx<T>* src = c + (int64_t)row * H;
    for (int k0 = 0; k0 < H; k0 += 64 * PK_U) {
      cpx<T> v[PK_U];
#pragma unroll
      for (int u = 0; u < PK_U; u++) {
        const int kx = k0 + lane * PK_U + u;
        v[u] = kx < H ? src[kx] : cpx<T>{0, 0};
      }
      int bin = -1;
      double sk = 0, sa = 0, sn = 0;
#pragma unroll
      for (int u = 0; u < PK_U; u++) {
        const int kx = k0 + lane * PK_U + u;
        bool ok = kx < H && !((kx == 0 || kx == nyq) && dup) && (kx | q2) != 0;
        const int qx = kx < nyq ? kx : kx - N;
        const float kr = sqrtf((float)(qx * qx + q2));
        const int ib = (int)floorf(kr + 0.5f);
        ok = ok && ib <= nbin;
        if (ok) {
          if (ib != bin) {
            if (bin >= 0) {
              atomicAdd(&sb[3 * bin], sn);
              atomicAdd(&sb[3 * bin + 1], sk);
              atomicAdd(&sb[3 * bin + 2], sa);
            }
            bin = ib;
            sk = sa = sn = 0;
          }
          const double sinc = win[abs(qx)] * wy * wz;
          const double re = (double)v[u].x * inv_norm, im = (double)v[u].y * inv_norm;
          const double s2 = sinc * sinc;
          sa += (re * re + im * im) / (s2 * s2) * 4.0 * M_PI * (double)kr * (double)kr * (double)kr;
          sk += (double)kr;
          sn += 1.0;
        }
      }
      if (bin >= 0) {
        atomicAdd(&sb[3 * bin], sn);
        atomicAdd(&sb[3 * bin + 1], sk);
        atomicAdd(&sb[3 * bin + 2], sa);
      }
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 3 * (nbin + 1); i += PK_NT)
    if (sb[i] != 0) atomicAdd(&bins[i], sb[i]);
}

// Scratch of cube_power_spectrum_noalloc: the per-bin partial sums (mode
// count, sum of |k|, sum of Delta^2 for bins 0..PK_MAXBIN), 48 KiB.  Every
// GPU the library runs on holds its own copy until the process ends.  In
// host code `scratch` only names the symbol; its device address on each
// GPU comes from hipGetSymbolAddress at cube_init (pk_scratch_setup).
static __device__ __align__(256) double scratch[3 * (PK_MAXBIN + 1)];
#define PK_MAX_DEVICES 64
static std::mutex g_scratch_mu;
static double* g_scratch_ptr[PK_MAX_DEVICES];

int pk_scratch_setup(cube_handle* h) {
  const int dev = h->p.device;
  if (dev < 0 || dev >= PK_MAX_DEVICES) return cube_fail(h, CUBE_ERR_ARG, "device %d outside [0, %d)", dev, PK_MAX_DEVICES);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (g_scratch_ptr[dev]) return 0;
  void* ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess || !ptr)
    return cube_fail(h, CUBE_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
  g_scratch_ptr[dev] = (double*)ptr;
  return 0;
}

__global__ void k_pk_zero(double* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0;
}

// Shared body of both entry points: argument checks, CIC density, R2C,
// binning into `bins` (3 doubles per bin 0..nbin, cleared here by a fill
// kernel), and bins 1..nbin into the caller's arrays.
static int pk_run(cube_handle* h, int nbin, double* modes, double* ksum, double* d2sum, double* bins) {
  const int64_t N = h->fine.N;
  const int want = (int)lrint((double)(N / 2) * sqrt(3.0));
  if (nbin != want)
    return cube_fail(h, CUBE_ERR_ARG, "nbin=%d; the linear binning of a %lld^3 mesh has nint(nyquist*sqrt(3))=%d bins", nbin,
                     (long long)N, want);
  if (nbin > PK_MAXBIN) return cube_fail(h, CUBE_ERR_ARG, "nbin=%d above %d", nbin, PK_MAXBIN);
  double mass = 0;
  int r = cic_fine(h, &mass);
  if (r) return r;
  if ((r = mesh_fft3_r2c(h, h->fine))) return r;
  const int nv = 3 * (nbin + 1);
  k_pk_zero<<<(nv + PK_NT - 1) / PK_NT, PK_NT, 0, h->stream>>>(bins, nv);
  HIP_TRY(h, hipGetLastError());
  const double mean = mass / ((double)N * N * N);
  const double inv_norm = 1.0 / ((double)N * N * N * mean);
  // a workgroup clears and folds its LDS bins once, so there are no more of
  // them than fill the GPU
  const unsigned grid = (unsigned)std::min<int64_t>((N * N + PK_NT / 64 - 1) / (PK_NT / 64), 2048);
  const size_t lds = sizeof(double) * (N / 2 + 1 + nv);
  if (h->prec == 4)
    k_pk_bin<float><<<grid, PK_NT, lds, h->stream>>>((const cpx<float>*)h->fine.R, (int)N, inv_norm, nbin, bins);
  else
    k_pk_bin<double><<<grid, PK_NT, lds, h->stream>>>((const cpx<double>*)h->fine.R, (int)N, inv_norm, nbin, bins);
  HIP_TRY(h, hipGetLastError());
  // one copy of all bins (a strided copy per field moves its rows one by
  // one: 9 ms at 443 bins).  The reference reports bins 1..nbin (xip=xi(:,1:));
  // field f of bin b is bins[3b+f].
  std::vector<double> hb(nv);
  HIP_TRY(h, hipMemcpyAsync(hb.data(), bins, sizeof(double) * nv, hipMemcpyDeviceToHost, h->stream));
  HIP_TRY(h, hipStreamSynchronize(h->stream));
  double* dst[3] = {modes, ksum, d2sum};
  for (int f = 0; f < 3; f++)
    for (int b = 1; b <= nbin; b++) dst[f][b - 1] = hb[3 * b + f];
  return CUBE_OK;
}

extern "C" int cube_power_spectrum(cube_handle* h, int nbin, double* modes, double* ksum, double* d2sum) {
  CUBE_EXCLUSIVE;
  if (!h || !modes || !ksum || !d2sum) return CUBE_ERR_ARG;
  if (hipSetDevice(h->p.device) != hipSuccess) return cube_fail(h, CUBE_ERR_HIP, "hipSetDevice failed");
  if (nbin < 1 || nbin > PK_MAXBIN) return cube_fail(h, CUBE_ERR_ARG, "nbin=%d outside [1, %d]", nbin, PK_MAXBIN);
  double* bins = nullptr;
  HIP_TRY(h, hipMalloc(&bins, sizeof(double) * 3 * (nbin + 1)));
  const int r = pk_run(h, nbin, modes, ksum, d2sum, bins);
  (void)hipStreamSynchronize(h->stream);
  (void)hipFree(bins);
  return r;
}

// The same estimator without any device allocation: the partial sums live
// in this file's static `scratch` array (at most PK_MAXBIN bins).  All calls
// on one GPU share that array, so calls that overlap on one GPU (several
// host threads, or handles on different streams) race; the bins are
// cleared at the start of every call.
extern "C" int cube_power_spectrum_noalloc(cube_handle* h, int nbin, double* modes, double* ksum, double* d2sum) {
  if (!h || !modes || !ksum || !d2sum) return CUBE_ERR_ARG;
  if (hipSetDevice(h->p.device) != hipSuccess) return cube_fail(h, CUBE_ERR_HIP, "hipSetDevice failed");
  if (nbin < 1 || nbin > PK_MAXBIN)
    return cube_fail(h, CUBE_ERR_ARG, "nbin=%d outside [1, %d] (the allocation-free scratch holds %d bins)", nbin,
                     PK_MAXBIN, PK_MAXBIN);
  double* bins = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    const int dev = h->p.device;
    if (dev >= 0 && dev < PK_MAX_DEVICES) bins = g_scratch_ptr[dev];
  }
  if (!bins) return cube_fail(h, CUBE_ERR_ARG, "no scratch address for device %d (cube_init sets it)", h->p.device);
  return pk_run(h, nbin, modes, ksum, d2sum, bins);
}
