// gfx950 engine of the elastic FWI operator: the time-step kernels, the plan
// (device-resident model, data and wavefields of one parameter file) and the
// job runner that drives one plan, or several plans on different grids,
// through one set of launches per time step.
//
// Device data layout (all FP32, z fastest so a wave64 row is 64 consecutive
// depth cells, one 256-byte coalesced access):
//   model      lam, mu, ave_mu, byc_a, byc_b          [NX][NZ]
//   wavefield  vz, vx, szz, sxx, sxz                  [shot][component][NX][NZ]
//   adjoint    same 5 components                      [shot][component][NX][NZ]
//   C-PML memory variables (8)                        [shot][variable][NX][NZ]
//   boundary ring, 5 layers x 4 sides, 5 components   [shot][step][component][ring slot]
//   seismograms syn/obs/res, time-major               [nSteps][all receivers]
//   gradient accumulators (5, summed over shots)      [NX][NZ]
//   exact adjoint only: transposed-update operands    [launch shot][slot][NX][NZ]
//
// Two adjoints: the reference's (el_velocity_adj / el_stress_adj, the default)
// and the exact one, the transpose of the forward step (a plan option, no
// reference counterpart; k_exact_a / k_exact_b).
//
// Arithmetic.  Every wavefield update evaluates the reference's expression in
// the reference's order and types, so that the fields follow its FP32
// arithmetic rather than a re-association of it:
//   * a stencil difference is DIVIDED by dz or dx, correctly rounded:
//     q = x*y + (x - d*(x*y))*y with y = RN(1/d), one Newton correction on a
//     correctly rounded reciprocal, which equals IEEE x/d for every normal x
//     when d passes the exhaustive check at plan creation (check_spacing);
//     C-PML K divisions take two corrections;
//   * the reference's double literals promote exactly where its source says
//     (2.0*mu, RSXXZZ*..., MEGA), so those terms are evaluated in FP64 and
//     rounded once to FP32 on assignment, as C++ does;
//   * no multiply-add contraction anywhere in this file.
// Gradient accumulators are the one place that sums in another order: the
// contributions of a launch's shots are added up first, in shot order, and the
// chain rule to (lambda, mu, rho) is applied once at the end.
//
// Reference kernels restated here: el_stress.cu:50-131, el_velocity.cu:45-117,
// el_velocity_adj.cu:22-108, el_stress_adj.cu:22-104, utilities.cu:125-205,
// 361-424, 506-593, 653-747; driver sequence libCUFD.cu:157-463.
#include <hip/hip_ext.h>
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "cond.hpp"
#include "engine.hpp"

#pragma clang fp contract(off)

// Device memory of the allocation-free entry point (fwiflow_cufd_noalloc):
// every buffer of such a call is carved out of this array, which each GPU
// the library runs on holds from module load to process end.  Host code
// never passes the array's name to a kernel or a copy (on the host it is a
// stand-in, not a device address): it uses the address that
// hipGetSymbolAddress returned for the current device (scratch_device).
static __device__ __align__(256) unsigned char scratch[FWIFLOW_SCRATCH_BYTES];

namespace fwiflow {

#define HIP_TRY(expr)                                                                    \
  do {                                                                                   \
    hipError_t e_ = (expr);                                                              \
    if (e_ != hipSuccess)                                                                \
      return Status::Err(FWIFLOW_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

#define TRY(expr)            \
  do {                       \
    Status s_ = (expr);      \
    if (!s_.ok()) return s_; \
  } while (0)

// 16-byte raw buffer load (the LLVM AMDGPU intrinsic, bound by name)
typedef float f4 __attribute__((ext_vector_type(4)));
__device__ f4 raw_load4(__amdgpu_buffer_rsrc_t r, int vo, int so, int aux) __asm(
    "llvm.amdgcn.raw.ptr.buffer.load.v4f32");

namespace {

constexpr int kBZ = 64;            // threads along z (one wave64 row)
constexpr int kCondBlocks = 512;   // misfit partial sums per shot of the conditioned residual
constexpr int kPartials = 1024;    // misfit partial sums of one residual launch
// el_stress.cu:42-43: float c1 = 9.0/8.0, c2 = 1.0/24.0
constexpr float kC1 = (float)(9.0 / 8.0);
constexpr float kC2 = (float)(1.0 / 24.0);
// add_source (utilities.cu:528): float scale = pow(1500.0, 2)
constexpr float kSrcScale = 2250000.0f;
// RSXXZZ (utilities.h:21) is the double literal 3.0
constexpr double kRS = 3.0;

// ------------------------------------------------------------ arithmetic
// x / d for d with the correctly rounded reciprocal y: one Newton correction
// (exact for every normal x when check_spacing(d) holds).
__device__ __forceinline__ float div1(float x, float d, float y) {
  const float q = x * y;
  return __builtin_fmaf(__builtin_fmaf(-d, q, x), y, q);
}
// two corrections: correctly rounded for any normal divisor (the first makes
// q faithful, the second rounds it)
__device__ __forceinline__ float div2(float x, float d, float y) {
  float q = x * y;
  q = __builtin_fmaf(__builtin_fmaf(-d, q, x), y, q);
  return __builtin_fmaf(__builtin_fmaf(-d, q, x), y, q);
}
__device__ __forceinline__ double ddiv2(double x, double d, double y) {
  double q = x * y;
  q = __builtin_fma(__builtin_fma(-d, q, x), y, q);
  return __builtin_fma(__builtin_fma(-d, q, x), y, q);
}

// ------------------------------------------------------------ descriptors
struct Geo {
  int nz, nx, nzA, nPml, nSteps;
  int ns;          // shots of this part in the launch
  int s0;          // plan index of its first shot
  long long N;     // cells per shot
  float dt, dz, dx, rdz, rdx;
  int ringW, ringH, ringlen;
  int R;           // receivers of the plan: row length of the time-major seismograms
  int rs0;         // ring: index of the part's first shot in the ring buffer
  int rnt;         // ring: steps held
};

struct Mdl {
  const float *lam, *mu, *amu, *ba, *bb;
};

// Wavefield arrays are [shot][component][cell]: the 5 components of a state
// (vz, vx, szz, sxx, sxz) and the 8 C-PML memory variables, named after the
// reference's d_mem_* arrays.
enum WaveComp { kVz = 0, kVx = 1, kSzz = 2, kSxx = 3, kSxz = 4, kWaveComps = 5 };
enum MemComp {
  kMvzz = 0,   // mem_dvz_dz
  kMvzx = 1,   // mem_dvz_dx
  kMvxz = 2,   // mem_dvx_dz
  kMvxx = 3,   // mem_dvx_dx
  kMszz = 4,   // mem_dszz_dz
  kMsxx = 5,   // mem_dsxx_dx
  kMsxzz = 6,  // mem_dsxz_dz
  kMsxzx = 7,  // mem_dsxz_dx
  kMemComps = 8
};

// Boundary ring (Boundary.cu:17-41, utilities.cu:361-424): rows and columns
// nPml-2 .. nPml+2 on each side of the interior, i.e. the band of width 5 of
// the rectangle [nPml-2, nzA-nPml+1] x [nPml-2, nx-nPml+1].  Slot numbering is
// this engine's own: top band [W][5], bottom band [W][5], left band [5][H-10],
// right band [5][H-10], z fastest inside each so a wave writes contiguously.
__host__ __device__ inline int ring_slot(int z, int x, const Geo& g) {
  const int zr = z - (g.nPml - 2), xr = x - (g.nPml - 2);
  const int H = g.ringH, W = g.ringW;
  if (zr < 0 || zr >= H || xr < 0 || xr >= W) return -1;
  if (zr < 5) return xr * 5 + zr;
  if (zr >= H - 5) return 5 * W + xr * 5 + (zr - (H - 5));
  const int hz = H - 10, zc = zr - 5;
  if (xr < 5) return 10 * W + xr * hz + zc;
  if (xr >= W - 5) return 10 * W + 5 * hz + (xr - (W - 5)) * hz + zc;
  return -1;
}

// Ring layout [ring shot][held step][component][slot], components szz, sxz,
// sxx, vz, vx.  The ring holds rnt consecutive steps: step it is row it % rnt
// (all steps of the sweep when rnt = nSteps - 1, one checkpoint segment
// otherwise).

// Stencil loads and stores go through buffer resources: one scalar resource
// per field of a part, the shot's byte offset in an SGPR (soffset) and the
// cell's per-lane byte offset in a VGPR, z neighbours in one 16-byte load.  A wave's addresses then cost no per-lane 64-bit arithmetic.
using Rsrc = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ Rsrc rsrc(const float* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), (short)0, (int)0xffffffff,
                                           0x00020000);
}
__device__ __forceinline__ float ldb(Rsrc r, int so, int vo) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, vo, so, 0));
}
// Column of the calling thread in a tile whose first column is x0.  A
// workgroup is 64 threads deep, so each wave64 is one column: the column
// is wave-uniform, and the x-direction C-PML coefficients and x branches it
// selects are scalar.
__device__ __forceinline__ int wave_col(int x0) {
  return __builtin_amdgcn_readfirstlane(x0 + (int)threadIdx.y);
}

// Staggered 4th-order differences as the reference writes them:
// forward / reverse (c1 (a - b) - c2 (c - d)) / h, adjoint (-c1 (a - b) + c2 (c - d)) / h.
__device__ __forceinline__ float dfw(float a, float b, float c, float d, float h, float rh) {
  return div1(kC1 * (a - b) - kC2 * (c - d), h, rh);
}
__device__ __forceinline__ float dad(float a, float b, float c, float d, float h, float rh) {
  return div1(-kC1 * (a - b) + kC2 * (c - d), h, rh);
}

#include "step_kernels.hpp"

// res_injection (utilities.cu:569-580) for surveys whose receivers are not one
// per cell in one row: one thread per injection cell adds its receivers'
// residuals in receiver order (szz_adj += res, sxx_adj += RSXXZZ res), the
// order in which the reference's per-receiver += lands on a shared cell when
// its threads run in index order.  cells[c] = (plan shot, z, x); receivers
// of cell c are rid[ptr[c] .. ptr[c+1]).
__global__ void k_res_inject(Geo g, float* __restrict__ adj, const int* __restrict__ cells,
                             const int* __restrict__ ptr, const int* __restrict__ rid, int c0,
                             int ncells, const float* __restrict__ row) {
  const int c = c0 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
  if (c >= c0 + ncells) return;
  float* a = adj + (size_t)cells[3 * c] * kWaveComps * g.N + (long long)cells[3 * c + 2] * g.nz +
             cells[3 * c + 1];
  float szz = a[kSzz * g.N], sxx = a[kSxx * g.N];
  for (int j = ptr[c]; j < ptr[c + 1]; ++j) {
    const float v = row[rid[j]];
    szz = szz + v;
    sxx = (float)((double)sxx + kRS * (double)v);
  }
  a[kSzz * g.N] = szz;
  a[kSxx * g.N] = sxx;
}

// Residual (libCUFD.cu:258-313 without the optional filters) over receivers
// [r0, r0 + nr) of the plan: window obs and syn with w^2, res = obs_w - syn_w
// (first sample 0, gpuMinus utilities.cu:154-167), sum res^2
// (cuda_cal_objective, here in FP64), then window res again.
__global__ __launch_bounds__(256) void k_residual(int nSteps, int R, int r0, int nr,
                                                  const float* __restrict__ w2,
                                                  const float* __restrict__ obs,
                                                  const float* __restrict__ syn,
                                                  float* __restrict__ res,
                                                  double* __restrict__ partial) {
  __shared__ double red[256];
  const size_t total = (size_t)nSteps * nr;
  double acc = 0.0;
  for (size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x; k < total;
       k += (size_t)gridDim.x * blockDim.x) {
    const int t = (int)(k / (size_t)nr);
    const size_t j = (size_t)t * R + r0 + (k - (size_t)t * nr);
    const float ww = w2[t];
    // obs and syn are windowed separately (two roundings, as the reference's
    // separate cuda_window launches do)
    const float ow = obs[j] * ww;
    const float sw = syn[j] * ww;
    const float rv = t > 0 ? ow - sw : 0.f;
    acc += (double)rv * (double)rv;
    res[j] = rv * ww;
  }
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}

__global__ void k_sum_partials(const double* __restrict__ partial, int n, double* out) {
  __shared__ double red[256];
  double acc = 0.0;
  for (int k = threadIdx.x; k < n; k += blockDim.x) acc += partial[k];
  red[threadIdx.x] = acc;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] += red[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

// Chain rule from the accumulated derivatives to (lambda, mu, rho), once per
// run.  Deterministic gather form of the reference's atomicAdd sprays
// (el_stress.cu:113-124, el_velocity.cu:104-112), with the same target
// conditions (including the always-true `gidx+1<=gidx<=nx-1-nPml`).  With
// `exact` (the exact adjoint) every cell of a harmonic or arithmetic average
// receives its share: the conditions that drop the last interior row and
// column's neighbours are not applied.
__global__ __launch_bounds__(256) void k_finalize(Geo g, Mdl m, const float* __restrict__ acc,
                                                  float* __restrict__ grad, int exact) {
  const int z = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int x = (int)blockIdx.y;
  if (z >= g.nz) return;
  const int nz = g.nz;
  const long long N = g.N;
  const float* acc_l = acc;
  const float* acc_m = acc + N;
  const float* acc_s = acc + 2 * N;
  const float* acc_a = acc + 3 * N;
  const float* acc_b = acc + 4 * N;
  const int z0 = g.nPml, z1 = g.nzA - 1 - g.nPml, x0 = g.nPml, x1 = g.nx - 1 - g.nPml;
  auto inI = [&](int zz, int xx) { return zz >= z0 && zz <= z1 && xx >= x0 && xx <= x1; };
  const long long i = (long long)x * nz + z;
  const float dt = g.dt;
  float gl = 0.f, gm = 0.f, gd = 0.f;
  if (inI(z, x)) {
    gl = -acc_l[i] * dt * 1.0e6f;
    gm = -2.f * acc_m[i] * dt * 1.0e6f;
  }
  auto shear = [&](int zz, int xx) -> float {
    const long long j = (long long)xx * nz + zz;
    const float am = m.amu[j];
    if (am == 0.f) return 0.f;
    const float S = 1.f / m.mu[j] + 1.f / m.mu[j + 1] + 1.f / m.mu[j + nz] + 1.f / m.mu[j + nz + 1];
    return -acc_s[j] * dt * am / S * 1.0e6f;
  };
  float t = 0.f;
  bool any = false;
  if (inI(z, x) && m.amu[i] != 0.f) t += shear(z, x), any = true;
  const bool zc = exact || z <= z1, xc = exact || x <= x1;
  if (inI(z - 1, x) && zc && m.amu[i - 1] != 0.f) t += shear(z - 1, x), any = true;
  if (inI(z, x - 1) && m.amu[i - nz] != 0.f) t += shear(z, x - 1), any = true;
  if (inI(z - 1, x - 1) && zc && xc && m.amu[i - nz - 1] != 0.f)
    t += shear(z - 1, x - 1), any = true;
  if (any) {
    const float mu = m.mu[i];
    gm += t / (mu * mu);
  }
  auto ga = [&](long long j) { const float b = m.ba[j]; return acc_a[j] * dt * (0.5f * b * b); };
  auto gb = [&](long long j) { const float b = m.bb[j]; return acc_b[j] * dt * (0.5f * b * b); };
  if (inI(z, x)) gd += ga(i) + gb(i);
  if (inI(z - 1, x) && zc) gd += ga(i - 1);
  if (inI(z, x - 1)) gd += gb(i - nz);
  grad[i] = gl;
  grad[N + i] = gm;
  grad[2 * N + i] = gd;
}

// aveMuInit / aveBycInit (utilities.cu:125-152) over [2, nz-3] x [2, nx-3];
// defaults 0 and 1/1000 elsewhere (Model.cu:67-73).
__global__ void k_model_init(Geo g, const float* __restrict__ mu, const float* __restrict__ den,
                             float* __restrict__ amu, float* __restrict__ ba,
                             float* __restrict__ bb) {
  const int z = (int)(blockIdx.x * blockDim.x + threadIdx.x);
  const int x = (int)blockIdx.y;
  if (z >= g.nz) return;
  const int nz = g.nz;
  const long long i = (long long)x * nz + z;
  float am = 0.f, fa = 1.f / 1000.f, fb = 1.f / 1000.f;
  if (z >= 2 && z <= g.nz - 3 && x >= 2 && x <= g.nx - 3) {
    const float A = mu[i], B = mu[i + 1], C = mu[i + nz], D = mu[i + nz + 1];
    if (A == 0.f || B == 0.f || C == 0.f || D == 0.f)
      am = 0.f;
    else
      am = (float)(4.0 / (1.0 / A + 1.0 / B + 1.0 / C + 1.0 / D));
    fa = (float)(2.0 / (double)(den[i + 1] + den[i]));
    fb = (float)(2.0 / (double)(den[i + nz] + den[i]));
  }
  amu[i] = am;
  ba[i] = fa;
  bb[i] = fb;
}

// [rows][cols] -> [cols][rows] through LDS tiles.
__global__ void k_transpose(const float* __restrict__ in, float* __restrict__ out, int rows,
                            int cols) {
  __shared__ float tile[32][33];
  const int c = blockIdx.x * 32 + threadIdx.x;
  const int r0 = blockIdx.y * 32;
  for (int k = threadIdx.y; k < 32; k += blockDim.y) {
    const int r = r0 + k;
    if (r < rows && c < cols) tile[k][threadIdx.x] = in[(size_t)r * cols + c];
  }
  __syncthreads();
  const int r = r0 + threadIdx.x;
  for (int k = threadIdx.y; k < 32; k += blockDim.y) {
    const int cc = blockIdx.x * 32 + k;
    if (r < rows && cc < cols) out[(size_t)cc * rows + r] = tile[threadIdx.x][k];
  }
}

// Model arrays in and gradients out: in [rows][cols] -> out [cols][rows], one
// array per blockIdx.z, in another type.  `scaled`: the first arrays in units of
// 1e6 (the caller's moduli are in MPa).
// Host arrays cross the bus as the caller has them and are turned here (TF's
// row-major [NZ][NX] to z-fastest, libCUFD.cu:72-78, and back, 480-486): the
// host's strided passes were bound by their cache misses.  A model of 608x1780
// 6.4 -> 0.8 ms, of 364x964 1.7 -> 0.3; gradients of the latter 1.3 -> 0.7.
struct Turn {
  const void* in[3];
  void* out[3];
};
template <typename TI, typename TO>
__global__ __launch_bounds__(256) void k_turn(Turn t, int rows, int cols, int scaled) {
  __shared__ TI tile[32][33];
  const TI* in = (const TI*)t.in[blockIdx.z];
  TO* out = (TO*)t.out[blockIdx.z];
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  for (int k = threadIdx.y; k < 32; k += 8)
    if (r0 + k < rows && c0 + (int)threadIdx.x < cols)
      tile[k][threadIdx.x] = in[(size_t)(r0 + k) * cols + c0 + threadIdx.x];
  __syncthreads();
  for (int k = threadIdx.y; k < 32; k += 8)
    if (c0 + k < cols && r0 + (int)threadIdx.x < rows) {
      const TI v = tile[threadIdx.x][k];
      out[(size_t)(c0 + k) * rows + r0 + threadIdx.x] = (int)blockIdx.z < scaled ? (TO)(v * 1e6) : (TO)v;
    }
}

// Largest Vp as velInit computes it (utilities.cu:119-121), one partial per
// workgroup; NaNs are passed over (the host looks at the first cell's itself).
__global__ __launch_bounds__(256) void k_vp_max(const double* __restrict__ lam, const double* __restrict__ mu,
                                                const double* __restrict__ den, size_t n,
                                                float* __restrict__ part) {
  __shared__ float red[256];
  float m = -1.f;  // below every square root
  for (size_t k = (size_t)blockIdx.x * 256 + threadIdx.x; k < n; k += (size_t)gridDim.x * 256) {
    const float l = (float)(lam[k] * 1e6), u = (float)(mu[k] * 1e6), d = (float)den[k];
    const float cp = (float)sqrt((l + 2.0 * u) / d);
    if (cp > m) m = cp;
  }
  red[threadIdx.x] = m;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) red[threadIdx.x] = fmaxf(red[threadIdx.x], red[threadIdx.x + s]);
    __syncthreads();
  }
  if (threadIdx.x == 0) part[blockIdx.x] = red[0];
}

}  // namespace

// ===================================================================== host
namespace {

int env_int(const char* name, int dflt) {
  const char* v = std::getenv(name);
  return v && *v ? std::atoi(v) : dflt;
}

// div1(x, d, RN(1/d)) == x / d for every normal x: checked over every
// mantissa of the binades [1, 2) and [2, 4) (the computation scales exactly
// with the exponent of x).  Cached per spacing; about 30 ms per new value.
bool spacing_ok(float d) {
  static std::mutex mu;
  static std::map<float, bool> seen;
  {
    std::lock_guard<std::mutex> lk(mu);
    auto it = seen.find(d);
    if (it != seen.end()) return it->second;
  }
  const float y = 1.0f / d;
  bool ok = std::isnormal(d) && std::isnormal(y);
  for (unsigned e = 127; e <= 128 && ok; ++e)
    for (unsigned m = 0; m < (1u << 23); ++m) {
      const unsigned u = e << 23 | m;
      float x;
      std::memcpy(&x, &u, 4);
      const float q = x * y;
      const float v = std::fma(std::fma(-d, q, x), y, q);
      if (v != x / d) {
        ok = false;
        break;
      }
    }
  std::lock_guard<std::mutex> lk(mu);
  seen[d] = ok;
  return ok;
}

}  // namespace

// A launch bracketed by timing events.
struct TimedLaunch {
  std::string name;
  hipEvent_t a, b;
  bool pooled = true;  // events go back to the pool (not those of a captured graph)
};

// A shot group's time loop captured as a graph, and its timed launches.
struct GraphEntry {
  hipGraphExec_t exec = nullptr;
  std::vector<TimedLaunch> recs;
};

// Bump allocator over a fixed device region (the scratch array of the
// allocation-free entry point): 256-byte aligned pieces, never returned
// before the region is dropped as a whole.
struct Arena {
  char* base = nullptr;
  size_t cap = 0, used = 0;
  Status take(void** p, size_t nb) {
    const size_t at = (used + 255) & ~(size_t)255;
    const size_t n = nb ? nb : 4;
    if (at > cap || n > cap - at)
      return Status::Err(FWIFLOW_ERR_MEMORY,
                         "device scratch exhausted: " + std::to_string(n) + " more bytes needed, " +
                             std::to_string(at) + " of the " + std::to_string(cap) +
                             " scratch bytes (FWIFLOW_SCRATCH_BYTES) in use");
    *p = base + at;
    used = at + n;
    return Status::Ok();
  }
  size_t free_bytes() const {
    const size_t at = (used + 255) & ~(size_t)255;
    return at < cap ? cap - at : 0;
  }
};

// Device-resident argument tables and captured time loops of a job, kept
// across runs.
struct JobCache {
  int dev = 0;
  Arena* arena = nullptr;  // device memory comes from here instead of hipMalloc when set
  StepArgs* steps = nullptr;  // forward and backward launch arguments of the last run
  BackArgs* backs = nullptr;
  size_t steps_cap = 0, backs_cap = 0;
  std::map<std::string, GraphEntry> graphs;
  ~JobCache() {
    (void)hipSetDevice(dev);
    clear_graphs();
    if (arena) return;
    if (steps) (void)hipFree(steps);
    if (backs) (void)hipFree(backs);
  }
  void clear_graphs() {
    for (auto& kv : graphs) {
      (void)hipGraphExecDestroy(kv.second.exec);
      for (auto& r : kv.second.recs) {
        (void)hipEventDestroy(r.a);
        (void)hipEventDestroy(r.b);
      }
    }
    graphs.clear();
  }
  template <typename T>
  Status reserve(size_t n, T*& dev_ptr, size_t& cap) {
    if (n <= cap) return Status::Ok();
    if (dev_ptr && !arena) HIP_TRY(hipFree(dev_ptr));
    dev_ptr = nullptr;
    cap = 0;
    if (arena)
      TRY(arena->take((void**)&dev_ptr, n * sizeof(T)));
    else
      HIP_TRY(hipMalloc((void**)&dev_ptr, n * sizeof(T)));
    cap = n;
    return Status::Ok();
  }
  template <typename T>
  Status upload(const std::vector<T>& a, T*& dev_ptr, size_t& cap) {
    TRY(reserve(a.size(), dev_ptr, cap));
    if (!a.empty()) HIP_TRY(hipMemcpy(dev_ptr, a.data(), a.size() * sizeof(T), hipMemcpyHostToDevice));
    return Status::Ok();
  }
};

// ===================================================================== device state
struct DeviceState {
  int dev = 0;
  hipStream_t stream = nullptr;
  Geo g{};  // whole plan: ns = plan shots, s0 = 0
  int R = 0;
  std::vector<int> roff;  // first receiver of each shot (+ total)
  // engine settings (environment variables read at plan creation)
  int tile_x = 4;          // columns of a half step's tile (blockDim.y) where chosen
  bool tile_auto = true;   // not chosen (tile_x is 4 then: such plans and those
                           // with 4 chosen may share a job)
  int shot_group = -1;     // shots per forward launch (0: all, -1: automatic)
  int shot_group_bwd = -1; // shots per backward launch (0: all, -1: automatic)
  bool fold_inject = true; // residual injection inside the adjoint stress update
  bool graphs = false;     // shot groups' time loops captured and replayed as graphs
                           // (measured no faster at 608x1780; timed runs stay eager)
  int ckpt_every = 0;      // 0: boundary ring every step; k > 0: checkpoints every k steps
  int adjoint = 0;         // 0: the reference's adjoint; 1: the exact adjoint
  double limit = 0;        // device bytes that the plan may hold (0: what the GPU has)
  double ring_budget = 32e9;  // device bytes a gradient run may hold for ring + checkpoints
  // model + tables
  float *lam = nullptr, *mu = nullptr, *den = nullptr, *amu = nullptr, *ba = nullptr,
        *bb = nullptr;
  // C-PML coefficients by row, then by column: K, 1/K, a, b and the half-cell
  // K, 1/K, a, b; and 1/K in double
  float* pmlc = nullptr;
  double* pml64 = nullptr;
  float* win2 = nullptr;  // nSteps
  int* src = nullptr;     // [ns][2]
  float* srcamp = nullptr;  // [ns][nSteps] windowed source rows
  float* srcwin = nullptr;  // [nSteps] the source rows' window (exact adjoint's stf gradient)
  int* rec = nullptr;     // [R][3] (z, x, plan shot)
  // residual injection: cells with their receivers (in receiver order), and by
  // shot and column
  int *icell = nullptr, *iptr = nullptr, *irid = nullptr;
  std::vector<int> coff;  // first injection cell of each shot (+ total)
  std::vector<int> icells, iptrs, irids;  // host copies until a gradient run needs them
  ColInj* inj = nullptr;
  bool inj_folded = false;  // the adjoint kernels inject (else k_res_inject does)
  // wavefields
  float *fwd = nullptr, *mem = nullptr, *adj = nullptr, *madj = nullptr;
  float* ring = nullptr;
  size_t ring_floats = 0;
  // second state of the whole-step launches, for the shots of one launch
  float *fwd2 = nullptr, *mem2 = nullptr, *adj2 = nullptr, *madj2 = nullptr;
  int shots2 = 0, mshots2 = 0, ashots2 = 0, xshots2 = 0;  // shots of each
  float* xt = nullptr;  // exact adjoint: operands [backward group shot][8][cell]
  size_t xt_floats = 0;
  float* snap = nullptr;
  size_t snap_floats = 0;
  float *syn = nullptr, *obs = nullptr, *res = nullptr, *stage = nullptr;
  float *acc = nullptr, *grad = nullptr, *stf_grad = nullptr, *illum = nullptr;
  double* partial = nullptr;
  int npartial = 0;
  double* misfit = nullptr;
  bool model_set = false, stf_set = false, obs_set = false;
  bool illum_on = false, illum_valid = false;
  double misfit_host = 0.0;
  // residual conditioning, shot by shot
  bool cond = false;
  FftDesc fft{};
  int* fperm = nullptr;
  float2* ftw = nullptr;
  float2* bpH = nullptr;
  float* wpad = nullptr;
  float *wst = nullptr, *wen = nullptr, *wwt = nullptr;
  float *cobs = nullptr, *csyn = nullptr;
  float2 *spo = nullptr, *spc = nullptr;
  float2* coef = nullptr;
  float* srcout = nullptr;
  double* cpart = nullptr;
  int nrec_max = 0;
  bool src_updated = false;
  std::vector<float> keep_obs, keep_syn;
  // last gradient run's memory plan and shot groups
  int last_k = 0, last_rows_sg = 0, last_groups_f = 0, last_groups_b = 0;
  int last_tile = 0;  // columns of the last run's half-step tiles (0: whole steps only)
  long long last_ring_bytes = 0, last_snap_bytes = 0;
  std::unique_ptr<JobCache> cache;  // maps of this plan's own runs
  std::vector<void*> allocs;
  long long bytes = 0;
  // allocation-free plans: buffers carved from the device scratch array, the
  // stream shared by all such plans of the device
  Arena arena_store;
  Arena* arena = nullptr;
  bool own_stream = true;
  // timing
  bool timing = false;
  using Rec = TimedLaunch;
  std::vector<Rec>* sink = nullptr;  // while a graph is captured: its sampled launches
  std::vector<Rec> pending;
  std::vector<hipEvent_t> pool;
  std::map<std::string, std::pair<double, long long>> totals;

  ~DeviceState() {
    if (stream) (void)hipSetDevice(dev);
    cache.reset();
    for (auto& r : pending) {
      if (!r.pooled) continue;  // owned by a captured graph
      (void)hipEventDestroy(r.a);
      (void)hipEventDestroy(r.b);
    }
    for (auto e : pool) (void)hipEventDestroy(e);
    for (void* p : allocs) (void)hipFree(p);
    if (stream && own_stream) (void)hipStreamDestroy(stream);
  }

  // The second states give way to every other buffer of the plan: none of its
  // runs is under way when it asks for one (a run allocates them last).
  template <typename T>
  Status alloc(T** p, size_t count) {
    Status s = take(p, count);
    if (s.code == FWIFLOW_ERR_MEMORY && drop_second()) s = take(p, count);
    return s;
  }
  bool drop_second() {
    if (!fwd2 && !mem2 && !adj2 && !madj2) return false;
    (void)hipGetLastError();
    const size_t N = (size_t)g.N;
    release(fwd2, (size_t)shots2 * kWaveComps * N);
    release(mem2, (size_t)mshots2 * kMemComps * N);
    release(adj2, (size_t)ashots2 * kWaveComps * N);
    release(madj2, (size_t)xshots2 * kMemComps * N);
    shots2 = mshots2 = ashots2 = xshots2 = 0;
    return true;
  }
  template <typename T>
  Status take(T** p, size_t count) {
    void* q = nullptr;
    const size_t nb = count * sizeof(T);
    if (arena) {
      TRY(arena->take(&q, nb));
      bytes += (long long)nb;
      *p = (T*)q;
      return Status::Ok();
    }
    if (limit > 0 && (double)bytes + (double)nb > limit)
      return Status::Err(FWIFLOW_ERR_MEMORY, std::to_string(nb) + " more bytes are over FWIFLOW_PLAN_BYTES, " +
                                                 std::to_string(bytes) + " in use");
    hipError_t e = hipMalloc(&q, nb ? nb : 4);
    if (e != hipSuccess)
      return Status::Err(e == hipErrorOutOfMemory ? FWIFLOW_ERR_MEMORY : FWIFLOW_ERR_HIP,
                         "hipMalloc(" + std::to_string(nb) + " bytes): " + hipGetErrorString(e));
    allocs.push_back(q);
    bytes += (long long)nb;
    *p = (T*)q;
    return Status::Ok();
  }
  template <typename T>
  void release(T*& p, size_t count) {
    if (!p) return;
    if (arena) {  // arena pieces are dropped with the plan
      bytes -= (long long)(count * sizeof(T));
      p = nullptr;
      return;
    }
    auto it = std::find(allocs.begin(), allocs.end(), (void*)p);
    if (it != allocs.end()) allocs.erase(it);
    (void)hipFree(p);
    bytes -= (long long)(count * sizeof(T));
    p = nullptr;
  }

  hipEvent_t take_event() {
    if (!pool.empty()) {
      hipEvent_t e = pool.back();
      pool.pop_back();
      return e;
    }
    hipEvent_t e = nullptr;
    (void)hipEventCreate(&e);
    return e;
  }
  // a sampled step launch passes these to hipExtLaunchKernel, which stamps
  // them when the kernel itself starts and ends (no launch gap inside)
  hipEvent_t kernel_start = nullptr, kernel_end = nullptr;
  template <typename F>
  void launch(const char* name, bool sample, F&& f) {
    if (timing && sample && !sink) {
      Rec r{name, take_event(), take_event(), true};
      kernel_start = r.a;
      kernel_end = r.b;
      f();
      kernel_start = kernel_end = nullptr;
      pending.push_back(r);
    } else if (timing && sample) {
      Rec r{name, take_event(), take_event(), false};
      (void)hipEventRecord(r.a, stream);
      f();
      (void)hipEventRecord(r.b, stream);
      sink->push_back(r);
    } else {
      f();
    }
  }
  void collect_timing() {
    for (auto& r : pending) {
      float ms = 0.f;
      (void)hipEventSynchronize(r.b);
      (void)hipEventElapsedTime(&ms, r.a, r.b);
      auto& t = totals[r.name];
      t.first += ms;
      t.second += 1;
      if (r.pooled) {
        pool.push_back(r.a);
        pool.push_back(r.b);
      }
    }
    pending.clear();
  }

  Mdl mdl() const { return Mdl{lam, mu, amu, ba, bb}; }
  size_t F() const { return (size_t)g.ns * g.N; }
  // first cell of shot s0 in a [shot][comps][cell] array
  float* shot(float* base, int comps, int s0) const { return base + (size_t)s0 * comps * g.N; }
  // ~40 B per cell and shot of forward state stay cache-resident from step to
  // step; the backward holds forward and adjoint state (~64 B), and the exact
  // adjoint its two operand sets besides (+32 B).  224 MB of the 256 MB
  // Infinity Cache for them (measured at 608x1780: 5 shots per forward
  // launch, 3 per backward launch; 2 for the exact adjoint, 4.87
  // shot-gradients/s against 4.37 with 3).
  double fwd_bytes_per_shot() const { return 40.0 * (double)g.N; }
  double bwd_bytes_per_shot() const { return (adjoint ? 96.0 : 64.0) * (double)g.N; }
  size_t ring_step_floats() const { return (size_t)5 * g.ringlen; }
  size_t snap_floats_per_shot() const { return (size_t)13 * g.N; }
  // zero shots [s0, s0+n) of a [shot][comps][cell] array
  // on stream st (the stream of the run, which may be another plan's)
  Status zero_shots(float* base, int comps, int s0, int n, hipStream_t st) {
    HIP_TRY(hipMemsetAsync(shot(base, comps, s0), 0, (size_t)n * comps * g.N * sizeof(float), st));
    return Status::Ok();
  }
};

// Address of the scratch array on each device and the stream of the
// allocation-free plans there, looked up once per device with that device
// current and kept until the process ends.
namespace {

struct ScratchDevice {
  bool ready = false;
  char* ptr = nullptr;
  hipStream_t stream = nullptr;
};
std::mutex g_scratch_mu;
std::vector<ScratchDevice> g_scratch_dev;

Status scratch_device(int dev, char** base, hipStream_t* stream) {
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if ((int)g_scratch_dev.size() <= dev) g_scratch_dev.resize(dev + 1);
  ScratchDevice& sd = g_scratch_dev[dev];
  if (!sd.ready) {
    HIP_TRY(hipSetDevice(dev));
    void* ptr = nullptr;
    HIP_TRY(hipGetSymbolAddress((void**)&ptr, HIP_SYMBOL(scratch)));
    HIP_TRY(hipStreamCreate(&sd.stream));
    sd.ptr = (char*)ptr;
    sd.ready = true;
  }
  *base = sd.ptr;
  *stream = sd.stream;
  return Status::Ok();
}

}  // namespace

Plan::Plan() = default;
Plan::~Plan() = default;

Status Plan::create(const std::string& para_fname, int gpu, int group_size, const int* shot_ids,
                    bool in_scratch) {
  TRY(parse_para(para_fname, para));
  TRY(parse_survey(para, group_size, shot_ids, survey));
  gpu_id = gpu;
  if (!spacing_ok(para.dz) || !spacing_ok(para.dx))
    return Status::Err(FWIFLOW_ERR_UNSUPPORTED,
                       "grid spacing: the reciprocal division of the stencils is not correctly "
                       "rounded for dz = " + std::to_string(para.dz) + " or dx = " +
                           std::to_string(para.dx));
  int ndev = 0;
  HIP_TRY(hipGetDeviceCount(&ndev));
  if (gpu < 0 || gpu >= ndev)
    return Status::Err(FWIFLOW_ERR_HIP, "gpu_id " + std::to_string(gpu) + " not present (" +
                                            std::to_string(ndev) + " devices)");
  d_.reset(new DeviceState());
  DeviceState& d = *d_;
  d.dev = gpu;
  d.tile_auto = !std::getenv("FWIFLOW_TILE_X");
  d.tile_x = std::max(1, std::min(4, env_int("FWIFLOW_TILE_X", 4)));  // <= 256 threads
  d.shot_group = std::max(-1, env_int("FWIFLOW_SHOT_GROUP", -1));
  d.shot_group_bwd = std::max(-1, env_int("FWIFLOW_SHOT_GROUP_BWD", -1));
  d.fold_inject = env_int("FWIFLOW_FOLD_INJECT", 1) != 0;
  d.graphs = env_int("FWIFLOW_GRAPHS", 0) != 0;
  d.adjoint = env_int("FWIFLOW_EXACT_ADJOINT", 0) != 0 ? 1 : 0;
  if (const char* v = std::getenv("FWIFLOW_PLAN_BYTES")) d.limit = std::atof(v);
  if (in_scratch) {
    // every buffer from the device's scratch array, no graphs (instantiating
    // one allocates), the device's shared stream
    char* base = nullptr;
    TRY(scratch_device(gpu, &base, &d.stream));
    d.own_stream = false;
    d.arena_store.base = base;
    d.arena_store.cap = FWIFLOW_SCRATCH_BYTES;
    d.arena = &d.arena_store;
    d.graphs = false;
  }
  HIP_TRY(hipSetDevice(gpu));
  if (!d.stream) HIP_TRY(hipStreamCreate(&d.stream));
  Geo& g = d.g;
  g.nz = para.nz;
  g.nx = para.nx;
  g.nzA = para.nzA();
  g.nPml = para.nPml;
  g.ns = group_size;
  g.s0 = 0;
  g.nSteps = para.nSteps;
  g.N = (long long)para.nz * para.nx;
  g.dt = para.dt;
  g.dz = para.dz;
  g.dx = para.dx;
  g.rdz = 1.f / para.dz;
  g.rdx = 1.f / para.dx;
  g.ringH = g.nzA - 2 * g.nPml + 4;
  g.ringW = g.nx - 2 * g.nPml + 4;
  g.ringlen = 10 * g.ringW + 10 * (g.ringH - 10);
  d.R = survey.total_rec();
  g.R = d.R;
  g.rs0 = 0;
  g.rnt = std::max(1, g.nSteps - 1);

  const size_t N = (size_t)g.N;
  // one array [lam, mu, amu, ba, bb, den][NX][NZ]: one base address in the kernels
  TRY(d.alloc(&d.lam, 6 * N));
  d.mu = d.lam + N, d.amu = d.lam + 2 * N, d.ba = d.lam + 3 * N, d.bb = d.lam + 4 * N;
  d.den = d.lam + 5 * N;
  {
    std::vector<float> tab(6 * ((size_t)g.nzA + g.nx)), c(8 * ((size_t)g.nzA + g.nx));
    std::vector<double> c64((size_t)g.nzA + g.nx);
    cpml_profiles(g.nzA, g.nPml, para.dz, para.f0, para.dt, tab.data());
    cpml_profiles(g.nx, g.nPml, para.dx, para.f0, para.dt, tab.data() + 6 * g.nzA);
    float* o = c.data();
    double* o64 = c64.data();
    for (int axis = 0; axis < 2; axis++) {
      const int n = axis ? g.nx : g.nzA;
      const float* p = tab.data() + (axis ? 6 * (size_t)g.nzA : 0);
      for (int i = 0; i < n; i++) {
        for (int h = 0; h < 2; h++, o += 4) {
          const float* q = p + 3 * (size_t)h * n + i;
          o[0] = q[0], o[1] = 1.f / q[0], o[2] = q[n], o[3] = q[2 * (size_t)n];
        }
        *o64++ = 1.0 / (double)p[i];
      }
    }
    TRY(d.alloc(&d.pmlc, c.size()));
    TRY(d.alloc(&d.pml64, c64.size()));
    HIP_TRY(hipMemcpy(d.pmlc, c.data(), c.size() * sizeof(float), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(d.pml64, c64.data(), c64.size() * sizeof(double), hipMemcpyHostToDevice));
  }
  std::vector<float> w2(g.nSteps);
  window_squared(g.nSteps, para.dt, 0.005f, w2.data());
  TRY(d.alloc(&d.win2, w2.size()));
  HIP_TRY(hipMemcpy(d.win2, w2.data(), w2.size() * sizeof(float), hipMemcpyHostToDevice));
  // the source rows' window (Src_Rec.cu:132-143): d(source amplitude)/d(stf)
  window_squared(g.nSteps, para.dt, 0.001f, w2.data());
  TRY(d.alloc(&d.srcwin, w2.size()));
  HIP_TRY(hipMemcpy(d.srcwin, w2.data(), w2.size() * sizeof(float), hipMemcpyHostToDevice));
  std::vector<int> src(2 * g.ns), rec(3 * (size_t)d.R);
  size_t r = 0;
  d.roff.assign(g.ns + 1, 0);
  for (int s = 0; s < g.ns; s++) {
    const Shot& sh = survey.shots[s];
    d.roff[s] = (int)r;
    src[2 * s] = sh.z_src;
    src[2 * s + 1] = sh.x_src;
    for (size_t k = 0; k < sh.z_rec.size(); k++, r++) {
      rec[3 * r] = sh.z_rec[k];
      rec[3 * r + 1] = sh.x_rec[k];
      rec[3 * r + 2] = s;
    }
  }
  d.roff[g.ns] = (int)r;
  {
    // injection cells of each shot, receivers of a cell in receiver order.  The
    // adjoint kernels inject where every receiver lies in the update region,
    // and for one-row surveys with one receiver per cell also where some do
    // not (those are then left out).
    bool one_row = d.R > 0, inside = true;
    d.iptrs.push_back(0);
    d.coff.assign(g.ns + 1, 0);
    for (int s = 0; s < g.ns; s++) {
      d.coff[s] = (int)d.icells.size() / 3;
      std::map<std::pair<int, int>, std::vector<int>> by;  // (x, z) -> receivers
      for (int k = d.roff[s]; k < d.roff[s + 1]; k++)
        by[{rec[3 * k + 1], rec[3 * k]}].push_back(k);
      for (auto& kv : by) {
        const int z = kv.first.second, x = kv.first.first;
        one_row = one_row && z == rec[0] && kv.second.size() == 1;
        inside = inside && z >= 2 && z <= g.nzA - 3 && x >= 2 && x <= g.nx - 3;
        d.icells.insert(d.icells.end(), {s, z, x});
        d.irids.insert(d.irids.end(), kv.second.begin(), kv.second.end());
        d.iptrs.push_back((int)d.irids.size());
      }
    }
    d.coff[g.ns] = (int)d.icells.size() / 3;
    d.inj_folded = d.fold_inject && (one_row || inside);
  }
  TRY(d.alloc(&d.src, src.size()));
  HIP_TRY(hipMemcpy(d.src, src.data(), src.size() * sizeof(int), hipMemcpyHostToDevice));
  TRY(d.alloc(&d.rec, std::max<size_t>(3, rec.size())));
  if (!rec.empty())
    HIP_TRY(hipMemcpy(d.rec, rec.data(), rec.size() * sizeof(int), hipMemcpyHostToDevice));
  TRY(d.alloc(&d.srcamp, (size_t)g.ns * g.nSteps));
  const size_t F = (size_t)g.ns * N;
  TRY(d.alloc(&d.fwd, 5 * F));
  TRY(d.alloc(&d.mem, 8 * F));
  d.cond = para.conditioned() || para.save_scratch;
  if (d.cond) {
    const int nt = g.nSteps, L = 2 * nt;
    for (int s = 0; s < g.ns; s++) d.nrec_max = std::max(d.nrec_max, d.roff[s + 1] - d.roff[s]);
    TRY(d.alloc(&d.cobs, (size_t)nt * d.nrec_max));
    TRY(d.alloc(&d.csyn, (size_t)nt * d.nrec_max));
    TRY(d.alloc(&d.cpart, (size_t)g.ns * kCondBlocks));
    if (para.if_win) {
      std::vector<float> a, b, c;
      for (const Shot& sh : survey.shots) {
        a.insert(a.end(), sh.win_start.begin(), sh.win_start.end());
        b.insert(b.end(), sh.win_end.begin(), sh.win_end.end());
        c.insert(c.end(), sh.weights.begin(), sh.weights.end());
      }
      TRY(d.alloc(&d.wst, a.size()));
      TRY(d.alloc(&d.wen, b.size()));
      TRY(d.alloc(&d.wwt, c.size()));
      HIP_TRY(hipMemcpy(d.wst, a.data(), a.size() * sizeof(float), hipMemcpyHostToDevice));
      HIP_TRY(hipMemcpy(d.wen, b.data(), b.size() * sizeof(float), hipMemcpyHostToDevice));
      HIP_TRY(hipMemcpy(d.wwt, c.data(), c.size() * sizeof(float), hipMemcpyHostToDevice));
    }
    if (para.if_filter || para.if_src_update) {
      std::vector<int> perm;
      std::vector<float2> tw;
      TRY(fft_plan(L, d.fft, perm, tw));
      TRY(d.alloc(&d.fperm, perm.size()));
      TRY(d.alloc(&d.ftw, tw.size()));
      HIP_TRY(hipMemcpy(d.fperm, perm.data(), perm.size() * sizeof(int), hipMemcpyHostToDevice));
      HIP_TRY(hipMemcpy(d.ftw, tw.data(), tw.size() * sizeof(float2), hipMemcpyHostToDevice));
    }
    if (para.if_filter) {
      std::vector<float2> H;
      bandpass_table(nt, para.dt, para.filter, H);
      TRY(d.alloc(&d.bpH, H.size()));
      HIP_TRY(hipMemcpy(d.bpH, H.data(), H.size() * sizeof(float2), hipMemcpyHostToDevice));
    }
    if (para.if_src_update) {
      std::vector<float> wp(L);
      window_squared(L, para.dt, 0.01f, wp.data());
      TRY(d.alloc(&d.wpad, wp.size()));
      HIP_TRY(hipMemcpy(d.wpad, wp.data(), wp.size() * sizeof(float), hipMemcpyHostToDevice));
      TRY(d.alloc(&d.spo, (size_t)d.nrec_max * (nt + 1)));
      TRY(d.alloc(&d.spc, (size_t)d.nrec_max * (nt + 1)));
      TRY(d.alloc(&d.coef, (size_t)nt + 1));
      TRY(d.alloc(&d.srcout, (size_t)g.ns * nt));
    }
  }
  TRY(d.alloc(&d.syn, std::max<size_t>(1, (size_t)g.nSteps * d.R)));
  TRY(d.alloc(&d.misfit, 1));
  return Status::Ok();
}

// injection tables, on the first gradient run
static Status ensure_injection(DeviceState& d) {
  if (d.inj) return Status::Ok();
  std::vector<ColInj> col((size_t)d.g.ns * d.g.nx, ColInj{0, 0, 0, -1});
  if (d.inj_folded)
    for (int c = 0; c < (int)d.icells.size() / 3; c++) {
      ColInj& q = col[(size_t)d.icells[3 * c] * d.g.nx + d.icells[3 * c + 2]];
      if (!q.n++) {
        q.first = c, q.z = d.icells[3 * c + 1];
        q.rid = d.iptrs[c + 1] - d.iptrs[c] == 1 ? d.irids[d.iptrs[c]] : -1;
      } else {
        q.rid = -1;
      }
    }
  auto put = [&](auto*& p, const auto& v) -> Status {
    if (!p) TRY(d.alloc(&p, std::max<size_t>(1, v.size())));
    if (!v.empty()) HIP_TRY(hipMemcpy(p, v.data(), v.size() * sizeof(v[0]), hipMemcpyHostToDevice));
    return Status::Ok();
  };
  TRY(put(d.icell, d.icells));
  TRY(put(d.iptr, d.iptrs));
  TRY(put(d.irid, d.irids));
  return put(d.inj, col);
}

Status Plan::set_model(const double* Lambda, const double* Mu, const double* Den, bool zfast) {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  if (!Lambda || !Mu || !Den) return Status::Err(FWIFLOW_ERR_ARG, "null model pointer");
  DeviceState& d = *d_;
  HIP_TRY(hipSetDevice(d.dev));
  // staged in the forward memory variables (32 bytes a cell; every run clears them)
  const size_t n = (size_t)d.g.N;
  double* const in = (double*)d.mem;
  const double* host[3] = {Lambda, Mu, Den};
  for (int k = 0; k < 3; k++)
    HIP_TRY(hipMemcpyAsync(in + k * n, host[k], n * sizeof(double), hipMemcpyHostToDevice, d.stream));
  const int blocks = (int)std::max<size_t>(1, std::min<size_t>(512, n / 512));
  float* const part = (float*)(in + 3 * n);
  hipLaunchKernelGGL(k_vp_max, dim3(blocks), dim3(256), 0, d.stream, in, in + n, in + 2 * n, n, part);
  HIP_TRY(hipGetLastError());
  std::vector<float> top(blocks);
  HIP_TRY(hipMemcpyAsync(top.data(), part, blocks * sizeof(float), hipMemcpyDeviceToHost, d.stream));
  HIP_TRY(hipStreamSynchronize(d.stream));
  const float first = (float)std::sqrt(((float)(Lambda[0] * 1e6) + 2.0 * (float)(Mu[0] * 1e6)) / (float)Den[0]);
  cp_max = std::isnan(first) ? first : *std::max_element(top.begin(), top.end());
  TRY(check_courant(para, cp_max));
  const dim3 blk(32, 8);
  const Turn t{{in, in + n, in + 2 * n}, {d.lam, d.mu, d.den}};
  const int rows = zfast ? 1 : d.g.nz, cols = zfast ? (int)n : d.g.nx;
  hipLaunchKernelGGL((k_turn<double, float>), dim3((cols + 31) / 32, (rows + 31) / 32, 3), blk, 0, d.stream, t,
                     rows, cols, 2);
  hipLaunchKernelGGL(k_model_init, dim3((d.g.nz + 255) / 256, d.g.nx), dim3(256), 0, d.stream,
                     d.g, d.mu, d.den, d.amu, d.ba, d.bb);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(d.stream));
  d.model_set = true;
  return Status::Ok();
}

Status Plan::set_stf(const double* stf) {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  if (!stf) return Status::Err(FWIFLOW_ERR_ARG, "null stf pointer");
  DeviceState& d = *d_;
  const int nSteps = d.g.nSteps;
  // Src_Rec.cu:132-143: row shot_id -> float -> window ratio 0.001
  std::vector<float> w2(nSteps), amps((size_t)d.g.ns * nSteps);
  window_squared(nSteps, para.dt, 0.001f, w2.data());
  for (int s = 0; s < d.g.ns; s++) {
    const double* row = stf + (size_t)survey.shots[s].id * nSteps;
    for (int it = 0; it < nSteps; it++) amps[(size_t)s * nSteps + it] = (float)row[it] * w2[it];
  }
  HIP_TRY(hipSetDevice(d.dev));
  HIP_TRY(hipMemcpy(d.srcamp, amps.data(), amps.size() * sizeof(float), hipMemcpyHostToDevice));
  d.stf_set = true;
  return Status::Ok();
}

static Status ensure_obs_buffers(DeviceState& d) {
  const size_t T = std::max<size_t>(1, (size_t)d.g.nSteps * d.R);
  if (!d.obs) TRY(d.alloc(&d.obs, T));
  if (!d.res) TRY(d.alloc(&d.res, T));
  if (!d.stage) TRY(d.alloc(&d.stage, T));
  return Status::Ok();
}

Status Plan::set_obs(const float* obs) {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  if (!obs) return Status::Err(FWIFLOW_ERR_ARG, "null obs pointer");
  DeviceState& d = *d_;
  HIP_TRY(hipSetDevice(d.dev));
  TRY(ensure_obs_buffers(d));
  const size_t T = (size_t)d.g.nSteps * d.R;
  // host [R][nSteps] (concatenated Shot files) -> device time-major [nSteps][R]
  HIP_TRY(hipMemcpyAsync(d.stage, obs, T * sizeof(float), hipMemcpyHostToDevice, d.stream));
  dim3 blk(32, 8), grd((d.g.nSteps + 31) / 32, (d.R + 31) / 32);
  hipLaunchKernelGGL(k_transpose, grd, blk, 0, d.stream, d.stage, d.obs, d.R, d.g.nSteps);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(d.stream));
  d.obs_set = true;
  return Status::Ok();
}

Status Plan::load_obs() {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  const int nSteps = para.nSteps;
  std::vector<float> host((size_t)nSteps * d_->R);
  size_t off = 0;
  for (const Shot& sh : survey.shots) {
    const std::string fn = para.data_dir + "/Shot" + std::to_string(sh.id) + ".bin";
    FILE* fp = std::fopen(fn.c_str(), "rb");
    if (!fp) return Status::Err(FWIFLOW_ERR_IO, "cannot open \"" + fn + "\"");
    const size_t n = sh.z_rec.size() * (size_t)nSteps;
    const size_t got = std::fread(host.data() + off, sizeof(float), n, fp);
    std::fclose(fp);
    if (got != n)
      return Status::Err(FWIFLOW_ERR_IO, "\"" + fn + "\" holds " + std::to_string(got) +
                                             " floats, expected " + std::to_string(n));
    off += n;
  }
  return set_obs(host.data());
}

Status Plan::set_checkpoint(int k) {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  if (k < 0) return Status::Err(FWIFLOW_ERR_ARG, "checkpoint interval must be >= 0");
  d_->ckpt_every = k;
  return Status::Ok();
}

Status Plan::set_adjoint(int mode) {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  if (mode != 0 && mode != 1) return Status::Err(FWIFLOW_ERR_ARG, "adjoint mode must be 0 or 1");
  d_->adjoint = mode;
  return Status::Ok();
}

int Plan::adjoint() const { return d_ ? d_->adjoint : 0; }

Status Plan::set_memory_budget(double bytes) {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  if (!(bytes > 0)) return Status::Err(FWIFLOW_ERR_ARG, "memory budget must be positive");
  d_->ring_budget = bytes;
  return Status::Ok();
}

Status Plan::set_launch(int tile_x, int shots_fwd, int shots_bwd) {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  if (tile_x != -1 && (tile_x < 1 || tile_x > 4))
    return Status::Err(FWIFLOW_ERR_ARG, "tile width must be 1..4, or -1 (automatic)");
  if (shots_fwd < -1 || shots_bwd < -1)
    return Status::Err(FWIFLOW_ERR_ARG, "shots per launch must be >= -1");
  d_->tile_auto = tile_x == -1;
  d_->tile_x = tile_x == -1 ? 4 : tile_x;
  d_->shot_group = shots_fwd;
  d_->shot_group_bwd = shots_bwd;
  if (d_->cache) d_->cache->clear_graphs();  // captured loops bake the old shape in
  return Status::Ok();
}

Status Plan::launch(int* tile_x, int* shots_fwd, int* shots_bwd) const {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  if (tile_x) *tile_x = d_->tile_auto ? -1 : d_->tile_x;
  if (shots_fwd) *shots_fwd = d_->shot_group;
  if (shots_bwd) *shots_bwd = d_->shot_group_bwd;
  return Status::Ok();
}

Status Plan::memory_plan(int* k, int* shots_per_sweep, long long* ring_bytes,
                         long long* checkpoint_bytes) const {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  if (k) *k = d_->last_k;
  if (shots_per_sweep) *shots_per_sweep = d_->last_rows_sg;
  if (ring_bytes) *ring_bytes = d_->last_ring_bytes;
  if (checkpoint_bytes) *checkpoint_bytes = d_->last_snap_bytes;
  return Status::Ok();
}

Status Plan::set_timing(bool on) {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  d_->timing = on;
  d_->totals.clear();
  return Status::Ok();
}

Status Plan::timing(const std::string& name, double* ms, long long* count) {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  auto it = d_->totals.find(name);
  if (ms) *ms = it == d_->totals.end() ? 0.0 : it->second.first;
  if (count) *count = it == d_->totals.end() ? 0 : it->second.second;
  return Status::Ok();
}

long long Plan::device_bytes() const { return d_ ? d_->bytes : 0; }

int Plan::shots_per_launch() const {
  if (!d_) return 0;
  return d_->last_groups_f > 0 ? (d_->g.ns + d_->last_groups_f - 1) / d_->last_groups_f : 0;
}
int Plan::shots_per_launch_bwd() const {
  if (!d_) return 0;
  return d_->last_groups_b > 0 ? (d_->g.ns + d_->last_groups_b - 1) / d_->last_groups_b : 0;
}
int Plan::tile_width() const { return d_ ? d_->last_tile : 0; }
int Plan::launch_groups(int backward) const {
  if (!d_) return 0;
  return backward ? d_->last_groups_b : d_->last_groups_f;
}

// Residual with the optional conditioning stages for shots [sb, se), one shot
// at a time (libCUFD.cu:254-313): window obs and syn (per-trace windows and
// weights, or the default ratio-0.005 window), band-pass both, source update
// (syn and the source row replaced), res = obs - syn and its misfit, then the
// adjoint stages on res: source-update filter, band-pass, window (ratio 0.1
// with per-trace windows).  `keep` copies the conditioned obs and syn to the
// host for the scratch files.
static Status condition_residual(DeviceState& d, const Para& para, bool keep, int sb, int se,
                                 hipStream_t st) {
  const Geo& g = d.g;
  const int nt = g.nSteps, nf = nt + 1, kc = touched_bins(nt);
  const float scale = 1.0f / (float)(2 * nt);
  const float dt = para.dt;
  if (keep && d.keep_obs.size() != (size_t)d.R * nt) {
    d.keep_obs.assign((size_t)d.R * nt, 0.f);
    d.keep_syn.assign((size_t)d.R * nt, 0.f);
  }
  std::vector<float> h;
  for (int s = sb; s < se; s++) {
    const int r0 = d.roff[s], n = d.roff[s + 1] - r0;
    const float* ws = para.if_win ? d.wst + r0 : nullptr;
    const float* we = para.if_win ? d.wen + r0 : nullptr;
    const float* wt = para.if_win ? d.wwt + r0 : nullptr;
    const TraceSet O{d.cobs, n, d.cobs, n, n}, Y{d.csyn, n, d.csyn, n, n};
    const TraceSet Rs{d.res + r0, d.R, d.res + r0, d.R, n};
    HIP_TRY(window_traces(st, nt, TraceSet{d.obs + r0, d.R, d.cobs, n, n}, d.win2, ws, we, wt,
                          0.005f, dt));
    HIP_TRY(window_traces(st, nt, TraceSet{d.syn + r0, d.R, d.csyn, n, n}, d.win2, ws, we, wt,
                          0.005f, dt));
    if (para.if_filter) {
      HIP_TRY(trace_filter(st, d.fft, d.fperm, d.ftw, nt, O, nullptr, d.bpH, kc, scale));
      HIP_TRY(trace_filter(st, d.fft, d.fperm, d.ftw, nt, Y, nullptr, d.bpH, kc, scale));
    }
    if (para.if_src_update) {
      HIP_TRY(trace_spectra(st, d.fft, d.fperm, d.ftw, nt, O, d.wpad, d.spo));
      HIP_TRY(trace_spectra(st, d.fft, d.fperm, d.ftw, nt, Y, d.wpad, d.spc));
      HIP_TRY(spectrum_ratio(st, d.spo, d.spc, n, nf, d.coef));
      HIP_TRY(trace_filter(st, d.fft, d.fperm, d.ftw, nt, Y, d.wpad, d.coef, nf, scale));
      const size_t so = (size_t)s * nt;
      HIP_TRY(trace_filter(st, d.fft, d.fperm, d.ftw, nt,
                           TraceSet{d.srcamp + so, 1, d.srcout + so, 1, 1}, nullptr, d.coef, nf,
                           scale));
    }
    HIP_TRY(shot_residual(st, nt, n, d.cobs, d.csyn, n, d.res + r0, d.R,
                          d.cpart + (size_t)s * kCondBlocks, kCondBlocks));
    if (para.if_src_update)
      HIP_TRY(trace_filter(st, d.fft, d.fperm, d.ftw, nt, Rs, d.wpad, d.coef, kc, scale));
    if (para.if_filter)
      HIP_TRY(trace_filter(st, d.fft, d.fperm, d.ftw, nt, Rs, nullptr, d.bpH, kc, scale));
    HIP_TRY(window_traces(st, nt, Rs, d.win2, ws, we, wt, 0.1f, dt));
    if (keep) {
      // [nSteps][n] -> [n][nSteps] (the Shot file layout)
      h.resize((size_t)nt * n);
      for (int q = 0; q < 2; q++) {
        HIP_TRY(hipMemcpyAsync(h.data(), q ? d.csyn : d.cobs, h.size() * sizeof(float),
                               hipMemcpyDeviceToHost, st));
        HIP_TRY(hipStreamSynchronize(st));
        float* dst = (q ? d.keep_syn.data() : d.keep_obs.data()) + (size_t)r0 * nt;
        for (int t = 0; t < nt; t++)
          for (int r = 0; r < n; r++) dst[(size_t)r * nt + t] = h[(size_t)t * n + r];
      }
    }
  }
  return Status::Ok();
}

// ===================================================================== job runner
// One run of calc_id over one or several plans on one device.  The plans'
// shots are lined up in rows (row r = shot r of every plan that has one); a
// launch of a time-step kernel covers a group of rows of every plan, each
// plan one part of the launch.
//
// Gradient runs take the rows in sweeps (super-groups): a sweep runs the
// forward of its rows, their residual and their backward before the next
// sweep starts, so the boundary store holds one sweep's shots, not all.
// The store is either the reference's ring of every step (k = 0) or
// checkpoints every k steps plus the ring of one k-step segment, the segment
// recomputed from its checkpoint in the backward sweep.
namespace {

struct Member {
  Plan* plan;
  DeviceState* d;
};

struct RowRange {
  int r0, r1;
};

std::vector<RowRange> split_even(int a, int b, int per) {
  std::vector<RowRange> v;
  if (b <= a) return v;
  const int n = (b - a + per - 1) / per;
  for (int k = 0; k < n; k++)
    v.push_back({a + (int)((long long)k * (b - a) / n), a + (int)((long long)(k + 1) * (b - a) / n)});
  return v;
}

// every 64th step of each launch kind is bracketed by timing events (when
// timing is on): events between launches cost the stream about 2% at every
// 8th step
constexpr int sample_every = 64;
constexpr int kMaxPartsTable = 31;  // plans of a job
// Where a time step is one launch instead of two, in columns of whole-step
// tiles over all shots (the waves that a launch without rims would need).
// Forward: one launch less and no second read of the first half's results,
// against the rim that is computed twice and a second copy of the state in the
// caches.  Measured, two launches / one, 500 steps: 672 columns 2.95 / 2.29 ms,
// 3168: 4.08 / 3.56, 3429: 4.22 / 3.53, 9144: 7.41 / 6.67, 12573: 8.86 / 7.87, 13720:
// 7.28 / 7.30, 14256: 9.78 / 9.41, 16002: 10.0 / 9.92, 16800: 8.10 / 8.88, 22272:
// 11.8 / 12.0, 27328: 11.3 / 12.3; one shot of 6860: 5.12 / 4.90, 11040: 7.62 /
// 7.12, 17800: 10.7 / 10.2.  (Worse inside the line: 20 shots of 600, 8.55 / 9.07.)
// Slices of two shots instead of one where one would need more than the 8192
// waves that the chip holds: 8 shots of 600 columns 4.95 / 4.53 ms, 10 of 792
// 6.61 / 6.33, 2 of 4200 5.75 / 5.49; below it one is better (6 of 1840 13.6 ms in
// twos, 14.2 in threes, 15.0 alone at 1000 steps).
//
// Backward (adjoint and reversal both recompute their rim, twice the state is
// copied, and the reversal's workgroups walk all shots, since their sums are
// taken in order), two launches / one, 400 steps: one shot of 84 columns 4.16 /
// 3.55 ms, 1023: 4.50 / 4.26, 1272: 5.08 / 4.83, 2080: 6.06 / 5.67, 3300: 11.7 /
// 12.0 (601 steps); two shots of 84: 4.68 / 3.72, 792: 15.0 / 14.7 (1000 steps),
// 1023: 5.56 / 5.75; three of 84: 5.33 / 4.30, 1023: 6.86 / 7.19; four of 84: 5.37 /
// 5.11, 368: 16.5 / 14.8 (1000 steps); six of 84: 6.18 / 6.32.
constexpr double kWholeFwdWaves = 16384, kWholeFwdWaves1 = 20480;  // several shots, one
constexpr double kChipWaves = 8192;
constexpr double kWholeBwdWaves = 1600, kWholeBwdWaves1 = 2304;  // several shots, one
constexpr int kWholeBwdShots = 4;

enum Phase { kPhFwd = 0, kPhRec = 1, kPhBwd = 2 };

// One group of rows in one phase: its parts (plan shots [s0, s0 + n) of a
// member) and their launch arguments.  steps / backs: index of the first
// part's entry in the argument tables; the entries of the whole-step launches,
// one set per combination of state buffers, follow those of the half steps.
struct GroupParts {
  std::vector<int> member, s0, n;
  std::vector<StepArgs> args;
  size_t steps = 0, backs = 0;
};

class Runner {
 public:
  Runner(std::vector<Member> m, JobCache& c) : M(std::move(m)), cache(c) {}
  Status run(int calc_id);

 private:
  std::vector<Member> M;
  JobCache& cache;
  DeviceState* d0 = nullptr;
  hipStream_t st = nullptr;
  int nSteps = 0, rows = 0, gf = 1, gb = 1, S = 1, K = 0, nsnap = 0;
  // shots per slice and slices of a forward launch and of a whole backward step,
  // threads per cell of a half one
  int sf_ = 1, nf_ = 1, sa_ = 1, na_ = 1, nb_ = 1;
  bool if_res = false, withAdj = false, ckpt = false;
  int tile_ = 2;  // columns of a half step's workgroup
  bool whole_f_ = false, whole_b_ = false;  // whole-step launches (forward, reference's adjoint)
  std::vector<StepArgs> steps_;             // host copies of the argument tables
  std::vector<BackArgs> backs_;
  float* xt_ = nullptr;                     // exact adjoint operands of the running group
  const float* srcwin_ = nullptr;           // and the source window

  int shots_in(const Member& m, int r) const { return std::min(r, m.d->g.ns); }
  GroupParts parts_of(RowRange rr, int sg0, Phase ph);
  double waves(int shots) const;
  void slice(int shots, int& per, int& n) const;
  int threads_per_cell(int shots) const;
  int ring_at(int it) const { return withAdj ? it % (ckpt ? K : std::max(1, nSteps - 1)) : -1; }

  // launches: half steps (in place)
  template <typename Ker, typename... A>
  void go(Ker k, dim3 grid, dim3 block, A... a) {
    if (d0->kernel_start)
      hipExtLaunchKernelGGL(k, grid, block, 0, st, d0->kernel_start, d0->kernel_end, 0, a...);
    else
      hipLaunchKernelGGL(k, grid, block, 0, st, a...);
  }
  // for half_chunk
  static unsigned inverse(int places) {
    return places > 1 ? (unsigned)(((1ull << 32) + places - 1) / places) : 0u;
  }
  // grid of a half-step launch: `kinds` strips per tile row, and rows for the
  // extra items (ring, receivers, illumination) of the parts
  dim3 half_grid(const GroupParts& gp, int kinds, bool ring, bool rec, bool illum, int places) const;
  void half_stress(const GroupParts& gp, int it, int ring);
  void half_vel(const GroupParts& gp, int it, int ring);
  void half_a(const GroupParts& gp, int it, int ring, int kinds);
  void half_b(const GroupParts& gp, int it, int ring, int kinds);
  void exact_a(const GroupParts& gp, int it, int first);
  void exact_b(const GroupParts& gp, int it);
  void ring_all(const GroupParts& gp, int it, int c0, int c1);
  // whole steps: `odd` launches read the second state buffers
  dim3 whole_grid(const GroupParts& gp, bool backward) const;
  void step_fwd(const GroupParts& gp, int odd, int it);
  void step_bwd(const GroupParts& gp, int fodd, int aodd, int it);
  void record_last(const GroupParts& gp, int it);
  void illum_last(const GroupParts& gp);
  Status second_states(DeviceState& d, int mf, int mb);
  Status clear_second(const GroupParts& gp);
  // forward steps [t0, t1) of a group, `before(it, odd)` before each; they end
  // in the main state buffers
  Status forward(const GroupParts& gp, int t0, int t1,
                 const std::function<Status(int, int)>& before);

  Status snapshot(const GroupParts& gp, int sg0, int j, bool save, int odd);
  // run `body` (launches only, no memsets) as a graph captured on first use
  Status replay(const std::string& key, const std::function<void()>& body);
  std::string graph_key(const char* phase, const GroupParts& gp) const;
};

std::string Runner::graph_key(const char* phase, const GroupParts& gp) const {
  // FNV-1a over everything the captured launches bake in
  unsigned long long h = 1469598103934665603ULL;
  auto mix = [&](const void* p, size_t n) {
    const unsigned char* b = (const unsigned char*)p;
    for (size_t i = 0; i < n; i++) h = (h ^ b[i]) * 1099511628211ULL;
  };
  mix(gp.args.data(), gp.args.size() * sizeof(StepArgs));
  const void* ptrs[4] = {cache.steps, cache.backs, xt_, srcwin_};
  mix(ptrs, sizeof(ptrs));
  const size_t offs[2] = {gp.steps, gp.backs};
  mix(offs, sizeof(offs));
  const int flags[] = {d0->timing ? 1 : 0, nSteps, sf_, nf_, sa_, na_, nb_, whole_f_, whole_b_,
                       tile_, withAdj};
  mix(flags, sizeof(flags));
  return std::string(phase) + "/" + std::to_string(h);
}

Status Runner::replay(const std::string& key, const std::function<void()>& body) {
  // events recorded inside a captured graph cannot be timed: timed runs are eager
  if (!d0->graphs || d0->timing) {
    body();
    return Status::Ok();
  }
  auto it = cache.graphs.find(key);
  if (it == cache.graphs.end()) {
    if (cache.graphs.size() >= 512) cache.clear_graphs();
    GraphEntry e;
    d0->sink = &e.recs;
    hipError_t err = hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed);
    if (err == hipSuccess) {
      body();
      hipGraph_t g = nullptr;
      err = hipStreamEndCapture(st, &g);
      if (err == hipSuccess) {
        err = hipGraphInstantiate(&e.exec, g, nullptr, nullptr, 0);
        (void)hipGraphDestroy(g);
      }
    }
    d0->sink = nullptr;
    if (err != hipSuccess) {
      for (auto& r : e.recs) {
        (void)hipEventDestroy(r.a);
        (void)hipEventDestroy(r.b);
      }
      return Status::Err(FWIFLOW_ERR_HIP, std::string("graph capture: ") + hipGetErrorString(err));
    }
    it = cache.graphs.emplace(key, std::move(e)).first;
  }
  HIP_TRY(hipGraphLaunch(it->second.exec, st));
  if (d0->timing)
    for (const TimedLaunch& r : it->second.recs) d0->pending.push_back(r);
  return Status::Ok();
}

double Runner::waves(int shots) const {
  double w = 0;
  for (const Member& m : M)
    w += (double)((m.d->g.nzA + kBZ - 1) / kBZ) * m.d->g.nx * std::min(shots, m.d->g.ns);
  return w;
}

// A forward launch's shots are cut into slices, each with its own workgroups,
// so that small grids bring enough waves to hide a cell's loads: about
// kSliceWaves, but slices of two shots at least once the chip's 1024 SIMDs
// have four waves each, since the second shot of a thread shares the first
// one's model loads and indexing.  224x448, 30 shots: objective 98.8 ms at
// 8192 waves, 96.8 at 16384, 97.3 at 32768, 102.3 at 65536; 6 shots of it in
// slices of two / one: gradient 39.2 / 41.8 ms; 580x1780 (17800 waves a shot):
// 58.7 ms at 8192 .. 32768, 60.1 at 65536.  Even slices above two: modelling
// of 22 shots of 224x448 19.6 -> 19.2 ms, 9 of 364x964 22.0 -> 21.7.
constexpr double kSliceWaves = 16384, kPairWaves = 4096;
void Runner::slice(int shots, int& per, int& n) const {
  n = std::max(1, std::min(shots, (int)std::ceil(kSliceWaves / waves(1))));
  per = (shots + n - 1) / n;
  if (per == 1 && waves(shots) >= 2 * kPairWaves) per = std::min(2, shots);
  if (n > 1 && per > 2 && per % 2) --per;  // the half steps take shots in pairs
  n = (shots + per - 1) / per;
}

// Threads per cell of a backward launch: its shots run side by side in a
// workgroup where one thread a cell would leave the SIMDs short of waves; 1, 2
// or 4 (a sum's round of 8 shots divides evenly), with two shots a thread at
// least.  1 / 2 / 4 threads, ms: 280 waves a shot, 24 shots 38.8 / 28.0 / 23.8
// (8: 23.4); 682, 20 shots 48.1 / 38.8 / 36.0 (8: 38.4); 1792, 15 shots, exact
// adjoint 113 / 107 / 99.6 (8: 112); 1792, 6 shots 39.6 / 39.3 / 43.7; 3300, 12
// shots 63.2 / 62.3 / 63.5; 4562, 8 shots 61.9 / 59.6 / 65.0; 5784, 4 shots
// 44.4 / 45.6 / 51.8; 17800, 3 shots 535 / 600 / 759.
int Runner::threads_per_cell(int shots) const {
  const double most = std::min({4.0, shots / 2.0, 10240 / waves(1), 16.0 / tile_});
  return most >= 4 ? 4 : most >= 2 ? 2 : 1;
}

GroupParts Runner::parts_of(RowRange rr, int sg0, Phase ph) {
  GroupParts gp;
  std::vector<BackArgs> back;
  for (size_t mi = 0; mi < M.size(); mi++) {
    DeviceState& d = *M[mi].d;
    const Geo& g = d.g;
    const int s0 = shots_in(M[mi], rr.r0), s1 = shots_in(M[mi], rr.r1);
    if (s1 <= s0) continue;
    gp.member.push_back((int)mi);
    gp.s0.push_back(s0);
    gp.n.push_back(s1 - s0);
    StepArgs a{};
    float* const mem = d.shot(ph == kPhBwd && ckpt ? d.madj : d.mem, kMemComps, s0);
    a.wo = d.shot(d.fwd, kWaveComps, s0), a.wi = a.wo;
    a.mo = mem, a.mi = mem;
    a.md = d.lam, a.zc = d.pmlc, a.xc = d.pmlc + 8 * (size_t)g.nzA;
    a.zx = d.src + 2 * s0;
    a.amp = (ph == kPhBwd && d.src_updated ? d.srcout : d.srcamp) + (size_t)s0 * nSteps;
    const bool ring = withAdj && ((ph == kPhFwd && !ckpt) || ph == kPhRec || ph == kPhBwd);
    a.ring = ring ? d.ring : nullptr;
    a.illum = ph == kPhFwd && d.illum_on ? d.illum : nullptr;
    a.rec = d.rec + 3 * (size_t)d.roff[s0];
    a.syn = d.syn + d.roff[s0];
    a.nz = g.nz, a.nx = g.nx, a.nzA = g.nzA, a.nPml = g.nPml;
    a.ns = s1 - s0, a.nSteps = nSteps, a.s0 = s0;
    a.nrec = ph == kPhFwd ? d.roff[s1] - d.roff[s0] : 0;  // recorded once
    a.dt = g.dt, a.dz = g.dz, a.dx = g.dx, a.rdz = g.rdz, a.rdx = g.rdx;
    a.Nb = (int)(g.N * 4), a.R = d.R, a.ringW = g.ringW, a.ringH = g.ringH, a.ringlen = g.ringlen;
    a.rs0 = s0 - shots_in(M[mi], sg0);
    a.rnt = ckpt ? K : std::max(1, nSteps - 1);
    a.gz = (g.nzA - 4 + kCoreZ - 1) / kCoreZ;
    a.gx = (g.nx - 4 + kCoreX - 1) / kCoreX;
    a.per = (a.gx + 7) / 8;
    a.hgz = (g.nzA + kBZ - 1) / kBZ;
    a.hgx = (g.nx - 4 + tile_ - 1) / tile_;
    a.hper = (a.hgx + 7) / 8;
    gp.args.push_back(a);
    if (ph != kPhBwd) continue;
    BackArgs b{};
    b.s = a;
    b.ao = d.shot(d.adj, kWaveComps, s0), b.ai = b.ao;
    b.zd = d.pml64, b.xd = d.pml64 + g.nzA;
    b.res = d.res, b.inj = d.inj, b.icell = d.icell, b.iptr = d.iptr, b.irid = d.irid;
    b.acc = d.acc, b.stf_grad = d.stf_grad + (size_t)s0 * nSteps;
    b.rgz = (g.ringH + kCoreZ - 1) / kCoreZ;
    b.rgx = (g.ringW + kCoreX - 1) / kCoreX;
    b.rper = (b.rgx + 7) / 8;
    back.push_back(b);
  }
  if (ph != kPhBwd) {
    gp.steps = steps_.size();
    steps_.insert(steps_.end(), gp.args.begin(), gp.args.end());
    for (int odd = 0; whole_f_ && odd < 2; odd++)
      for (size_t q = 0; q < gp.args.size(); q++) {
        const DeviceState& d = *M[gp.member[q]].d;
        StepArgs a = gp.args[q];
        if (odd)
          a.wi = d.fwd2, a.mi = d.mem2;
        else
          a.wo = d.fwd2, a.mo = d.mem2;
        steps_.push_back(a);
      }
  } else {
    gp.backs = backs_.size();
    backs_.insert(backs_.end(), back.begin(), back.end());
    for (int v = 0; whole_b_ && v < 4; v++)
      for (size_t q = 0; q < back.size(); q++) {
        const DeviceState& d = *M[gp.member[q]].d;
        BackArgs b = back[q];
        float* const m2 = ckpt ? d.madj2 : d.mem2;
        if (v & 1)
          b.s.wi = d.fwd2;
        else
          b.s.wo = d.fwd2;
        if (v & 2)
          b.s.mi = m2, b.ai = d.adj2;
        else
          b.s.mo = m2, b.ao = d.adj2;
        backs_.push_back(b);
      }
  }
  return gp;
}

// Columns of a chunk: a strip's rim is read again by the strips above and
// below it, from the L2 if they run soon enough.  580x1780, ms: no chunks
// gradient 531, modelling 59.0; 128 columns 510 / 58.3, 32: 501 / 58.1, 16:
// 496 / 57.7, 8: 497 / 57.6, 2: 528 / 58.4.  Smaller grids: 364x964 44.5 -> 43.8,
// the two-grid job 59.7 -> 57.3, 224x448 x 30 shots 99.2 -> 96.2.
constexpr int kChunk = 16;
dim3 Runner::half_grid(const GroupParts& gp, int kinds, bool ring, bool rec, bool illum,
                       int places) const {
  int per = 1, y = 1;
  for (const StepArgs& a : gp.args) per = std::max(per, a.hper);
  // chunks of at most kChunk columns, evenly filled
  const int most = std::max(1, kChunk / tile_), n = (per + most - 1) / most;
  const int x = (per + n - 1) / n, chunks = (per + x - 1) / x;
  const int row = kBZ * tile_ * 8 * x * chunks;  // items of a grid row of every chunk
  for (const StepArgs& a : gp.args) {
    const int items = ((ring || rec || illum) && a.ring ? (a.ringlen + 63) / 64 * 64 : 0) +
                      (rec ? a.nrec : 0) + (illum && a.illum && nf_ > 1 ? a.Nb / 4 : 0);
    y = std::max(y, kinds * a.hgz + (items + row - 1) / row);
  }
  return dim3((unsigned)(8 * x), (unsigned)y, (unsigned)(chunks * places));
}
void Runner::half_stress(const GroupParts& gp, int it, int ring) {
  const int pf = nf_ * (int)gp.args.size();
  go(k_half_stress<2>, half_grid(gp, 1, ring >= 0, false, true, pf), dim3(kBZ, tile_),
     cache.steps + gp.steps, it, ring, nf_, sf_, pf, inverse(pf));
}
void Runner::half_vel(const GroupParts& gp, int it, int ring) {
  const int pf = nf_ * (int)gp.args.size();
  go(k_half_vel<2>, half_grid(gp, 1, ring >= 0, true, false, pf), dim3(kBZ, tile_),
     cache.steps + gp.steps, it, ring, nf_, sf_, pf, inverse(pf));
}
void Runner::half_a(const GroupParts& gp, int it, int ring, int kinds) {
  const int parts = (int)gp.args.size();
  go(nb_ > 1 ? k_half_bwd_a<true> : k_half_bwd_a<false>, half_grid(gp, 2, ring >= 0, false, false, parts),
     dim3(kBZ, tile_, nb_), cache.backs + gp.backs, it, ring, kinds, parts, inverse(parts));
}
void Runner::half_b(const GroupParts& gp, int it, int ring, int kinds) {
  const int parts = (int)gp.args.size();
  go(nb_ > 1 ? k_half_bwd_b<true> : k_half_bwd_b<false>, half_grid(gp, 2, ring >= 0, false, false, parts),
     dim3(kBZ, tile_, nb_), cache.backs + gp.backs, it, ring, kinds, parts, inverse(parts));
}
// exact adjoint (with the reversal of the step)
void Runner::exact_a(const GroupParts& gp, int it, int first) {
  const int parts = (int)gp.args.size();
  go(nb_ > 1 ? k_exact_a<true> : k_exact_a<false>, half_grid(gp, 1, true, false, false, parts),
     dim3(kBZ, tile_, nb_), cache.backs + gp.backs, xt_, it, ring_at(it), first,
     parts, inverse(parts));
}
void Runner::exact_b(const GroupParts& gp, int it) {
  const int parts = (int)gp.args.size();
  go(nb_ > 1 ? k_exact_b<true> : k_exact_b<false>, half_grid(gp, 1, true, false, false, parts),
     dim3(kBZ, tile_, nb_), cache.backs + gp.backs, xt_, srcwin_, it, ring_at(it),
     parts, inverse(parts));
}

dim3 Runner::whole_grid(const GroupParts& gp, bool backward) const {
  int x = 8, y = 1;
  for (size_t q = 0; q < gp.args.size(); q++) {
    const StepArgs& a = gp.args[q];
    x = std::max(x, 8 * a.per);
    if (backward) y = std::max(y, a.gz + backs_[gp.backs + q].rgz);
  }
  if (!backward) {
    const int row = kBZ * kStepW * x;
    for (const StepArgs& a : gp.args) {
      const int items = (a.ring ? (a.ringlen + 63) / 64 * 64 : 0) + (a.nrec + 63) / 64 * 64 +
                        (a.illum && nf_ > 1 ? a.Nb / 4 : 0);
      y = std::max(y, a.gz + (items + row - 1) / row);
    }
  }
  return dim3((unsigned)x, (unsigned)y, (unsigned)((backward ? na_ : nf_) * (int)gp.args.size()));
}
void Runner::step_fwd(const GroupParts& gp, int odd, int it) {
  const StepArgs* t = cache.steps + gp.steps + (size_t)(1 + odd) * gp.args.size();
  const dim3 grid = whole_grid(gp, false), b(kBZ, kStepW);
  const int ring = gp.args[0].ring ? ring_at(it) : -1;
  go(k_step_fwd, grid, b, t, it, ring, nf_, sf_);
}
void Runner::step_bwd(const GroupParts& gp, int fodd, int aodd, int it) {
  const BackArgs* t = cache.backs + gp.backs + (size_t)(1 + fodd + 2 * aodd) * gp.args.size();
  const dim3 grid = whole_grid(gp, true), b(kBZ, kStepW);
  go(k_step_bwd, grid, b, t, it, ring_at(it), na_, sa_);
}

Status Runner::forward(const GroupParts& gp, int t0, int t1,
                       const std::function<Status(int, int)>& before) {
  const bool ring = !gp.args.empty() && gp.args[0].ring;
  auto row = [&](int it) { return ring ? ring_at(it) : -1; };
  if (!whole_f_ && ring && t1 > t0) ring_all(gp, t0, 0, 3);  // the stresses that step t0 reads
  for (int it = t0; it < t1; it++) {
    const bool smp = it % sample_every == 0;
    const int odd = whole_f_ ? (t1 - it) & 1 : 0;
    TRY(before(it, odd));
    if (whole_f_) {
      d0->launch("step_fwd", smp, [&] { step_fwd(gp, odd, it); });
    } else {
      d0->launch("stress_fwd", smp, [&] { half_stress(gp, it, row(it)); });
      d0->launch("vel_fwd", smp, [&] { half_vel(gp, it, it + 1 < t1 ? row(it + 1) : -1); });
    }
  }
  return Status::Ok();
}

// ring components [c0, c1) of step it saved from the main state buffers
void Runner::ring_all(const GroupParts& gp, int it, int c0, int c1) {
  int n = 0;
  for (const StepArgs& a : gp.args) n = std::max(n, a.ringlen);
  hipLaunchKernelGGL(k_ring, dim3((n + 255) / 256, 1, (unsigned)gp.args.size()), dim3(256), 0,
                     st, cache.steps + gp.steps, ring_at(it), c0, c1);
}

void Runner::record_last(const GroupParts& gp, int it) {
  int n = 0;
  for (const StepArgs& a : gp.args) n = std::max(n, a.nrec);
  if (n)
    hipLaunchKernelGGL(k_record, dim3((n + 255) / 256, 1, (unsigned)gp.args.size()), dim3(256), 0, st,
                       cache.steps + gp.steps, it);
}

void Runner::illum_last(const GroupParts& gp) {
  int n = 0;
  for (const StepArgs& a : gp.args) n = std::max(n, a.illum ? a.Nb / 4 : 0);
  if (n)
    hipLaunchKernelGGL(k_illum, dim3((n + 255) / 256, 1, (unsigned)gp.args.size()), dim3(256), 0, st,
                       cache.steps + gp.steps);
}

// Room for the second states of the launches that take whole steps; they start
// out zero and stay zero outside the update region.
Status Runner::second_states(DeviceState& d, int mf, int mb) {
  auto room = [&](float*& p, int& have, int need, int comps) -> Status {
    need = std::min(need, d.g.ns);
    if (have >= need) return Status::Ok();
    const size_t n = (size_t)comps * d.g.N;
    d.release(p, have * n);
    have = 0;
    TRY(d.take(&p, need * n));
    have = need;
    HIP_TRY(hipMemsetAsync(p, 0, need * n * sizeof(float), st));
    return Status::Ok();
  };
  const int f = whole_f_ ? mf : 0, b = whole_b_ ? mb : 0;
  TRY(room(d.fwd2, d.shots2, std::max(f, b), kWaveComps));
  TRY(room(d.mem2, d.mshots2, std::max(f, ckpt ? 0 : b), kMemComps));
  TRY(room(d.adj2, d.ashots2, b, kWaveComps));
  TRY(room(d.madj2, d.xshots2, ckpt ? b : 0, kMemComps));
  return Status::Ok();
}

Status Runner::clear_second(const GroupParts& gp) {
  for (size_t q = 0; q < gp.member.size(); q++) {
    DeviceState& d = *M[gp.member[q]].d;
    const size_t n = (size_t)gp.n[q] * d.g.N * sizeof(float);
    HIP_TRY(hipMemsetAsync(d.fwd2, 0, kWaveComps * n, st));
    HIP_TRY(hipMemsetAsync(d.mem2, 0, kMemComps * n, st));
  }
  return Status::Ok();
}

// Checkpoint j >= 1 of the shots of a group: the 5 wavefield components and
// the 8 forward C-PML memory variables before forward step j * K.  Layout
// [j-1] x {wavefields [shot of the sweep][5][cell], memory variables
// [shot of the sweep][8][cell]}: a group's shots are one contiguous block of
// each.
Status Runner::snapshot(const GroupParts& gp, int sg0, int j, bool save, int odd) {
  for (size_t q = 0; q < gp.member.size(); q++) {
    DeviceState& d = *M[gp.member[q]].d;
    const int s0 = gp.s0[q], n = gp.n[q];
    const int rows_m = std::min(S, d.g.ns), rs = s0 - shots_in(M[gp.member[q]], sg0);
    const size_t N = (size_t)d.g.N;
    float* cp = d.snap + (size_t)(j - 1) * (kWaveComps + kMemComps) * rows_m * N;
    float* cw = cp + (size_t)rs * kWaveComps * N;
    float* cm = cp + (size_t)rows_m * kWaveComps * N + (size_t)rs * kMemComps * N;
    float* fw = odd ? d.fwd2 : d.shot(d.fwd, kWaveComps, s0);
    float* fm = odd ? d.mem2 : d.shot(d.mem, kMemComps, s0);
    const size_t bw = (size_t)n * kWaveComps * N * sizeof(float);
    const size_t bm = (size_t)n * kMemComps * N * sizeof(float);
    HIP_TRY(hipMemcpyAsync(save ? cw : fw, save ? fw : cw, bw, hipMemcpyDeviceToDevice, st));
    HIP_TRY(hipMemcpyAsync(save ? cm : fm, save ? fm : cm, bm, hipMemcpyDeviceToDevice, st));
  }
  return Status::Ok();
}

Status Runner::run(int calc_id) {
  TRY(check_calc_id(calc_id));
  if (M.empty()) return Status::Err(FWIFLOW_ERR_ARG, "no plans to run");
  d0 = M[0].d;
  for (const Member& m : M) {
    if (!m.d) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
    if (!m.d->model_set) return Status::Err(FWIFLOW_ERR_ARG, "model not set");
    if (!m.d->stf_set) return Status::Err(FWIFLOW_ERR_ARG, "source time functions not set");
    if (calc_id != 2 && !m.d->obs_set) return Status::Err(FWIFLOW_ERR_ARG, "observed data not set");
    if (m.d->dev != d0->dev) return Status::Err(FWIFLOW_ERR_ARG, "plans of a job must share the GPU");
    if (m.d->g.nSteps != d0->g.nSteps)
      return Status::Err(FWIFLOW_ERR_ARG, "plans of a job must share nSteps");
    if (m.d->tile_x != d0->tile_x)
      return Status::Err(FWIFLOW_ERR_ARG, "plans of a job must share the tile width");
    if (m.d->adjoint && M.size() > 1)
      return Status::Err(FWIFLOW_ERR_UNSUPPORTED, "the exact adjoint runs one plan at a time");
    if (m.d->adjoint && calc_id == 1 && m.plan->para.if_src_update)
      return Status::Err(FWIFLOW_ERR_UNSUPPORTED,
                         "the exact adjoint does not take the source update (if_src_update)");
    m.d->illum_valid = false;
    m.plan->last_calc = -1;
  }
  if (M.size() > 1 && M.size() > (size_t)kMaxPartsTable)
    return Status::Err(FWIFLOW_ERR_ARG, "at most " + std::to_string(kMaxPartsTable) + " plans per job");
  HIP_TRY(hipSetDevice(d0->dev));
  st = d0->stream;
  nSteps = d0->g.nSteps;
  if_res = calc_id != 2;
  withAdj = calc_id == 1;
  rows = 0;
  double rowf = 0, rowb = 0, ring_row = 0, snap_row = 0;
  for (const Member& m : M) {
    rows = std::max(rows, m.d->g.ns);
    rowf += m.d->fwd_bytes_per_shot();
    rowb += m.d->bwd_bytes_per_shot();
    ring_row += 4.0 * m.d->ring_step_floats();
    snap_row += 4.0 * m.d->snap_floats_per_shot();
  }
  // rows per launch: forward and backward state of a group kept in the
  // Infinity Cache from step to step
  const DeviceState& c0 = *d0;
  auto autosize = [&](double per_row) {
    return std::max(1, std::min(rows, (int)std::lround(224e6 / per_row)));
  };
  gf = c0.shot_group == 0 ? rows : c0.shot_group > 0 ? std::min(c0.shot_group, rows) : autosize(rowf);
  if (c0.shot_group_bwd == 0)
    gb = rows;
  else if (c0.shot_group_bwd > 0)
    gb = std::min(c0.shot_group_bwd, rows);
  else if (c0.shot_group >= 0)
    gb = gf;
  else
    gb = autosize(rowb);
  // the kernels address a part's arrays with 32-bit byte offsets: one part's
  // C-PML memory variables (8 arrays per shot) must stay below 2^31 bytes
  int cap = rows;
  for (const Member& m : M)
    cap = std::min(cap, (int)(2147483647LL / ((long long)kMemComps * 4 * m.d->g.N)));
  if (cap < 1) return Status::Err(FWIFLOW_ERR_SHAPE, "grid too large for one shot per launch");
  gf = std::min(gf, cap);
  gb = std::min(gb, cap);
  // memory plan of a gradient run: rows per sweep S and checkpoint interval K
  const int steps = std::max(1, nSteps - 1);  // forward steps 0 .. nSteps-2
  double budget = c0.ring_budget;
  if (withAdj && c0.arena && M.size() == 1) {
    // scratch-backed plan: ring + checkpoints get what the scratch array has
    // left after the gradient run's other buffers (adjoint fields, C-PML
    // adjoint memory variables, accumulators, misfit partials, injection and
    // argument tables)
    const DeviceState& d = c0;
    const double N = (double)d.g.N, F = (double)d.F();
    const double other = 4.0 * ((d.adj ? 0 : 5 * F) + (d.madj ? 0 : 8 * F) +
                                (d.acc ? 0 : 5 * N) + (d.grad ? 0 : 3 * N) +
                                (d.stf_grad ? 0 : (double)d.g.ns * nSteps) +
                                (d.illum_on && !d.illum ? N : 0)) +
                         (d.inj ? 0 : sizeof(ColInj) * (double)d.g.ns * d.g.nx +
                                          4.0 * (d.icells.size() + d.iptrs.size() + d.irids.size())) +
                         (2 * sizeof(StepArgs) + sizeof(BackArgs)) * (double)rows +
                         8.0 * rows * kPartials + (1 << 20);
    budget = std::min(budget, std::max(1.0, (double)d.arena->free_bytes() - other));
  }
  K = withAdj ? c0.ckpt_every : 0;
  if (K >= steps) K = 0;
  S = rows;
  if (withAdj) {
    const int l = gf / std::__gcd(gf, gb) * gb;
    auto fit = [&](double per_row) {
      // the most rows within the budget, a multiple of both group sizes if
      // possible (no partial groups inside a sweep), else of the backward's
      int n = (int)std::floor(budget / per_row);
      if (n >= l) n = n / l * l;
      else if (n >= gb) n = n / gb * gb;
      return std::max(1, std::min(rows, n));
    };
    const double full = ring_row * steps;
    if (K == 0 && full * std::min(rows, gb) > budget && steps > 1) {
      // the full ring of one backward group does not fit: checkpoints, at the
      // interval that minimises ring + checkpoint memory
      K = (int)std::lround(std::sqrt((double)steps * snap_row / ring_row));
      K = std::max(1, std::min(K, steps - 1));
    }
    ckpt = K > 0;
    if (ckpt) {
      nsnap = (steps + K - 1) / K - 1;
      S = fit(K * ring_row + nsnap * snap_row);
    } else {
      nsnap = 0;
      S = fit(full);
    }
  }
  // sweeps (super-groups) and their launch groups, as row ranges
  std::vector<RowRange> sweeps;
  for (int a = 0; a < rows; a += S) sweeps.push_back({a, std::min(rows, a + S)});
  std::vector<std::vector<RowRange>> FR(sweeps.size()), BR(sweeps.size());
  for (size_t j = 0; j < sweeps.size(); j++) {
    FR[j] = split_even(sweeps[j].r0, sweeps[j].r1, gf);
    if (withAdj) BR[j] = split_even(sweeps[j].r0, sweeps[j].r1, gb);
  }
  // launch forms, by the most rows that a forward launch (of a checkpointed run
  // also the recomputation of a backward group) and a backward launch hold
  int mf = 1, mb = 1;
  for (size_t j = 0; j < sweeps.size(); j++) {
    for (RowRange rr : FR[j]) mf = std::max(mf, rr.r1 - rr.r0);
    for (RowRange rr : BR[j]) mb = std::max(mb, rr.r1 - rr.r0);
  }
  if (ckpt) mf = std::max(mf, mb);
  // two columns a workgroup unless the caller chose: against four, 580x1780
  // 59.5 / 59.8 ms, 364x964 44.4 / 45.2, 224x448 39.6 / 41.8 (smaller steps of
  // the work that the SIMDs share out)
  tile_ = c0.tile_auto ? 2 : c0.tile_x;
  slice(mf, sf_, nf_);
  slice(mb, sa_, na_);
  nb_ = threads_per_cell(mb);
  // a workgroup of four threads a cell is one column wide: exact adjoint of 15
  // shots of 224x448 96.0 -> 94.0 ms, 20 shots of 224x520 68.8 -> 66.5, reference's
  // adjoint of 20 shots of 127x341 36.7 -> 36.0
  if (c0.tile_auto && withAdj && nb_ == 4) tile_ = 1;
  auto tiles = [&](int shots) {  // columns of whole-step tiles, each a wave of its core
    double t = 0;
    for (const Member& m : M)
      t += (double)((m.d->g.nzA - 4 + kCoreZ - 1) / kCoreZ) * m.d->g.nx * std::min(shots, m.d->g.ns);
    return t;
  };
  whole_f_ = !c0.arena && tiles(mf) <= (mf == 1 ? kWholeFwdWaves1 : kWholeFwdWaves);
  if (whole_f_) {
    sf_ = kStepW / kCoreX * tiles(mf) > kChipWaves ? std::min(2, mf) : 1;
    nf_ = (mf + sf_ - 1) / sf_;
  }
  whole_b_ = !c0.arena && withAdj && mb <= kWholeBwdShots &&
             tiles(mb) <= (mb == 1 ? kWholeBwdWaves1 : kWholeBwdWaves);
  for (const Member& m : M) whole_b_ = whole_b_ && !m.d->adjoint && m.d->inj_folded;
  // buffers; where a plan of a job has no room for its own, the second states
  // that others hold from earlier runs give way
  auto buffers = [&]() -> Status {
    for (const Member& m : M) {
      DeviceState& d = *m.d;
      const size_t N = (size_t)d.g.N, F = d.F();
      if (withAdj) {
        if (!d.adj) TRY(d.alloc(&d.adj, 5 * F));
        if (ckpt && !d.madj) TRY(d.alloc(&d.madj, 8 * F));
        if (!d.acc) TRY(d.alloc(&d.acc, 5 * N));
        if (!d.grad) TRY(d.alloc(&d.grad, 3 * N));
        if (!d.stf_grad) TRY(d.alloc(&d.stf_grad, (size_t)d.g.ns * nSteps));
        if (d.adjoint) {
          const size_t xf = (size_t)std::min(gb, d.g.ns) * 8 * N;
          if (d.xt_floats < xf) {
            d.release(d.xt, d.xt_floats);
            d.xt_floats = 0;
            TRY(d.alloc(&d.xt, xf));
            d.xt_floats = xf;
          }
        }
        const int rows_m = std::min(S, d.g.ns);
        const size_t rf = (size_t)rows_m * (ckpt ? K : steps) * d.ring_step_floats();
        if (d.ring_floats < rf || d.ring_floats > 2 * rf + (1u << 20)) {
          d.release(d.ring, d.ring_floats);
          d.ring_floats = 0;
          TRY(d.alloc(&d.ring, rf));
          d.ring_floats = rf;
        }
        const size_t sf = ckpt ? (size_t)nsnap * 13 * rows_m * N : 0;
        if (d.snap_floats < sf || (sf == 0 && d.snap)) {
          d.release(d.snap, d.snap_floats);
          d.snap_floats = 0;
          if (sf) {
            TRY(d.alloc(&d.snap, sf));
            d.snap_floats = sf;
          }
        }
        d.last_k = K;
        d.last_rows_sg = rows_m;
        d.last_ring_bytes = (long long)(rf * sizeof(float));
        d.last_snap_bytes = (long long)(sf * sizeof(float));
      }
      if (withAdj) TRY(ensure_injection(d));
      const int npart = (int)sweeps.size() * kPartials;
      if (d.npartial < npart) {
        d.release(d.partial, (size_t)d.npartial);
        d.npartial = 0;
        TRY(d.alloc(&d.partial, (size_t)npart));
        d.npartial = npart;
      }
      if (d.illum_on && !d.illum) TRY(d.alloc(&d.illum, N));
      d.src_updated = if_res && d.cond && m.plan->para.if_src_update;
      d.last_groups_f = 0;
      d.last_groups_b = 0;
      for (size_t j = 0; j < sweeps.size(); j++) {
        for (RowRange rr : FR[j]) d.last_groups_f += shots_in(m, rr.r1) > shots_in(m, rr.r0);
        for (RowRange rr : BR[j]) d.last_groups_b += shots_in(m, rr.r1) > shots_in(m, rr.r0);
      }
    }
    size_t nf = 0, nb = 0;  // argument table entries
    for (size_t j = 0; j < sweeps.size(); j++) {
      nf += FR[j].size() + (ckpt ? BR[j].size() : 0);
      nb += BR[j].size();
    }
    TRY(cache.reserve(nf * M.size() * (whole_f_ ? 3 : 1), cache.steps, cache.steps_cap));
    return cache.reserve(nb * M.size() * (whole_b_ ? 5 : 1), cache.backs, cache.backs_cap);
  };
  if (Status s = buffers(); !s.ok()) {
    bool held = false;
    for (const Member& m : M) held = m.d->drop_second() || held;
    if (!held) return s;
    TRY(buffers());
  }
  // The second states come last: a run without them takes two launches a step,
  // all members alike.
  Status second = Status::Ok();
  for (const Member& m : M)
    if (second.ok()) second = second_states(*m.d, mf, mb);
  if (!second.ok()) {
    if (second.code != FWIFLOW_ERR_MEMORY) return second;
    (void)hipGetLastError();
    for (const Member& m : M) m.d->drop_second();
    whole_f_ = whole_b_ = false;
    slice(mf, sf_, nf_);
  }
  for (const Member& m : M) m.d->last_tile = whole_f_ && (whole_b_ || !withAdj) ? 0 : tile_;
  // parts of every group (pointing at the buffers above)
  std::vector<std::vector<GroupParts>> FG(sweeps.size()), RG(sweeps.size()), BG(sweeps.size());
  for (size_t j = 0; j < sweeps.size(); j++) {
    for (RowRange rr : FR[j]) FG[j].push_back(parts_of(rr, sweeps[j].r0, kPhFwd));
    for (RowRange rr : BR[j]) {
      BG[j].push_back(parts_of(rr, sweeps[j].r0, kPhBwd));
      if (ckpt) RG[j].push_back(parts_of(rr, sweeps[j].r0, kPhRec));
    }
  }
  TRY(cache.upload(steps_, cache.steps, cache.steps_cap));
  TRY(cache.upload(backs_, cache.backs, cache.backs_cap));
  // clear the run's state
  for (const Member& m : M) {
    DeviceState& d = *m.d;
    const size_t N = (size_t)d.g.N, F = d.F();
    HIP_TRY(hipMemsetAsync(d.fwd, 0, 5 * F * sizeof(float), st));
    HIP_TRY(hipMemsetAsync(d.mem, 0, 8 * F * sizeof(float), st));
    HIP_TRY(hipMemsetAsync(d.syn, 0, (size_t)nSteps * d.R * sizeof(float), st));
    HIP_TRY(hipMemsetAsync(d.partial, 0, (size_t)d.npartial * sizeof(double), st));
    if (d.illum_on) HIP_TRY(hipMemsetAsync(d.illum, 0, N * sizeof(float), st));
    if (withAdj) {
      HIP_TRY(hipMemsetAsync(d.acc, 0, 5 * N * sizeof(float), st));
      HIP_TRY(hipMemsetAsync(d.stf_grad, 0, (size_t)d.g.ns * nSteps * sizeof(float), st));
    }
  }
  for (size_t j = 0; j < sweeps.size(); j++) {
    const RowRange sw = sweeps[j];
    // ------------------------------------------------------ forward
    for (const GroupParts& gp : FG[j]) {
      if (whole_f_ && (steps & 1)) TRY(clear_second(gp));
      auto save = [&](int it, int odd) -> Status {
        return ckpt && it > 0 && it % K == 0 ? snapshot(gp, sw.r0, it / K, true, odd) : Status::Ok();
      };
      if (ckpt)  // checkpoint copies between the steps: no graph
        TRY(forward(gp, 0, nSteps - 1, save));
      else
        TRY(replay(graph_key("F", gp), [&] { (void)forward(gp, 0, nSteps - 1, save); }));
      if (whole_f_) record_last(gp, nSteps - 1);
      if (nf_ > 1 && nSteps > 1) illum_last(gp);
    }
    HIP_TRY(hipGetLastError());
    // ------------------------------------------------------ residual
    if (if_res) {
      for (const Member& m : M) {
        DeviceState& d = *m.d;
        const int sa = shots_in(m, sw.r0), sb = shots_in(m, sw.r1);
        if (sb <= sa) continue;
        if (d.cond) {
          TRY(condition_residual(d, m.plan->para, m.plan->para.save_scratch && withAdj, sa, sb,
                                 st));
        } else {
          const int r0 = d.roff[sa], nr = d.roff[sb] - r0;
          hipLaunchKernelGGL(k_residual, dim3(kPartials), dim3(256), 0, st, nSteps, d.R, r0, nr,
                             d.win2, d.obs, d.syn, d.res, d.partial + j * kPartials);
        }
      }
      HIP_TRY(hipGetLastError());
    }
    if (!withAdj) continue;
    // ------------------------------------------------------ backward
    for (size_t q = 0; q < BG[j].size(); q++) {
      const GroupParts& gp = BG[j][q];
      for (size_t p = 0; p < gp.member.size(); p++) {
        DeviceState& d = *M[gp.member[p]].d;
        const int s0 = gp.s0[p], n = gp.n[p];
        TRY(d.zero_shots(d.adj, kWaveComps, s0, n, st));
        TRY(d.zero_shots(ckpt ? d.madj : d.mem, kMemComps, s0, n, st));
      }
      // residual injection of step t for plans without the folded injection
      auto inject = [&](int t) {
        for (size_t p = 0; p < gp.member.size(); p++) {
          DeviceState& d = *M[gp.member[p]].d;
          if (d.inj_folded) continue;
          const int c0 = d.coff[gp.s0[p]], nc = d.coff[gp.s0[p] + gp.n[p]] - c0;
          if (nc > 0)
            hipLaunchKernelGGL(k_res_inject, dim3((nc + 255) / 256), dim3(256), 0, st, d.g,
                               d.adj, d.icell, d.iptr, d.irid, c0, nc,
                               d.res + (size_t)t * d.R);
        }
      };
      // exact adjoint, reverse steps t1-1 .. t0 of a segment: the forward
      // state enters as (v, sigma) after step t1-1 and each reverse step it
      // re-materialises (v^it, sigma^it) in its two launches.  No initial
      // adjoint step: sample 0 is not recorded, and sample it+1 enters at
      // reverse step it.
      auto xsegment = [&](int t0, int t1) {
        for (int it = t1 - 1; it >= t0; it--) {
          const bool smp = it % sample_every == 0;
          d0->launch("exact_a", smp, [&] { exact_a(gp, it, it == nSteps - 2 ? 1 : 0); });
          inject(it + 1);
          d0->launch("exact_b", smp, [&] { exact_b(gp, it); });
        }
      };
      if (d0->adjoint) {
        for (size_t p = 0; p < gp.member.size(); p++) {
          DeviceState& d = *M[gp.member[p]].d;
          HIP_TRY(hipMemsetAsync(d.xt, 0, (size_t)gp.n[p] * 8 * d.g.N * sizeof(float), st));
        }
        xt_ = d0->xt;
        srcwin_ = d0->srcwin;
      }
      if (d0->adjoint && !ckpt) {
        if (nSteps >= 2) TRY(replay(graph_key("X", gp), [&] { xsegment(0, steps); }));
        HIP_TRY(hipGetLastError());
        continue;
      }
      // the initial adjoint step at t = nSteps-1 (libCUFD.cu:353-373), in place;
      // adj_stress shares its launch with the first reversal where half steps follow
      auto initial = [&] {
        half_a(gp, nSteps - 1, -1, 1);
        inject(nSteps - 1);
        if (nSteps < 2 || whole_b_) half_b(gp, nSteps - 1, -1, 1);
      };
      // reverse steps t1-1 .. t0 of one segment; `last` is the segment that
      // ends at nSteps-1
      int aodd = 0;  // whole steps: the adjoint state is in its second buffers
      auto segment = [&](int t0, int t1, bool last) {
        if (whole_b_) {
          int fodd = 0;
          for (int it = t1 - 1; it >= t0; it--, fodd ^= 1, aodd ^= 1)
            d0->launch("step_bwd", it % sample_every == 0, [&] { step_bwd(gp, fodd, aodd, it); });
          return;
        }
        // adj_stress(nSteps-1) + rev_vel(nSteps-2), or rev_vel(t1-1)
        half_b(gp, t1, ring_at(t1 - 1), last ? 3 : 2);
        for (int it = t1 - 1; it >= t0; it--) {
          const bool smp = it % sample_every == 0;
          d0->launch("bwd_pair_a", smp, [&] { half_a(gp, it, ring_at(it), 3); });
          inject(it);
          if (it > t0)
            d0->launch("bwd_pair_b", smp, [&] { half_b(gp, it, ring_at(it - 1), 3); });
          else
            half_b(gp, it, -1, 1);
        }
      };
      if (!ckpt) {
        TRY(replay(graph_key("B", gp), [&] {
          initial();
          if (nSteps >= 2) segment(0, steps, true);
        }));
        HIP_TRY(hipGetLastError());
        continue;
      }
      // checkpoints: each segment is recomputed from its checkpoint, then
      // reversed with its ring
      if (!d0->adjoint) initial();
      if (nSteps < 2) continue;
      const GroupParts& rg = RG[j][q];
      const int nseg = (steps + K - 1) / K;
      for (int jj = nseg - 1; jj >= 0; jj--) {
        const int t0 = jj * K, t1 = std::min(t0 + K, steps);
        const int odd = whole_f_ ? (t1 - t0) & 1 : 0;  // the buffers that the segment starts from
        if (jj == 0) {
          for (size_t p = 0; p < gp.member.size(); p++) {
            DeviceState& d = *M[gp.member[p]].d;
            TRY(d.zero_shots(d.fwd, kWaveComps, gp.s0[p], gp.n[p], st));
            TRY(d.zero_shots(d.mem, kMemComps, gp.s0[p], gp.n[p], st));
          }
          if (odd) TRY(clear_second(rg));
        } else {
          TRY(snapshot(rg, sw.r0, jj, false, odd));
        }
        TRY(forward(rg, t0, t1, [](int, int) { return Status::Ok(); }));
        if (d0->adjoint)
          xsegment(t0, t1);
        else
          segment(t0, t1, jj == nseg - 1);
      }
      HIP_TRY(hipGetLastError());
    }
  }
  // misfit and gradients
  for (const Member& m : M) {
    DeviceState& d = *m.d;
    if (if_res) {
      if (d.cond)
        hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, st, d.cpart,
                           d.g.ns * kCondBlocks, d.misfit);
      else
        hipLaunchKernelGGL(k_sum_partials, dim3(1), dim3(256), 0, st, d.partial,
                           (int)sweeps.size() * kPartials, d.misfit);
    }
    if (withAdj)
      hipLaunchKernelGGL(k_finalize, dim3((d.g.nz + 255) / 256, d.g.nx), dim3(256), 0, st, d.g,
                         d.mdl(), d.acc, d.grad, d.adjoint);
  }
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipStreamSynchronize(st));
  if (d0->timing) d0->collect_timing();
  for (const Member& m : M) {
    DeviceState& d = *m.d;
    if (if_res) HIP_TRY(hipMemcpy(&d.misfit_host, d.misfit, sizeof(double), hipMemcpyDeviceToHost));
    m.plan->last_calc = calc_id;
    d.illum_valid = d.illum_on;
  }
  return Status::Ok();
}

}  // namespace

Status Plan::run(int calc_id) {
  TRY(check_calc_id(calc_id));
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  HIP_TRY(hipSetDevice(d_->dev));
  if (!d_->cache) {
    d_->cache.reset(new JobCache());
    d_->cache->dev = d_->dev;
    d_->cache->arena = d_->arena;
  }
  Runner r({Member{this, d_.get()}}, *d_->cache);
  return r.run(calc_id);
}

Job::Job() = default;
Job::~Job() {
  if (cache_) {
    (void)hipSetDevice(cache_->dev);
    cache_.reset();
  }
}

Status Job::add(Plan* p) {
  if (!p || !p->d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  if ((int)plans_.size() >= kMaxPartsTable)
    return Status::Err(FWIFLOW_ERR_ARG, "at most " + std::to_string(kMaxPartsTable) + " plans per job");
  for (Plan* q : plans_)
    if (q == p) return Status::Err(FWIFLOW_ERR_ARG, "plan already in the job");
  if (p->d_->arena)
    return Status::Err(FWIFLOW_ERR_ARG, "a plan in the device scratch cannot join a job");
  if (!plans_.empty()) {
    const DeviceState& a = *plans_[0]->d_;
    if (p->d_->dev != a.dev) return Status::Err(FWIFLOW_ERR_ARG, "plans of a job must share the GPU");
    if (p->d_->g.nSteps != a.g.nSteps)
      return Status::Err(FWIFLOW_ERR_ARG, "plans of a job must share nSteps");
  }
  plans_.push_back(p);
  cache_.reset();  // maps depend on the members
  return Status::Ok();
}

Status Job::run(int calc_id) {
  if (plans_.empty()) return Status::Err(FWIFLOW_ERR_ARG, "empty job");
  HIP_TRY(hipSetDevice(plans_[0]->d_->dev));
  // Fused launches (every launch covers a group of shots of every plan) or
  // the plans one after another.  The fused groups are sized by the
  // Infinity-Cache rule on the plans' summed bytes per shot, so a fused
  // backward launch holds fewer shots of each plan than that plan's own
  // launches would, and every launch re-reads every plan's model and
  // gradient accumulators for those few shots.  Fusing pays only where the
  // plans are small enough that their own launches would be no larger;
  // FWIFLOW_JOB_FUSE = 1 / 0 forces either.
  int fuse = env_int("FWIFLOW_JOB_FUSE", -1);
  if (fuse < 0 && plans_.size() > 1) {
    auto group = [](double bytes_per_row, int rows) {
      return std::max(1, std::min(rows, (int)std::lround(224e6 / bytes_per_row)));
    };
    double sum = 0;
    int rows = 0, solo = 1 << 30;
    for (Plan* p : plans_) {
      const DeviceState& d = *p->d_;
      sum += d.bwd_bytes_per_shot();
      rows = std::max(rows, d.g.ns);
      solo = std::min(solo, d.shot_group_bwd > 0 ? std::min(d.shot_group_bwd, d.g.ns)
                                                 : group(d.bwd_bytes_per_shot(), d.g.ns));
    }
    const int fused = plans_[0]->d_->shot_group_bwd > 0
                          ? std::min(plans_[0]->d_->shot_group_bwd, rows)
                          : group(sum, rows);
    fuse = fused >= solo ? 1 : 0;
  }
  // the exact adjoint runs one plan at a time
  for (Plan* p : plans_)
    if (p->d_->adjoint) fuse = 0;
  last_fused_ = fuse != 0 || plans_.size() == 1;
  if (!last_fused_) {
    for (Plan* p : plans_) TRY(p->run(calc_id));
    return Status::Ok();
  }
  if (!cache_) {
    cache_.reset(new JobCache());
    cache_->dev = plans_[0]->d_->dev;
  }
  std::vector<Member> m;
  for (Plan* p : plans_) m.push_back(Member{p, p->d_.get()});
  Runner r(std::move(m), *cache_);
  return r.run(calc_id);
}

int Job::size() const { return (int)plans_.size(); }
bool Job::fused() const { return last_fused_; }

Status Plan::misfit(double* out) {
  if (!d_ || (last_calc != 0 && last_calc != 1))
    return Status::Err(FWIFLOW_ERR_ARG, "no calc_id 0 or 1 result");
  if (out) *out = 0.5 * d_->misfit_host;
  return Status::Ok();
}

// Arrays of the grid, one after another at `in`, to the caller's doubles (null:
// not asked for): z fastest -> row-major [NZ][NX] (libCUFD.cu:480-486).
// Small grids come over as they are in one copy and are turned here: a kernel
// and a copy an array take longer.  Gradients, us, turned on the device / here:
// 8064 cells 66 / 39, 11904 71 / 42, 15872 75 / 54, 28672 91 / 101; illumination
// 27 / 13, 28 / 15, 30 / 19, 35 / 39.
constexpr size_t kHostTurn = 20480;  // cells
static Status fetch_turned(DeviceState& d, const float* in, std::vector<double*> outs) {
  const size_t nz = (size_t)d.g.nz, nx = (size_t)d.g.nx, N = (size_t)d.g.N, n = outs.size();
  if (N <= kHostTurn) {
    std::vector<float> h(n * N);
    HIP_TRY(hipMemcpyAsync(h.data(), in, h.size() * sizeof(float), hipMemcpyDeviceToHost, d.stream));
    HIP_TRY(hipStreamSynchronize(d.stream));
    for (size_t k = 0; k < n; k++)
      for (size_t z = 0; outs[k] && z < nz; z++)
        for (size_t x = 0; x < nx; x++) outs[k][z * nx + x] = h[k * N + x * nz + z];
    return Status::Ok();
  }
  double* const out = (double*)d.mem;  // every run clears it
  Turn t{};
  for (size_t k = 0; k < n; k++) t.in[k] = in + k * N, t.out[k] = out + k * N;
  hipLaunchKernelGGL((k_turn<float, double>), dim3((d.g.nz + 31) / 32, (d.g.nx + 31) / 32, (unsigned)n),
                     dim3(32, 8), 0, d.stream, t, d.g.nx, d.g.nz, 0);
  HIP_TRY(hipGetLastError());
  for (size_t k = 0; k < n; k++)
    if (outs[k])
      HIP_TRY(hipMemcpyAsync(outs[k], out + k * N, N * sizeof(double), hipMemcpyDeviceToHost, d.stream));
  HIP_TRY(hipStreamSynchronize(d.stream));
  return Status::Ok();
}

Status Plan::gradients(double* gL, double* gM, double* gD, double* gS) {
  if (!d_ || last_calc != 1) return Status::Err(FWIFLOW_ERR_ARG, "no calc_id 1 result");
  DeviceState& d = *d_;
  HIP_TRY(hipSetDevice(d.dev));
  TRY(fetch_turned(d, d.grad, {gL, gM, gD}));
  if (gS) {
    std::vector<float> s((size_t)d.g.ns * d.g.nSteps);
    HIP_TRY(hipMemcpy(s.data(), d.stf_grad, s.size() * sizeof(float), hipMemcpyDeviceToHost));
    for (size_t k = 0; k < s.size(); k++) gS[k] = s[k];
  }
  return Status::Ok();
}

Status Plan::set_illumination(bool on) {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  d_->illum_on = on;
  return Status::Ok();
}

Status Plan::illumination(double* out) {
  if (!d_ || !d_->illum_valid)
    return Status::Err(FWIFLOW_ERR_ARG, "no run with the illumination enabled");
  if (!out) return Status::Err(FWIFLOW_ERR_ARG, "null output pointer");
  DeviceState& d = *d_;
  HIP_TRY(hipSetDevice(d.dev));
  return fetch_turned(d, d.illum, {out});
}

Status Plan::data(float* syn) {
  if (!d_ || last_calc < 0) return Status::Err(FWIFLOW_ERR_ARG, "no run result");
  if (!syn) return Status::Err(FWIFLOW_ERR_ARG, "null output pointer");
  DeviceState& d = *d_;
  HIP_TRY(hipSetDevice(d.dev));
  TRY(ensure_obs_buffers(d));
  const size_t T = (size_t)d.g.nSteps * d.R;
  // time-major [nSteps][R] -> [R][nSteps] (Shot file layout, utilities.cu:557-567)
  dim3 blk(32, 8), grd((d.R + 31) / 32, (d.g.nSteps + 31) / 32);
  hipLaunchKernelGGL(k_transpose, grd, blk, 0, d.stream, d.syn, d.stage, d.g.nSteps, d.R);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(syn, d.stage, T * sizeof(float), hipMemcpyDeviceToHost, d.stream));
  HIP_TRY(hipStreamSynchronize(d.stream));
  return Status::Ok();
}

Status Plan::write_data() {
  if (!d_) return Status::Err(FWIFLOW_ERR_ARG, "plan not created");
  std::vector<float> h((size_t)para.nSteps * d_->R);
  TRY(data(h.data()));
  size_t off = 0;
  for (const Shot& sh : survey.shots) {
    const std::string fn = para.data_dir + "/Shot" + std::to_string(sh.id) + ".bin";
    FILE* fp = std::fopen(fn.c_str(), "wb");
    if (!fp) return Status::Err(FWIFLOW_ERR_IO, "cannot write \"" + fn + "\"");
    const size_t n = sh.z_rec.size() * (size_t)para.nSteps;
    const size_t put = std::fwrite(h.data() + off, sizeof(float), n, fp);
    std::fclose(fp);
    if (put != n) return Status::Err(FWIFLOW_ERR_IO, "short write to \"" + fn + "\"");
    off += n;
  }
  return Status::Ok();
}

Status Plan::residual(float* res) {
  if (!d_ || (last_calc != 0 && last_calc != 1))
    return Status::Err(FWIFLOW_ERR_ARG, "no calc_id 0 or 1 result");
  if (!res) return Status::Err(FWIFLOW_ERR_ARG, "null output pointer");
  DeviceState& d = *d_;
  HIP_TRY(hipSetDevice(d.dev));
  const size_t T = (size_t)d.g.nSteps * d.R;
  dim3 blk(32, 8), grd((d.R + 31) / 32, (d.g.nSteps + 31) / 32);
  hipLaunchKernelGGL(k_transpose, grd, blk, 0, d.stream, d.res, d.stage, d.g.nSteps, d.R);
  HIP_TRY(hipGetLastError());
  HIP_TRY(hipMemcpyAsync(res, d.stage, T * sizeof(float), hipMemcpyDeviceToHost, d.stream));
  HIP_TRY(hipStreamSynchronize(d.stream));
  return Status::Ok();
}

Status Plan::source(float* rows) {
  if (!d_ || !d_->stf_set) return Status::Err(FWIFLOW_ERR_ARG, "no source set");
  if (!rows) return Status::Err(FWIFLOW_ERR_ARG, "null output pointer");
  DeviceState& d = *d_;
  HIP_TRY(hipSetDevice(d.dev));
  const float* p = d.src_updated ? d.srcout : d.srcamp;
  HIP_TRY(hipMemcpy(rows, p, (size_t)d.g.ns * d.g.nSteps * sizeof(float), hipMemcpyDeviceToHost));
  return Status::Ok();
}

// libCUFD.cu:493-511: after a gradient run, per shot the residual, the
// conditioned synthetic and observed data and the source row.
Status Plan::write_scratch() {
  if (!d_ || last_calc != 1) return Status::Err(FWIFLOW_ERR_ARG, "no calc_id 1 result");
  DeviceState& d = *d_;
  if (!para.save_scratch) return Status::Ok();
  const int nt = para.nSteps;
  if (d.keep_obs.size() != (size_t)d.R * nt)
    return Status::Err(FWIFLOW_ERR_ARG, "conditioned data of the last run were not kept");
  std::vector<float> res((size_t)d.R * nt), src((size_t)d.g.ns * nt);
  TRY(residual(res.data()));
  TRY(source(src.data()));
  auto put = [&](const std::string& fn, const float* p, size_t n) -> Status {
    FILE* fp = std::fopen(fn.c_str(), "wb");
    if (!fp) return Status::Err(FWIFLOW_ERR_IO, "cannot write \"" + fn + "\"");
    const size_t w = std::fwrite(p, sizeof(float), n, fp);
    std::fclose(fp);
    if (w != n) return Status::Err(FWIFLOW_ERR_IO, "short write to \"" + fn + "\"");
    return Status::Ok();
  };
  for (int s = 0; s < d.g.ns; s++) {
    const std::string id = std::to_string(survey.shots[s].id), dir = para.scratch_dir + "/";
    const size_t off = (size_t)d.roff[s] * nt, n = (size_t)(d.roff[s + 1] - d.roff[s]) * nt;
    TRY(put(dir + "Residual_Shot" + id + ".bin", res.data() + off, n));
    TRY(put(dir + "Syn_Shot" + id + ".bin", d.keep_syn.data() + off, n));
    TRY(put(dir + "CondObs_Shot" + id + ".bin", d.keep_obs.data() + off, n));
    TRY(put(dir + "src_updated" + id + ".bin", src.data() + (size_t)s * nt, (size_t)nt));
  }
  return Status::Ok();
}

}  // namespace fwiflow
