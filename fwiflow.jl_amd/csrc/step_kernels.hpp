// Whole-step kernels: one launch per time step (included by engine.hip, inside
// its anonymous namespace, after the arithmetic and addressing helpers).
//
// A workgroup of 64 x 8 threads owns a tile of 64 depth cells x 8 columns, one
// cell per thread, and walks the shots of its slice.  Per shot it applies the
// first half of the step to the whole tile from the state in memory, leaves
// what the second half differentiates in LDS, and applies the second half to
// the tile's core, 60 x 4 cells.  The first half's results in the 2-cell rim
// are the neighbouring tiles' own: they are computed again here, by the same
// operations on the same values.  The new state goes to a second set of
// buffers, which the next step reads, since a neighbour may still read the old
// one.
//
// These launches serve grids that do not fill the chip, where a launch is all
// latency: the host's 2.5 us to send it, then the workgroup's chain of argument,
// coefficient and state loads.  Half the launches and no second read of the
// first half's results, arguments in cached device memory and tiles by index
// arithmetic (a map of tiles and arguments in the uncached kernel argument
// segment cost 440 scalar instructions a wave): modelling of 2 shots of 64x84
// 2.9 -> 1.18 ms for 300 steps, 164x264 x 1 shot 9.0 -> 4.25 ms for 1000, its
// gradient 18.7 -> 10.2 ms.  6, 10, 12 or 16 columns a tile: 14, 2, 8, 15% slower.

constexpr int kStepW = 8;         // columns of a tile
constexpr int kCoreZ = kBZ - 4;   // depth cells of its core
constexpr int kCoreX = kStepW - 4;  // and columns

// One plan's shots in one whole-step launch.  Read through scalar loads from
// cached device memory: as a kernel argument the same fields cost a chain of
// uncached scalar loads in every workgroup.
struct StepArgs {
  const float* wi;   // state read: [shot][5][cell] from the part's first shot
  float* wo;         // state written
  const float* mi;   // C-PML memory variables read / written: [shot][8][cell]
  float* mo;
  const float* md;   // [lam, mu, amu, ba, bb][cell]
  const float* zc;   // C-PML coefficients of row z: K, 1/K, a, b, Kh, 1/Kh, ah, bh
  const float* xc;   // ... of column x
  const int* zx;     // source cell of each shot
  const float* amp;  // source rows
  float* ring;       // boundary ring (null: not saved)
  float* illum;      // forward illumination planes (null: off)
  const int* rec;    // receivers (z, x, plan shot)
  float* syn;
  int nz, nx, nzA, nPml;
  int ns, nSteps, nrec, s0;
  float dt, dz, dx, rdz, rdx;
  int Nb;            // bytes of one array
  int R, ringW, ringH, ringlen, rs0, rnt;
  int gz;            // strips of tiles along z
  int per;           // tiles along x of one XCD
  int gx;            // tiles along x
  int hgz, hper, hgx;  // the same of the half steps' 64 x 4 tiles
};
typedef const __attribute__((address_space(4))) StepArgs CStep;
typedef const __attribute__((address_space(4))) float CFloat;
typedef const __attribute__((address_space(4))) int CInt;

// C-PML coefficients of one row or column
struct Coef {
  float K, r, a, b, Kh, rh, ah, bh;
};
__device__ __forceinline__ Coef coef_row(const float* zc, int z) {
  const f4 p = *(const f4*)(zc + 8 * z), q = *(const f4*)(zc + 8 * z + 4);
  return Coef{p[0], p[1], p[2], p[3], q[0], q[1], q[2], q[3]};
}
__device__ __forceinline__ Coef coef_col(const float* xc, int x) {  // wave-uniform x
  CFloat* c = (CFloat*)xc + 8 * x;
  return Coef{c[0], c[1], c[2], c[3], c[4], c[5], c[6], c[7]};
}
__device__ __forceinline__ float kdiv(float x, float K, float r) {
  return K == 1.f ? x : div2(x, K, r);
}
__device__ __forceinline__ void stb(Rsrc r, int so, int vo, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, vo, so, 0);
}
__device__ __forceinline__ f4 ldb4(Rsrc r, int so, int vo) { return raw_load4(r, vo, so, 0); }

// Where a forward workgroup works: x tiles in XCD bands (workgroup b runs on
// XCD b % 8 when gridDim.x is a multiple of 8), strips along y, slices of shots
// and parts along z.
struct Place {
  int part, slice, lo, hi;
};
__device__ __forceinline__ Place place_of(int k, int slices, int per_slice) {
  int part = 0;
  while (k >= slices) k -= slices, ++part;
  return Place{part, k, k * per_slice, (k + 1) * per_slice};
}

// Sums over a launch's shots are taken in shot order, so that they do not
// depend on how the shots are spread over waves.  Sliced: the workgroup holds
// blockDim.z threads per cell; in rounds of kSumShots shots each takes a run of
// them and leaves its contributions in LDS, which then are added up in order,
// thread k % blockDim.z of a cell adding sum k.  body(s, c) handles shot s and
// sets its contributions c; it is called by `live` threads, and the sums go to
// acc[k][cell] (byte offset v0) where `in`.
constexpr int kSumShots = 8;  // 8 shots x 3 sums x 256 cells: 24 KB of LDS
constexpr int kSumCells = kBZ * 4;
template <int C, bool Sliced, typename F>
__device__ __forceinline__ void sum_shots(int ns, bool live, bool in, float* lds, Rsrc acc, int first,
                                          int Nb, int v0, F&& body) {
  const int S = Sliced ? (int)blockDim.z : 1;
  const int tz = Sliced ? __builtin_amdgcn_readfirstlane((int)threadIdx.z) : 0;
  float g0[C] = {}, g[C] = {};
  if (in)
#pragma unroll
    for (int k = 0; k < C; ++k)
      if (k % S == tz) g0[k] = ldb(acc, (first + k) * Nb, v0);
  if (!Sliced) {
    if (live)
      for (int s = 0; s < ns; ++s) {
        float c[C] = {};
        body(s, c);
#pragma unroll
        for (int k = 0; k < C; ++k) g[k] += c[k];
      }
  } else {
    float* const own = lds + (int)threadIdx.y * kBZ + (int)threadIdx.x;
    for (int base = 0; base < ns; base += kSumShots) {
      const int n = min(kSumShots, ns - base), per = (n + S - 1) / S;
      if (live)
        for (int i = tz * per; i < min(n, (tz + 1) * per); ++i) {
          float c[C] = {};
          body(base + i, c);
#pragma unroll
          for (int k = 0; k < C; ++k) own[(i * C + k) * kSumCells] = c[k];
        }
      __syncthreads();
      if (in)
#pragma unroll
        for (int k = 0; k < C; ++k)
          if (k % S == tz)
            for (int i = 0; i < n; ++i) g[k] += own[(i * C + k) * kSumCells];
      if (base + kSumShots < ns) __syncthreads();
    }
  }
  if (in)
#pragma unroll
    for (int k = 0; k < C; ++k)
      if (k % S == tz) stb(acc, (first + k) * Nb, v0, g0[k] + g[k]);
}
// the shots [lo, hi) of a thread where nothing is summed
template <bool Sliced>
__device__ __forceinline__ void own_shots(int ns, int& lo, int& hi) {
  lo = 0, hi = ns;
  if (Sliced) {
    const int S = (int)blockDim.z, per = (ns + S - 1) / S;
    lo = __builtin_amdgcn_readfirstlane((int)threadIdx.z) * per, hi = min(ns, lo + per);
  }
}

// The forward illumination of launches whose shots are spread over workgroups:
// sum over shots of vz^2 + vx^2 of the state that the launch reads (a launch in
// which one thread walks all shots of a cell adds its results itself).
__device__ __forceinline__ void illum_cell(CStep& A, int i) {
  const int N = A.Nb / 4, x = i / A.nz, z = i - x * A.nz;
  if (i >= N || z < 2 || z > A.nzA - 3 || x < 2 || x > A.nx - 3) return;
  const float* w = A.wi + i;
  float il = 0.f;
#pragma unroll 4
  for (int s = 0; s < A.ns; ++s, w += (size_t)kWaveComps * N) {
    const float vz = w[kVz * (size_t)N], vx = w[kVx * (size_t)N];
    il += vz * vz + vx * vx;
  }
  A.illum[i] += il;
}

// receiver r of the part: sample it of its trace (recording, utilities.cu:557-567)
__device__ __forceinline__ void record_cell(CStep& A, int r, int it) {
  if (r >= A.nrec) return;
  const size_t N = (size_t)(A.Nb / 4);
  const int z = A.rec[3 * r], x = A.rec[3 * r + 1], s = A.rec[3 * r + 2] - A.s0;
  const float* w = A.wi + (size_t)s * kWaveComps * N + (size_t)x * A.nz + z;
  A.syn[(size_t)it * A.R + r] = (float)((double)w[kSzz * N] + kRS * (double)w[kSxx * N]);
}

__device__ __forceinline__ Geo ring_geo(CStep& A) {
  Geo g{};
  g.nz = A.nz, g.nx = A.nx, g.nzA = A.nzA, g.nPml = A.nPml;
  g.ringW = A.ringW, g.ringH = A.ringH, g.ringlen = A.ringlen, g.rs0 = A.rs0, g.rnt = A.rnt;
  return g;
}
// cell of a ring slot (the inverse of ring_slot)
__device__ __forceinline__ void ring_cell(const Geo& g, int slot, int& z, int& x) {
  const int W = g.ringW, hz = g.ringH - 10;
  int zr, xr;
  if (slot < 10 * W) {
    const int q = slot < 5 * W ? slot : slot - 5 * W;
    xr = q / 5;
    zr = q - 5 * xr + (slot < 5 * W ? 0 : g.ringH - 5);
  } else {
    const int q = slot - 10 * W, c = q / hz;
    zr = q - c * hz + 5;
    xr = c < 5 ? c : W - 10 + c;
  }
  z = zr + g.nPml - 2;
  x = xr + g.nPml - 2;
}
// components [c0, c1) of ring slot i, row `row` of the ring: saved from (Save,
// from_bnd, utilities.cu:361-391) or restored to (to_bnd, 394-424) `state`.
// Ring order: szz, sxz, sxx, vz, vx.
template <bool Save>
__device__ __forceinline__ void ring_move(CStep& A, float* state, int i, int lo, int hi, int row,
                                          int c0, int c1) {
  if (!A.ring || row < 0 || i < 0 || i >= A.ringlen) return;
  const Geo g = ring_geo(A);
  int z, x;
  ring_cell(g, i, z, x);
  constexpr int comp[5] = {kSzz, kSxz, kSxx, kVz, kVx};
  const size_t N = (size_t)(A.Nb / 4);
  for (int s = lo; s < hi; ++s) {
    float* w = state + (size_t)s * kWaveComps * N + (size_t)x * A.nz + z;
    float* r = A.ring + (((size_t)A.rs0 + s) * A.rnt + row) * 5 * (size_t)A.ringlen + i;
#pragma unroll
    for (int c = 0; c < 5; ++c)
      if (c >= c0 && c < c1) {
        if (Save)
          r[(size_t)c * A.ringlen] = w[comp[c] * N];
        else
          w[comp[c] * N] = r[(size_t)c * A.ringlen];
      }
  }
}

// Forward step it: el_stress.cu:50-88 + add_source (utilities.cu:521-555), then
// el_velocity.cu:45-82.  The grid's rows beyond the strips save the boundary
// ring and record, both from the state that the step reads: the ring of step
// it and sample it (the last sample is recorded by k_record).
__global__ __launch_bounds__(64 * kStepW) void k_step_fwd(const StepArgs* __restrict__ args, int it,
                                                     int ring, int slices, int per_slice) {
  __shared__ float ss[2][3][kStepW][kBZ];  // new stresses of the shot at hand, two buffers
  const Place pl = place_of((int)blockIdx.z, slices, per_slice);
  CStep& A = ((CStep*)args)[pl.part];
  const int hi = min(pl.hi, A.ns);
  const int lane = (int)threadIdx.x, j = wave_col(0), strip = (int)blockIdx.y;
  const int bx = ((int)blockIdx.x & 7) * A.per + ((int)blockIdx.x >> 3);
  if (strip >= A.gz) {
    const int i = (((strip - A.gz) * (int)gridDim.x + (int)blockIdx.x) * kStepW + j) * 64 + lane;
    const int ringpad = A.ring ? (A.ringlen + 63) & ~63 : 0;
    const int recpad = ringpad + ((A.nrec + 63) & ~63);
    if (i < ringpad)
      ring_move<true>(A, const_cast<float*>(A.wi), i, pl.lo, hi, ring, 0, 5);
    else if (i < recpad && !pl.slice)
      record_cell(A, i - ringpad, it);
    else if (A.illum && slices > 1 && !pl.slice)
      illum_cell(A, i - recpad);
    return;
  }
  if (((int)blockIdx.x >> 3) >= A.per || bx >= A.gx) return;
  const int nz = A.nz, nx = A.nx, nzA = A.nzA, nPml = A.nPml, Nb = A.Nb;
  const float dt = A.dt, dz = A.dz, dx = A.dx, rdz = A.rdz, rdx = A.rdx;
  const double dt64 = (double)dt;
  const int z0 = strip * kCoreZ, z = z0 + lane, x = bx * kCoreX + j;
  // loads of lanes and columns outside the update region are moved inside it;
  // their results are dropped
  const int xl = min(max(x, 2), nx - 3), zl = min(max(z, 2), nzA - 3);
  const bool valid = z == zl && x == xl;
  const bool core = valid && lane >= 2 && lane < kBZ - 2 && j >= 2 && j < kStepW - 2;
  const bool E = z0 < nPml || z0 + kBZ > nzA - nPml;  // the tile holds C-PML rows
  const bool pz = E && (zl < nPml || zl > nzA - nPml - 1);
  const bool px = xl < nPml || xl > nx - nPml - 1;    // el_stress's gate
  const bool pv = xl < nPml || xl > nx - nPml;        // el_velocity's gate
  const int v0 = 4 * (xl * nz + zl), cb = 4 * nz;
  const int vm1 = v0 - cb, vm2 = vm1 - cb, vp1 = v0 + cb, vp2 = vp1 + cb;
  const Rsrc wi = rsrc(A.wi), wo = rsrc(A.wo), mi = rsrc(A.mi), mo = rsrc(A.mo), md = rsrc(A.md);
  const float lam = ldb(md, 0, v0), mu = ldb(md, Nb, v0), amu = ldb(md, 2 * Nb, v0),
              ba = ldb(md, 3 * Nb, v0), bb = ldb(md, 4 * Nb, v0);
  const double l2m = (double)lam + 2.0 * (double)mu;  // (d_Lambda + 2.0*d_Mu)
  Coef Z{}, X{};
  if (pz) Z = coef_row(A.zc, zl);
  if (px) X = coef_col(A.xc, xl);  // px holds wherever pv does
  float il = 0.f;
  int buf = 0;
  for (int s = pl.lo; s < hi; ++s, buf ^= 1) {
    const int sw = s * kWaveComps * Nb, sm = s * kMemComps * Nb;
    const f4 vzc = ldb4(wi, sw + kVz * Nb, v0 - 8), vxc = ldb4(wi, sw + kVx * Nb, v0 - 4);
    const float vzp = ldb(wi, sw + kVz * Nb, vp1), vzp2 = ldb(wi, sw + kVz * Nb, vp2),
                vzm = ldb(wi, sw + kVz * Nb, vm1);
    const float vxm = ldb(wi, sw + kVx * Nb, vm1), vxp = ldb(wi, sw + kVx * Nb, vp1),
                vxm2 = ldb(wi, sw + kVx * Nb, vm2);
    float szz = ldb(wi, sw + kSzz * Nb, v0), sxx = ldb(wi, sw + kSxx * Nb, v0),
          sxz = ldb(wi, sw + kSxz * Nb, v0);
    float m0 = 0.f, m1 = 0.f, n0 = 0.f, n1 = 0.f;
    if (pz) m0 = ldb(mi, sm + kMvzz * Nb, v0), m1 = ldb(mi, sm + kMvxz * Nb, v0);
    if (px) n0 = ldb(mi, sm + kMvxx * Nb, v0), n1 = ldb(mi, sm + kMvzx * Nb, v0);
    const float vz0 = vzc[2], vx0 = vxc[1];
    float dvz_dz = dfw(vz0, vzc[1], vzc[3], vzc[0], dz, rdz);
    float dvx_dx = dfw(vx0, vxm, vxp, vxm2, dx, rdx);
    float dvx_dz = dfw(vxc[2], vx0, vxc[3], vxc[0], dz, rdz);
    float dvz_dx = dfw(vzp, vz0, vzp2, vzm, dx, rdx);
    if (pz) {
      m0 = Z.b * m0 + Z.a * dvz_dz;
      dvz_dz = kdiv(dvz_dz, Z.K, Z.r) + m0;
      m1 = Z.bh * m1 + Z.ah * dvx_dz;
      dvx_dz = kdiv(dvx_dz, Z.Kh, Z.rh) + m1;
    }
    if (px) {
      n0 = X.b * n0 + X.a * dvx_dx;
      dvx_dx = kdiv(dvx_dx, X.K, X.r) + n0;
      n1 = X.bh * n1 + X.ah * dvz_dx;
      dvz_dx = kdiv(dvz_dx, X.Kh, X.rh) + n1;
    }
    szz = (float)((double)szz + (l2m * (double)dvz_dz + (double)(lam * dvx_dx)) * dt64);
    sxx = (float)((double)sxx + ((double)(lam * dvz_dz) + l2m * (double)dvx_dx) * dt64);
    sxz = sxz + amu * (dvx_dz + dvz_dx) * dt;
    if (x == ((CInt*)A.zx)[2 * s + 1] && z == ((CInt*)A.zx)[2 * s]) {
      // add_source: szz += scale*amp*dt*gauss (float), sxx += RSXXZZ*scale*amp*dt*gauss
      // (double); the 9x9 Gaussian is 1 at the centre and 0 elsewhere in FP32
      const float amp = A.amp[(size_t)s * A.nSteps + it];
      szz = szz + kSrcScale * amp * dt;
      sxx = (float)((double)sxx + kRS * (double)kSrcScale * (double)amp * dt64);
    }
    ss[buf][0][j][lane] = valid ? szz : 0.f;
    ss[buf][1][j][lane] = valid ? sxx : 0.f;
    ss[buf][2][j][lane] = valid ? sxz : 0.f;
    if (core) {
      stb(wo, sw + kSzz * Nb, v0, szz);
      stb(wo, sw + kSxx * Nb, v0, sxx);
      stb(wo, sw + kSxz * Nb, v0, sxz);
      if (pz) stb(mo, sm + kMvzz * Nb, v0, m0), stb(mo, sm + kMvxz * Nb, v0, m1);
      if (px) stb(mo, sm + kMvxx * Nb, v0, n0), stb(mo, sm + kMvzx * Nb, v0, n1);
      if (pz) m0 = ldb(mi, sm + kMszz * Nb, v0), m1 = ldb(mi, sm + kMsxzz * Nb, v0);
      if (pv) n0 = ldb(mi, sm + kMsxzx * Nb, v0), n1 = ldb(mi, sm + kMsxx * Nb, v0);
    }
    __syncthreads();
    if (core) {
      const float *tz = &ss[buf][0][j][lane], *tx = &ss[buf][1][j][lane], *ts = &ss[buf][2][j][lane];
      float dszz_dz = dfw(tz[1], tz[0], tz[2], tz[-1], dz, rdz);
      float dsxz_dx = dfw(sxz, ts[-kBZ], ts[kBZ], ts[-2 * kBZ], dx, rdx);
      float dsxz_dz = dfw(sxz, ts[-1], ts[1], ts[-2], dz, rdz);
      float dsxx_dx = dfw(tx[kBZ], sxx, tx[2 * kBZ], tx[-kBZ], dx, rdx);
      if (pz) {
        m0 = Z.bh * m0 + Z.ah * dszz_dz;
        stb(mo, sm + kMszz * Nb, v0, m0);
        dszz_dz = kdiv(dszz_dz, Z.Kh, Z.rh) + m0;
        m1 = Z.b * m1 + Z.a * dsxz_dz;
        stb(mo, sm + kMsxzz * Nb, v0, m1);
        dsxz_dz = kdiv(dsxz_dz, Z.K, Z.r) + m1;
      }
      if (pv) {
        n0 = X.b * n0 + X.a * dsxz_dx;
        stb(mo, sm + kMsxzx * Nb, v0, n0);
        dsxz_dx = kdiv(dsxz_dx, X.K, X.r) + n0;
        n1 = X.bh * n1 + X.ah * dsxx_dx;
        stb(mo, sm + kMsxx * Nb, v0, n1);
        dsxx_dx = kdiv(dsxx_dx, X.Kh, X.rh) + n1;
      }
      const float vz = vz0 + (dszz_dz + dsxz_dx) * ba * dt;
      const float vx = vx0 + (dsxz_dz + dsxx_dx) * bb * dt;
      stb(wo, sw + kVz * Nb, v0, vz);
      stb(wo, sw + kVx * Nb, v0, vx);
      il += vz * vz + vx * vx;
    }
  }
  if (A.illum && slices == 1 && core) A.illum[x * nz + z] += il;
}

// the stresses that the last step left, recorded as sample it
__global__ __launch_bounds__(256) void k_record(const StepArgs* __restrict__ args, int it) {
  record_cell(((CStep*)args)[blockIdx.z], (int)(blockIdx.x * 256 + threadIdx.x), it);
}
// and its velocities, where the step's launch did not add them itself
__global__ __launch_bounds__(256) void k_illum(const StepArgs* __restrict__ args) {
  CStep& A = ((CStep*)args)[blockIdx.z];
  if (A.illum) illum_cell(A, (int)(blockIdx.x * 256 + threadIdx.x));
}

// ------------------------------------------------------------------ backward
// Residual entering a column of one shot: its injection cells (sorted by row)
// from `first`; with exactly one receiver in the column, its row and index.
struct ColInj {
  int first, n, z, rid;
};

struct BackArgs {
  StepArgs s;        // wi / wo: forward state, mi / mo: adjoint memory variables
  const float* ai;   // adjoint state read / written
  float* ao;
  const double *zd, *xd;  // 1 / K in double by row and column
  const float* res;  // time-major residual
  const ColInj* inj; // [shot][column]
  const int *icell, *iptr, *irid;
  float* acc;        // gradient accumulators [5][cell]
  int rgz, rper, rgx;  // tiles of the ring rectangle: strips, along x of one XCD, along x
  float* stf_grad;
};
typedef const __attribute__((address_space(4))) BackArgs CBack;

// The adjoint half of a backward step, update region, tiles as the forward's:
// el_velocity_adj.cu:22-108 with source_grad (utilities.cu:582-593) on the
// tile, then the residual of sample it (res_injection, utilities.cu:569-580)
// and el_stress_adj.cu:22-104 on the core.  The memory variables of the
// stress update are kept where they are ever read with a non-zero coefficient:
// the C-PML layers and the stencil's 2-cell reach.
__device__ __forceinline__ void step_adj(CBack& B, int lo, int hi, int strip, int bx, int it,
                                         float (&lds)[6][kStepW][kBZ]) {
  const auto& A = B.s;
  const int lane = (int)threadIdx.x, j = wave_col(0);
  const int nz = A.nz, nx = A.nx, nzA = A.nzA, nPml = A.nPml, Nb = A.Nb;
  const float dt = A.dt, dz = A.dz, dx = A.dx, rdz = A.rdz, rdx = A.rdx;
  const double dt64 = (double)dt;
  const int z0 = strip * kCoreZ, z = z0 + lane, x = bx * kCoreX + j;
  const int xl = min(max(x, 2), nx - 3), zl = min(max(z, 2), nzA - 3);
  const bool valid = z == zl && x == xl;
  const bool core = valid && lane >= 2 && lane < kBZ - 2 && j >= 2 && j < kStepW - 2;
  const bool E = z0 < nPml + 2 || z0 + kBZ > nzA - nPml - 2;  // the tile holds live rows
  const bool pz = E && (zl < nPml || zl > nzA - nPml - 1);
  const bool px = xl < nPml || xl > nx - nPml - 1;
  const bool zlive = E && (zl <= nPml + 1 || zl >= nzA - nPml - 2);
  const bool xlive = xl <= nPml + 1 || xl >= nx - nPml - 2;
  const int v0 = 4 * (xl * nz + zl), cb = 4 * nz;
  const int vm1 = v0 - cb, vm2 = vm1 - cb, vp1 = v0 + cb, vp2 = vp1 + cb;
  const Rsrc ai = rsrc(B.ai), ao = rsrc(B.ao), mi = rsrc(A.mi), mo = rsrc(A.mo), md = rsrc(A.md);
  const float lam = ldb(md, 0, v0), mu = ldb(md, Nb, v0), amu = ldb(md, 2 * Nb, v0),
              ba = ldb(md, 3 * Nb, v0), bb = ldb(md, 4 * Nb, v0);
  Coef Z{1.f, 1.f, 0.f, 0.f, 1.f, 1.f, 0.f, 0.f}, X = Z;
  double zr64 = 1.0, xr64 = 1.0;
  if (zlive) Z = coef_row(A.zc, zl), zr64 = B.zd[zl];
  if (xlive) X = coef_col(A.xc, xl), xr64 = ((const __attribute__((address_space(4))) double*)B.xd)[xl];
  const double l2m = (double)lam + 2.0 * (double)mu;
  const float amu_kzh = kdiv(amu, Z.Kh, Z.rh), amu_kxh = kdiv(amu, X.Kh, X.rh);
  auto kd64 = [](double v, float K, double r) { return K == 1.f ? v : ddiv2(v, (double)K, r); };
  const float* const row = B.res + (size_t)it * A.R;
  for (int s = lo; s < hi; ++s) {
    const int sw = s * kWaveComps * Nb, sm = s * kMemComps * Nb;
    const int zs = ((CInt*)A.zx)[2 * s], xs = ((CInt*)A.zx)[2 * s + 1];
    const __attribute__((address_space(4))) ColInj* ci =
        (const __attribute__((address_space(4))) ColInj*)B.inj + (size_t)(A.s0 + s) * nx + xl;
    const int cfirst = ci->first, cn = ci->n, cz = ci->z, crid = ci->rid;
    // every load of the shot
    const f4 szc = ldb4(ai, sw + kSzz * Nb, v0 - 4), sxc = ldb4(ai, sw + kSxx * Nb, v0 - 4),
             xzc = ldb4(ai, sw + kSxz * Nb, v0 - 8);
    const float szzp = ldb(ai, sw + kSzz * Nb, vp1), szzp2 = ldb(ai, sw + kSzz * Nb, vp2),
                szzm = ldb(ai, sw + kSzz * Nb, vm1);
    const float sxxp = ldb(ai, sw + kSxx * Nb, vp1), sxxp2 = ldb(ai, sw + kSxx * Nb, vp2),
                sxxm = ldb(ai, sw + kSxx * Nb, vm1);
    const float sxzm = ldb(ai, sw + kSxz * Nb, vm1), sxzp = ldb(ai, sw + kSxz * Nb, vp1),
                sxzm2 = ldb(ai, sw + kSxz * Nb, vm2);
    float vz = ldb(ai, sw + kVz * Nb, v0), vx = ldb(ai, sw + kVx * Nb, v0);
    float hxx = 0.f, hzx = 0.f, hzz = 0.f, hxz = 0.f;  // the stress update's own memory variables
    float pxx[3] = {}, pzx[3] = {}, q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
    f4 pxz{}, pzz{};
    if (xlive) hxx = ldb(mi, sm + kMvxx * Nb, v0), hzx = ldb(mi, sm + kMvzx * Nb, v0);
    if (zlive) hzz = ldb(mi, sm + kMvzz * Nb, v0), hxz = ldb(mi, sm + kMvxz * Nb, v0);
    if (px) {
      pxx[0] = ldb(mi, sm + kMvxx * Nb, vp1), pxx[1] = ldb(mi, sm + kMvxx * Nb, vp2);
      pxx[2] = ldb(mi, sm + kMvxx * Nb, vm1);
      pzx[0] = ldb(mi, sm + kMvzx * Nb, vm1), pzx[1] = ldb(mi, sm + kMvzx * Nb, vp1);
      pzx[2] = ldb(mi, sm + kMvzx * Nb, vm2);
      q0 = ldb(mi, sm + kMsxzx * Nb, v0), q1 = ldb(mi, sm + kMsxx * Nb, v0);
    }
    if (pz) {
      pxz = ldb4(mi, sm + kMvxz * Nb, v0 - 8), pzz = ldb4(mi, sm + kMvzz * Nb, v0 - 4);
      q2 = ldb(mi, sm + kMsxzz * Nb, v0), q3 = ldb(mi, sm + kMszz * Nb, v0);
    }
    const float cres = cn == 1 && crid >= 0 ? ((CFloat*)row)[crid] : 0.f;
    float szz = szc[1], sxx = sxc[1], sxz = xzc[2];
    if (B.stf_grad && core && x == xs && z == zs)  // -(szz_adj + RSXXZZ sxx_adj) dt, double, stored as float
      B.stf_grad[(size_t)s * A.nSteps + it] = (float)(-((double)szz + kRS * (double)sxx) * dt64);
    {
      // vx: a_x dpsi_xx/dx + lambda dszz/dx / K_x dt + (lambda + 2.0 mu) dsxx/dx / K_x dt
      //     + a_z_half dpsi_xz/dz + ave_mu / K_z_half dsxz/dz dt
      const float dszz_dx = dad(szzp, szz, szzp2, szzm, dx, rdx);
      const float dsxx_dx = dad(sxxp, sxx, sxxp2, sxxm, dx, rdx);
      const float dsxz_dz = dad(sxz, xzc[1], xzc[3], xzc[0], dz, rdz);
      float t = kdiv(lam * dszz_dx, X.K, X.r) * dt;
      if (px && X.a != 0.f)  // psi_vxx at x+1, x, x+2, x-1
        t = X.a * dad(pxx[0], hxx, pxx[1], pxx[2], dx, rdx) + t;
      double S = (double)t + kd64(l2m * (double)dsxx_dx, X.K, xr64) * dt64;
      if (pz && Z.ah != 0.f)  // psi_vxz at z, z-1, z+1, z-2
        S = S + (double)(Z.ah * dad(pxz[2], pxz[1], pxz[3], pxz[0], dz, rdz));
      S = S + (double)(amu_kzh * dsxz_dz * dt);
      vx = (float)((double)vx + S);
      // vz: a_z dpsi_zz/dz + (lambda + 2.0 mu) dszz/dz / K_z dt + lambda dsxx/dz / K_z dt
      //     + a_x_half dpsi_zx/dx + ave_mu / K_x_half dsxz/dx dt
      const float dszz_dz = dad(szc[2], szz, szc[3], szc[0], dz, rdz);
      const float dsxx_dz = dad(sxc[2], sxx, sxc[3], sxc[0], dz, rdz);
      const float dsxz_dx = dad(sxz, sxzm, sxzp, sxzm2, dx, rdx);
      S = kd64(l2m * (double)dszz_dz, Z.K, zr64) * dt64;
      if (pz && Z.a != 0.f)  // psi_vzz at z+1, z, z+2, z-1
        S = (double)(Z.a * dad(pzz[2], pzz[1], pzz[3], pzz[0], dz, rdz)) + S;
      S = S + (double)(kdiv(lam * dsxx_dz, Z.K, Z.r) * dt);
      if (px && X.ah != 0.f)  // psi_vzx at x, x-1, x+1, x-2
        S = S + (double)(X.ah * dad(hzx, pzx[0], pzx[1], pzx[2], dx, rdx));
      S = S + (double)(amu_kxh * dsxz_dx * dt);
      vz = (float)((double)vz + S);
      if (px) {
        q0 = X.b * q0 + ba * vz * dt;
        q1 = X.bh * q1 + bb * vx * dt;
        lds[2][j][lane] = valid ? q0 : 0.f, lds[3][j][lane] = valid ? q1 : 0.f;
      } else {
        lds[2][j][lane] = 0.f, lds[3][j][lane] = 0.f;
      }
      if (pz) {
        q2 = Z.b * q2 + bb * vx * dt;
        q3 = Z.bh * q3 + ba * vz * dt;
      }
      if (E) lds[4][j][lane] = valid ? q2 : 0.f, lds[5][j][lane] = valid ? q3 : 0.f;
      lds[0][j][lane] = valid ? vz : 0.f;
      lds[1][j][lane] = valid ? vx : 0.f;
      if (core) {
        stb(ao, sw + kVz * Nb, v0, vz);
        stb(ao, sw + kVx * Nb, v0, vx);
        if (px) stb(mo, sm + kMsxzx * Nb, v0, q0), stb(mo, sm + kMsxx * Nb, v0, q1);
        if (pz) stb(mo, sm + kMsxzz * Nb, v0, q2), stb(mo, sm + kMszz * Nb, v0, q3);
      }
    }
    __syncthreads();
    if (core) {
      const float *tz = &lds[0][j][lane], *tx = &lds[1][j][lane];
      const float *c0 = &lds[2][j][lane], *c1 = &lds[3][j][lane], *c2 = &lds[4][j][lane],
                  *c3 = &lds[5][j][lane];
      // sxz += a_x dphi_xz_x/dx + dvz/dx / K_x ba dt + a_z dphi_xz_z/dz + dvx/dz / K_z bb dt
      const float dvz_dx = dad(tz[kBZ], vz, tz[2 * kBZ], tz[-kBZ], dx, rdx);
      const float dvx_dz = dad(tx[1], vx, tx[2], tx[-1], dz, rdz);
      float e = kdiv(dvz_dx, X.K, X.r) * ba * dt;
      if (px && X.a != 0.f) e = X.a * dad(c0[kBZ], c0[0], c0[2 * kBZ], c0[-kBZ], dx, rdx) + e;
      if (pz && Z.a != 0.f) e = e + Z.a * dad(c2[1], c2[0], c2[2], c2[-1], dz, rdz);
      e = e + kdiv(dvx_dz, Z.K, Z.r) * bb * dt;
      sxz = sxz + e;
      stb(ao, sw + kSxz * Nb, v0, sxz);
      if (cn) {
        if (crid >= 0) {
          if (z == cz) {
            szz = szz + cres;
            sxx = (float)((double)sxx + kRS * (double)cres);
          }
        } else {  // several receivers in the column: each cell's in receiver order
          for (int c = cfirst; c < cfirst + cn; ++c)
            if (z == B.icell[3 * c + 1])
              for (int q = B.iptr[c]; q < B.iptr[c + 1]; ++q) {
                const float v = row[B.irid[q]];
                szz = szz + v;
                sxx = (float)((double)sxx + kRS * (double)v);
              }
        }
      }
      // sxx += a_x_half dphi_xx/dx + bb dvx/dx / K_x_half dt; szz likewise in z
      const float dvx_dx = dad(vx, tx[-kBZ], tx[kBZ], tx[-2 * kBZ], dx, rdx);
      const float dvz_dz = dad(vz, tz[-1], tz[1], tz[-2], dz, rdz);
      float t = kdiv(bb * dvx_dx, X.Kh, X.rh) * dt;
      if (px && X.ah != 0.f) t = X.ah * dad(c1[0], c1[-kBZ], c1[kBZ], c1[-2 * kBZ], dx, rdx) + t;
      sxx = sxx + t;
      t = kdiv(ba * dvz_dz, Z.Kh, Z.rh) * dt;
      if (pz && Z.ah != 0.f) t = Z.ah * dad(c3[0], c3[-1], c3[1], c3[-2], dz, rdz) + t;
      szz = szz + t;
      stb(ao, sw + kSxx * Nb, v0, sxx);
      stb(ao, sw + kSzz * Nb, v0, szz);
      // psi_xx = b_x psi + lambda szz dt + (lambda + 2.0 mu) sxx dt;
      // psi_zz = b_z psi + (lambda + 2.0 mu) szz dt + lambda sxx dt
      if (xlive) {
        stb(mo, sm + kMvzx * Nb, v0, X.bh * hzx + sxz * amu * dt);
        stb(mo, sm + kMvxx * Nb, v0, (float)((double)(X.b * hxx + lam * szz * dt) + l2m * (double)sxx * dt64));
      }
      if (zlive) {
        stb(mo, sm + kMvxz * Nb, v0, Z.bh * hxz + sxz * amu * dt);
        stb(mo, sm + kMvzz * Nb, v0,
            (float)((double)(Z.b * hzz) + l2m * (double)szz * dt64 + (double)(lam * sxx * dt)));
      }
    }
    if (s + 1 < hi) __syncthreads();  // the next shot's first half overwrites the tile
  }
}

// The reversal half of a backward step, tiles over the ring rectangle: forward
// velocities of step it from the stresses of it + 1 (el_velocity.cu:84-117,
// isFor = false) on the tile, then the stresses of step it (el_stress.cu:90-131)
// on the core; ring cells take the stored values; the gradient sums take the
// adjoint state that step it starts from.
__device__ __forceinline__ void step_rev(CBack& B, int strip, int bx, int it,
                                         int itr, float (&lds)[6][kStepW][kBZ]) {
  const auto& A = B.s;
  const int hi = A.ns;
  const int lane = (int)threadIdx.x, j = wave_col(0);
  const int nz = A.nz, nx = A.nx, nzA = A.nzA, nPml = A.nPml, Nb = A.Nb;
  const float dt = A.dt, dz = A.dz, dx = A.dx, rdz = A.rdz, rdx = A.rdx;
  const double dt64 = (double)dt;
  const int z = nPml - 4 + strip * kCoreZ + lane, x = nPml - 4 + bx * kCoreX + j;
  // loads of cells outside the interior are moved inside it; their results are dropped
  const int xl = min(max(x, nPml), nx - 1 - nPml), zl = min(max(z, nPml), nzA - 1 - nPml);
  const bool in = z == zl && x == xl;
  const int slot = ring_slot(z, x, ring_geo(A));
  const bool core = lane >= 2 && lane < kBZ - 2 && j >= 2 && j < kStepW - 2 && (in || slot >= 0);
  const int v0 = 4 * (xl * nz + zl), cb = 4 * nz, vo = 4 * (x * nz + z);
  const int vm1 = v0 - cb, vm2 = vm1 - cb, vp1 = v0 + cb, vp2 = vp1 + cb;
  const Rsrc wi = rsrc(A.wi), wo = rsrc(A.wo), ai = rsrc(B.ai), md = rsrc(A.md);
  const float lam = ldb(md, 0, v0), mu = ldb(md, Nb, v0), amu = ldb(md, 2 * Nb, v0),
              ba = ldb(md, 3 * Nb, v0), bb = ldb(md, 4 * Nb, v0);
  const double l2m = (double)lam + 2.0 * (double)mu;
  const Rsrc ac = rsrc(B.acc);
  float gl = ldb(ac, 0, v0), gm = ldb(ac, Nb, v0), gs = ldb(ac, 2 * Nb, v0), ga = ldb(ac, 3 * Nb, v0),
        gb = ldb(ac, 4 * Nb, v0);
  float dl = 0.f, dm = 0.f, ds = 0.f, da = 0.f, db = 0.f;  // this launch's sums
  const size_t ring_step = (size_t)A.rnt * 5 * A.ringlen, rl = (size_t)A.ringlen;
  const float* rp = A.ring + (size_t)A.rs0 * ring_step + (size_t)itr * 5 * rl + max(slot, 0);
  for (int s = 0; s < hi; ++s, rp += ring_step) {
    const int sw = s * kWaveComps * Nb;
    const int zs = ((CInt*)A.zx)[2 * s], xs = ((CInt*)A.zx)[2 * s + 1];
    // every load of the shot
    const f4 szc = ldb4(wi, sw + kSzz * Nb, v0 - 4), xzc = ldb4(wi, sw + kSxz * Nb, v0 - 8);
    const float sxzm = ldb(wi, sw + kSxz * Nb, vm1), sxzp = ldb(wi, sw + kSxz * Nb, vp1),
                sxzm2 = ldb(wi, sw + kSxz * Nb, vm2);
    const float sxxp = ldb(wi, sw + kSxx * Nb, vp1), sxx0 = ldb(wi, sw + kSxx * Nb, v0),
                sxxp2 = ldb(wi, sw + kSxx * Nb, vp2), sxxm = ldb(wi, sw + kSxx * Nb, vm1);
    float vz = ldb(wi, sw + kVz * Nb, v0), vx = ldb(wi, sw + kVx * Nb, v0);
    const float avz = ldb(ai, sw + kVz * Nb, v0), avx = ldb(ai, sw + kVx * Nb, v0);
    const float azz = ldb(ai, sw + kSzz * Nb, v0), axx = ldb(ai, sw + kSxx * Nb, v0),
                axz = ldb(ai, sw + kSxz * Nb, v0);
    float szz = szc[1], sxx = sxx0, sxz = xzc[2], rvz = 0.f, rvx = 0.f;
    if (slot >= 0) szz = rp[0], sxz = rp[rl], sxx = rp[2 * rl], rvz = rp[3 * rl], rvx = rp[4 * rl];
    {
      const float dszz_dz = dfw(szc[2], szc[1], szc[3], szc[0], dz, rdz);
      const float dsxz_dx = dfw(xzc[2], sxzm, sxzp, sxzm2, dx, rdx);
      const float dsxz_dz = dfw(xzc[2], xzc[1], xzc[3], xzc[0], dz, rdz);
      const float dsxx_dx = dfw(sxxp, sxx0, sxxp2, sxxm, dx, rdx);
      const float fz = dszz_dz + dsxz_dx, fx = dsxz_dz + dsxx_dx;
      da += avz * fz;
      db += avx * fx;
      vz = slot >= 0 ? rvz : vz - fz * ba * dt;
      vx = slot >= 0 ? rvx : vx - fx * bb * dt;
    }
    const bool known = in || slot >= 0;
    lds[0][j][lane] = known ? vz : 0.f;
    lds[1][j][lane] = known ? vx : 0.f;
    if (core) {
      stb(wo, sw + kVz * Nb, vo, vz);
      stb(wo, sw + kVx * Nb, vo, vx);
    }
    __syncthreads();
    if (core) {
      const float *tz = &lds[0][j][lane], *tx = &lds[1][j][lane];
      const float dvz_dz = dfw(vz, tz[-1], tz[1], tz[-2], dz, rdz);
      const float dvx_dx = dfw(vx, tx[-kBZ], tx[kBZ], tx[-2 * kBZ], dx, rdx);
      const float dvx_dz = dfw(tx[1], vx, tx[2], tx[-1], dz, rdz);
      const float dvz_dx = dfw(tz[kBZ], vz, tz[2 * kBZ], tz[-kBZ], dx, rdx);
      dl += (azz + axx) * (dvz_dz + dvx_dx);
      dm += azz * dvz_dz + axx * dvx_dx;
      ds += axz * (dvx_dz + dvz_dx);
      if (slot < 0) {
        if (x == xs && z == zs) {  // add_source(-)
          const float amp = A.amp[(size_t)s * A.nSteps + it];
          szz = szz - kSrcScale * amp * dt;
          sxx = (float)((double)sxx - kRS * (double)kSrcScale * (double)amp * dt64);
        }
        szz = (float)((double)szz - (l2m * (double)dvz_dz + (double)(lam * dvx_dx)) * dt64);
        sxx = (float)((double)sxx - ((double)(lam * dvz_dz) + l2m * (double)dvx_dx) * dt64);
        sxz = sxz - amu * (dvx_dz + dvz_dx) * dt;
      }
      stb(wo, sw + kSzz * Nb, vo, szz);
      stb(wo, sw + kSxx * Nb, vo, sxx);
      stb(wo, sw + kSxz * Nb, vo, sxz);
    }
    if (s + 1 < hi) __syncthreads();  // the next shot's first half overwrites the tile
  }
  if (in && core) {
    stb(ac, 0, v0, gl + dl);
    stb(ac, Nb, v0, gm + dm);
    stb(ac, 2 * Nb, v0, gs + ds);
    stb(ac, 3 * Nb, v0, ga + da);
    stb(ac, 4 * Nb, v0, gb + db);
  }
}

// One backward step in one launch.  The two halves touch different state (the
// reversal reads the adjoint state of its own cell, which the adjoint half
// does not write in place), so they are workgroups of their own: the first
// rows of the grid the adjoint's tiles, the rest the reversal's.
__global__ __launch_bounds__(64 * kStepW) void k_step_bwd(const BackArgs* __restrict__ args, int it,
                                                     int itr, int slices, int per_slice) {
  // velocities z, x, and the adjoint's memory variables sxzx, sxx, sxzz, szz
  __shared__ float lds[6][kStepW][kBZ];
  const Place pl = place_of((int)blockIdx.z, slices, per_slice);
  CBack& B = ((CBack*)args)[pl.part];
  const int xcd = (int)blockIdx.x & 7, q = (int)blockIdx.x >> 3;
  int strip = (int)blockIdx.y;
  if (strip < B.s.gz) {
    const int bx = xcd * B.s.per + q;
    if (q >= B.s.per || bx >= B.s.gx) return;
    step_adj(B, pl.lo, min(pl.hi, B.s.ns), strip, bx, it, lds);
  } else if (!pl.slice) {  // all shots: their sums are taken in order
    strip -= B.s.gz;
    const int bx = xcd * B.rper + q;
    if (strip >= B.rgz || q >= B.rper || bx >= B.rgx) return;
    step_rev(B, strip, bx, it, itr, lds);
  }
}

// ------------------------------------------------------------------ half steps
// The same updates in place, one launch per half of a step: for grids that
// fill the chip, where a second copy of the state would overflow the Infinity
// Cache and recomputing the rim costs more than a launch.  A workgroup is 64
// depth cells x 1..4 columns, a thread one cell of all shots of its slice.
// Workgroups of extra grid rows move the boundary ring and record, always
// arrays that the launch's other workgroups only read or do not touch.
//
// Bound by the traffic between L2 and the Infinity Cache on large grids
// (580x1780, 4 shots a launch: 5.6-6.4 TB/s) and by the loads' latency on small
// ones; a kernel's registers are left to its loads (limited to 64, for 8 waves
// a SIMD, the gradient there takes 618 ms instead of 531).  Microseconds a
// launch at 580x1780, as one launch per half with tiles from a map before and
// here: stress 30.8 -> 28.5, velocity 24.4 -> 24.7 (4 shots), adjoint velocity
// with reverse stress 40.0 -> 36.5, adjoint stress with reverse velocity 33.6 ->
// 31.9 (2.7 shots).
//
// The grid: x tiles in XCD bands, each band in chunks of gridDim.x / 8 tiles;
// strips along y, chunks x places (slices and parts) along z, chunks outermost.
// Workgroups start in that order, so that a strip's neighbours run while its
// rim is still in the XCD's L2.
struct HalfTile {
  int z, x;
};
// chunk of the workgroup; k: its place.  inv = ceil(2^32 / places) (0 for one
// place): the high half of b times it is b / places for 16-bit numbers.  Counted
// off in a loop, a grid of 84 x 60024 (469 chunks) took 15.5 ms instead of 5.0
// for 60 steps.
__device__ __forceinline__ int half_chunk(int places, unsigned inv, int& k) {
  const unsigned b = blockIdx.z, chunk = inv ? __umulhi(b, inv) : b;
  k = (int)(b - chunk * (unsigned)places);
  return (int)chunk;
}
// false: the workgroup is past the tiles
__device__ __forceinline__ bool half_tile(CStep& A, int strip, int chunk, HalfTile& t) {
  const int q = chunk * ((int)gridDim.x >> 3) + ((int)blockIdx.x >> 3);
  const int bx = ((int)blockIdx.x & 7) * A.hper + q;
  if (q >= A.hper || bx >= A.hgx) return false;
  t.z = strip * kBZ + (int)threadIdx.x;
  t.x = wave_col(2 + bx * (int)blockDim.y);
  return true;
}
// linear item of a thread in the grid rows from row `first` on
__device__ __forceinline__ int extra_item(int first, int chunk) {
  const int row = chunk * ((int)gridDim.y - first) + (int)blockIdx.y - first;
  return ((row * (int)gridDim.x + (int)blockIdx.x) * (int)blockDim.y + (int)threadIdx.y) * kBZ + (int)threadIdx.x;
}

// ring components [c0, c1) of a run's or segment's first step
__global__ __launch_bounds__(256) void k_ring(const StepArgs* __restrict__ args, int row, int c0, int c1) {
  CStep& A = ((CStep*)args)[blockIdx.z];
  ring_move<true>(A, A.wo, (int)(blockIdx.x * 256 + threadIdx.x), 0, A.ns, row, c0, c1);
}

// el_stress.cu:50-88 + add_source (utilities.cu:521-555).  Extra rows save the
// velocities of the ring (row `ring`, -1: none) and add the illumination of the
// step before.
template <int U>
__global__ __launch_bounds__(256) void k_half_stress(const StepArgs* __restrict__ args, int it,
                                                     int ring, int slices, int per_slice, int places,
                                                     unsigned inv) {
  int k;
  const int chunk = half_chunk(places, inv, k);
  const Place pl = place_of(k, slices, per_slice);
  CStep& A = ((CStep*)args)[pl.part];
  const int hi = min(pl.hi, A.ns), strip = (int)blockIdx.y;
  if (strip >= A.hgz) {
    const int i = extra_item(A.hgz, chunk), pad = A.ring ? (A.ringlen + 63) & ~63 : 0;
    if (i < pad)
      ring_move<true>(A, A.wo, i, pl.lo, hi, ring, 3, 5);
    else if (A.illum && slices > 1 && !pl.slice)
      illum_cell(A, i - pad);
    return;
  }
  HalfTile t;
  if (!half_tile(A, strip, chunk, t)) return;
  const int z = t.z, x = t.x, nz = A.nz, nx = A.nx, nzA = A.nzA, nPml = A.nPml, Nb = A.Nb;
  if (z < 2 || z > nzA - 3 || x > nx - 3) return;
  const float dt = A.dt, dz = A.dz, dx = A.dx, rdz = A.rdz, rdx = A.rdx;
  const double dt64 = (double)dt;
  const bool pz = z < nPml || z > nzA - nPml - 1;
  const bool px = x < nPml || x > nx - nPml - 1;
  const int v0 = 4 * (x * nz + z), cb = 4 * nz;
  const int vm1 = v0 - cb, vm2 = vm1 - cb, vp1 = v0 + cb, vp2 = vp1 + cb;
  const Rsrc w = rsrc(A.wo), m = rsrc(A.mo), md = rsrc(A.md);
  const float lam = ldb(md, 0, v0), mu = ldb(md, Nb, v0), amu = ldb(md, 2 * Nb, v0);
  const double l2m = (double)lam + 2.0 * (double)mu;  // (d_Lambda + 2.0*d_Mu)
  Coef Z{}, X{};
  if (pz) Z = coef_row(A.zc, z);
  if (px) X = coef_col(A.xc, x);
  for (int s0 = pl.lo; s0 < hi; s0 += U) {
    f4 vzc[U], vxc[U];
    float vzp[U], vzp2[U], vzm[U], vxm[U], vxp[U], vxm2[U], szz[U], sxx[U], sxz[U];
    float m0[U], m1[U], n0[U], n1[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u;
      if (s >= hi) break;
      const int sw = s * kWaveComps * Nb, sm = s * kMemComps * Nb;
      vzc[u] = ldb4(w, sw + kVz * Nb, v0 - 8), vxc[u] = ldb4(w, sw + kVx * Nb, v0 - 4);
      vzp[u] = ldb(w, sw + kVz * Nb, vp1), vzp2[u] = ldb(w, sw + kVz * Nb, vp2), vzm[u] = ldb(w, sw + kVz * Nb, vm1);
      vxm[u] = ldb(w, sw + kVx * Nb, vm1), vxp[u] = ldb(w, sw + kVx * Nb, vp1), vxm2[u] = ldb(w, sw + kVx * Nb, vm2);
      szz[u] = ldb(w, sw + kSzz * Nb, v0), sxx[u] = ldb(w, sw + kSxx * Nb, v0), sxz[u] = ldb(w, sw + kSxz * Nb, v0);
      m0[u] = m1[u] = n0[u] = n1[u] = 0.f;
      if (pz) m0[u] = ldb(m, sm + kMvzz * Nb, v0), m1[u] = ldb(m, sm + kMvxz * Nb, v0);
      if (px) n0[u] = ldb(m, sm + kMvxx * Nb, v0), n1[u] = ldb(m, sm + kMvzx * Nb, v0);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u;
      if (s >= hi) break;
      const int sw = s * kWaveComps * Nb, sm = s * kMemComps * Nb;
      const float vz0 = vzc[u][2], vx0 = vxc[u][1];
      float dvz_dz = dfw(vz0, vzc[u][1], vzc[u][3], vzc[u][0], dz, rdz);
      float dvx_dx = dfw(vx0, vxm[u], vxp[u], vxm2[u], dx, rdx);
      float dvx_dz = dfw(vxc[u][2], vx0, vxc[u][3], vxc[u][0], dz, rdz);
      float dvz_dx = dfw(vzp[u], vz0, vzp2[u], vzm[u], dx, rdx);
      if (pz) {
        const float p = Z.b * m0[u] + Z.a * dvz_dz, q = Z.bh * m1[u] + Z.ah * dvx_dz;
        stb(m, sm + kMvzz * Nb, v0, p), stb(m, sm + kMvxz * Nb, v0, q);
        dvz_dz = kdiv(dvz_dz, Z.K, Z.r) + p;
        dvx_dz = kdiv(dvx_dz, Z.Kh, Z.rh) + q;
      }
      if (px) {
        const float p = X.b * n0[u] + X.a * dvx_dx, q = X.bh * n1[u] + X.ah * dvz_dx;
        stb(m, sm + kMvxx * Nb, v0, p), stb(m, sm + kMvzx * Nb, v0, q);
        dvx_dx = kdiv(dvx_dx, X.K, X.r) + p;
        dvz_dx = kdiv(dvz_dx, X.Kh, X.rh) + q;
      }
      float fzz = (float)((double)szz[u] + (l2m * (double)dvz_dz + (double)(lam * dvx_dx)) * dt64);
      float fxx = (float)((double)sxx[u] + ((double)(lam * dvz_dz) + l2m * (double)dvx_dx) * dt64);
      if (x == ((CInt*)A.zx)[2 * s + 1] && z == ((CInt*)A.zx)[2 * s]) {
        const float amp = A.amp[(size_t)s * A.nSteps + it];
        fzz = fzz + kSrcScale * amp * dt;
        fxx = (float)((double)fxx + kRS * (double)kSrcScale * (double)amp * dt64);
      }
      stb(w, sw + kSzz * Nb, v0, fzz);
      stb(w, sw + kSxx * Nb, v0, fxx);
      stb(w, sw + kSxz * Nb, v0, sxz[u] + amu * (dvx_dz + dvz_dx) * dt);
    }
  }
}

// el_velocity.cu:45-82.  Extra rows record sample it + 1 and save the stresses
// of the ring (row `ring`, that of step it + 1; -1: none).
template <int U>
__global__ __launch_bounds__(256) void k_half_vel(const StepArgs* __restrict__ args, int it, int ring,
                                                  int slices, int per_slice, int places, unsigned inv) {
  int k;
  const int chunk = half_chunk(places, inv, k);
  const Place pl = place_of(k, slices, per_slice);
  CStep& A = ((CStep*)args)[pl.part];
  const int hi = min(pl.hi, A.ns), strip = (int)blockIdx.y;
  if (strip >= A.hgz) {
    const int i = extra_item(A.hgz, chunk), pad = A.ring ? (A.ringlen + 63) & ~63 : 0;
    if (i < pad)
      ring_move<true>(A, A.wo, i, pl.lo, hi, ring, 0, 3);
    else if (!pl.slice)
      record_cell(A, i - pad, it + 1);
    return;
  }
  HalfTile t;
  if (!half_tile(A, strip, chunk, t)) return;
  const int z = t.z, x = t.x, nz = A.nz, nx = A.nx, nzA = A.nzA, nPml = A.nPml, Nb = A.Nb;
  if (z < 2 || z > nzA - 3 || x > nx - 3) return;
  const float dt = A.dt, dz = A.dz, dx = A.dx, rdz = A.rdz, rdx = A.rdx;
  const bool pz = z < nPml || z > nzA - nPml - 1;
  const bool pv = x < nPml || x > nx - nPml;  // el_velocity.cu:56,71
  const int v0 = 4 * (x * nz + z), cb = 4 * nz;
  const int vm1 = v0 - cb, vm2 = vm1 - cb, vp1 = v0 + cb, vp2 = vp1 + cb;
  const Rsrc w = rsrc(A.wo), m = rsrc(A.mo), md = rsrc(A.md);
  const float ba = ldb(md, 3 * Nb, v0), bb = ldb(md, 4 * Nb, v0);
  Coef Z{}, X{};
  if (pz) Z = coef_row(A.zc, z);
  if (pv) X = coef_col(A.xc, x);
  float il = 0.f;
  for (int s0 = pl.lo; s0 < hi; s0 += U) {
    f4 szc[U], sxc[U];
    float sxzm[U], sxzp[U], sxzm2[U], sxxp[U], sxx0[U], sxxp2[U], sxxm[U], vz[U], vx[U];
    float m0[U], m1[U], n0[U], n1[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u;
      if (s >= hi) break;
      const int sw = s * kWaveComps * Nb, sm = s * kMemComps * Nb;
      szc[u] = ldb4(w, sw + kSzz * Nb, v0 - 4), sxc[u] = ldb4(w, sw + kSxz * Nb, v0 - 8);
      sxzm[u] = ldb(w, sw + kSxz * Nb, vm1), sxzp[u] = ldb(w, sw + kSxz * Nb, vp1), sxzm2[u] = ldb(w, sw + kSxz * Nb, vm2);
      sxxp[u] = ldb(w, sw + kSxx * Nb, vp1), sxx0[u] = ldb(w, sw + kSxx * Nb, v0);
      sxxp2[u] = ldb(w, sw + kSxx * Nb, vp2), sxxm[u] = ldb(w, sw + kSxx * Nb, vm1);
      vz[u] = ldb(w, sw + kVz * Nb, v0), vx[u] = ldb(w, sw + kVx * Nb, v0);
      m0[u] = m1[u] = n0[u] = n1[u] = 0.f;
      if (pz) m0[u] = ldb(m, sm + kMszz * Nb, v0), m1[u] = ldb(m, sm + kMsxzz * Nb, v0);
      if (pv) n0[u] = ldb(m, sm + kMsxzx * Nb, v0), n1[u] = ldb(m, sm + kMsxx * Nb, v0);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int s = s0 + u;
      if (s >= hi) break;
      const int sw = s * kWaveComps * Nb, sm = s * kMemComps * Nb;
      float dszz_dz = dfw(szc[u][2], szc[u][1], szc[u][3], szc[u][0], dz, rdz);
      float dsxz_dx = dfw(sxc[u][2], sxzm[u], sxzp[u], sxzm2[u], dx, rdx);
      float dsxz_dz = dfw(sxc[u][2], sxc[u][1], sxc[u][3], sxc[u][0], dz, rdz);
      float dsxx_dx = dfw(sxxp[u], sxx0[u], sxxp2[u], sxxm[u], dx, rdx);
      if (pz) {
        const float p = Z.bh * m0[u] + Z.ah * dszz_dz, q = Z.b * m1[u] + Z.a * dsxz_dz;
        stb(m, sm + kMszz * Nb, v0, p), stb(m, sm + kMsxzz * Nb, v0, q);
        dszz_dz = kdiv(dszz_dz, Z.Kh, Z.rh) + p;
        dsxz_dz = kdiv(dsxz_dz, Z.K, Z.r) + q;
      }
      if (pv) {
        const float p = X.b * n0[u] + X.a * dsxz_dx, q = X.bh * n1[u] + X.ah * dsxx_dx;
        stb(m, sm + kMsxzx * Nb, v0, p), stb(m, sm + kMsxx * Nb, v0, q);
        dsxz_dx = kdiv(dsxz_dx, X.K, X.r) + p;
        dsxx_dx = kdiv(dsxx_dx, X.Kh, X.rh) + q;
      }
      const float fvz = vz[u] + (dszz_dz + dsxz_dx) * ba * dt;
      const float fvx = vx[u] + (dsxz_dz + dsxx_dx) * bb * dt;
      stb(w, sw + kVz * Nb, v0, fvz);
      stb(w, sw + kVx * Nb, v0, fvx);
      il += fvz * fvz + fvx * fvx;
    }
  }
  if (A.illum && slices == 1) A.illum[x * nz + z] += il;
}

// el_velocity_adj.cu:22-108, plus source_grad (utilities.cu:582-593) where
// `stf`.  The C-PML memory terms a*dpsi are evaluated only where a != 0;
// elsewhere they are exactly zero in the reference as well.
template <bool Sliced>
__device__ __forceinline__ void half_adj_vel(CBack& B, const HalfTile& t,
                                             int it, bool stf) {
  const auto& A = B.s;
  const int z = t.z, x = t.x, nz = A.nz, nx = A.nx, nzA = A.nzA, nPml = A.nPml, Nb = A.Nb;
  if (z < 2 || z > nzA - 3 || x > nx - 3) return;
  const float dt = A.dt, dz = A.dz, dx = A.dx, rdz = A.rdz, rdx = A.rdx;
  const double dt64 = (double)dt;
  const bool E = __builtin_amdgcn_readfirstlane(z - (int)threadIdx.x < nPml || z - (int)threadIdx.x + kBZ > nzA - nPml);
  const bool pz = z < nPml || z > nzA - nPml - 1;
  const bool px = x < nPml || x > nx - nPml - 1;
  const int v0 = 4 * (x * nz + z), cb = 4 * nz;
  const int vm1 = v0 - cb, vm2 = vm1 - cb, vp1 = v0 + cb, vp2 = vp1 + cb;
  const Rsrc a = rsrc(B.ao), m = rsrc(A.mo), md = rsrc(A.md);
  const float lam = ldb(md, 0, v0), mu = ldb(md, Nb, v0), amu = ldb(md, 2 * Nb, v0),
              ba = ldb(md, 3 * Nb, v0), bb = ldb(md, 4 * Nb, v0);
  const double l2m = (double)lam + 2.0 * (double)mu;
  Coef Z{1.f, 1.f, 0.f, 0.f, 1.f, 1.f, 0.f, 0.f}, X = Z;
  double zr64 = 1.0, xr64 = 1.0;
  if (pz) Z = coef_row(A.zc, z), zr64 = B.zd[z];
  if (px) X = coef_col(A.xc, x), xr64 = ((const __attribute__((address_space(4))) double*)B.xd)[x];
  const float amu_kzh = kdiv(amu, Z.Kh, Z.rh), amu_kxh = kdiv(amu, X.Kh, X.rh);
  int lo, hi;
  own_shots<Sliced>(A.ns, lo, hi);
  for (int s = lo; s < hi; ++s) {
    const int sw = s * kWaveComps * Nb, sm = s * kMemComps * Nb;
    const f4 szc = ldb4(a, sw + kSzz * Nb, v0 - 4), sxc = ldb4(a, sw + kSxx * Nb, v0 - 4),
             xzc = ldb4(a, sw + kSxz * Nb, v0 - 8);
    const float szzp = ldb(a, sw + kSzz * Nb, vp1), szzp2 = ldb(a, sw + kSzz * Nb, vp2),
                szzm = ldb(a, sw + kSzz * Nb, vm1);
    const float sxxp = ldb(a, sw + kSxx * Nb, vp1), sxxp2 = ldb(a, sw + kSxx * Nb, vp2),
                sxxm = ldb(a, sw + kSxx * Nb, vm1);
    const float sxzm = ldb(a, sw + kSxz * Nb, vm1), sxzp = ldb(a, sw + kSxz * Nb, vp1),
                sxzm2 = ldb(a, sw + kSxz * Nb, vm2);
    float vz = ldb(a, sw + kVz * Nb, v0), vx = ldb(a, sw + kVx * Nb, v0);
    float pxx[4] = {}, pzx[4] = {}, q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
    f4 pxz{}, pzz{};
    if (px) {
      pxx[0] = ldb(m, sm + kMvxx * Nb, vp1), pxx[1] = ldb(m, sm + kMvxx * Nb, v0);
      pxx[2] = ldb(m, sm + kMvxx * Nb, vp2), pxx[3] = ldb(m, sm + kMvxx * Nb, vm1);
      pzx[0] = ldb(m, sm + kMvzx * Nb, v0), pzx[1] = ldb(m, sm + kMvzx * Nb, vm1);
      pzx[2] = ldb(m, sm + kMvzx * Nb, vp1), pzx[3] = ldb(m, sm + kMvzx * Nb, vm2);
      q0 = ldb(m, sm + kMsxzx * Nb, v0), q1 = ldb(m, sm + kMsxx * Nb, v0);
    }
    if (pz) {
      pxz = ldb4(m, sm + kMvxz * Nb, v0 - 8), pzz = ldb4(m, sm + kMvzz * Nb, v0 - 4);
      q2 = ldb(m, sm + kMsxzz * Nb, v0), q3 = ldb(m, sm + kMszz * Nb, v0);
    }
    const float szz = szc[1], sxx = sxc[1], sxz = xzc[2];
    if (stf && B.stf_grad && x == ((CInt*)A.zx)[2 * s + 1] && z == ((CInt*)A.zx)[2 * s])
      B.stf_grad[(size_t)s * A.nSteps + it] = (float)(-((double)szz + kRS * (double)sxx) * dt64);
    const float dszz_dx = dad(szzp, szz, szzp2, szzm, dx, rdx);
    const float dsxx_dx = dad(sxxp, sxx, sxxp2, sxxm, dx, rdx);
    const float dsxz_dz = dad(sxz, xzc[1], xzc[3], xzc[0], dz, rdz);
    // wave-uniform branches skip the divisions outside the C-PML
    float tx = lam * dszz_dx;
    double t64 = l2m * (double)dsxx_dx;
    if (px) {
      tx = kdiv(tx, X.K, X.r);
      t64 = X.K == 1.f ? t64 : ddiv2(t64, (double)X.K, xr64);
    }
    tx = tx * dt;
    if (px && X.a != 0.f) tx = X.a * dad(pxx[0], pxx[1], pxx[2], pxx[3], dx, rdx) + tx;
    double S = (double)tx + t64 * dt64;
    if (E && Z.ah != 0.f) S = S + (double)(Z.ah * dad(pxz[2], pxz[1], pxz[3], pxz[0], dz, rdz));
    S = S + (double)(amu_kzh * dsxz_dz * dt);
    vx = (float)((double)vx + S);
    stb(a, sw + kVx * Nb, v0, vx);
    const float dszz_dz = dad(szc[2], szz, szc[3], szc[0], dz, rdz);
    const float dsxx_dz = dad(sxc[2], sxx, sxc[3], sxc[0], dz, rdz);
    const float dsxz_dx = dad(sxz, sxzm, sxzp, sxzm2, dx, rdx);
    t64 = l2m * (double)dszz_dz;
    float tz = lam * dsxx_dz;
    if (E) {
      t64 = Z.K == 1.f ? t64 : ddiv2(t64, (double)Z.K, zr64);
      tz = kdiv(tz, Z.K, Z.r);
    }
    S = t64 * dt64;
    if (E && Z.a != 0.f) S = (double)(Z.a * dad(pzz[2], pzz[1], pzz[3], pzz[0], dz, rdz)) + S;
    S = S + (double)(tz * dt);
    if (px && X.ah != 0.f) S = S + (double)(X.ah * dad(pzx[0], pzx[1], pzx[2], pzx[3], dx, rdx));
    S = S + (double)(amu_kxh * dsxz_dx * dt);
    vz = (float)((double)vz + S);
    stb(a, sw + kVz * Nb, v0, vz);
    if (px) {
      stb(m, sm + kMsxzx * Nb, v0, X.b * q0 + ba * vz * dt);
      stb(m, sm + kMsxx * Nb, v0, X.bh * q1 + bb * vx * dt);
    }
    if (pz) {
      stb(m, sm + kMsxzz * Nb, v0, Z.b * q2 + bb * vx * dt);
      stb(m, sm + kMszz * Nb, v0, Z.bh * q3 + ba * vz * dt);
    }
  }
}

// the residual of sample it (res_injection, utilities.cu:569-580), then
// el_stress_adj.cu:22-104
template <bool Sliced>
__device__ __forceinline__ void half_adj_stress(CBack& B, const HalfTile& t,
                                                int it) {
  const auto& A = B.s;
  const int z = t.z, x = t.x, nz = A.nz, nx = A.nx, nzA = A.nzA, nPml = A.nPml, Nb = A.Nb;
  if (z < 2 || z > nzA - 3 || x > nx - 3) return;
  const float dt = A.dt, dz = A.dz, dx = A.dx, rdz = A.rdz, rdx = A.rdx;
  const double dt64 = (double)dt;
  const bool E = __builtin_amdgcn_readfirstlane(z - (int)threadIdx.x < nPml || z - (int)threadIdx.x + kBZ > nzA - nPml);
  const bool pz = z < nPml || z > nzA - nPml - 1;
  const bool px = x < nPml || x > nx - nPml - 1;
  const bool zlive = z <= nPml + 1 || z >= nzA - nPml - 2;
  const bool xlive = x <= nPml + 1 || x >= nx - nPml - 2;
  const int v0 = 4 * (x * nz + z), cb = 4 * nz;
  const int vm1 = v0 - cb, vm2 = vm1 - cb, vp1 = v0 + cb, vp2 = vp1 + cb;
  const Rsrc a = rsrc(B.ao), m = rsrc(A.mo), md = rsrc(A.md);
  const float lam = ldb(md, 0, v0), mu = ldb(md, Nb, v0), amu = ldb(md, 2 * Nb, v0),
              ba = ldb(md, 3 * Nb, v0), bb = ldb(md, 4 * Nb, v0);
  const double l2m = (double)lam + 2.0 * (double)mu;
  Coef Z{1.f, 1.f, 0.f, 0.f, 1.f, 1.f, 0.f, 0.f}, X = Z;
  if (zlive) Z = coef_row(A.zc, z);
  if (xlive) X = coef_col(A.xc, x);
  const float* const row = B.res + (size_t)it * A.R;
  int lo, hi;
  own_shots<Sliced>(A.ns, lo, hi);
  for (int s = lo; s < hi; ++s) {
    const int sw = s * kWaveComps * Nb, sm = s * kMemComps * Nb;
    const __attribute__((address_space(4))) ColInj* ci =
        (const __attribute__((address_space(4))) ColInj*)B.inj + (size_t)(A.s0 + s) * nx + x;
    const int cfirst = ci->first, cn = ci->n, cz = ci->z, crid = ci->rid;
    const f4 vzc = ldb4(a, sw + kVz * Nb, v0 - 8), vxc = ldb4(a, sw + kVx * Nb, v0 - 4);
    const float vzp = ldb(a, sw + kVz * Nb, vp1), vzp2 = ldb(a, sw + kVz * Nb, vp2), vzm = ldb(a, sw + kVz * Nb, vm1);
    const float vxm = ldb(a, sw + kVx * Nb, vm1), vxp = ldb(a, sw + kVx * Nb, vp1), vxm2 = ldb(a, sw + kVx * Nb, vm2);
    float szz = ldb(a, sw + kSzz * Nb, v0), sxx = ldb(a, sw + kSxx * Nb, v0), sxz = ldb(a, sw + kSxz * Nb, v0);
    float q1[4] = {}, q3[4] = {}, hzx = 0.f, hxx = 0.f, hxz = 0.f, hzz = 0.f;
    f4 q2{}, q4{};
    if (px) {
      q1[0] = ldb(m, sm + kMsxzx * Nb, vp1), q1[1] = ldb(m, sm + kMsxzx * Nb, v0);
      q1[2] = ldb(m, sm + kMsxzx * Nb, vp2), q1[3] = ldb(m, sm + kMsxzx * Nb, vm1);
      q3[0] = ldb(m, sm + kMsxx * Nb, v0), q3[1] = ldb(m, sm + kMsxx * Nb, vm1);
      q3[2] = ldb(m, sm + kMsxx * Nb, vp1), q3[3] = ldb(m, sm + kMsxx * Nb, vm2);
    }
    if (pz) q2 = ldb4(m, sm + kMsxzz * Nb, v0 - 4), q4 = ldb4(m, sm + kMszz * Nb, v0 - 8);
    if (xlive) hzx = ldb(m, sm + kMvzx * Nb, v0), hxx = ldb(m, sm + kMvxx * Nb, v0);
    if (zlive) hxz = ldb(m, sm + kMvxz * Nb, v0), hzz = ldb(m, sm + kMvzz * Nb, v0);
    const float cres = cn == 1 && crid >= 0 ? ((CFloat*)row)[crid] : 0.f;
    const float vz0 = vzc[2], vx0 = vxc[1];
    // sxz += a_x dphi_xz_x/dx + dvz/dx / K_x ba dt + a_z dphi_xz_z/dz + dvx/dz / K_z bb dt
    float dvz_dx = dad(vzp, vz0, vzp2, vzm, dx, rdx);
    float dvx_dz = dad(vxc[2], vx0, vxc[3], vxc[0], dz, rdz);
    if (px) dvz_dx = kdiv(dvz_dx, X.K, X.r);
    if (E) dvx_dz = kdiv(dvx_dz, Z.K, Z.r);
    float e = dvz_dx * ba * dt;
    if (px && X.a != 0.f) e = X.a * dad(q1[0], q1[1], q1[2], q1[3], dx, rdx) + e;
    if (E && Z.a != 0.f) e = e + Z.a * dad(q2[2], q2[1], q2[3], q2[0], dz, rdz);
    e = e + dvx_dz * bb * dt;
    sxz = sxz + e;
    stb(a, sw + kSxz * Nb, v0, sxz);
    if (cn) {
      if (crid >= 0) {
        if (z == cz) {
          szz = szz + cres;
          sxx = (float)((double)sxx + kRS * (double)cres);
        }
      } else {  // several receivers in the column: each cell's in receiver order
        for (int c = cfirst; c < cfirst + cn; ++c)
          if (z == B.icell[3 * c + 1])
            for (int q = B.iptr[c]; q < B.iptr[c + 1]; ++q) {
              const float v = row[B.irid[q]];
              szz = szz + v;
              sxx = (float)((double)sxx + kRS * (double)v);
            }
      }
    }
    // sxx += a_x_half dphi_xx/dx + bb dvx/dx / K_x_half dt; szz likewise in z
    float tx = bb * dad(vx0, vxm, vxp, vxm2, dx, rdx);
    float tz = ba * dad(vz0, vzc[1], vzc[3], vzc[0], dz, rdz);
    if (px) tx = kdiv(tx, X.Kh, X.rh);
    if (E) tz = kdiv(tz, Z.Kh, Z.rh);
    tx = tx * dt;
    tz = tz * dt;
    if (px && X.ah != 0.f) tx = X.ah * dad(q3[0], q3[1], q3[2], q3[3], dx, rdx) + tx;
    if (E && Z.ah != 0.f) tz = Z.ah * dad(q4[2], q4[1], q4[3], q4[0], dz, rdz) + tz;
    sxx = sxx + tx;
    szz = szz + tz;
    stb(a, sw + kSxx * Nb, v0, sxx);
    stb(a, sw + kSzz * Nb, v0, szz);
    // psi_xx = b_x psi + lambda szz dt + (lambda + 2.0 mu) sxx dt;
    // psi_zz = b_z psi + (lambda + 2.0 mu) szz dt + lambda sxx dt
    if (xlive) {
      stb(m, sm + kMvzx * Nb, v0, X.bh * hzx + sxz * amu * dt);
      stb(m, sm + kMvxx * Nb, v0, (float)((double)(X.b * hxx + lam * szz * dt) + l2m * (double)sxx * dt64));
    }
    if (zlive) {
      stb(m, sm + kMvxz * Nb, v0, Z.bh * hxz + sxz * amu * dt);
      stb(m, sm + kMvzz * Nb, v0,
          (float)((double)(Z.b * hzz) + l2m * (double)szz * dt64 + (double)(lam * sxx * dt)));
    }
  }
}

// el_velocity.cu:84-117 (isFor = false) on the interior, with the density sums;
// ring cells inside the interior add to the sums, their velocities are
// restored by other workgroups
template <bool Sliced>
__device__ __forceinline__ void half_rev_vel(CBack& B, const HalfTile& t, float* lds) {
  const auto& A = B.s;
  const int z = t.z, x = t.x, nz = A.nz, nx = A.nx, nzA = A.nzA, nPml = A.nPml, Nb = A.Nb;
  const bool in = z >= nPml && z <= nzA - 1 - nPml && x >= nPml && x <= nx - 1 - nPml;
  const bool inner = z > nPml + 2 && z < nzA - nPml - 3 && x > nPml + 2 && x < nx - nPml - 3;
  const float dt = A.dt, dz = A.dz, dx = A.dx, rdz = A.rdz, rdx = A.rdx;
  const int v0 = 4 * (x * nz + z), cb = 4 * nz;
  const int vm1 = v0 - cb, vm2 = vm1 - cb, vp1 = v0 + cb, vp2 = vp1 + cb;
  const Rsrc w = rsrc(A.wo), a = rsrc(B.ai), md = rsrc(A.md);
  float ba = 0.f, bb = 0.f;
  if (in) ba = ldb(md, 3 * Nb, v0), bb = ldb(md, 4 * Nb, v0);
  sum_shots<2, Sliced>(A.ns, in, in, lds, rsrc(B.acc), 3, Nb, v0, [&](int s, float (&c)[2]) {
    const int sw = s * kWaveComps * Nb;
    const f4 szc = ldb4(w, sw + kSzz * Nb, v0 - 4), xzc = ldb4(w, sw + kSxz * Nb, v0 - 8);
    const float sxzm = ldb(w, sw + kSxz * Nb, vm1), sxzp = ldb(w, sw + kSxz * Nb, vp1), sxzm2 = ldb(w, sw + kSxz * Nb, vm2);
    const float sxxp = ldb(w, sw + kSxx * Nb, vp1), sxx0 = ldb(w, sw + kSxx * Nb, v0),
                sxxp2 = ldb(w, sw + kSxx * Nb, vp2), sxxm = ldb(w, sw + kSxx * Nb, vm1);
    const float avz = ldb(a, sw + kVz * Nb, v0), avx = ldb(a, sw + kVx * Nb, v0);
    const float vz = ldb(w, sw + kVz * Nb, v0), vx = ldb(w, sw + kVx * Nb, v0);
    const float dszz_dz = dfw(szc[2], szc[1], szc[3], szc[0], dz, rdz);
    const float dsxz_dx = dfw(xzc[2], sxzm, sxzp, sxzm2, dx, rdx);
    const float dsxz_dz = dfw(xzc[2], xzc[1], xzc[3], xzc[0], dz, rdz);
    const float dsxx_dx = dfw(sxxp, sxx0, sxxp2, sxxm, dx, rdx);
    const float fz = dszz_dz + dsxz_dx, fx = dsxz_dz + dsxx_dx;
    c[0] = avz * fz;
    c[1] = avx * fx;
    if (inner) {
      stb(w, sw + kVz * Nb, v0, vz - fz * ba * dt);
      stb(w, sw + kVx * Nb, v0, vx - fx * bb * dt);
    }
  });
}

// add_source(-) and el_stress.cu:90-131 (isFor = false) on the interior, with
// the lambda / mu sums; ring cells as above
template <bool Sliced>
__device__ __forceinline__ void half_rev_stress(CBack& B, const HalfTile& t, int it, float* lds) {
  const auto& A = B.s;
  const int z = t.z, x = t.x, nz = A.nz, nx = A.nx, nzA = A.nzA, nPml = A.nPml, Nb = A.Nb;
  const bool in = z >= nPml && z <= nzA - 1 - nPml && x >= nPml && x <= nx - 1 - nPml;
  const bool inner = z > nPml + 2 && z < nzA - nPml - 3 && x > nPml + 2 && x < nx - nPml - 3;
  const float dt = A.dt, dz = A.dz, dx = A.dx, rdz = A.rdz, rdx = A.rdx;
  const double dt64 = (double)dt;
  const int v0 = 4 * (x * nz + z), cb = 4 * nz;
  const int vm1 = v0 - cb, vm2 = vm1 - cb, vp1 = v0 + cb, vp2 = vp1 + cb;
  const Rsrc w = rsrc(A.wo), a = rsrc(B.ai), md = rsrc(A.md);
  float lam = 0.f, mu = 0.f, amu = 0.f;
  if (in) lam = ldb(md, 0, v0), mu = ldb(md, Nb, v0), amu = ldb(md, 2 * Nb, v0);
  const double l2m = (double)lam + 2.0 * (double)mu;
  sum_shots<3, Sliced>(A.ns, in, in, lds, rsrc(B.acc), 0, Nb, v0, [&](int s, float (&c)[3]) {
    const int sw = s * kWaveComps * Nb;
    const f4 vzc = ldb4(w, sw + kVz * Nb, v0 - 8), vxc = ldb4(w, sw + kVx * Nb, v0 - 4);
    const float vzp = ldb(w, sw + kVz * Nb, vp1), vzp2 = ldb(w, sw + kVz * Nb, vp2), vzm = ldb(w, sw + kVz * Nb, vm1);
    const float vxm = ldb(w, sw + kVx * Nb, vm1), vxp = ldb(w, sw + kVx * Nb, vp1), vxm2 = ldb(w, sw + kVx * Nb, vm2);
    const float azz = ldb(a, sw + kSzz * Nb, v0), axx = ldb(a, sw + kSxx * Nb, v0), axz = ldb(a, sw + kSxz * Nb, v0);
    float szz = ldb(w, sw + kSzz * Nb, v0), sxx = ldb(w, sw + kSxx * Nb, v0), sxz = ldb(w, sw + kSxz * Nb, v0);
    const float vz0 = vzc[2], vx0 = vxc[1];
    const float dvz_dz = dfw(vz0, vzc[1], vzc[3], vzc[0], dz, rdz);
    const float dvx_dx = dfw(vx0, vxm, vxp, vxm2, dx, rdx);
    const float dvx_dz = dfw(vxc[2], vx0, vxc[3], vxc[0], dz, rdz);
    const float dvz_dx = dfw(vzp, vz0, vzp2, vzm, dx, rdx);
    c[0] = (azz + axx) * (dvz_dz + dvx_dx);
    c[1] = azz * dvz_dz + axx * dvx_dx;
    c[2] = axz * (dvx_dz + dvz_dx);
    if (inner) {
      if (x == ((CInt*)A.zx)[2 * s + 1] && z == ((CInt*)A.zx)[2 * s]) {
        const float amp = A.amp[(size_t)s * A.nSteps + it];
        szz = szz - kSrcScale * amp * dt;
        sxx = (float)((double)sxx - kRS * (double)kSrcScale * (double)amp * dt64);
      }
      stb(w, sw + kSzz * Nb, v0,
          (float)((double)szz - (l2m * (double)dvz_dz + (double)(lam * dvx_dx)) * dt64));
      stb(w, sw + kSxx * Nb, v0,
          (float)((double)sxx - ((double)(lam * dvz_dz) + l2m * (double)dvx_dx) * dt64));
      stb(w, sw + kSxz * Nb, v0, sxz - amu * (dvx_dz + dvz_dx) * dt);
    }
  });
}

// Backward pairs with disjoint reads and writes share a launch, strip by strip:
//   a: adj_vel(it) + rev_stress(it) (rev_stress reads the adjoint stress that
//      adj_vel also only reads), the ring's stresses of step it restored;
//   b: adj_stress(it) + rev_vel(it-1) (rev_vel reads the adjoint velocity that
//      adj_stress also only reads), the ring's velocities of it - 1 restored.
// kinds: 1 the adjoint half, 2 the reversal, 3 both.
template <bool Sliced>
__global__ __launch_bounds__(Sliced ? 1024 : 256) void k_half_bwd_a(
    const BackArgs* __restrict__ args, int it, int ring, int kinds, int places, unsigned inv) {
  __shared__ float lds[Sliced ? kSumShots * 3 * kSumCells : 1];
  int part;
  const int chunk = half_chunk(places, inv, part);
  CBack& B = ((CBack*)args)[part];
  const auto& A = B.s;
  const int row = (int)blockIdx.y;
  if (row >= 2 * A.hgz) {
    int lo, hi;
    own_shots<Sliced>(A.ns, lo, hi);
    if (kinds & 2) ring_move<false>(A, A.wo, extra_item(2 * A.hgz, chunk), lo, hi, ring, 0, 3);
    return;
  }
  HalfTile t;
  if (!half_tile(A, row >> 1, chunk, t)) return;
  if (row & 1) {
    if (kinds & 2) half_rev_stress<Sliced>(B, t, it, lds);
  } else if (kinds & 1) {
    half_adj_vel<Sliced>(B, t, it, it < A.nSteps - 1);
  }
}

template <bool Sliced>
__global__ __launch_bounds__(Sliced ? 1024 : 256) void k_half_bwd_b(
    const BackArgs* __restrict__ args, int it, int ring, int kinds, int places, unsigned inv) {
  __shared__ float lds[Sliced ? kSumShots * 2 * kSumCells : 1];
  int part;
  const int chunk = half_chunk(places, inv, part);
  CBack& B = ((CBack*)args)[part];
  const auto& A = B.s;
  const int row = (int)blockIdx.y;
  if (row >= 2 * A.hgz) {
    int lo, hi;
    own_shots<Sliced>(A.ns, lo, hi);
    if (kinds & 2) ring_move<false>(A, A.wo, extra_item(2 * A.hgz, chunk), lo, hi, ring, 3, 5);
    return;
  }
  HalfTile t;
  if (!half_tile(A, row >> 1, chunk, t)) return;
  if (row & 1) {
    if (kinds & 2) half_rev_vel<Sliced>(B, t, lds);
  } else if (kinds & 1) {
    half_adj_stress<Sliced>(B, t, it);
  }
}

// ------------------------------------------------------------ exact adjoint
// No reference counterpart: the transpose of the forward time step
// (el_stress_fwd, add_source, el_velocity_fwd, recording), taken operation by
// operation, so that the gradient is the derivative of the discrete misfit
// also where waves enter the C-PML and in zero-shear layers.  The adjoint
// state keeps the reference's sign (the residual is injected with +, so it is
// -dJ/d(state)) and the gradient sums keep the meaning of the reference
// mode's, so k_finalize turns both into (lambda, mu, rho) gradients.
//
// A stencil difference f -> D f of the forward step becomes its transpose
// acting on the coefficient-weighted adjoint, and a C-PML term
// d~ = d / K + psi', psi' = b psi + a d becomes, for the adjoint P of psi,
// d_adj = g / K + a (g + P), P <- b (g + P) (only where the forward updates
// psi, with the forward's gates, including el_velocity.cu:56,71's
// x > nx - nPml).  Each transposed update runs as two passes over the
// update region: the first forms the weighted operands of every cell
// (xt, zero outside the update region), the second applies the transposed
// stencils to them.  The second pass of one update and the first of the next
// touch only their own cell's adjoint, so they share a launch, and so does
// the reverse re-materialisation step that reads the same forward field:
//   k_exact_a(it): reverse velocity step it (v^{it+1} -> v^it from
//     sigma^{it+1}), transposed stress update of step it+1 into v_adj,
//     velocity operands of step it and the density sums from sigma^{it+1};
//   k_exact_b(it): residual of sample it+1 (folded injection), transposed
//     velocity update of step it into sigma_adj, stf gradient, stress
//     operands of step it and the lambda / mu sums from v^it, reverse stress
//     step it (sigma^{it+1} -> sigma^it from v^it).
// Each reversal writes only its cell's own forward field, which the adjoint
// half of its launch does not read; ring cells are restored by the workgroups
// of the extra grid rows.  xt holds two operand sets per shot
// (slots 0-3: Azz, Axx, Axz, Azx of the stress update; 4-7: Bz, Bzx, Bxz, Bx
// of the velocity update).  Outside the C-PML frame (cells whose row or
// column is gated) Azx = Axz, Bzx = Bz and Bx = Bxz, so slots 3, 5 and 7 are
// written and read only inside the frame, and a reader takes slots 2, 4 and 6
// for neighbours outside it.
// Bound by L2-miss traffic on large grids (580x1780, 2 shots: 33.1 -> 28.8 us and
// 39.9 -> 33.3 us a launch, at 5.7 and 6.0 TB/s) and by latency on small ones,
// where 71 and 95 registers leave 7 and 5 waves a SIMD (224x448, 15 shots, four
// threads a cell: 25.2 and 28.9 us; an objective there 143 -> 92.5 ms).  Fewer
// registers make it slower (85 for k_exact_b: 114 ms), and so do more, for the
// next shot's loads (107 ms).
__device__ __forceinline__ float pml_t(float g, float K, float r, float a, float b, float& P) {
  const float tot = g + P;
  P = b * tot;
  return kdiv(g, K, r) + a * tot;
}
// The transposed differences are written through dfw: for a stride st,
// (D+)^T B at j = (c1 (B[j-st] - B[j]) - c2 (B[j-2st] - B[j+st])) / h and
// (D-)^T B at j = (c1 (B[j] - B[j+st]) - c2 (B[j-st] - B[j+2st])) / h, for
// D+ f = (c1 (f[k+1] - f[k]) - c2 (f[k+2] - f[k-1])) / h and
// D- f = (c1 (f[k] - f[k-1]) - c2 (f[k+1] - f[k-2])) / h.


// x neighbour of a cell (byte offset v) from operand slot `own` when the
// neighbour lies in the C-PML frame (`f`), else from slot `base`; the slot
// goes into the per-lane offset, so `f` may differ between lanes.
__device__ __forceinline__ float ldf(Rsrc X, int sx, int Nb, int own, int base, int v, bool f) {
  return ldb(X, sx, v + (f ? own : base) * Nb);
}

template <bool Sliced>
__global__ __launch_bounds__(Sliced ? 1024 : 256) void k_exact_a(const BackArgs* __restrict__ args,
                                                 float* __restrict__ xt, int it, int ring, int first,
                                                 int places, unsigned inv) {
  __shared__ float lds[Sliced ? kSumShots * 2 * kSumCells : 1];
  int part;
  const int chunk = half_chunk(places, inv, part);
  CBack& B = ((CBack*)args)[part];
  const auto& A = B.s;
  const int strip = (int)blockIdx.y;
  if (strip >= A.hgz) {
    int lo, hi;
    own_shots<Sliced>(A.ns, lo, hi);
    ring_move<false>(A, A.wo, extra_item(A.hgz, chunk), lo, hi, ring, 3, 5);
    return;
  }
  HalfTile t;
  if (!half_tile(A, strip, chunk, t)) return;
  const int z = t.z, x = t.x, nz = A.nz, nx = A.nx, nzA = A.nzA, nPml = A.nPml, Nb = A.Nb;
  const bool live = z >= 2 && z <= nzA - 3 && x <= nx - 3;
  const float dt = A.dt, dz = A.dz, dx = A.dx, rdz = A.rdz, rdx = A.rdx;
  const bool in = z >= nPml && z <= nzA - 1 - nPml && x >= nPml && x <= nx - 1 - nPml;
  const bool inner = z > nPml + 2 && z < nzA - nPml - 3 && x > nPml + 2 && x < nx - nPml - 3;
  const bool pz = z < nPml || z > nzA - nPml - 1;
  const bool px = x < nPml || x > nx - nPml;  // el_velocity's gate
  const int v0 = 4 * (x * nz + z), cb = 4 * nz;
  const int vm1 = v0 - cb, vm2 = vm1 - cb, vp1 = v0 + cb, vp2 = vp1 + cb;
  const Rsrc W = rsrc(A.wo), Ad = rsrc(B.ao), M = rsrc(A.mo), X = rsrc(xt), md = rsrc(A.md);
  float ba = 0.f, bb = 0.f;
  if (live) ba = ldb(md, 3 * Nb, v0), bb = ldb(md, 4 * Nb, v0);
  Coef Z{}, Xc{};
  if (live && pz) Z = coef_row(A.zc, z);
  if (x <= nx - 3 && px) Xc = coef_col(A.xc, x);
  // Azx: slot 3 in the stress update's frame, else Axz
  auto fs = [&](int k) { return pz || x + k < nPml || x + k > nx - nPml - 1; };
  const bool fm2 = fs(-2), fm1 = fs(-1), f0 = fs(0), fp1 = fs(1);
  sum_shots<2, Sliced>(A.ns, live, in, lds, rsrc(B.acc), 3, Nb, v0, [&](int s, float (&c)[2]) {
    const int sw = s * kWaveComps * Nb, sm = s * kMemComps * Nb, sx = s * 8 * Nb;
    // forward stresses sigma^{it+1} around the cell (interior cells)
    f4 szc{}, sxc{};
    float sxzmx = 0.f, sxzpx = 0.f, sxzm2x = 0.f, sxxpx = 0.f, sxx0 = 0.f, sxxp2x = 0.f, sxxmx = 0.f,
          wvz = 0.f, wvx = 0.f;
    if (in) {
      szc = ldb4(W, sw + kSzz * Nb, v0 - 4), sxc = ldb4(W, sw + kSxz * Nb, v0 - 8);
      sxzmx = ldb(W, sw + kSxz * Nb, vm1), sxzpx = ldb(W, sw + kSxz * Nb, vp1), sxzm2x = ldb(W, sw + kSxz * Nb, vm2);
      sxxpx = ldb(W, sw + kSxx * Nb, vp1), sxx0 = ldb(W, sw + kSxx * Nb, v0);
      sxxp2x = ldb(W, sw + kSxx * Nb, vp2), sxxmx = ldb(W, sw + kSxx * Nb, vm1);
      wvz = ldb(W, sw + kVz * Nb, v0), wvx = ldb(W, sw + kVx * Nb, v0);
    }
    float vz = ldb(Ad, sw + kVz * Nb, v0), vx = ldb(Ad, sw + kVx * Nb, v0);
    float q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
    if (pz) q0 = ldb(M, sm + kMszz * Nb, v0), q1 = ldb(M, sm + kMsxzz * Nb, v0);
    if (px) q2 = ldb(M, sm + kMsxzx * Nb, v0), q3 = ldb(M, sm + kMsxx * Nb, v0);
    if (!first) {
      const f4 azz = ldb4(X, sx, v0 - 4);           // Azz at z-1 .. z+2
      const f4 axz = ldb4(X, sx + 2 * Nb, v0 - 8);  // Axz at z-2 .. z+1
      const float azxm = ldf(X, sx, Nb, 3, 2, vm1, fm1), azx0 = ldf(X, sx, Nb, 3, 2, v0, f0),
                  azxm2 = ldf(X, sx, Nb, 3, 2, vm2, fm2), azxp = ldf(X, sx, Nb, 3, 2, vp1, fp1);
      const float axx0 = ldb(X, sx + Nb, v0), axxp = ldb(X, sx + Nb, vp1),
                  axxm = ldb(X, sx + Nb, vm1), axxp2 = ldb(X, sx + Nb, vp2);
      // (D-)^T Azz along z + (D+)^T Azx along x; (D-)^T Axx along x + (D+)^T Axz along z
      vz = vz + (dfw(azz[1], azz[2], azz[0], azz[3], dz, rdz) + dfw(azxm, azx0, azxm2, azxp, dx, rdx));
      vx = vx + (dfw(axx0, axxp, axxm, axxp2, dx, rdx) + dfw(axz[1], axz[2], axz[0], axz[3], dz, rdz));
      stb(Ad, sw + kVz * Nb, v0, vz);
      stb(Ad, sw + kVx * Nb, v0, vx);
    }
    const float gz = dt * ba * vz, gx = dt * bb * vx;
    float oz = gz, ozx = gz, oxz = gx, ox = gx;
    if (pz) {
      oz = pml_t(gz, Z.Kh, Z.rh, Z.ah, Z.bh, q0);
      stb(M, sm + kMszz * Nb, v0, q0);
      oxz = pml_t(gx, Z.K, Z.r, Z.a, Z.b, q1);
      stb(M, sm + kMsxzz * Nb, v0, q1);
    }
    if (px) {
      ozx = pml_t(gz, Xc.K, Xc.r, Xc.a, Xc.b, q2);
      stb(M, sm + kMsxzx * Nb, v0, q2);
      ox = pml_t(gx, Xc.Kh, Xc.rh, Xc.ah, Xc.bh, q3);
      stb(M, sm + kMsxx * Nb, v0, q3);
    }
    stb(X, sx + 4 * Nb, v0, oz);
    stb(X, sx + 6 * Nb, v0, oxz);
    if (pz || px) {  // the velocity update's frame
      stb(X, sx + 5 * Nb, v0, ozx);
      stb(X, sx + 7 * Nb, v0, ox);
    }
    if (in) {
      const float dszz_dz = dfw(szc[2], szc[1], szc[3], szc[0], dz, rdz);
      const float dsxz_dx = dfw(sxc[2], sxzmx, sxzpx, sxzm2x, dx, rdx);
      const float dsxz_dz = dfw(sxc[2], sxc[1], sxc[3], sxc[0], dz, rdz);
      const float dsxx_dx = dfw(sxxpx, sxx0, sxxp2x, sxxmx, dx, rdx);
      const float fz = dszz_dz + dsxz_dx, fx = dsxz_dz + dsxx_dx;
      c[0] = vz * fz;
      c[1] = vx * fx;
      if (inner) {  // el_velocity.cu:84-117, isFor = false
        stb(W, sw + kVz * Nb, v0, wvz - fz * ba * dt);
        stb(W, sw + kVx * Nb, v0, wvx - fx * bb * dt);
      }
    }
  });
}

template <bool Sliced>
__global__ __launch_bounds__(Sliced ? 1024 : 256) void k_exact_b(const BackArgs* __restrict__ args,
                                                 float* __restrict__ xt,
                                                 const float* __restrict__ srcwin, int it, int ring,
                                                 int places, unsigned inv) {
  __shared__ float lds[Sliced ? kSumShots * 3 * kSumCells : 1];
  int part;
  const int chunk = half_chunk(places, inv, part);
  CBack& B = ((CBack*)args)[part];
  const auto& A = B.s;
  const int strip = (int)blockIdx.y;
  if (strip >= A.hgz) {
    int lo, hi;
    own_shots<Sliced>(A.ns, lo, hi);
    ring_move<false>(A, A.wo, extra_item(A.hgz, chunk), lo, hi, ring, 0, 3);
    return;
  }
  HalfTile t;
  if (!half_tile(A, strip, chunk, t)) return;
  const int z = t.z, x = t.x, nz = A.nz, nx = A.nx, nzA = A.nzA, nPml = A.nPml, Nb = A.Nb;
  const bool live = z >= 2 && z <= nzA - 3 && x <= nx - 3;
  const float dt = A.dt, dz = A.dz, dx = A.dx, rdz = A.rdz, rdx = A.rdx;
  const double dt64 = (double)dt;
  const bool in = z >= nPml && z <= nzA - 1 - nPml && x >= nPml && x <= nx - 1 - nPml;
  const bool inner = z > nPml + 2 && z < nzA - nPml - 3 && x > nPml + 2 && x < nx - nPml - 3;
  const bool pz = z < nPml || z > nzA - nPml - 1;
  const bool px = x < nPml || x > nx - nPml - 1;  // el_stress's gate
  const int v0 = 4 * (x * nz + z), cb = 4 * nz;
  const int vm1 = v0 - cb, vm2 = vm1 - cb, vp1 = v0 + cb, vp2 = vp1 + cb;
  const Rsrc W = rsrc(A.wo), Ad = rsrc(B.ao), M = rsrc(A.mo), X = rsrc(xt), md = rsrc(A.md);
  float lam = 0.f, mu = 0.f, amu = 0.f;
  if (live) lam = ldb(md, 0, v0), mu = ldb(md, Nb, v0), amu = ldb(md, 2 * Nb, v0);
  Coef Z{}, Xc{};
  if (live && pz) Z = coef_row(A.zc, z);
  if (x <= nx - 3 && px) Xc = coef_col(A.xc, x);
  const double l2m64 = (double)lam + 2.0 * (double)mu;
  const float l2m = (float)l2m64;
  // Bzx and Bx: slots 5 and 7 in the velocity update's frame, else Bz and Bxz
  auto fv = [&](int k) { return pz || x + k < nPml || x + k > nx - nPml; };
  const bool fm2 = fv(-2), fm1 = fv(-1), f0 = fv(0), fp1 = fv(1), fp2 = fv(2);
  const float* const row = B.res + (size_t)(it + 1) * A.R;
  sum_shots<3, Sliced>(A.ns, live, in, lds, rsrc(B.acc), 0, Nb, v0, [&](int s, float (&c)[3]) {
    const int sw = s * kWaveComps * Nb, sm = s * kMemComps * Nb, sx = s * 8 * Nb;
    const int zs = ((CInt*)A.zx)[2 * s], xs = ((CInt*)A.zx)[2 * s + 1];
    const __attribute__((address_space(4))) ColInj* ci =
        (const __attribute__((address_space(4))) ColInj*)B.inj + (size_t)(A.s0 + s) * nx + x;
    const int cfirst = ci->first, cn = ci->n, cz = ci->z, crid = ci->rid;
    // forward velocities v^it around the cell (interior cells)
    f4 vzc{}, vxc{};
    float vzpx = 0.f, vzp2x = 0.f, vzmx = 0.f, vxmx = 0.f, vxpx = 0.f, vxm2x = 0.f, wszz = 0.f,
          wsxx = 0.f, wsxz = 0.f;
    if (in) {
      vzc = ldb4(W, sw + kVz * Nb, v0 - 8), vxc = ldb4(W, sw + kVx * Nb, v0 - 4);
      vzpx = ldb(W, sw + kVz * Nb, vp1), vzp2x = ldb(W, sw + kVz * Nb, vp2), vzmx = ldb(W, sw + kVz * Nb, vm1);
      vxmx = ldb(W, sw + kVx * Nb, vm1), vxpx = ldb(W, sw + kVx * Nb, vp1), vxm2x = ldb(W, sw + kVx * Nb, vm2);
      wszz = ldb(W, sw + kSzz * Nb, v0), wsxx = ldb(W, sw + kSxx * Nb, v0), wsxz = ldb(W, sw + kSxz * Nb, v0);
    }
    float szz = ldb(Ad, sw + kSzz * Nb, v0), sxx = ldb(Ad, sw + kSxx * Nb, v0), sxz = ldb(Ad, sw + kSxz * Nb, v0);
    float q0 = 0.f, q1 = 0.f, q2 = 0.f, q3 = 0.f;
    if (pz) q0 = ldb(M, sm + kMvzz * Nb, v0), q1 = ldb(M, sm + kMvxz * Nb, v0);
    if (px) q2 = ldb(M, sm + kMvxx * Nb, v0), q3 = ldb(M, sm + kMvzx * Nb, v0);
    const f4 bzc = ldb4(X, sx + 4 * Nb, v0 - 8);   // Bz at z-2 .. z+1
    const f4 bxzc = ldb4(X, sx + 6 * Nb, v0 - 4);  // Bxz at z-1 .. z+2
    const float bzx0 = ldf(X, sx, Nb, 5, 4, v0, f0), bzxp = ldf(X, sx, Nb, 5, 4, vp1, fp1),
                bzxm = ldf(X, sx, Nb, 5, 4, vm1, fm1), bzxp2 = ldf(X, sx, Nb, 5, 4, vp2, fp2);
    const float bxm = ldf(X, sx, Nb, 7, 6, vm1, fm1), bx0 = ldf(X, sx, Nb, 7, 6, v0, f0),
                bxm2 = ldf(X, sx, Nb, 7, 6, vm2, fm2), bxp = ldf(X, sx, Nb, 7, 6, vp1, fp1);
    if (cn) {
      if (crid >= 0) {
        if (z == cz) {
          const float v = row[crid];
          szz = szz + v;
          sxx = (float)((double)sxx + kRS * (double)v);
        }
      } else {  // several receivers in the column: each cell's in receiver order
        for (int k = cfirst; k < cfirst + cn; ++k)
          if (z == B.icell[3 * k + 1])
            for (int q = B.iptr[k]; q < B.iptr[k + 1]; ++q) {
              const float v = row[B.irid[q]];
              szz = szz + v;
              sxx = (float)((double)sxx + kRS * (double)v);
            }
      }
    }
    // (D+)^T Bz along z; (D-)^T Bzx along x + (D-)^T Bxz along z; (D+)^T Bx along x
    szz = szz + dfw(bzc[1], bzc[2], bzc[0], bzc[3], dz, rdz);
    sxz = sxz + (dfw(bzx0, bzxp, bzxm, bzxp2, dx, rdx) + dfw(bxzc[1], bxzc[2], bxzc[0], bxzc[3], dz, rdz));
    sxx = sxx + dfw(bxm, bx0, bxm2, bxp, dx, rdx);
    stb(Ad, sw + kSzz * Nb, v0, szz);
    stb(Ad, sw + kSxx * Nb, v0, sxx);
    stb(Ad, sw + kSxz * Nb, v0, sxz);
    // d(szz, sxx)/d(stf) at the source: 1500^2 dt and the window (add_source)
    const bool at_src = x == xs && z == zs;
    if (at_src && B.stf_grad)
      B.stf_grad[(size_t)s * A.nSteps + it] = (float)(-(double)kSrcScale * dt64 *
                                                      ((double)szz + kRS * (double)sxx) * (double)srcwin[it]);
    const float Gzz = dt * (l2m * szz + lam * sxx);
    const float Gxx = dt * (lam * szz + l2m * sxx);
    const float Gs = dt * amu * sxz;
    float ozz = Gzz, oxx = Gxx, oxz = Gs, ozx = Gs;
    if (pz) {
      ozz = pml_t(Gzz, Z.K, Z.r, Z.a, Z.b, q0);
      stb(M, sm + kMvzz * Nb, v0, q0);
      oxz = pml_t(Gs, Z.Kh, Z.rh, Z.ah, Z.bh, q1);
      stb(M, sm + kMvxz * Nb, v0, q1);
    }
    if (px) {
      oxx = pml_t(Gxx, Xc.K, Xc.r, Xc.a, Xc.b, q2);
      stb(M, sm + kMvxx * Nb, v0, q2);
      ozx = pml_t(Gs, Xc.Kh, Xc.rh, Xc.ah, Xc.bh, q3);
      stb(M, sm + kMvzx * Nb, v0, q3);
    }
    stb(X, sx, v0, ozz);
    stb(X, sx + Nb, v0, oxx);
    stb(X, sx + 2 * Nb, v0, oxz);
    if (pz || px) stb(X, sx + 3 * Nb, v0, ozx);  // the stress update's frame
    if (in) {
      const float dvz_dz = dfw(vzc[2], vzc[1], vzc[3], vzc[0], dz, rdz);
      const float dvx_dx = dfw(vxc[1], vxmx, vxpx, vxm2x, dx, rdx);
      const float dvx_dz = dfw(vxc[2], vxc[1], vxc[3], vxc[0], dz, rdz);
      const float dvz_dx = dfw(vzpx, vzc[2], vzp2x, vzmx, dx, rdx);
      c[0] = (szz + sxx) * (dvz_dz + dvx_dx);
      c[1] = szz * dvz_dz + sxx * dvx_dx;
      c[2] = sxz * (dvx_dz + dvz_dx);
      if (inner) {  // add_source(-) then el_stress.cu:90-131, isFor = false
        if (at_src) {
          const float amp = A.amp[(size_t)s * A.nSteps + it];
          wszz = wszz - kSrcScale * amp * dt;
          wsxx = (float)((double)wsxx - kRS * (double)kSrcScale * (double)amp * dt64);
        }
        stb(W, sw + kSzz * Nb, v0, (float)((double)wszz - (l2m64 * (double)dvz_dz + (double)(lam * dvx_dx)) * dt64));
        stb(W, sw + kSxx * Nb, v0, (float)((double)wsxx - ((double)(lam * dvz_dz) + l2m64 * (double)dvx_dx) * dt64));
        stb(W, sw + kSxz * Nb, v0, wsxz - amu * (dvx_dz + dvz_dx) * dt);
      }
    }
  });
}
