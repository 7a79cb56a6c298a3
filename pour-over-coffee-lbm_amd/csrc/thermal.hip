// Thermal D3Q7 lattice Boltzmann step (temperature populations) for gfx950.
//
// Replaces (reference): src/physics/thermal_lbm.py
//   :186-201 equilibrium g_eq = w_q T; :203-229 BGK collision with the heat
//   source; :231-253 streaming (an out-of-box source keeps the cell's own
//   value); :255-266 temperature; :268-286 heat flux -k grad T; :288-346
//   Dirichlet / Neumann / convective boundary forms; :348-376 stability test;
//   :378-394 min / max / mean; :518-538 convection source -u.grad T.
//
// The reference collides locally and then pull-streams in a second pass.
// Here one kernel collides and pushes: cell x reads its 7 streamed
// populations (coalesced), forms T, S and g*, and writes g*_q to x + e_q, or
// to itself when x - e_q lies outside the box -- the reference's boundary
// rule, every destination written exactly once.  A second kernel forms the
// new temperature (the reference's compute_temperature) with the stability
// test fused in; in a run of pure-diffusion steps the second kernel runs
// once, after the last step, and the last collide pass stores the
// temperature of its input state.  Temperature buffers ping-pong, so
// temperature_old needs no copy.  The arithmetic follows the reference's FP32 expressions operation by
// operation with contraction off:
//   T = ((((((0 + g0) + g1) + g2) + g3) + g4) + g5) + g6
//   g* = (g - omega (g - w T)) + (w S) 1
//   dT/dx = (T[x+1] - T[x-1]) / 2,  S += -((ux dTdx + uy dTdy) + uz dTdz)
// so an FP32 numpy restatement of the same expressions agrees bit for bit.
// With a base heat source bound (hsb) every step starts from it, S = base
// (+ convection), and writes S to the heat source: the coupled loop's
// reset_heat_source_to_base (thermal_fluid_coupled.py:193-194) at no extra
// pass.
#include <algorithm>

#include "engine.h"

namespace pol {

constexpr int TQ = 7;
__host__ __device__ constexpr int TEX(int q) { return q == 1 ? 1 : (q == 2 ? -1 : 0); }
__host__ __device__ constexpr int TEY(int q) { return q == 3 ? 1 : (q == 4 ? -1 : 0); }
__host__ __device__ constexpr int TEZ(int q) { return q == 5 ? 1 : (q == 6 ? -1 : 0); }
template <typename R>
__host__ __device__ constexpr R TW(int q) {
  return q == 0 ? R(0.25) : R(0.125);
}

constexpr uint32_t STAT_BLOCKS = 1024;
constexpr int STAT_ROW = 4;

// |u| > 1.  The rounded square root of s exceeds 1 exactly when s is above the
// first value after 1 (sqrt(1 + eps) rounds to 1), so none is taken.
template <typename R>
__device__ inline bool faster_than_one(R x, R y, R z) {
#pragma clang fp contract(off)
  constexpr R after_one = R(1) + (sizeof(R) == 4 ? R(0x1p-23) : R(0x1p-52));
  return (x * x + y * y) + z * z > after_one;
}

template <typename R>
__device__ inline R omega_of(const ThermalArgs& a) {
  if constexpr (sizeof(R) == 4) return a.omega_f;
  else return a.omega_d;
}

__device__ inline void decompose(const ThermalArgs& a, uint32_t i, uint32_t& x, uint32_t& y, uint32_t& z) {
  const uint32_t yz = fdiv(i, a.dnx);
  x = i - yz * a.nx;
  z = fdiv(yz, a.dny);
  y = yz - z * a.ny;
}

// WT: also store T = sum_q g_q of the input state into its temperature slot
// (a.T) -- the value the previous step's temperature pass would have
// written.  In a run of pure-diffusion steps only the last step does so (its
// input state's temperature is the one a caller can still read afterwards).
// HAND: the velocity comes from a.u_src (the fluid's field) and is stored to
// a.u beside the step, instead of a copy before it (270 MB and 0.085 ms at
// 224^3; here its read is the one the convection needs anyway, 0.03 ms more).
// NT (populations above the last-level cache): what this pass reads for the
// last time or writes for a later step bypasses the cache: the populations it
// reads, the rest and the y and z populations it writes, the sources, the
// velocity handed over.  The temperature's neighbours and the x populations
// written stay cached (their one-cell shift splits a sector at both ends of
// every wave: streamed as well, diffusion at 187 x 150 x 201 63.2 us, convection
// collide pass at 224^3 173 -> 187).  Stores alone: diffusion 66.4 -> 61.1 us,
// 224^3 135.3 -> 132.7.  Loads and the velocity too, coupled step at 224^3: this
// pass 173 -> 160 us, the fluid step after it 116 -> 108.
template <typename R, bool CONV, bool WT, bool HAND, bool NT>
__global__ void __launch_bounds__(256) k_thermal_collide(const ThermalArgs a) {
#pragma clang fp contract(off)
  const uint32_t lblk = ordered_block(a.ord);
  if (lblk >= a.ord.nblk) return;
  const uint32_t i = lblk * 256u + threadIdx.x;
  if (i >= a.N) return;
  if (i == 0) *a.bad = 0u;  // counted by the temperature pass that follows
  uint32_t x, y, z;
  decompose(a, i, x, y, z);
  const R* __restrict__ gin = (const R*)a.gin;
  R* __restrict__ gout = (R*)a.gout;
  const size_t N = a.N;
  R g[TQ];
#pragma unroll
  for (int q = 0; q < TQ; ++q) g[q] = load_as<NT>(gin + q * N + i);
  R T = R(0);
#pragma unroll
  for (int q = 0; q < TQ; ++q) T = T + g[q];
  if constexpr (WT) ((R*)a.T)[i] = T;
  R* __restrict__ hs = (R*)a.hs;
  const R* __restrict__ hsb = (const R*)a.hsb;
  R S = hsb ? load_as<NT>(hsb + i) : hs[i];
  bool write_s = hsb != nullptr;
  R v0 = R(0), v1 = R(0), v2 = R(0);
  if constexpr (HAND) {  // each cell reads and writes its own elements only: u_src may be u
    const R* us = (const R*)a.u_src;
    v0 = load_as<NT>(us + i);
    v1 = load_as<NT>(us + N + i);
    v2 = load_as<NT>(us + 2 * N + i);
    R* u = (R*)a.u;
    store_as<NT>(u + i, v0);
    store_as<NT>(u + N + i, v1);
    store_as<NT>(u + 2 * N + i, v2);
    if (a.report) {  // cells with |u| > 1: zero on entry, taken and cleared by the fold
      const bool fast = faster_than_one(v0, v1, v2);
      const uint64_t cells = __ballot(fast);
      if (fast && (cells & ((1ull << (threadIdx.x & 63)) - 1ull)) == 0ull) atomicAdd(a.bad + 1, (uint32_t)__popcll(cells));
    }
  }
  if constexpr (CONV) {
    if (x >= 1 && x + 1 < a.nx && y >= 1 && y + 1 < a.ny && z >= 1 && z + 1 < a.nz) {
      const R* __restrict__ Tf = (const R*)a.T;
      if constexpr (!HAND) {
        const R* __restrict__ u = (const R*)a.u;
        v0 = u[i];
        v1 = u[N + i];
        v2 = u[2 * N + i];
      }
      const R dTdx = (Tf[i + 1] - Tf[i - 1]) / R(2);
      const R dTdy = (Tf[i + a.nx] - Tf[i - a.nx]) / R(2);
      const R dTdz = (Tf[i + a.nxy] - Tf[i - a.nxy]) / R(2);
      const R conv = -((v0 * dTdx + v1 * dTdy) + v2 * dTdz);
      S = S + conv;
      write_s = true;
    }
  }
  if (write_s) store_as<NT>(hs + i, S);
  const R om = omega_of<R>(a);
#pragma unroll
  for (int q = 0; q < TQ; ++q) {
    const R w = TW<R>(q);
    const R geq = w * T;
    const R gs = (g[q] - om * (g[q] - geq)) + (w * S) * R(1);
    const int ex = TEX(q), ey = TEY(q), ez = TEZ(q);
    // destination x + e_q when inside the box
    const bool to_in = (ex == 0 || (ex > 0 ? x + 1 < a.nx : x >= 1)) && (ey == 0 || (ey > 0 ? y + 1 < a.ny : y >= 1)) &&
                       (ez == 0 || (ez > 0 ? z + 1 < a.nz : z >= 1));
    // own slot when the source x - e_q lies outside the box
    const bool from_out = (ex > 0 && x == 0) || (ex < 0 && x + 1 == a.nx) || (ey > 0 && y == 0) ||
                          (ey < 0 && y + 1 == a.ny) || (ez > 0 && z == 0) || (ez < 0 && z + 1 == a.nz);
    const int64_t off = (int64_t)ex + (int64_t)ey * a.nx + (int64_t)ez * a.nxy;
    if (q == 0) {
      store_as<NT>(gout + i, gs);
    } else {
      if (to_in) {
        R* p = gout + q * N + (size_t)((int64_t)i + off);
        if (ex != 0) *p = gs;
        else store_as<NT>(p, gs);
      }
      if (from_out) gout[q * N + i] = gs;
    }
  }
}

// {min, max, sum, count} of the block's lanes into its row of partial.
__device__ inline void stat_row(double mn, double mx, double sm, double c, double* __restrict__ partial) {
  mn = wave_min(mn);
  mx = wave_max(mx);
  sm = wave_sum(sm);
  c = wave_sum(c);
  __shared__ double sh[4][STAT_ROW];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane == 0) {
    sh[wid][0] = mn;
    sh[wid][1] = mx;
    sh[wid][2] = sm;
    sh[wid][3] = c;
  }
  __syncthreads();
  if (threadIdx.x < STAT_ROW) {
    const int s = threadIdx.x;
    double r = sh[0][s];
    for (int w = 1; w < 4; ++w) r = s == 0 ? fmin(r, sh[w][s]) : (s == 1 ? fmax(r, sh[w][s]) : r + sh[w][s]);
    partial[(size_t)blockIdx.x * STAT_ROW + s] = r;
  }
}

template <typename R>
struct Vec16;  // 16 bytes
template <>
struct Vec16<float> {
  typedef float type __attribute__((ext_vector_type(4)));
};
template <>
struct Vec16<double> {
  typedef double type __attribute__((ext_vector_type(2)));
};
// Values 4 j .. 4 j + 3 of p (16-byte aligned).
template <bool NT = false, typename R>
__device__ inline void load_quad(const R* __restrict__ p, uint32_t j, R (&v)[4]) {
  using V = typename Vec16<R>::type;
  constexpr int W = 16 / sizeof(R);
#pragma unroll
  for (int k = 0; k < 4; k += W) {
    const V t = load_as<NT>((const V*)(p + 4 * (size_t)j + k));
#pragma unroll
    for (int l = 0; l < W; ++l) v[k + l] = t[l];
  }
}
template <bool NT, typename R>
__device__ inline void store_quad(R* __restrict__ p, uint32_t j, const R (&v)[4]) {
  using V = typename Vec16<R>::type;
  constexpr int W = 16 / sizeof(R);
#pragma unroll
  for (int k = 0; k < 4; k += W) {
    V t;
#pragma unroll
    for (int l = 0; l < W; ++l) t[l] = v[k + l];
    store_as<NT>((V*)(p + 4 * (size_t)j + k), t);
  }
}

// T' = sum_q g'_q and the stability test, W cells a lane and load.  Bound by
// reading the populations (360 MB at 224^3).  Failing cells are counted in
// *a.bad, which the collide pass before has set to zero: a wave without one
// (every wave of a stable state) neither reduces nor stores anything.
// REP: also the block's {min, max, sum} of T', while they are in registers
// (a statistics pass over T and u after the step took 0.033 ms at 224^3).
// NT (populations above the last-level cache): loads and stores bypass it.  In
// the coupled loop nothing here is read again before the cache has turned over
// (reporting pass at 224^3 85 -> 67 us; cached, its loads also evict what the
// fluid step that follows would find).  In a run with convection the next
// collide pass reads T at once, from HBM then, and the step still gains: what T
// (45 of 405 MB at 224^3) would keep out of the cache is more (16 steps at
// 200^3 2586 -> 2284 us, both passes streamed).
template <typename R, int W, bool REP, bool NT>
__global__ void __launch_bounds__(256) k_thermal_temperature(const ThermalArgs a, double* __restrict__ partial) {
#pragma clang fp contract(off)
  const R* __restrict__ gp = (const R*)a.gout;
  R* __restrict__ Tout = (R*)a.Tout;
  const size_t N = a.N;
  const uint32_t items = a.N / W;
  double mn = 1.0e300, mx = -1.0e300, sm = 0.0;
  uint32_t nbad = 0;
  for (uint32_t j = blockIdx.x * 256u + threadIdx.x; j < items; j += gridDim.x * 256u) {
    R g[TQ][W], T[W];
#pragma unroll
    for (int q = 0; q < TQ; ++q) {
      if constexpr (W == 4) load_quad<NT>(gp + q * N, j, g[q]);
      else g[q][0] = load_as<NT>(gp + q * N + j);
    }
#pragma unroll
    for (int k = 0; k < W; ++k) {
      T[k] = R(0);
      bool bad = false;
#pragma unroll
      for (int q = 0; q < TQ; ++q) {
        const R v = g[q][k];
        T[k] = T[k] + v;
        bad = bad || !(v == v) || fabs(v) > R(1000);
      }
      bad = bad || T[k] < R(-50) || T[k] > R(150) || !(T[k] == T[k]);
      nbad += bad ? 1u : 0u;
      if constexpr (REP) {
        const double d = (double)T[k];
        mn = fmin(mn, d);
        mx = fmax(mx, d);
        sm += d;
      }
    }
    if constexpr (W == 4) store_quad<NT>(Tout, j, T);
    else store_as<NT>(Tout + j, T[0]);
  }
  if (__ballot(nbad != 0u) != 0ull) {
    const double n = wave_sum((double)nbad);
    if ((threadIdx.x & 63) == 0) atomicAdd(a.bad, (uint32_t)n);
  }
  if constexpr (REP) stat_row(mn, mx, sm, 0.0, partial);
}

// {min, max, sum} of T and, with a velocity, the number of cells with |u| > 1:
// up to STAT_BLOCKS blocks stride over the field, four values a lane and load
// where the field's size allows it, and keep their lanes' results in
// registers, so the field is read at memory speed and 1024 rows are left to
// fold.  (One value a lane with a row per 256 cells was bound by its FP64
// shuffles: 0.074 ms for 45 MB, and 0.057 ms to fold 43 904 rows.)
template <typename R, int W>
__global__ void __launch_bounds__(256) k_thermal_stats(const R* __restrict__ T, const R* __restrict__ u, uint32_t N,
                                                       double* __restrict__ partial) {
#pragma clang fp contract(off)
  double mn = 1.0e300, mx = -1.0e300, sm = 0.0;
  uint32_t fast = 0;
  const uint32_t items = N / W;
  auto one = [&](R t) {
    const double d = (double)t;
    mn = fmin(mn, d);
    mx = fmax(mx, d);
    sm += d;
  };
  auto speed = [&](R x, R y, R z) { fast += faster_than_one(x, y, z) ? 1u : 0u; };
  for (uint32_t j = blockIdx.x * 256u + threadIdx.x; j < items; j += gridDim.x * 256u) {
    if constexpr (W == 4) {
      R t[4];
      load_quad(T, j, t);
#pragma unroll
      for (int k = 0; k < 4; ++k) one(t[k]);
      if (u) {
        R x[4], y[4], z[4];
        load_quad(u, j, x);
        load_quad(u + N, j, y);
        load_quad(u + 2 * (size_t)N, j, z);
#pragma unroll
        for (int k = 0; k < 4; ++k) speed(x[k], y[k], z[k]);
      }
    } else {
      one(T[j]);
      if (u) speed(u[j], u[(size_t)N + j], u[2 * (size_t)N + j]);
    }
  }
  stat_row(mn, mx, sm, (double)fast, partial);
}

// Fold of at most STAT_BLOCKS rows {min, max, sum, count} into out (pinned host
// memory): four rows of loads in flight per lane, then across the lanes that
// hold the same column.  count: {unstable, fast} cells of a reporting step;
// the fast ones become the fourth value, are cleared for the next step, and
// the unstable ones follow in out[4].
__global__ void __launch_bounds__(256) k_thermal_fold(const double* __restrict__ partial, uint32_t rows,
                                                      double* __restrict__ out, uint32_t* __restrict__ count) {
  __shared__ double sh[4][STAT_ROW];
  const int s = threadIdx.x & 3, j = threadIdx.x >> 2;
  auto add = [&](double r, double p) { return s == 0 ? fmin(r, p) : (s == 1 ? fmax(r, p) : r + p); };
  const double id = s == 0 ? 1.0e300 : (s == 1 ? -1.0e300 : 0.0);
  double v = id;
  for (uint32_t b = j; b < rows; b += 256) {
    double t[4];
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) t[k] = b + 64 * k < rows ? partial[(size_t)(b + 64 * k) * STAT_ROW + s] : id;
#pragma unroll
    for (int k = 0; k < 4; ++k) v = add(v, t[k]);
  }
  double x, y;
  lane_pair<32>(v, x, y);
  v = add(x, y);
  lane_pair<16>(v, x, y);
  v = add(x, y);
  lane_pair<8>(v, x, y);
  v = add(x, y);
  lane_pair<4>(v, x, y);
  v = add(x, y);
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  if (lane < STAT_ROW) sh[wid][lane] = v;
  __syncthreads();
  if (threadIdx.x < STAT_ROW) {
    double r = add(add(sh[0][s], sh[1][s]), add(sh[2][s], sh[3][s]));
    if (count && s == 3) {
      // one exchange: a plain load here is a scalar one, which the store of
      // the zero does not wait for
      r = (double)atomicExch(count + 1, 0u);
      out[4] = (double)count[0];
    }
    out[s] = r;
  }
}

template <typename R>
__global__ void __launch_bounds__(256) k_thermal_flux(const ThermalArgs a, R* __restrict__ flux) {
#pragma clang fp contract(off)
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= a.N) return;
  uint32_t x, y, z;
  decompose(a, i, x, y, z);
  const size_t N = a.N;
  R q0 = R(0), q1 = R(0), q2 = R(0);
  if (x >= 1 && x + 1 < a.nx && y >= 1 && y + 1 < a.ny && z >= 1 && z + 1 < a.nz) {
    const R* __restrict__ Tf = (const R*)a.T;
    const R dTdx = (Tf[i + 1] - Tf[i - 1]) / R(2);
    const R dTdy = (Tf[i + a.nx] - Tf[i - a.nx]) / R(2);
    const R dTdz = (Tf[i + a.nxy] - Tf[i - a.nxy]) / R(2);
    const R k = a.k ? ((const R*)a.k)[i] : R(0.68);
    q0 = -k * dTdx;
    q1 = -k * dTdy;
    q2 = -k * dTdz;
  }
  flux[i] = q0;
  flux[N + i] = q1;
  flux[2 * N + i] = q2;
}

template <typename R>
__global__ void __launch_bounds__(256) k_thermal_init(const ThermalArgs a) {
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= a.N) return;
  const R T = ((const R*)a.T)[i];
  R* __restrict__ g = (R*)a.gout;
#pragma unroll
  for (int q = 0; q < TQ; ++q) g[(size_t)q * a.N + i] = TW<R>(q) * T;
}

template <typename R>
__global__ void __launch_bounds__(256) k_thermal_boundary(const ThermalArgs a, int kind, const uint8_t* __restrict__ mask,
                                                          R va, R vb) {
#pragma clang fp contract(off)
  const uint32_t i = blockIdx.x * 256u + threadIdx.x;
  if (i >= a.N || !mask[i]) return;
  if (kind == 1) {
    ((R*)a.Tout)[i] = va;
    R* __restrict__ g = (R*)a.gout;
#pragma unroll
    for (int q = 0; q < TQ; ++q) g[(size_t)q * a.N + i] = TW<R>(q) * va;
  } else if (kind == 2) {
    ((R*)a.hs)[i] = va;
  } else {
    const R Ts = ((const R*)a.T)[i];
    ((R*)a.hs)[i] = -(va * (Ts - vb));
  }
}

// ---- launchers ----------------------------------------------------------------
template <typename R, bool NT>
static void thermal_collide(const ThermalArgs& a, bool first, bool last, dim3 grid, hipStream_t s) {
  if (a.conv && a.u_src && first)
    hipLaunchKernelGGL((k_thermal_collide<R, true, false, true, NT>), grid, dim3(256), 0, s, a);
  else if (a.conv)
    hipLaunchKernelGGL((k_thermal_collide<R, true, false, false, NT>), grid, dim3(256), 0, s, a);
  else if (first || !last)
    hipLaunchKernelGGL((k_thermal_collide<R, false, false, false, NT>), grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL((k_thermal_collide<R, false, true, false, NT>), grid, dim3(256), 0, s, a);
}

// Blocks of a pass that strides over the field, W cells a lane.
static uint32_t stride_blocks(uint32_t N, uint32_t W) { return std::min((N / W + 255u) / 256u, STAT_BLOCKS); }

static bool quad_aligned(const void* p) { return ((uintptr_t)p & 15) == 0; }

// The temperature pass: with its statistics (partial not null) striding, four
// cells a lane where every plane starts on a 16-byte boundary, so that few
// rows are left to fold; else one cell a lane (striding: 31.3 -> 33.8 us at
// 187 x 150 x 201).
template <typename R, bool NT>
static void thermal_temperature(const ThermalArgs& a, double* partial, double* out, hipStream_t s) {
  if (!partial) {
    hipLaunchKernelGGL((k_thermal_temperature<R, 1, false, NT>), dim3((a.N + 255) / 256), dim3(256), 0, s, a, nullptr);
    return;
  }
  const bool quad = a.N % 4 == 0 && quad_aligned(a.gout) && quad_aligned(a.Tout);
  const uint32_t blocks = stride_blocks(a.N, quad ? 4 : 1);
  if (quad) hipLaunchKernelGGL((k_thermal_temperature<R, 4, true, NT>), dim3(blocks), dim3(256), 0, s, a, partial);
  else hipLaunchKernelGGL((k_thermal_temperature<R, 1, true, NT>), dim3(blocks), dim3(256), 0, s, a, partial);
  hipLaunchKernelGGL(k_thermal_fold, dim3(1), dim3(256), 0, s, partial, blocks, out, a.bad);
}

template <typename R>
static hipError_t thermal_steps(const ThermalArgs& base, void* const g[2], void* const T[2], int& gcur, int& tcur,
                                int nsteps, double* partial, double* out, hipStream_t s) {
  // With convection a step's source needs the whole temperature field of its
  // input state before it starts, so every step runs the temperature pass.
  // Pure diffusion reads only the cell's own populations: the temperature
  // pass (with the stability test that is reported) runs after the last step
  // only, and the last step's collide pass stores T of its input state
  // itself.  The steps between store none (two temperature buffers: each
  // would be overwritten unread, 4 of 64 B per cell).  A run's first step
  // leaves the input state's temperature as the caller set it (it may be a
  // boundary value rather than sum g).
  // convection reads the temperature's neighbours (populations, T, u and the
  // sources, 80 B a cell); pure diffusion reads only the cell's own values
  const BlockOrder ord = base.conv ? stencil_order(base.N, 20ull * sizeof(R) * base.N, CONVECTION_LINEAR_BYTES)
                                   : linear_order(base.N);
  const dim3 cgrid(launch_blocks(ord));
  // Both population buffers above the last-level cache (168^3 FP32, 133^3 FP64):
  // where diffusion starts to gain.  Runs of 16 steps, cached / streamed (us):
  // FP32 160^3 632 / 755, 168^3 801 / 823, 170^3 895 / 892, 176^3 1028 / 959;
  // FP64 128^3 681 / 861, 134^3 854 / 859, 136^3 944 / 959, 140^3 1098 / 991.
  // Convection gains from a little below on (FP64 112^3 778 / 849, 120^3 1087 /
  // 1055, 134^3 1498 / 1390; FP32 168^3 1431 / 1381, 176^3 1647 / 1517), the
  // coupled loop too (five steps FP32 160^3 983 / 858, 170^3 1118 / 1056).
  const bool nt = 2ull * TQ * sizeof(R) * base.N > LAST_LEVEL_BYTES;
  for (int n = 0; n < nsteps; ++n) {
    ThermalArgs a = base;
    a.ord = ord;
    a.gin = g[gcur];
    a.gout = g[1 - gcur];
    a.T = T[tcur];
    a.Tout = T[1 - tcur];
    const bool last = n + 1 == nsteps;
    if (nt) thermal_collide<R, true>(a, n == 0, last, cgrid, s);
    else thermal_collide<R, false>(a, n == 0, last, cgrid, s);
    double* const rows = last && a.report ? partial : nullptr;
    if (a.conv || last) {
      if (nt) thermal_temperature<R, true>(a, rows, out, s);
      else thermal_temperature<R, false>(a, rows, out, s);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    gcur = 1 - gcur;
    tcur = 1 - tcur;
  }
  return hipSuccess;
}

hipError_t launch_thermal_steps(bool dbl, const ThermalArgs& base, void* const g[2], void* const T[2], int& gcur,
                                int& tcur, int nsteps, double* partial, double* out, hipStream_t s) {
  return dbl ? thermal_steps<double>(base, g, T, gcur, tcur, nsteps, partial, out, s)
             : thermal_steps<float>(base, g, T, gcur, tcur, nsteps, partial, out, s);
}

template <typename R>
static hipError_t thermal_stats(const void* T, const void* u, uint32_t N, double* partial, double* out, hipStream_t s) {
  // four values a load when every component of u starts on a 16-byte
  // boundary (N % 4; the bases are allocations or whole multiples of it)
  const bool quad = N % 4 == 0 && quad_aligned(T) && quad_aligned(u);
  const uint32_t blocks = stride_blocks(N, quad ? 4 : 1);
  if (quad)
    hipLaunchKernelGGL((k_thermal_stats<R, 4>), dim3(blocks), dim3(256), 0, s, (const R*)T, (const R*)u, N, partial);
  else
    hipLaunchKernelGGL((k_thermal_stats<R, 1>), dim3(blocks), dim3(256), 0, s, (const R*)T, (const R*)u, N, partial);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_thermal_fold, dim3(1), dim3(256), 0, s, partial, blocks, out, (uint32_t*)nullptr);
  return hipGetLastError();
}

hipError_t launch_thermal_stats(bool dbl, const void* T, const void* u, uint32_t N, double* partial, double* out,
                                hipStream_t s) {
  return dbl ? thermal_stats<double>(T, u, N, partial, out, s) : thermal_stats<float>(T, u, N, partial, out, s);
}

hipError_t launch_thermal_flux(bool dbl, const ThermalArgs& a, void* flux, hipStream_t s) {
  const dim3 grid((a.N + 255) / 256);
  if (dbl)
    hipLaunchKernelGGL(k_thermal_flux<double>, grid, dim3(256), 0, s, a, (double*)flux);
  else
    hipLaunchKernelGGL(k_thermal_flux<float>, grid, dim3(256), 0, s, a, (float*)flux);
  return hipGetLastError();
}

hipError_t launch_thermal_init(bool dbl, const ThermalArgs& a, hipStream_t s) {
  const dim3 grid((a.N + 255) / 256);
  if (dbl)
    hipLaunchKernelGGL(k_thermal_init<double>, grid, dim3(256), 0, s, a);
  else
    hipLaunchKernelGGL(k_thermal_init<float>, grid, dim3(256), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_thermal_boundary(bool dbl, const ThermalArgs& a, int kind, const uint8_t* mask, double va, double vb,
                                   hipStream_t s) {
  const dim3 grid((a.N + 255) / 256);
  if (dbl)
    hipLaunchKernelGGL(k_thermal_boundary<double>, grid, dim3(256), 0, s, a, kind, mask, va, vb);
  else
    hipLaunchKernelGGL(k_thermal_boundary<float>, grid, dim3(256), 0, s, a, kind, mask, (float)va, (float)vb);
  return hipGetLastError();
}

}  // namespace pol
