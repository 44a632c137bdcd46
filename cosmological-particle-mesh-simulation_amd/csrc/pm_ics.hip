// The two ends of the PM step on the device: Zel'dovich initial conditions from a Gaussian
// random field (the work of gaussian_random_field.py + zeldovich.py) and the shell-binned
// matter power spectrum of the density grid.
//
// Initial conditions, for an N_PARTS^3 lattice (n below) of a sim on an N_CELLS grid:
//   1. white noise w on the n^3 lattice, [i][j][k] order (i slowest): Philox4x32-10 counters
//      (Salmon, Moraes, Dror & Shaw, SC'11) and the Box-Muller transform, or a caller's field;
//   2. its half spectrum W(k) (forward R2C, the FFT passes of the Poisson solve);
//   3. per displacement component d: Psi_d(k) = i m_d / |m|^2 * A(|m|^2) * W(k) * scale, with
//      A = sqrt(P(k) n^3 / V) D(a) tabulated on the host per integer |m|^2, the Nyquist plane of
//      axis d and k = 0 zeroed; inverse C2R; then s_d = Psi_d and v_d = c_v Psi_d written to
//      the particles in slot order (lattice axis d = positions[d], zeldovich.py:79-83).
// Lattice axis i is the grid's slowest axis here, so component 0 differentiates along the
// spectrum's z index and component 2 along its half (x) axis.
#include "pm_ics.h"

namespace pm {

namespace {

constexpr int kB = 256;

inline unsigned grid_for(long n, long per_thread = 1) {
  const long t = (n + per_thread - 1) / per_thread;
  const long g = (t + kB - 1) / kB;
  return (unsigned)(g < 1 ? 1 : g);
}

template <typename R>
__global__ __launch_bounds__(kB) void k_white_noise(R* out, long n3, uint64_t seed) {
  const long g = blockIdx.x * (long)kB + threadIdx.x;
  if (4 * g >= n3) return;
  double z[4];
  white4(g, seed, z);
#pragma unroll
  for (int r = 0; r < 4; ++r)
    if (4 * g + r < n3) out[4 * g + r] = R(z[r]);
}

template <typename Tin, typename R>
__global__ __launch_bounds__(kB) void k_copy_field(const Tin* __restrict__ in, R* __restrict__ out, long n3) {
  const long i = blockIdx.x * (long)kB + threadIdx.x;
  if (i < n3) out[i] = R(in[i]);
}

// signed mode number of index i on an n-point axis (numpy.fft.fftfreq order)
__device__ __forceinline__ int signed_mode(int i, int n) { return i < n / 2 ? i : i - n; }

// amp[m2] -> scale * amp[m2] / m2 (0 for m2 = 0), in place: one division per |m|^2 instead of one per
// mode and component
__global__ __launch_bounds__(kB) void k_amplitude_scale(double* __restrict__ amp, long count, double scale) {
  const long i = blockIdx.x * (long)kB + threadIdx.x;
  if (i < count) amp[i] = i ? scale * amp[i] / (double)i : 0.0;
}

// one displacement component's half spectrum from the noise spectrum W (H part + Nyquist plane); a
// thread takes two neighbouring modes of a row, the last blocks the Nyquist plane.  With 64-bit
// divisions, an FP64 one and one mode per thread: 46 us at 256^3 for 134 MB of traffic, now 40 (one
// thread for the four mirrored modes of a table value: 52).
template <typename R>
__global__ __launch_bounds__(kB) void k_zeldovich_component(const cpx<R>* __restrict__ WH, const cpx<R>* __restrict__ WQ,
                                                           cpx<R>* __restrict__ H, cpx<R>* __restrict__ Q,
                                                           const double* __restrict__ amp, int n, FastDiv by_n,
                                                           FastDiv by_pairs, uint32_t main_blocks, int d) {
  struct alignas(2 * sizeof(cpx<R>)) Pair {
    cpx<R> v[2];
  };
  const uint32_t pairs = by_pairs.d, rows = (uint32_t)n * (uint32_t)n;
  const bool main = blockIdx.x < main_blocks;
  const uint32_t idx = (main ? blockIdx.x : blockIdx.x - main_blocks) * (uint32_t)kB + threadIdx.x;
  if (idx >= (main ? rows * pairs : rows)) return;
  const uint32_t row = main ? by_pairs.div(idx) : idx;
  const int kx = main ? 2 * (int)(idx - row * pairs) : n / 2;
  const int z = (int)by_n.div(row), y = (int)(row - (uint32_t)z * (uint32_t)n);
  const int mz = signed_mode(z, n), my = signed_mode(y, n);
  auto mode = [&](int mx, cpx<R> w) {
    // component d: derivative along lattice axis d = spectrum axis z, y, x for d = 0, 1, 2; its Nyquist
    // plane is zero
    const int md = d == 0 ? mz : (d == 1 ? my : mx);
    const double f = (d == 0 ? z : d == 1 ? y : mx) == n / 2 ? 0.0 : amp[mx * mx + my * my + mz * mz] * (double)md;
    return cmake<cpx<R>>(R(-f * (double)w.y), R(f * (double)w.x));  // i f w
  };
  if (main) {
    Pair p = reinterpret_cast<const Pair*>(WH)[idx];
    p.v[0] = mode(kx, p.v[0]);
    p.v[1] = mode(kx + 1, p.v[1]);
    reinterpret_cast<Pair*>(H)[idx] = p;
  } else {
    Q[row] = mode(kx, WQ[row]);
  }
}

// particles of the lattice take component d of the displacement field (real [i][j][k] grid)
template <typename R>
__global__ __launch_bounds__(kB) void k_zeldovich_particles(const R* __restrict__ psi, R* __restrict__ s, R* __restrict__ v,
                                                           Lattice L, int d, double vel_factor) {
  const long slot = blockIdx.x * (long)kB + threadIdx.x;
  if (slot >= L.np) return;
  int i, j, k;
  slot_to_ijk(slot, L, i, j, k);
  const long p = ((long)i * L.np_side + j) * L.np_side + k;  // reference particle index
  const R x = psi[p];
  s[d * L.np + slot] = wrap_disp<R>(x, R(L.n));
  v[d * L.np + slot] = R(vel_factor * (double)x);
}

// the same for lattices of 4^3 blocks, through LDS in whole cache lines (see kSlotK; 48 -> 30 us at 256^3)
template <typename R>
__global__ __launch_bounds__(kB) void k_zeldovich_slots(const R* __restrict__ psi, R* __restrict__ s, R* __restrict__ v,
                                                        Lattice L, int d, double vel_factor) {
  constexpr int PER = 16 * kSlotK / kB;
  __shared__ R t[kSlotK * kSlotPitch];
  const SlotRegion r = slot_region(L, blockIdx.x);
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    int ijk[3], at;
    long p;
    if (slot_ref(L, r, u * kB + threadIdx.x, ijk, p, at)) t[at] = psi[p];
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < PER; ++u) {
    int at;
    long slot;
    if (slot_dev(L, r, u * kB + threadIdx.x, slot, at)) {
      const R x = t[at];
      s[d * L.np + slot] = wrap_disp<R>(x, R(L.n));
      v[d * L.np + slot] = R(vel_factor * (double)x);
    }
  }
}

// ---------------------------------------------------------------- power spectrum
// FP64 sum of n values in 16-byte loads, kSumU of them in flight per thread; few blocks, since each
// ends with an atomic at one address (134 MB of FP64: 43 us with one load in flight and 2048 blocks, now
// 24 us)
constexpr int kSumU = 8, kSumBlocks = 512;
template <typename R>
__global__ __launch_bounds__(kB) void k_sum(const R* __restrict__ x, long n, double* out) {
  constexpr int V = 16 / sizeof(R);
  struct alignas(16) Vec {
    R v[V];
  };
  __shared__ double sh[kB / 64];
  const Vec* xv = reinterpret_cast<const Vec*>(x);
  const long nv = n / V, step = (long)gridDim.x * kB;
  double acc[V] = {};
  long i = blockIdx.x * (long)kB + threadIdx.x;
  for (; i + (kSumU - 1) * step < nv; i += kSumU * step) {
    Vec u[kSumU];
#pragma unroll
    for (int k = 0; k < kSumU; ++k) u[k] = xv[i + k * step];
#pragma unroll
    for (int k = 0; k < kSumU; ++k)
#pragma unroll
      for (int q = 0; q < V; ++q) acc[q] += (double)u[k].v[q];
  }
  for (; i < nv; i += step) {
    const Vec u = xv[i];
#pragma unroll
    for (int q = 0; q < V; ++q) acc[q] += (double)u.v[q];
  }
  double sum = 0.0;
#pragma unroll
  for (int q = 0; q < V; ++q) sum += acc[q];
  if (blockIdx.x == 0 && threadIdx.x < n - nv * V) sum += (double)x[nv * V + threadIdx.x];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_down(sum, o);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kB / 64; ++w) sum += sh[w];
    atomicAdd(out, sum);
  }
}

// shell sums over the half spectrum: bins[0..nb] of {sum w|F|^2, sum w|m|, sum w}, bin
// floor(|m| + 0.5); weight 2 for 0 < kx < n/2 (each stands for its conjugate), else 1.
// A thread takes the modes (kx, +-my, +-mz) together: one root and one LDS atomic per sum for up to
// four modes, and modes beyond the last shell are not read.  Few blocks: each adds its 3 (nb + 1) sums
// to the same addresses.  256^3 FP64 to nb = 128: 75 -> 40 us.
constexpr int kShellBlocks = 1024;
template <typename R>
__global__ __launch_bounds__(kB) void k_shell_sums(const cpx<R>* __restrict__ H, const cpx<R>* __restrict__ Q, int n,
                                                  int nb, FastDiv side, uint32_t total, double* __restrict__ bins) {
  extern __shared__ double lb[];  // 3 * (nb + 1)
  for (int i = threadIdx.x; i < 3 * (nb + 1); i += kB) lb[i] = 0.0;
  __syncthreads();
  const int h = n / 2;
  for (uint32_t idx = blockIdx.x * kB + threadIdx.x; idx < total; idx += gridDim.x * kB) {
    const uint32_t row = side.div(idx), zr = side.div(row);
    const int kx = (int)(idx - row * side.d), y = (int)(row - zr * side.d), z = (int)zr;
    const long m2 = (long)kx * kx + (long)y * y + (long)z * z;
    const double mr = sqrt((double)m2);
    const int ib = (int)floor(mr + 0.5);
    if (ib < 1 || ib > nb) continue;
    const bool y2 = y != 0 && y != h, z2 = z != 0 && z != h;  // the mirrored row is another one
    auto row_at = [&](int zz, int yy) {
      const size_t r = (size_t)zz * n + yy;
      return kx < h ? H[r * h + kx] : Q[r];
    };
    cpx<R> f[4] = {row_at(z, y), cmake<cpx<R>>(R(0), R(0)), cmake<cpx<R>>(R(0), R(0)), cmake<cpx<R>>(R(0), R(0))};
    if (y2) f[1] = row_at(z, n - y);
    if (z2) f[2] = row_at(n - z, y);
    if (y2 && z2) f[3] = row_at(n - z, n - y);
    double p2 = 0.0;
#pragma unroll
    for (int q = 0; q < 4; ++q) p2 += (double)f[q].x * (double)f[q].x + (double)f[q].y * (double)f[q].y;
    const double w = (kx == 0 || kx == h) ? 1.0 : 2.0, wm = w * (y2 ? 2.0 : 1.0) * (z2 ? 2.0 : 1.0);
    __hip_atomic_fetch_add(&lb[ib], w * p2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(&lb[(nb + 1) + ib], wm * mr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(&lb[2 * (nb + 1) + ib], wm, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 3 * (nb + 1); i += kB)
    if (lb[i] != 0.0) atomicAdd(&bins[i], lb[i]);
}

}  // namespace

hipError_t white_noise(void* out, int prec, long n3, uint64_t seed, hipStream_t st) {
  if (n3 <= 0) return hipSuccess;
  if (prec == 8) k_white_noise<double><<<grid_for(n3, 4), kB, 0, st>>>((double*)out, n3, seed);
  else k_white_noise<float><<<grid_for(n3, 4), kB, 0, st>>>((float*)out, n3, seed);
  return hipGetLastError();
}

template <typename R>
hipError_t zeldovich_ics(const void* noise, int noise_bytes, uint64_t seed, double* d_amp, double scale,
                         double vel_factor, const Lattice& L, const FftTables& t, R* s, R* v, R* wbuf, R* hbuf,
                         cpx<R>* qbuf, hipStream_t st) {
  const int n = L.np_side;
  const long n3 = (long)n * n * n;
  // 1. white noise as a real n^3 grid in hbuf
  if (noise) {
    if (noise_bytes == 8) k_copy_field<double, R><<<grid_for(n3), kB, 0, st>>>((const double*)noise, hbuf, n3);
    else k_copy_field<float, R><<<grid_for(n3), kB, 0, st>>>((const float*)noise, hbuf, n3);
  } else {
    k_white_noise<R><<<grid_for(n3, 4), kB, 0, st>>>(hbuf, n3, seed);
  }
  if (hipError_t e = hipGetLastError()) return e;
  // 2. its half spectrum in wbuf (H part, then the Nyquist plane)
  cpx<R>* WH = reinterpret_cast<cpx<R>*>(wbuf);
  cpx<R>* WQ = WH + (long)n * n * (n / 2);
  if (hipError_t e = fft_forward_xy<R, R>(hbuf, WH, WQ, n, t, st)) return e;
  if (hipError_t e = fft_c2c_z<R>(WH, WQ, n, -1, t, st)) return e;
  // 3. per component: k-space operator, inverse transform, particles
  cpx<R>* H = reinterpret_cast<cpx<R>*>(hbuf);
  const unsigned main_blocks = grid_for((long)n * n * (n / 4));  // (n is a multiple of 8)
  const long n_amp = 3L * (n / 2) * (n / 2) + 1;
  k_amplitude_scale<<<grid_for(n_amp), kB, 0, st>>>(d_amp, n_amp, scale);
  for (int d = 0; d < 3; ++d) {
    k_zeldovich_component<R><<<main_blocks + grid_for((long)n * n), kB, 0, st>>>(
        WH, WQ, H, qbuf, d_amp, n, FastDiv((uint32_t)n), FastDiv((uint32_t)n / 4), main_blocks, d);
    if (hipError_t e = hipGetLastError()) return e;
    if (hipError_t e = fft_c2c_z<R>(H, qbuf, n, +1, t, st)) return e;
    if (hipError_t e = fft_inverse_yx<R, R>(H, qbuf, hbuf, n, t, st)) return e;
    if (slot_regions(L)) k_zeldovich_slots<R><<<slot_blocks(L), kB, 0, st>>>(hbuf, s, v, L, d, vel_factor);
    else k_zeldovich_particles<R><<<grid_for(L.np), kB, 0, st>>>(hbuf, s, v, L, d, vel_factor);
    if (hipError_t e = hipGetLastError()) return e;
  }
  return hipSuccess;
}

template <typename R>
hipError_t grid_sum(const R* x, long n, double* d_out, hipStream_t st) {
  const unsigned g = std::min(grid_for(n, 4 * kSumU), (unsigned)kSumBlocks);
  k_sum<R><<<g, kB, 0, st>>>(x, n, d_out);
  return hipGetLastError();
}

template <typename R>
hipError_t shell_sums(const cpx<R>* H, const cpx<R>* Q, int n, int nb, double* d_bins, hipStream_t st) {
  const uint32_t side = (uint32_t)n / 2 + 1, total = side * side * side;  // (n <= 1024: below 2^31)
  const unsigned g = std::min(grid_for(total, 4), (unsigned)kShellBlocks);
  k_shell_sums<R><<<g, kB, 3 * (nb + 1) * sizeof(double), st>>>(H, Q, n, nb, FastDiv(side), total, d_bins);
  return hipGetLastError();
}

#define PM_INST(R)                                                                                                \
  template hipError_t zeldovich_ics<R>(const void*, int, uint64_t, double*, double, double, const Lattice&, \
                                       const FftTables&, R*, R*, R*, R*, cpx<R>*, hipStream_t);                   \
  template hipError_t grid_sum<R>(const R*, long, double*, hipStream_t);                                          \
  template hipError_t shell_sums<R>(const cpx<R>*, const cpx<R>*, int, int, double*, hipStream_t);
PM_INST(float)
PM_INST(double)
#undef PM_INST

}  // namespace pm
