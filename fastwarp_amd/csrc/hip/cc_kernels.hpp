// The fused CC kernels, templates over the window's radius. cc.hip instantiates one radius per object, so
// that the eight compile side by side.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "device_common.hpp"
#include "kernels.hpp"

namespace fw::hip {

// ------------------------------------------------------------------------------------------
// CC pair (metric/cc.rs:170-321 and wgpu_backend.rs:1354-1520 semantics, fused).
//
// The window sums of a, b, aa, bb and ab are taken in f64, every window from its own terms: the
// product of two f32 values is exact in f64, and no sum is ever formed by subtracting a plane that
// has left the window. So a window of zeros sums to exactly zero (which decides the degenerate
// windows of cc.rs:270-300), a window of tiny values (the smoothed edge of a zero-padded region,
// local variance 1e-12, where the coefficient is the largest of the image) keeps its relative
// precision, and no scale of the image enters. The centred moments, the local CC and the
// coefficients follow in f64 from one reciprocal; the derivative is the coefficient times the f32
// central difference, rounded once to f32. Each output voxel writes both derivative directions;
// localCC is symmetric, so one value partial serves both.
//
// A block owns a 32 x 8 (x, y) tile over a run of tile_z planes and takes the planes z0 - R ..
// z1 - 1 + R in turn. A plane's tile and halo are staged in LDS as f32 (the next plane's loads are in
// flight meanwhile); the x pass forms the products and sums them over x, eight outputs a lane, whose
// windows share their middle (2.6 additions an output where the plain sum takes 8), a wave for each
// of (a, aa), (b, bb), (ab); the y pass adds 2R + 1 rows of x sums per output voxel; the z pass
// keeps the last planes' x/y sums of the thread's one output column in registers and forms the
// running window from partial sums (three or four additions a plane, CcWindow).
//
// Bound by the latency of its f64 chains at two waves a SIMD (vector instructions fill a third of the
// time, the LDS reads of the y pass another). 182 x 218 x 182, radius 4, with the value's sum: 156 us;
// sums of split values, running along z with the leaving plane subtracted, on 64 x 8 tiles: 375 us
// (radius 2: 120 for 305, radius 8: 329 for 952; 45 x 54 x 45 at radius 4: 22 for 51).
// ------------------------------------------------------------------------------------------
constexpr int kCcTX = kCcTileX, kCcTY = kCcTileY, kCcThreads = kCcTX * kCcTY;
constexpr int kCcRun = 8;  // outputs along x of one lane of the x pass

template <int R>
struct CcTile {
  static constexpr int W = 2 * R + 1;
  static constexpr int LX = kCcTX + 2 * R, LY = kCcTY + 2 * R;
  // a row is read in 16-byte vectors; an odd number of them a row keeps neighbouring rows' reads
  // on different banks
  static constexpr int VEC = (LX + 3) / 4;
  static constexpr int PITCH = 4 * (VEC % 2 ? VEC : VEC + 1);
  static constexpr int PER = (LX * LY + kCcThreads - 1) / kCcThreads;  // elements a thread stages
  static constexpr int RUNS = kCcTX / kCcRun, JOBS = RUNS * LY;
  // Column tx of row ly of the x sums is stored in another 16-byte place of its 64 bytes: the lanes
  // of the x pass store 64 bytes apart, and the exchange spreads eight of them (four runs of two
  // rows) over all banks. A row stays the same 256 bytes, so the y pass reads it without conflicts.
  static __device__ __forceinline__ int swap_of(int ly, int run) { return (run >> 1) | ((ly & 1) << 1); }
  static __device__ __forceinline__ int column(int ly, int tx) {
    return tx ^ (swap_of(ly, tx / kCcRun) << 1);
  }
  // the f32 inputs of a run of outputs
  static constexpr int N = kCcRun + 2 * R;
  static __device__ __forceinline__ void read_run(const float* p, float (&f)[(N + 3) / 4 * 4]) {
#pragma unroll
    for (int q = 0; q < (N + 3) / 4; ++q) *reinterpret_cast<float4*>(f + 4 * q) = *reinterpret_cast<const float4*>(p + 4 * q);
  }
  static __device__ __forceinline__ void write_run(double* row, int ly, int run, const double (&o)[kCcRun]) {
    const int s = swap_of(ly, run);
#pragma unroll
    for (int p = 0; p < kCcRun / 2; ++p)
      *reinterpret_cast<double2*>(row + run * kCcRun + 2 * (p ^ s)) = make_double2(o[2 * p], o[2 * p + 1]);
  }
};

// o[i] = sum of the terms i .. i + W - 1: groups of at most W outputs share the middle of their
// windows and add running sums of the ends to it. add(t, s) gives s plus term t (a product goes
// into the sum by one fma, so it is not rounded by itself), first(t) the term alone.
template <int N, int W, typename V, typename First, typename Add>
__device__ __forceinline__ void window_sums(First first, Add add, V (&o)[N]) {
#pragma unroll
  for (int base = 0; base < N; base += W) {
    const int n = N - base < W ? N - base : W;
    V left = first(base + n - 1);
#pragma unroll
    for (int t = n; t < W; ++t) left = add(base + t, left);
    o[base + n - 1] = left;
#pragma unroll
    for (int i = n - 2; i >= 0; --i) {
      left = add(base + i, left);
      o[base + i] = left;
    }
    V right = V(0);
#pragma unroll
    for (int i = 1; i < n; ++i) {
      right = i == 1 ? first(base + W) : add(base + W - 1 + i, right);
      o[base + i] += right;
    }
  }
}

// The running window of the z pass over W planes of one sum: step<J>(w), J the plane's place in a cycle
// of CYCLE planes, turns a plane's sum into the sum of the last W planes. With `pre` (the sum of this
// cycle's planes) and, in slot j, the sum of the last cycle's planes j .. W - 1 before step j and this
// cycle's plane j after it: about three additions a plane and W + 1 values held.
template <int W, typename V>
struct CcWindow {
  static constexpr int CYCLE = W;
  V ring[W], pre;
  __device__ __forceinline__ void clear() {
    pre = V(0);
#pragma unroll
    for (int j = 0; j < W; ++j) ring[j] = V(0);
  }
  template <int J>
  __device__ __forceinline__ V step(V plane) {
    pre += plane;
    V w = pre;
    if constexpr (J + 1 < W) w += ring[J + 1];
    ring[J] = plane;
    if constexpr (J + 1 == W) {
#pragma unroll
      for (int i = W - 2; i >= 1; --i) ring[i] += ring[i + 1];
      pre = V(0);
    }
    return w;
  }
};

// Nine planes (radius 4) as three sums of three: four additions a plane and eight values held
// (ten by the general scheme; the shorter cycle also keeps the code in the instruction cache).
template <typename V>
struct CcWindow<9, V> {
  static constexpr int CYCLE = 6;
  V last[2], three[6];  // by plane number modulo 2 and 6
  __device__ __forceinline__ void clear() {
    last[0] = last[1] = V(0);
#pragma unroll
    for (int j = 0; j < 6; ++j) three[j] = V(0);
  }
  template <int J>
  __device__ __forceinline__ V step(V plane) {
    const V s = (last[0] + last[1]) + plane;
    last[J % 2] = plane;
    const V w = (s + three[(J + 3) % 6]) + three[J];
    three[J] = s;
    return w;
  }
};

// step(J, zin + J) for J = 0 .. CYCLE - 1, each with its own J at compile time.
template <int CYCLE, int J = 0, typename Step>
__device__ __forceinline__ void cc_cycle(Step& step, int zin) {
  if constexpr (J < CYCLE) {
    step(std::integral_constant<int, J>{}, zin + J);
    cc_cycle<CYCLE, J + 1>(step, zin);
  }
}

// 1 / v for normal v by the hardware's approximation and two Newton steps (within two units in the last
// place; the IEEE division takes twice the instructions).
__device__ __forceinline__ double reciprocal(double v) {
  double r = __builtin_amdgcn_rcp(v);
  r = fma(fma(-v, r, 1.0), r, r);
  return fma(fma(-v, r, 1.0), r, r);
}

// sum / count by the count's reciprocal and one correction: exact where the quotient is (a window of
// one value has that value as its mean, so its variance is zero, not a rounding error).
__device__ __forceinline__ double mean_of(double sum, double count, double inv_count) {
  const double q = sum * inv_count;
  return fma(fma(-q, count, sum), inv_count, q);
}

static __device__ float block_sum_f64(double v) {
  __shared__ double red[16];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) red[w] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0)
    for (int q = 0; q < (int)(blockDim.x >> 6); ++q) t += red[q];
  return (float)t;
}

// Waves per SIMD the registers are held to. At radius 4 the windows take 80 registers and the kernel
// 187: held to 168 for three blocks a CU it spills 21 of them and takes 199 us at 1 mm for 156 us.
template <int R>
constexpr int cc_waves() {
  return R <= 3 ? 3 : 2;
}

template <int R, bool MASKED, bool DIAGONAL>
__global__ __launch_bounds__(kCcThreads, cc_waves<R>()) void k_cc2(CcArgs a) {
#define FW_CC2_TILE xcd_block()
#include "cc2_body.inc"
#undef FW_CC2_TILE
}

// Several unmasked CC pairs on one grid: the grid's z blocks repeat once per item, and item q's
// blocks are the blocks of its own launch (the same tiles, partials at the same indices of its
// own partial buffers).
template <int R, bool DIAGONAL>
__global__ __launch_bounds__(kCcThreads, cc_waves<R>()) void k_cc2_items(CcItems c) {
  constexpr bool MASKED = false;
  const unsigned gz = gridDim.z / (unsigned)c.count;
  const unsigned q = xcd_block().z / gz;
  const CcArgs& a = c.a[q];
#define FW_CC2_TILE make_uint3(xcd_block().x, xcd_block().y, xcd_block().z - q * gz)
#include "cc2_body.inc"
#undef FW_CC2_TILE
}

template <int R, bool M>
static void launch_cc_r(const CcArgs& a, hipStream_t s) {
  if (a.probes.diagonal) launch((k_cc2<R, M, true>), cc_grid(a.d, a.tile_z), dim3(kCcThreads), 0, s, a);
  else launch((k_cc2<R, M, false>), cc_grid(a.d, a.tile_z), dim3(kCcThreads), 0, s, a);
}

template <int R>
void launch_cc_radius(const CcArgs& a, hipStream_t s) {
  if (a.valid != nullptr) launch_cc_r<R, true>(a, s);
  else launch_cc_r<R, false>(a, s);
}

template <int R>
void launch_cc_items_radius(const CcItems& c, hipStream_t s) {
  const CcArgs& a = c.a[0];
  dim3 g = cc_grid(a.d, a.tile_z);
  g.z *= (unsigned)c.count;
  if (a.probes.diagonal) launch((k_cc2_items<R, true>), g, dim3(kCcThreads), 0, s, c);
  else launch((k_cc2_items<R, false>), g, dim3(kCcThreads), 0, s, c);
}

}  // namespace fw::hip
