// The fused CC kernels, templates over the window's radius. cc.hip instantiates one radius of one launch per
// object, so that they compile side by side.
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
// has left the window. So a window of zeros sums to exactly zero (and is a degenerate window of
// cc.rs:270-300; one of another value is so within its sums' rounding, mean_of), a window of tiny
// values (the smoothed edge of a zero-padded region, local variance 1e-12, where the coefficient is
// the largest of the image) keeps its relative precision, and no scale of the image enters. The centred moments, the local CC and the
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
// time, the LDS reads of the y pass another). 182 x 218 x 182, radius 4, inputs in cache: 147 us; sums of
// split values, running along z with the leaving plane subtracted, on 64 x 8 tiles: 337 us (radius 2: 118
// for 262, radius 8: 323 for 947). With the value's sum and inputs from HBM: 177 us for 391.
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

// sum / count by the count's reciprocal and one correction: exact where the quotient is (a window of one value
// has that value as its mean, so its centred moments are zero up to the rounding of the sums of squares, n v^2
// 2^-53 a few times; exactly zero where those sums fit 53 bits).
__device__ __forceinline__ double mean_of(double sum, double count, double inv_count) {
  const double q = sum * inv_count;
  return fma(fma(-q, count, sum), inv_count, q);
}

// A window's means, centred moments and local CC from its five sums (cc.rs:270-300), and the
// coefficients of the two derivative directions at its centre values.
struct CcPoint {
  double fmean, mmean, s_ff, s_mm, s_fm, r, cc;
  __device__ __forceinline__ CcPoint(const double (&w)[5], double count, double inv_count)
      : fmean(mean_of(w[0], count, inv_count)), mmean(mean_of(w[1], count, inv_count)) {
    s_ff = fma(-fmean, w[0], w[2]);
    s_mm = fma(-mmean, w[1], w[3]);
    s_fm = fma(-fmean, w[1], w[4]);
    const double product = s_ff * s_mm;
    r = reciprocal(product);
    cc = fabs(product) > (double)kEps64 ? s_fm * s_fm * r : 1.0;
  }
  __device__ __forceinline__ bool varies() const { return s_ff > (double)kEps64 && s_mm > (double)kEps64; }
  // 2 s_fm / (s_ff s_mm) and the regression slopes s_fm / s_mm, s_fm / s_ff from one reciprocal
  __device__ __forceinline__ void coefficients(double fc, double mc, double& cf, double& cm) const {
    const double fi = fc - fmean, mi = mc - mmean;
    const double k1 = s_fm * r;
    cf = 2.0 * k1 * fma(-k1 * s_ff, mi, fi);
    cm = 2.0 * k1 * fma(-k1 * s_mm, fi, mi);
  }
};

// Along grid axis g of an axis-aligned grid: the factor of the difference of the two neighbours, and the
// plane (physical axis) its product goes to.
struct CcAxes {
  float fac[3] = {0.0f, 0.0f, 0.0f};
  int plane[3] = {0, 1, 2};
  __device__ __forceinline__ explicit CcAxes(const Probes& pr) {
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int g = 0; g < 3; ++g)
        if (pr.o[p][g] != 0.0f) {
          fac[g] = (pr.o[p][g] > 0.0f ? 0.5f : -0.5f) * pr.inv_spacing[p];
          plane[g] = p;
        }
  }
};

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
// 187: held to 168 for three blocks a CU it spills 21 of them and takes 199 us at 1 mm for 156 us. Up to
// radius 3 an axis-aligned grid's kernel fits 168 (110 to 165). From radius 7 on (6 with a mask, 4 oblique with
// one) the windows exceed the 256 of two waves and 4 to 120 registers are spilled.
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

// ------------------------------------------------------------------------------------------
// The same pair one plane at a time, where the grid gives too few blocks for long walks (cc_plan). Each
// thread sums its columns of the tile and halo over the window's planes first, with all loads independent
// of each other, then the x and y passes run once, in place, where k_cc2 runs them for every plane of the
// window. The sums are the same terms in f64 in another order, none subtracted.
//
// Bound by the z pass (2R + 1 planes of 2.5 columns a thread at radius 4, from L2) where the chip is full
// and by one chain of loads, three barriers and the f64 sums where it is not: at radius 4 7.9 us at
// 24 x 28 x 24 (k_cc2 15.8), 11.6 at 45 x 54 x 45 (19).
// ------------------------------------------------------------------------------------------
template <int R, bool MASKED, bool DIAGONAL>
__device__ __forceinline__ void cc_plane(const CcArgs& a, uint3 bl) {
  using T = CcTile<R>;
  constexpr int W = T::W, SUMS = MASKED ? 6 : 5;
  // odd, so that the x pass's eight rows a half-wave lie on different banks
  constexpr int PITCH = T::LX | 1;
  constexpr int ROWS = SUMS * T::LY * T::RUNS, JOBS = (ROWS + kCcThreads - 1) / kCcThreads;
  __shared__ double sums[SUMS][T::LY * PITCH];
  const Dims d = a.d;
  const int x0 = bl.x * kCcTX, y0 = bl.y * kCcTY, z0 = bl.z * a.tile_z, z1 = min(z0 + a.tile_z, d.nz);
  const long long plane = (long long)d.nx * d.ny, n3 = d.n();

  const CcAxes axes(a.probes);
  double cc_sum = 0.0;
  int counted = 0;
#pragma unroll 1
  for (int z = z0; z < z1; ++z) {
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // offsets are formed for each plane: hoisted, they take the registers of two waves
    // z pass
#pragma unroll
    for (int q = 0; q < T::PER; ++q) {
      const int e = tid + kCcThreads * q;
      const int ly = e / T::LX, lx = e % T::LX;
      const int gx = x0 - R + lx, gy = y0 - R + ly;
      const int cx = min(max(gx, 0), d.nx - 1), cy = min(max(gy, 0), d.ny - 1);
      const long long o = (long long)cx + (long long)d.nx * cy;
      double s[SUMS] = {};
#pragma unroll
      for (int t = 0; t < W; ++t) {
        const int k = z - R + t;
        const long long at = o + plane * min(max(k, 0), d.nz - 1);
        float u = a.fixed[at], v = a.moving[at];
        bool in = k >= 0 && k < d.nz;
        if constexpr (MASKED) in = in && a.valid[at] != 0.0f;
        u = in ? u : 0.0f;
        v = in ? v : 0.0f;
        s[0] += (double)u;
        s[1] += (double)v;
        s[2] = fma((double)u, (double)u, s[2]);
        s[3] = fma((double)v, (double)v, s[3]);
        s[4] = fma((double)u, (double)v, s[4]);
        if constexpr (MASKED) s[5] += in ? 1.0 : 0.0;
      }
      if (T::LX * T::LY % kCcThreads == 0 || e < T::LX * T::LY) {
        const bool in = gx == cx && gy == cy;
#pragma unroll
        for (int c = 0; c < SUMS; ++c) sums[c][ly * PITCH + lx] = in ? s[c] : 0.0;
      }
    }
    __syncthreads();
    // x pass: runs of kCcRun outputs of one row of one sum, written over the row once all are read
    double o[JOBS][kCcRun];
#pragma unroll
    for (int q = 0; q < JOBS; ++q) {
      const int e = min(tid + kCcThreads * q, ROWS - 1);
      const double* row = &sums[0][0] + (e / T::RUNS) * PITCH + (e % T::RUNS) * kCcRun;
      window_sums<kCcRun, W>([&](int t) { return row[t]; }, [&](int t, double v) { return v + row[t]; }, o[q]);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < JOBS; ++q) {
      const int e = tid + kCcThreads * q;
      if (e < ROWS) {
        double* row = &sums[0][0] + (e / T::RUNS) * PITCH + (e % T::RUNS) * kCcRun;
#pragma unroll
        for (int t = 0; t < kCcRun; ++t) row[t] = o[q][t];
      }
    }
    __syncthreads();
    // y pass and output
    const int tx = tid & (kCcTX - 1), ty = tid / kCcTX;
    const int x = x0 + tx, y = y0 + ty;
    if (x < d.nx && y < d.ny) {
      const long long at = lin(d, x, y, z);
      float df[3] = {0.0f, 0.0f, 0.0f}, dm[3] = {0.0f, 0.0f, 0.0f};
      if (!MASKED || a.valid[at] != 0.0f) {
        double w[SUMS];
#pragma unroll
        for (int q = 0; q < SUMS; ++q) {
          double s = 0.0;
#pragma unroll
          for (int t = 0; t < W; ++t) s += sums[q][(ty + t) * PITCH + tx];
          w[q] = s;
        }
        double count;
        if constexpr (MASKED) count = w[5];
        else count = (double)(window_count(x, d.nx, R) * window_count(y, d.ny, R) * window_count(z, d.nz, R));
        const double five[5] = {w[0], w[1], w[2], w[3], w[4]};
        const CcPoint p(five, count, 1.0 / count);
        cc_sum += p.cc;
        counted += 1;
        if (p.varies()) {
          float gm[3], gf[3];
          if constexpr (DIAGONAL) {
            // the two neighbours along each grid axis, at the edges as k_cc2 reads them
            const long long step[3] = {1, d.nx, plane};
            const int pos[3] = {x, y, z}, len[3] = {d.nx, d.ny, d.nz};
#pragma unroll
            for (int q = 0; q < 3; ++q) {
              const long long up = pos[q] + 1 < len[q] ? step[q] : 0, down = pos[q] >= 1 && pos[q] + 1 < len[q] ? step[q] : 0;
              gm[q] = (a.moving[at + up] - a.moving[at - down]) * axes.fac[q];
              gf[q] = (a.fixed[at + up] - a.fixed[at - down]) * axes.fac[q];
            }
          } else {
#pragma unroll 1
            for (int q = 0; q < 3; ++q) {
              gm[q] = central_difference(a.moving, d, a.probes, q, x, y, z);
              gf[q] = central_difference(a.fixed, d, a.probes, q, x, y, z);
            }
          }
          double cf, cm;
          p.coefficients((double)a.fixed[at], (double)a.moving[at], cf, cm);
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            df[q] = (float)(cf * (double)gm[q]);
            dm[q] = (float)(cm * (double)gf[q]);
          }
        }
      }
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const long long to = at + n3 * (DIAGONAL ? axes.plane[q] : q);
        a.d_fixed[to] = df[q];
        a.d_moving[to] = dm[q];
      }
    }
    __syncthreads();  // the y pass has read the plane's sums
  }
  const float total = block_sum_f64(cc_sum);
  const float cnt = block_sum((float)counted);
  if (threadIdx.x == 0) {
    const unsigned b = bl.x + gridDim.x * (bl.y + gridDim.y * bl.z);
    a.partial_cc[b] = total;
    a.partial_count[b] = (int)cnt;
  }
}

template <int R, bool MASKED, bool DIAGONAL>
__global__ __launch_bounds__(kCcThreads) void k_cc2_plane(CcArgs a) {
  cc_plane<R, MASKED, DIAGONAL>(a, xcd_block());
}

template <int R, bool DIAGONAL>
__global__ __launch_bounds__(kCcThreads) void k_cc2_plane_items(CcItems c) {
  const unsigned gz = gridDim.z / (unsigned)c.count;
  const uint3 bl = xcd_block();
  const unsigned q = bl.z / gz;
  cc_plane<R, false, DIAGONAL>(c.a[q], make_uint3(bl.x, bl.y, bl.z - q * gz));
}

// Whether k_cc2 is there for a radius: on oblique grids, whose gradient gathers leave it too few
// registers, only where it is the faster one on large grids (cc_plan).
template <int R, bool M, bool DIAGONAL>
constexpr bool cc_walks() {
  return DIAGONAL || R >= (M ? kCcObliqueMasked : kCcObliquePlain);
}

template <int R, bool M, bool DIAGONAL>
static void launch_cc_one(const CcArgs& a, hipStream_t s) {
  const dim3 g = cc_grid(a.d, a.tile_z), t(kCcThreads);
  if constexpr (cc_walks<R, M, DIAGONAL>()) {
    if (!a.plane) {
      launch((k_cc2<R, M, DIAGONAL>), g, t, 0, s, a);
      return;
    }
  }
  launch((k_cc2_plane<R, M, DIAGONAL>), g, t, 0, s, a);
}

template <int R, bool MASKED>
void launch_cc_radius(const CcArgs& a, hipStream_t s) {
  if (a.probes.diagonal) launch_cc_one<R, MASKED, true>(a, s);
  else launch_cc_one<R, MASKED, false>(a, s);
}

template <int R, bool DIAGONAL>
static void launch_cc_items_one(const CcItems& c, hipStream_t s) {
  const CcArgs& a = c.a[0];
  const dim3 t(kCcThreads);
  dim3 g = cc_grid(a.d, a.tile_z);
  g.z *= (unsigned)c.count;
  if constexpr (cc_walks<R, false, DIAGONAL>()) {
    if (!a.plane) {
      launch((k_cc2_items<R, DIAGONAL>), g, t, 0, s, c);
      return;
    }
  }
  launch((k_cc2_plane_items<R, DIAGONAL>), g, t, 0, s, c);
}

template <int R>
void launch_cc_items_radius(const CcItems& c, hipStream_t s) {
  if (c.a[0].probes.diagonal) launch_cc_items_one<R, true>(c, s);
  else launch_cc_items_one<R, false>(c, s);
}

}  // namespace fw::hip
