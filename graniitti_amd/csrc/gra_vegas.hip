// VEGAS accumulation, grid-map and unweighting kernels (mode independent).
#include <hip/hip_runtime.h>

#include "gra_device.h"
#include "gra_kernels.h"

namespace {

using gra_hip::kIterScalars;

// Deterministic accumulation of one iteration. Each block owns a contiguous
// range of points and has kAccWaves waves that walk the same points; wave w
// owns the dimensions w, w + kAccWaves, ... and keeps their histograms of f and
// f^2 in its own LDS slice. For each batch of 64 points and each owned dimension
// seven ballots, one a bit of the bin, give every lane the mask of the lanes that
// share its bin; f and f^2 are summed over these by doubling the distance to the lane
// before, and the last of them adds the sums to its bin. The order of every addition
// is fixed by the points, so the histograms are the same on every run, without
// atomics. Wave 0 also sums the scalars.
// Bins are uniform on the VEGAS map, so 64 points put at most about four in one of 128
// bins and two doublings do, at most six. Bound by instruction issue: about 300 a batch
// for two dimensions, with the next batch's loads in flight; three waits in a row for W,
// flags and bins made 2^20 points in 8 dimensions 43 us, now 36. Sorting (bin, lane) keys
// with a bitonic network and scanning runs of equal bins took 97: 54 lane exchanges a
// batch and dimension for 12 here. 80 registers; a bound of 64 for full occupancy spills
// the time back (65 us).
constexpr int kAccWave = 64;
constexpr int kAccWaves = 4;

// The scalars of one iteration: sums with their compensations (value fs - fc), maxima, counts
struct IterScal {
  double fs = 0, fc = 0, f2s = 0, f2c = 0, mW = 0, mf = 0;
  uint64_t kin = 0, fid = 0, val = 0, nan = 0, inf = 0;
  // (s, c) += (os, oc): two-sum of the sums, carrying the compensations
  static __device__ __forceinline__ void merge(double& s, double& c, double os, double oc) {
    const double t = s + os, bp = t - s, e = (s - (t - bp)) + (os - bp);
    s = t;
    c = c + oc - e;
  }
  __device__ __forceinline__ void add(const double* p) {
    merge(fs, fc, p[0], p[1]);
    merge(f2s, f2c, p[2], p[3]);
    mW = p[4] > mW ? p[4] : mW;
    mf = p[5] > mf ? p[5] : mf;
    kin += (uint64_t)p[6];
    fid += (uint64_t)p[7];
    val += (uint64_t)p[8];
    nan += (uint64_t)p[9];
    inf += (uint64_t)p[10];
  }
  // Over the wave in a fixed lane order, into lane 0
  __device__ __forceinline__ void reduce() {
    for (int off = kAccWave / 2; off > 0; off >>= 1) {
      const double ofs = __shfl_down(fs, off), ofc = __shfl_down(fc, off);
      const double of2s = __shfl_down(f2s, off), of2c = __shfl_down(f2c, off);
      merge(fs, fc, ofs, ofc);
      merge(f2s, f2c, of2s, of2c);
      const double omW = __shfl_down(mW, off), omf = __shfl_down(mf, off);
      mW = omW > mW ? omW : mW;
      mf = omf > mf ? omf : mf;
      kin += __shfl_down(kin, off);
      fid += __shfl_down(fid, off);
      val += __shfl_down(val, off);
      nan += __shfl_down(nan, off);
      inf += __shfl_down(inf, off);
    }
  }
  __device__ __forceinline__ void store(double* o) const {
    o[0] = fs;
    o[1] = fc;
    o[2] = f2s;
    o[3] = f2c;
    o[4] = mW;
    o[5] = mf;
    o[6] = (double)kin;
    o[7] = (double)fid;
    o[8] = (double)val;
    o[9] = (double)nan;
    o[10] = (double)inf;
  }
};

// The lanes of the mask act whose 7-bit bin is this lane's
__device__ __forceinline__ uint64_t wave_match(int bin, uint64_t act) {
  uint32_t lo = (uint32_t)act, hi = (uint32_t)(act >> 32);
#pragma unroll
  for (int k = 0; k < 7; ++k) {
    const int sign = (bin << (31 - k)) >> 31;  // all ones where the bit is set
    const uint64_t set = __ballot(sign < 0);
    lo &= ~((uint32_t)set ^ (uint32_t)sign);
    hi &= ~((uint32_t)(set >> 32) ^ (uint32_t)sign);
  }
  return (uint64_t)hi << 32 | lo;
}

template <int DT>
__global__ __launch_bounds__(kAccWave* kAccWaves) void k_accumulate(
    const double* __restrict__ W, const double* __restrict__ vw, const uint8_t* __restrict__ bins,
    const uint8_t* __restrict__ flags, uint64_t n, uint64_t chunk, int D,
    double* __restrict__ part_hist, double* __restrict__ part_scal) {
  constexpr int DPW = (DT + kAccWaves - 1) / kAccWaves;  // dimensions per wave
  constexpr int NB = GRA_VEGAS_BINS;
  static_assert(NB == 128, "wave_match compares seven bits");
  __shared__ double2 hist[kAccWaves][DPW][NB];
  const int lane = threadIdx.x & (kAccWave - 1);
  const int wave = threadIdx.x / kAccWave;  // wave-uniform
  double2(*hw)[NB] = hist[wave];
#pragma unroll
  for (int q = 0; q < DPW; ++q)
    for (int b = lane; b < NB; b += kAccWave) hw[q][b] = make_double2(0.0, 0.0);
  const uint64_t p0 = (uint64_t)blockIdx.x * chunk;
  uint64_t p1 = p0 + chunk;
  if (p1 > n) p1 = n;
  IterScal scal;
  struct Batch {
    double W, vw;
    uint8_t fl, bin[DPW];
  };
  // the lane's point of a batch; a lane past the last reads the last point again, a
  // dimension past the last the last dimension
  const auto load = [&](uint64_t base, Batch& v) {
    const uint64_t i = min(base + lane, p1 - 1);
    v.W = W[i];
    v.vw = vw[i];
    v.fl = flags[i];
#pragma unroll
    for (int q = 0; q < DPW; ++q) v.bin[q] = bins[i * D + min(wave + q * kAccWaves, D - 1)];
  };
  Batch next;
  if (p0 < p1) load(p0, next);
  for (uint64_t base = p0; base < p1; base += kAccWave) {
    const Batch v = next;
    if (base + kAccWave < p1) load(base + kAccWave, next);  // in flight while this one is summed
    const bool in = base + lane < p1;
    const double f = in ? v.W * v.vw : 0.0;
    if (wave == 0 && in) {
      const double f2 = f * f;
      double y = f - scal.fc, t = scal.fs + y;
      scal.fc = (t - scal.fs) - y;
      scal.fs = t;
      y = f2 - scal.f2c;
      t = scal.f2s + y;
      scal.f2c = (t - scal.f2s) - y;
      scal.f2s = t;
      scal.mW = v.W > scal.mW ? v.W : scal.mW;
      scal.mf = f > scal.mf ? f : scal.mf;
      const uint8_t fl = v.fl;
      scal.kin += (fl & GRA_FLAG_KIN_OK) ? 1 : 0;
      scal.fid += (fl & GRA_FLAG_FID_OK) ? 1 : 0;
      scal.val += ((fl & GRA_FLAG_KIN_OK) && (fl & GRA_FLAG_FID_OK) && (fl & GRA_FLAG_VETO_OK)) ? 1
                                                                                             : 0;
      const bool bad = !(fl & GRA_FLAG_AMP_OK);
      scal.nan += (bad && !(fl & GRA_FLAG_INF)) ? 1 : 0;
      scal.inf += (bad && (fl & GRA_FLAG_INF)) ? 1 : 0;
    }
    const uint64_t act = __ballot(f != 0.0);
    if (act == 0) continue;  // wave-uniform
    double s[DPW], s2[DPW];
    int prev[DPW];  // the lane before in this lane's bin; its own where there is none
    bool tail[DPW];
    const uint64_t below = (1ull << lane) - 1;
    bool more = false;
#pragma unroll
    for (int q = 0; q < DPW; ++q) {
      s[q] = f;
      s2[q] = f * f;
      // zero contributions are dropped, and so are dimensions past the last
      const bool on = f != 0.0 && wave + q * kAccWaves < D;
      const uint64_t same = wave_match(v.bin[q], act);
      tail[q] = on && (same >> lane) == 1;
      prev[q] = on && (same & below) ? 63 - __clzll(same & below) : lane;
      more |= prev[q] != lane;
    }
    while (__ballot(more) != 0) {  // six times at most
      more = false;
#pragma unroll
      for (int q = 0; q < DPW; ++q) {
        const double os = __shfl(s[q], prev[q]), os2 = __shfl(s2[q], prev[q]);
        const int op = __shfl(prev[q], prev[q]);
        if (prev[q] != lane) {
          s[q] += os;
          s2[q] += os2;
        }
        // past the first of the bin's lanes there is no lane to add
        prev[q] = op != prev[q] ? op : lane;
        more |= prev[q] != lane;
      }
    }
#pragma unroll
    for (int q = 0; q < DPW; ++q)
      if (tail[q]) {
        const double2 h = hw[q][v.bin[q]];
        hw[q][v.bin[q]] = make_double2(h.x + s[q], h.y + s2[q]);
      }
    // the next batch's lanes read what this one's wrote
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
  const uint64_t H = 2 * (uint64_t)D * NB;
  double* ph = part_hist + (uint64_t)blockIdx.x * H;
#pragma unroll
  for (int q = 0; q < DPW; ++q) {
    const int j = wave + q * kAccWaves;
    if (j < D)
      for (int b = lane; b < NB; b += kAccWave) {
        ph[j * NB + b] = hw[q][b].x;
        ph[(D + j) * NB + b] = hw[q][b].y;
      }
  }
  if (wave != 0) return;
  scal.reduce();
  if (lane == 0) scal.store(part_scal + (uint64_t)blockIdx.x * kIterScalars);
}

// Reduction of the nblk block partials in a fixed order into gra_iter_stats layout:
// out[0 .. kIterScalars - 1] scalars, then the histograms [2][D][128]. A block takes
// kRedCols columns (128 bytes of each row): group g of kRedGroups sums the partials
// [g nblk / G, (g + 1) nblk / G) of a column in order, then the groups are summed in
// order. The block past the last column reduces the scalars. Bound by reading the
// partials once, 16 loads of a thread in flight: 9 us for 2^20 points (2048 partials,
// 34 MB), where two launches with a load at a time took 29 + 7; 6 us, a chain of waits,
// for small passes.
constexpr int kRedCols = 16;
constexpr int kRedGroups = 32;

__global__ __launch_bounds__(kRedCols* kRedGroups) void k_reduce(
    const double* __restrict__ part_hist, const double* __restrict__ part_scal, int nblk, int H,
    double* __restrict__ out) {
  __shared__ double sum[kRedGroups][kRedCols];
  __shared__ double sums[kRedCols * kRedGroups / kAccWave][kIterScalars];
  const int t = threadIdx.x;
  if ((int)blockIdx.x * kRedCols < H) {  // block-uniform; H is a multiple of kRedCols
    const int c = t % kRedCols, g = t / kRedCols;
    const int b0 = (int)((long long)nblk * g / kRedGroups);
    const int b1 = (int)((long long)nblk * (g + 1) / kRedGroups);
    const double* p = part_hist + (uint64_t)blockIdx.x * kRedCols + c;
    double s = 0.0;
    int b = b0;
    for (; b + 16 <= b1; b += 16) {
      double v[16];
#pragma unroll
      for (int k = 0; k < 16; ++k) v[k] = p[(uint64_t)(b + k) * H];
#pragma unroll
      for (int k = 0; k < 16; ++k) s += v[k];
    }
    for (; b < b1; ++b) s += p[(uint64_t)b * H];
    sum[g][c] = s;
    __syncthreads();
    if (g != 0) return;
    s = 0.0;
#pragma unroll
    for (int k = 0; k < kRedGroups; ++k) s += sum[k][c];
    out[kIterScalars + blockIdx.x * kRedCols + c] = s;
    return;
  }
  const int lane = t & (kAccWave - 1), wave = t / kAccWave;
  IterScal a;
  for (int b = t; b < nblk; b += kRedCols * kRedGroups)
    a.add(part_scal + (uint64_t)b * kIterScalars);
  a.reduce();
  if (lane == 0) a.store(sums[wave]);
  __syncthreads();
  if (wave != 0) return;
  IterScal w;
  if (lane < kRedCols * kRedGroups / kAccWave) w.add(sums[lane]);
  w.reduce();
  if (lane == 0) w.store(out);
}

// Map only (tests of the VEGAS map)
__global__ void k_map(const double* __restrict__ grid, int D, unsigned int bins,
                      const double* __restrict__ u, uint64_t n, double* __restrict__ x,
                      double* __restrict__ vw, int32_t* __restrict__ b) {
  __shared__ double xm[GRA_MAX_DIM * GRA_VEGAS_BINS];
  for (int k = threadIdx.x; k < D * GRA_VEGAS_BINS; k += blockDim.x) xm[k] = grid[k];
  __syncthreads();
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double uu[GRA_MAX_DIM], xx[GRA_MAX_DIM];
  uint8_t bb[GRA_MAX_DIM];
  for (int j = 0; j < D; ++j) uu[j] = u[i * D + j];
  vw[i] = vegas_map(xm, D, bins, uu, xx, bb);
  for (int j = 0; j < D; ++j) {
    x[i * D + j] = xx[j];
    b[i * D + j] = (int32_t)bb[j] + 1;
  }
}

// Hit-or-miss unweighting, MGraniitti::SaveEvent (src/MGraniitti.cc:1651-1663):
// accept = U < w / wmax, overflow when w > wmax (then rejected).
__global__ void k_unweight(const double* __restrict__ w, uint64_t n, double wmax, uint64_t seed,
                           uint8_t* __restrict__ acc, unsigned long long* __restrict__ counts) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool hit = false, over = false;
  if (i < n) {
    double u;
    point_uniforms(seed, 0xFFFFFFFFu, i, 1, &u);
    hit = u < (w[i] / wmax);
    if (w[i] > wmax) {
      over = true;
      hit = false;
    }
    acc[i] = hit ? 1 : 0;
  }
  const uint64_t mh = __ballot(hit), mo = __ballot(over);
  if ((threadIdx.x & 63) == 0) {
    if (mh) atomicAdd(&counts[0], (unsigned long long)__popcll(mh));
    if (mo) atomicAdd(&counts[1], (unsigned long long)__popcll(mo));
  }
}

// Hit-or-miss of the generation pass: f = W vw of valid points against maxf.
// Each wave stores five ballots of its 64 points (word 5 g + m of masks for
// group g): hits, valid points, overflows (f > maxf), NaN weights and Inf
// weights. k_tile_count, k_tile_scan and k_tile_write then count them and
// compact the hit indices in index order, with no atomics, so the result does
// not depend on the schedule.
constexpr int kAccMasks = 5;
__global__ void k_accept(const double* __restrict__ W, const double* __restrict__ vw,
                         const uint8_t* __restrict__ flags, uint64_t n, double maxf, uint64_t seed,
                         uint32_t iter, uint64_t first, uint64_t* __restrict__ masks) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool valid = false, hit = false, over = false, is_nan = false, is_inf = false;
  if (i < n) {
    const uint8_t fl = flags[i];
    is_nan = !(fl & GRA_FLAG_AMP_OK) && !(fl & GRA_FLAG_INF);
    is_inf = !(fl & GRA_FLAG_AMP_OK) && (fl & GRA_FLAG_INF);
    valid = (fl & (GRA_FLAG_KIN_OK | GRA_FLAG_FID_OK | GRA_FLAG_VETO_OK)) ==
            (GRA_FLAG_KIN_OK | GRA_FLAG_FID_OK | GRA_FLAG_VETO_OK);
    const double f = vw ? W[i] * vw[i] : W[i];
    double u;
    point_uniforms(seed, 0xC0000000u | (iter & 0x3FFFFFFFu), first + i, 1, &u);
    hit = u < (f / maxf);
    if (f > maxf) {
      over = true;
      hit = false;
    }
    hit = hit && valid;
  }
  const uint64_t m[kAccMasks] = {__ballot(hit), __ballot(valid), __ballot(over), __ballot(is_nan),
                                 __ballot(is_inf)};
  const int lane = threadIdx.x & 63;
  // lane 0 holds the wave's smallest index: the wave has points iff lane 0 does
  if (lane < kAccMasks && (i - lane) < n) {
    uint64_t v = m[0];
#pragma unroll
    for (int k = 1; k < kAccMasks; ++k) v = (lane == k) ? m[k] : v;
    masks[kAccMasks * ((i - lane) >> 6) + lane] = v;
  }
}

// Ordered compaction of the hit masks: a tile is 256 wpt groups of 64 points
// (one block of 256 threads, wpt consecutive groups per thread). wpt is 1 up to
// 2^28 points, so that a pass of 2^20 points spreads over 64 blocks, and 16
// above (accept_wpt)
constexpr int kAccMaxTiles = 1024 * 16;  // k_tile_scan: 1024 threads x 16 tiles

// Exclusive prefix sum of v over the 256 threads of a block; total in *tot.
// sh holds 4 entries; a second call in the same kernel must follow a barrier.
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* sh, uint32_t* tot) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  if (lane == 63) sh[wave] = x;
  __syncthreads();
  uint32_t base = 0, all = 0;
  for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
    if (w < wave) base += sh[w];
    all += sh[w];
  }
  *tot = all;
  return base + x - v;
}

// Per tile: the five mask counts (tile_cnt[5 t + m])
__global__ __launch_bounds__(256) void k_tile_count(const uint64_t* __restrict__ masks,
                                                    uint64_t ngroups, int wpt,
                                                    uint32_t* __restrict__ tile_cnt) {
  __shared__ uint32_t sh[kAccMasks][4];
  const uint64_t g0 = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * wpt;
  uint32_t c[kAccMasks] = {};
  for (int j = 0; j < wpt; ++j) {
    if (g0 + j >= ngroups) break;
#pragma unroll
    for (int k = 0; k < kAccMasks; ++k) c[k] += (uint32_t)__popcll(masks[kAccMasks * (g0 + j) + k]);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < kAccMasks; ++k) {
    uint32_t x = c[k];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) x += __shfl_xor(x, d);
    if (lane == 0) sh[k][wave] = x;
  }
  __syncthreads();
  if (threadIdx.x < kAccMasks)
    tile_cnt[kAccMasks * blockIdx.x + threadIdx.x] =
        sh[threadIdx.x][0] + sh[threadIdx.x][1] + sh[threadIdx.x][2] + sh[threadIdx.x][3];
}

// One block: exclusive offsets of the tiles' hits, and the pass counters
// (trials, valid, accepted, overflow, NaN, Inf)
__global__ __launch_bounds__(1024) void k_tile_scan(const uint32_t* __restrict__ tile_cnt,
                                                    int ntiles, uint64_t n,
                                                    uint32_t* __restrict__ tile_off,
                                                    unsigned long long* __restrict__ counts) {
  __shared__ uint32_t sh[16];
  __shared__ unsigned long long tot[kAccMasks];
  if (threadIdx.x < kAccMasks) tot[threadIdx.x] = 0;
  const int t0 = threadIdx.x * 16;
  uint32_t c = 0;
  unsigned long long o[kAccMasks - 1] = {};
  for (int j = 0; j < 16; ++j)
    if (t0 + j < ntiles) {
      c += tile_cnt[kAccMasks * (t0 + j)];
#pragma unroll
      for (int k = 1; k < kAccMasks; ++k) o[k - 1] += tile_cnt[kAccMasks * (t0 + j) + k];
    }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  uint32_t x = c;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const uint32_t y = __shfl_up(x, d);
    if (lane >= d) x += y;
  }
  if (lane == 63) sh[wave] = x;
  __syncthreads();
#pragma unroll
  for (int k = 1; k < kAccMasks; ++k)
    if (o[k - 1]) atomicAdd(&tot[k], o[k - 1]);
  uint32_t base = 0, all = 0;
  for (int w = 0; w < 16; ++w) {
    if (w < wave) base += sh[w];
    all += sh[w];
  }
  uint32_t run = base + x - c;
  for (int j = 0; j < 16; ++j)
    if (t0 + j < ntiles) {
      tile_off[t0 + j] = run;
      run += tile_cnt[kAccMasks * (t0 + j)];
    }
  __syncthreads();
  if (threadIdx.x == 0) {
    counts[0] = n;
    counts[1] = tot[1];
    counts[2] = all;
    counts[3] = tot[2];
    counts[4] = tot[3];
    counts[5] = tot[4];
  }
}

__global__ __launch_bounds__(256) void k_tile_write(const uint64_t* __restrict__ masks,
                                                    uint64_t ngroups, int wpt,
                                                    const uint32_t* __restrict__ tile_off,
                                                    uint64_t* __restrict__ idx, uint64_t max_out) {
  __shared__ uint32_t sh[4];
  const uint64_t g0 = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * wpt;
  uint32_t c = 0;
  for (int j = 0; j < wpt; ++j) {
    if (g0 + j >= ngroups) break;
    c += (uint32_t)__popcll(masks[kAccMasks * (g0 + j)]);
  }
  uint32_t tot;
  uint64_t pos = (uint64_t)tile_off[blockIdx.x] + block_exclusive_scan(c, sh, &tot);
  for (int j = 0; j < wpt; ++j) {
    if (g0 + j >= ngroups || pos >= max_out) break;
    uint64_t m = masks[kAccMasks * (g0 + j)];
    while (m) {
      const int b = __ffsll((unsigned long long)m) - 1;
      if (pos < max_out) idx[pos] = ((g0 + j) << 6) + (uint64_t)b;
      ++pos;
      m &= m - 1;
    }
  }
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t v, uint64_t n) {
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

}  // namespace

namespace gra_hip {

hipError_t launch_fill_u32(uint32_t* p, uint32_t v, size_t n, hipStream_t st) {
  if (n == 0) return hipSuccess;
  const unsigned int nb = (unsigned int)((n + 255) / 256);
  hipLaunchKernelGGL(k_fill_u32, dim3(nb), dim3(256), 0, st, p, v, (uint64_t)n);
  return hipGetLastError();
}

size_t accept_mask_words(uint64_t n) { return kAccMasks * (size_t)((n + 63) / 64); }
static int accept_wpt(uint64_t n) { return n <= (1ull << 28) ? 1 : 16; }
static size_t accept_tiles(uint64_t n) {
  const uint64_t tile_words = 256 * (uint64_t)accept_wpt(n);
  return (size_t)(((n + 63) / 64 + tile_words - 1) / tile_words);
}
size_t accept_tile_words(uint64_t n) { return (kAccMasks + 1) * accept_tiles(n); }

hipError_t launch_accept(const double* W, const double* vw, const uint8_t* flags, uint64_t n,
                         double maxf, uint64_t seed, uint32_t iter, uint64_t first, uint64_t* masks,
                         uint32_t* tiles, uint64_t* idx, uint64_t max_out,
                         unsigned long long* counts, hipStream_t st) {
  if (n == 0 || n > 0xFFFFFFFFull) return hipErrorInvalidValue;
  const uint64_t ng = (n + 63) / 64;
  const size_t nt = accept_tiles(n);
  if (nt > (size_t)kAccMaxTiles) return hipErrorInvalidValue;
  const unsigned int nb = (unsigned int)((n + 255) / 256);
  hipLaunchKernelGGL(k_accept, dim3(nb), dim3(256), 0, st, W, vw, flags, n, maxf, seed, iter, first,
                     masks);
  const int wpt = accept_wpt(n);
  hipLaunchKernelGGL(k_tile_count, dim3((unsigned int)nt), dim3(256), 0, st, masks, ng, wpt, tiles);
  uint32_t* off = tiles + kAccMasks * nt;
  hipLaunchKernelGGL(k_tile_scan, dim3(1), dim3(1024), 0, st, tiles, (int)nt, n, off, counts);
  hipLaunchKernelGGL(k_tile_write, dim3((unsigned int)nt), dim3(256), 0, st, masks, ng, wpt, off,
                     idx, max_out);
  return hipGetLastError();
}

hipError_t launch_accumulate(const double* W, const double* vw, const uint8_t* bins,
                             const uint8_t* flags, uint64_t n, int D, int nblk, double* part_hist,
                             double* part_scal, double* out, hipStream_t st) {
  const uint64_t chunk = (n + nblk - 1) / nblk;
  if (D <= 8)
    hipLaunchKernelGGL(k_accumulate<8>, dim3(nblk), dim3(kAccWave * kAccWaves), 0, st, W, vw,
                       bins, flags, n, chunk, D, part_hist, part_scal);
  else if (D <= 14)
    hipLaunchKernelGGL(k_accumulate<14>, dim3(nblk), dim3(kAccWave * kAccWaves), 0, st, W, vw,
                       bins, flags, n, chunk, D, part_hist, part_scal);
  else
    hipLaunchKernelGGL(k_accumulate<16>, dim3(nblk), dim3(kAccWave * kAccWaves), 0, st, W, vw,
                       bins, flags, n, chunk, D, part_hist, part_scal);
  const int H = 2 * D * GRA_VEGAS_BINS;
  hipLaunchKernelGGL(k_reduce, dim3(H / kRedCols + 1), dim3(kRedCols * kRedGroups), 0, st, part_hist,
                     part_scal, nblk, H, out);
  return hipGetLastError();
}

hipError_t launch_map(const double* grid, int D, unsigned int bins, const double* u, uint64_t n,
                      double* x, double* vw, int32_t* b, hipStream_t st) {
  const unsigned int nb = (unsigned int)((n + 255) / 256);
  hipLaunchKernelGGL(k_map, dim3(nb), dim3(256), 0, st, grid, D, bins, u, n, x, vw, b);
  return hipGetLastError();
}

hipError_t launch_unweight(const double* w, uint64_t n, double wmax, uint64_t seed, uint8_t* acc,
                           unsigned long long* counts, hipStream_t st) {
  const unsigned int nb = (unsigned int)((n + 255) / 256);
  hipLaunchKernelGGL(k_unweight, dim3(nb), dim3(256), 0, st, w, n, wmax, seed, acc, counts);
  return hipGetLastError();
}

}  // namespace gra_hip
