// Device bodies of the one-launch projections of small calls, single slices
// whose projection takes less time than the launches around it.  They read the
// caller's image or sinogram as it lies (any strides): no copies before, no
// partial sums after; what the larger paths stage in memory each wave stages in
// its own part of LDS.
#pragma once

#include "stack.h"

namespace gt {

// LDS accesses of a wave are served in order: what its lanes wrote is there
// for all of them, the compiler only has to keep the order.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ double read_lane(double v, int lane) {
  const int2 b = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(b.x, lane),
                                              __builtin_amdgcn_readlane(b.y, lane)));
}

// Forward: 64 neighbouring rays of one angle, the rows of their frame split
// over WV waves, whose sums meet in LDS.  A wave copies windows of kSmallRows
// rows into LDS, lanes along the axis that is contiguous in memory, and walks
// them as the slice-batched forward does.
constexpr int kSmallRows = 8;

template <typename real, int WV, int CAP>
struct SmallFwdShared {
  real buf[WV][CAP];
  real sum[WV][64];
};

template <typename real, bool FAN, int WV, int CAP>
__device__ __forceinline__ void fwd_small_block(const Job<real> &J, Strides3 ii, int rb, int a, int z,
                                                SmallFwdShared<real, WV, CAP> &sh) {
  using LdsReal = const __attribute__((address_space(3))) real *;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int first = rb * 64, nray = min(64, J.Ns - first);
  const int s_own = first + lane, s = min(s_own, J.Ns - 1);
  const double s_mid = first + 0.5 * (nray - 1);
  FwdAngle g = fwd_angle(J, a);
  const bool flip = strip_flipped(J, g, s_mid);
  const StripRay R = strip_ray<real, FAN>(J, g, s, flip);
  bool ok = g.scale > 0 && fabs(R.m) < 4 && fabs(R.n) < 4 && fabs(R.u0) < 1e6 && fabs(R.v0) < 1e6;
  ok = ok && (!FAN || strip_forward(J, g, s, flip));
  const bool irregular = __ballot(!ok) != 0;
  const real *img = J.src + z * ii.s2;
  // pixels of a frame, zero outside the row
  struct Frame {
    const real *p;
    int64_t sx, sy;
    int nx, ny;
  };
  auto frame = [&](bool f) {
    return f ? Frame{img, ii.s1, ii.s0, J.Ny, J.Nx} : Frame{img, ii.s0, ii.s1, J.Nx, J.Ny};
  };
  auto rows = [&](const Frame &F, int w) { return (int)((int64_t)F.ny * w / WV); };
  auto direct = [&](const StripRay &r, const Frame &F, int ya, int yb, real (&sum)[1][1]) {
    strip_direct<real, FAN>(
        r, ya, yb, F.nx,
        [&](int, int y, int x) { return Slices<real, 1>{{F.p[y * F.sy + x * F.sx]}}; }, sum);
  };
  real tot = 0;
  bool again = irregular;
  if (!irregular) {
    const Frame F = frame(flip);
    const double m0 = read_lane(R.m, 0), m1 = read_lane(R.m, 63), u0 = read_lane(R.u0, 0),
                 u1 = read_lane(R.u0, 63), n0 = read_lane(R.n, 0), n1 = read_lane(R.n, 63),
                 v0 = read_lane(R.v0, 0), v1 = read_lane(R.v0, 63);
    real *buf = sh.buf[wv];
    const bool along = F.sx <= F.sy;  // rows lie along memory
    const int y1 = rows(F, wv + 1);
    for (int y = rows(F, wv); y < y1;) {
      // The window of the next rows: the edge rays are the extremes and linear
      // along the rows; one whole column to spare on each side for the rounding.
      FwdChunk c{y, min(kSmallRows, y1 - y), 0, 0, 0};
      double lo = 1e30, hi = -1e30, w = 0, xr = -1e30;
      for (int end = 0; end < 2; ++end) {
        const double ye = end ? y + c.rows - 1 : y;
        const double ua = fma(m0, ye, u0), ub = fma(m1, ye, u1), va = fma(n0, ye, v0), vb = fma(n1, ye, v1);
        lo = fmin(lo, fmin(ua, ub));
        hi = fmax(hi, fmax(ua, ub));
        xr = fmax(xr, fmax(va, vb));
        w = fmax(w, fmax(va - ua, vb - ub));
      }
      c.lo = __builtin_amdgcn_readfirstlane((int)floor(lo) - 1);
      c.taps = __builtin_amdgcn_readfirstlane((int)floor(w + 1e-3) + 1);
      c.pitch = __builtin_amdgcn_readfirstlane((int)floor(hi) + c.taps + 2 - c.lo);
      y += c.rows;
      if (!(xr > -1 && lo < F.nx)) continue;
      if (c.pitch > CAP) {
        again = true;
        break;
      }
      if (c.pitch * c.rows > CAP) {
        y -= c.rows;
        c.rows = CAP / c.pitch;
        y += c.rows;
      }
      wave_lds_fence();
      // lanes: 64 columns of a row, or 8 rows of 8 columns
      const int lr = along ? 0 : lane & 7, lc = along ? lane : lane >> 3;
      const int dr = along ? 1 : 8, dc = along ? 64 : 8;
      for (int r0 = 0; r0 < c.rows; r0 += dr) {
        const int r = r0 + lr;
        const real *p = F.p + (c.y + r) * F.sy + c.lo * F.sx;
#pragma unroll 4
        for (int j = lc; j < c.pitch; j += dc) {
          const int x = c.lo + j;
          const real v = r < c.rows && (unsigned)x < (unsigned)F.nx ? p[j * F.sx] : (real)0;
          if (r < c.rows) buf[r * c.pitch + j] = v;
        }
      }
      wave_lds_fence();
      LaneRay<real> ray;
      ray.start(R, c.y);
      real acc[1][1] = {};
      const LdsReal win = (LdsReal)buf;
      switch (c.taps) {
        case 2:
          strip_rows<real, FAN, 1, 2>(ray, c, 0, 0, win, 0, acc);
          break;
        case 3:
          strip_rows<real, FAN, 1, 3>(ray, c, 0, 0, win, 0, acc);
          break;
        default:
          strip_rows<real, FAN, 1, 0>(ray, c, 0, 0, win, 0, acc);
      }
      tot += acc[0][0];
    }
    // a value which is not finite may come from a tap of zero weight outside the strip
    again = again || tot * (real)0 != (real)0;
    tot *= (real)g.scale;
  }
  if (again) {
    // rays that leave the block's frame take their own, in every wave alike
    const bool f = irregular ? strip_flipped(J, g, s) : flip;
    const Frame F = frame(f);
    g.scale = 1;
    real sum[1][1] = {};
    direct(strip_ray<real, FAN>(J, g, s, f), F, rows(F, wv), rows(F, wv + 1), sum);
    tot = sum[0][0];
  }
  sh.sum[wv][lane] = tot;
  __syncthreads();
  if (wv == 0 && s_own < J.Ns) {
    real v = 0;
#pragma unroll
    for (int i = 0; i < WV; ++i) v += sh.sum[i][lane];
    if (FAN)
      fan_store(J, s, a, z, v);
    else
      store_fwd(J, s, a, z, v * radon_scale(J));
  }
}

// Backprojection: a tile of RP x 64 pixels, the angles split over WV waves,
// whose sums meet in LDS.  A wave takes NA angles at a time: a lane
// makes an angle's window, the wave copies the bins, weighted, into LDS
// (padded: lanes along the angles write neighbouring banks), then each lane
// adds them to its RP pixels, 8 apart.
template <typename real, int WV, int NA, int CAP>
struct SmallBackShared {
  real buf[WV][NA * (CAP + 1)];
  TileWindow<real> win[WV][NA];
  real weight[WV][NA];
};

template <typename real, bool FAN, int RP, int WV, int NA, int CAP>
__device__ __forceinline__ void back_small_tile(const Job<real> &J, int bx, int by, int z,
                                                SmallBackShared<real, WV, NA, CAP> &sh) {
  using LdsReal = const __attribute__((address_space(3))) real *;
  constexpr int TX = RP > 1 ? 16 : 8, TY = RP > 2 ? 16 : 8, P = CAP + 1;
  static_assert(64 * RP <= NA * P && NA <= 16, "the wave's sums reuse its windows");
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xa = bx * TX, ya = by * TY;
  const real dx = (real)(lane & 7), dy = (real)(lane >> 3);
  const real hi = (real)J.Ns + (real)2.5, mid = FAN ? J.geo[5] + (real)2 : (real)0;
  const real *sino = J.sino + z * J.so.s2;
  const bool along = J.so.s0 <= J.so.s1;  // bins lie along memory
  real *buf = sh.buf[wv];
  // bin s of angle a with its weights, zero outside the detector
  auto value = [&](int s, int a, real weight) {
    if ((unsigned)s >= (unsigned)J.Ns) return (real)0;
    const real v = sino[s * J.so.s0 + a * J.so.s1];
    return FAN ? v * J.sdpd[s] * weight : v * weight;
  };
  real acc[RP][1][1];
#pragma unroll
  for (int r = 0; r < RP; ++r) acc[r][0][0] = 0;
  const int a1 = (int)((int64_t)J.Na * (wv + 1) / WV);
  for (int a0 = (int)((int64_t)J.Na * wv / WV); a0 < a1; a0 += NA) {
    const int na = min(NA, a1 - a0);
    int n = 0;
    wave_lds_fence();
    if (lane < na) {
      const int a = a0 + lane;
      AngleRec<real> c[1];
      back_table_entry(c, J.ofs + 8 * (int64_t)a, J.geo, FAN, 0);
      const TileWindow<real> W = tile_window<real, FAN, TX, TY>(J, c[0], xa, ya, CAP);
      sh.win[wv][lane] = W;
      sh.weight[wv][lane] = FAN ? J.ofs[8 * (int64_t)a + 6] / J.geo[0] : J.ofs[8 * (int64_t)a + 4];
      n = W.n;
    }
    const uint64_t none = __ballot(lane < na && n == 0);
#pragma unroll
    for (int o = 8; o; o >>= 1) n = max(n, __shfl_xor(n, o, 64));
    const int widest = __builtin_amdgcn_readfirstlane(n);
    wave_lds_fence();
    if (along) {
#pragma unroll 4
      for (int k = 0; k < na; ++k)
        for (int j = lane; j < widest; j += 64)
          buf[k * P + j] = value(sh.win[wv][k].w0 + j - 2, a0 + k, sh.weight[wv][k]);
    } else {
      const int k = lane & (NA - 1);
      if (k < na) {
        const int w0 = sh.win[wv][k].w0;
        const real weight = sh.weight[wv][k];
#pragma unroll 4
        for (int j = lane / NA; j < widest; j += 64 / NA)
          buf[k * P + j] = value(w0 + j - 2, a0 + k, weight);
      }
    }
    wave_lds_fence();
    if (none == 0) {
#pragma unroll 2
      for (int k = 0; k < na; ++k)
        stack_angle<real, FAN, 1, RP, true>(sh.win[wv][k], dx, dy, (LdsReal)(buf + k * P), 0, nullptr, mid, hi,
                                            acc);
    } else {
#pragma unroll 1
      for (int k = 0; k < na; ++k) {
        if ((none >> k) & 1)
          stack_angle<real, FAN, 1, RP, false>(
              sh.win[wv][k], dx, dy, LdsReal(), 0,
              [&](int, int i) { return Slices<real, 1>{{value(i - 2, a0 + k, sh.weight[wv][k])}}; }, mid, hi,
              acc);
        else
          stack_angle<real, FAN, 1, RP, true>(sh.win[wv][k], dx, dy, (LdsReal)(buf + k * P), 0, nullptr, mid,
                                              hi, acc);
      }
    }
  }
  wave_lds_fence();
#pragma unroll
  for (int r = 0; r < RP; ++r)
    buf[(((lane >> 3) + 8 * (r >> 1)) * TX) + (lane & 7) + 8 * (r & 1)] = acc[r][0][0];
  __syncthreads();
  for (int i = tid; i < 64 * RP; i += 64 * WV) {
    const int x = xa + i % TX, y = ya + i / TX;
    if (x >= J.Nx || y >= J.Ny) continue;
    real v = 0;
#pragma unroll
    for (int w = 0; w < WV; ++w) v += sh.buf[w][i];
    store_back(J, x, y, z, v);
  }
}

}  // namespace gt
