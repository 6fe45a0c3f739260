// Device bodies of the slice-batched projections: stacks of slices share one
// geometry, so a lane computes each pixel's detector coordinate (or each
// ray's strip) once and applies it to several slices.  The slices travel in
// 16-byte entries of kSlices<real> values (4 float32 or 2 float64), the
// widest LDS access.
#pragma once

#include "kernels.h"

namespace gt {

template <typename real>
constexpr int kSlices = 16 / (int)sizeof(real);

// kSlices slices of one detector bin or pixel
template <typename real>
struct alignas(16) Entry {
  real v[kSlices<real>];
};

template <typename real>
using LdsEntry = const __attribute__((address_space(3))) Entry<real> *;

// What one LDS read of a strip walk returns: an entry of slices, or a single
// slice's value.
template <typename real, int Z>
struct Slices {
  real v[Z];
};

template <typename real>
__device__ __forceinline__ Slices<real, kSlices<real>> lds_slices(LdsEntry<real> p) {
  typedef real vec __attribute__((ext_vector_type(kSlices<real>)));
  return __builtin_bit_cast(Slices<real, kSlices<real>>, *(const __attribute__((address_space(3))) vec *)p);
}

template <typename real>
__device__ __forceinline__ Slices<real, 1> lds_slices(const __attribute__((address_space(3))) real *p) {
  return {{*p}};
}

// ---------------------------------------------------------------------------
// Backprojection.
// ---------------------------------------------------------------------------
// Padded, pre-weighted sinogram of the slice groups: entry
// S[(q Na + a)(Ns + 4) + 2 + s] holds the q-th kSlices slices of bin s at angle a
// times the angle's weight (and sdpd[s]/R for fanbeam), zeros past the last
// slice and in the two entries at each end.

// Geometry of a backprojection tile: 4 waves of 8*RPX x 8*RPY pixels in a 2 x 2
// square.  A lane owns RPX x RPY pixels, 8 apart, so that the 64 lanes of one
// tap read span 8 x 8 pixels: at most 16 neighbouring entries while a pixel is
// at most 1.2 bins wide, which 64 banks serve without conflicts.  (64 lanes in
// two rows of 32 pixels span up to 45 entries.  Measured on LDS reads alone,
// GB/s per CU: 16-byte entries 200-300 in a row against 515 as 8 x 8.)
template <int RP>
struct StackTile {
  static constexpr int kRX = 2, kRY = RP / 2;
  static constexpr int kX = 16 * kRX, kY = 16 * kRY;
};

// One angle's window for one tile: the constants of StageWindow (kernels.h),
// relative to the tile's corner pixel.  n = 0: read from memory (fan: q = ss).
template <typename real>
struct alignas(sizeof(real) * 8) TileWindow {
  real c0, c1, k0, k1, k3, k4;
  int w0, n;
};

template <typename real, bool FAN, int TX, int TY>
__device__ __forceinline__ TileWindow<real> tile_window(const Job<real> &J, const AngleRec<real> &c, int xa,
                                                        int ya, int cap) {
  const double mid = FAN ? (double)J.geo[5] + 2.0 : 0.0;
  const double c0 = c.c[0], c1 = c.c[1], c2 = c.c[2];
  const double c3 = c.c[3], c4 = c.c[4], c5 = c.c[5];
  double pmin = 0, pmax = 0;
  bool ok = true;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const double x = (k & 1) ? xa + TX - 1 : xa, y = (k & 2) ? ya + TY - 1 : ya;
    double p = c0 * x + c1 * y + c2;
    if (FAN) {
      ok = ok && p > 0;
      p = (c3 * x + c4 * y + c5) / p + mid;
    }
    pmin = k == 0 ? p : fmin(pmin, p);
    pmax = k == 0 ? p : fmax(pmax, p);
  }
  TileWindow<real> W;
  const double span = pmax - pmin;
  ok = ok && span == span && span < cap - 5 && fabs(pmin) < 1e8;
  W.w0 = ok ? (int)floor(pmin) - 1 : 0;
  W.n = ok ? (int)floor(pmax) + 3 - W.w0 : 0;
  const double pc = c0 * xa + c1 * ya + c2;
  W.c0 = c.c[0];
  W.c1 = c.c[1];
  if (FAN) {
    const double sc = c3 * xa + c4 * ya + c5;
    const double k = ok ? mid - W.w0 : 0.0;  // window shift folded into q
    W.k0 = (real)pc;
    W.k1 = (real)(sc + k * pc);
    W.k3 = (real)(c3 + k * c0);
    W.k4 = (real)(c4 + k * c1);
  } else {
    W.k0 = (real)(pc - W.w0);
    W.k1 = W.k3 = W.k4 = (real)0;
  }
  return W;
}

// Adds one angle to the lane's RP pixels of G slice groups.  STAGED:
// win is the angle's window in LDS (planes of `plane` entries per group);
// otherwise bin(g, i) reads entry i of group g's padded sinogram row from
// memory, with the coordinate clamped to [0.5, Ns + 2.5].
template <typename real, bool FAN, int G, int RP, bool STAGED, typename Lds, typename Bin, int Z>
__device__ __forceinline__ void stack_angle(const TileWindow<real> &W, real dx, real dy, Lds win, int plane,
                                            Bin bin, real mid, real hi, real (&acc)[RP][G][Z]) {
  using A = Arith<real>;
  const real t0 = fma(W.c0, dx, fma(W.c1, dy, W.k0));
  const real q0 = FAN ? fma(W.k3, dx, fma(W.k4, dy, W.k1)) : t0;
  const real qx = FAN ? W.k3 : W.c0, qy = FAN ? W.k4 : W.c1;
  real w0[RP], w1[RP];
  int ix[RP];
#pragma unroll
  for (int r = 0; r < RP; ++r) {
    const real ox = (real)(8 * (r & 1)), oy = (real)(8 * (r >> 1));
    // one FMA per offset axis from the lane's first pixel (no running sums)
    real q = q0, t = t0;
    if (r >> 1) q = fma(qy, oy, q);
    if (r & 1) q = fma(qx, ox, q);
    real p = q, w = 1;
    if (FAN) {
      if (r >> 1) t = fma(W.c1, oy, t);
      if (r & 1) t = fma(W.c0, ox, t);
      w = STAGED ? A::rcp_positive(t) : A::rcp(t);
      p = STAGED ? q * w : fma(q, w, mid);
    }
    if (!STAGED) p = A::clamp(p, (real)0.5, hi);
    const real f = A::fract(p);
    ix[r] = (int)p;
    w1[r] = FAN ? f * w : f;
    w0[r] = w - w1[r];
  }
#pragma unroll
  for (int g = 0; g < G; ++g) {
    Slices<real, Z> e0[RP], e1[RP];
#pragma unroll
    for (int r = 0; r < RP; ++r) {
      if constexpr (STAGED) {
        e0[r] = lds_slices<real>(win + g * plane + ix[r]);
        e1[r] = lds_slices<real>(win + g * plane + ix[r] + 1);
      } else {
        e0[r] = bin(g, ix[r]);
        e1[r] = bin(g, ix[r] + 1);
      }
    }
#pragma unroll
    for (int r = 0; r < RP; ++r)
#pragma unroll
      for (int z = 0; z < Z; ++z)
        acc[r][g][z] = fma(w1[r], e1[r].v[z], fma(w0[r], e0[r].v[z], acc[r][g][z]));
  }
}

constexpr int kStackBatch = 128;  // angles per window table

// LDS of one block
template <typename real, int G, int CAP>
struct StackShared {
  Entry<real> buf[2][G * CAP];
  TileWindow<real> win[kStackBatch];
  int widest[4], direct[4];
};

// Backprojection of one tile in G slice groups, angles [a0, a1).  Per batch of
// kStackBatch angles a window table is made in LDS, one angle per thread.
// The batch then runs in chunks of as many angles as fit the buffer at the
// batch's widest window.  The windows of the chunk after the current one are
// copied by loads that write LDS directly (no registers, no LDS store
// instructions) while the current one is summed, so a chunk costs one barrier.
// The batch's sums are added to the totals at its end: the rounding then
// grows with the batch length and not with the number of angles.
template <typename real, bool FAN, int G, int RP, int CAP>
__device__ __forceinline__ void back_stack_tile(const Job<real> &J, int bx, int by, int zb, int a0,
                                                int a1, real *part, int band,
                                                StackShared<real, G, CAP> &sh) {
  using E = Entry<real>;
  using T = StackTile<RP>;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int xa = bx * T::kX, ya = by * T::kY;
  // the lane's first pixel relative to the tile's corner
  const int px = (wv & 1) * 8 * T::kRX + (lane & 7), py = (wv >> 1) * 8 * T::kRY + (lane >> 3);
  const real dx = (real)px, dy = (real)py;
  const int Nsp = J.Ns + 4;
  const int64_t quad = (int64_t)J.Na * Nsp;  // entries per slice group
  const E *S = reinterpret_cast<const E *>(J.S) + (int64_t)zb * G * quad;
  const real hi = (real)J.Ns + (real)2.5, mid = FAN ? J.geo[5] + (real)2 : (real)0;
  constexpr int ZV = kSlices<real>;
  real acc[RP][G][ZV], tot[RP][G][ZV];
#pragma unroll
  for (int r = 0; r < RP; ++r)
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int z = 0; z < ZV; ++z) acc[r][g][z] = tot[r][g][z] = 0;

  for (int ab = a0; ab < a1; ab += kStackBatch) {
    const int nb = min(kStackBatch, a1 - ab);
    __syncthreads();  // the previous batch is summed
    {
      int n = 0;
      if (tid < nb) {
        const TileWindow<real> W = tile_window<real, FAN, T::kX, T::kY>(J, J.tab[ab + tid], xa, ya, CAP);
        sh.win[tid] = W;
        n = W.n;
      }
      const uint64_t none = __ballot(tid < nb && n == 0);
#pragma unroll
      for (int o = 32; o; o >>= 1) n = max(n, __shfl_xor(n, o, 64));
      if (lane == 0) {
        sh.widest[wv] = n;
        sh.direct[wv] = none != 0;
      }
    }
    __syncthreads();
    const int width = __builtin_amdgcn_readfirstlane(
        max(max(sh.widest[0], sh.widest[1]), max(max(sh.widest[2], sh.widest[3]), 1)));
    const bool direct = __builtin_amdgcn_readfirstlane(sh.direct[0] | sh.direct[1] | sh.direct[2] |
                                                       sh.direct[3]) != 0;
    const int per = CAP / width;  // angles per chunk (width <= CAP)

    // item (angle k of the chunk, group g) is copied by wave (k G + g) % 4;
    // indices outside the padded row take one of its zero end entries
    auto stage = [&](int i0, E *dst) {
      const int items = min(per, nb - i0) * G;
      for (int it = wv; it < items; it += 4) {
        const int k = it / G, g = it % G;
        const int w0 = sh.win[i0 + k].w0, n = sh.win[i0 + k].n;
        E *to = dst + g * CAP + k * width;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(S + g * quad + (int64_t)(ab + i0 + k) * Nsp), (short)0, Nsp * (int)sizeof(E),
            0x00020000);
        for (int base = 0; base < width; base += 64) {
          const int j = base + lane;
          if (j < n) {
            const int e = min(max(w0 + j, 0), Nsp - 1);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                rs, (__attribute__((address_space(3))) void *)(to + base), 16, e * 16, 0, 0, 0);
          }
        }
      }
    };
    int which = 0;
    stage(0, sh.buf[0]);
    for (int i0 = 0; i0 < nb; i0 += per) {
      __builtin_amdgcn_s_waitcnt(0x0f70);  // this wave's copies have landed
      __syncthreads();                     // everybody's have; the other buffer is free
      if (i0 + per < nb) stage(i0 + per, sh.buf[which ^ 1]);
      LdsEntry<real> cur = (LdsEntry<real>)sh.buf[which];
      const int end = min(i0 + per, nb);
      if (!direct) {
#pragma unroll 1
        for (int l = i0; l < end; ++l, cur += width)
          stack_angle<real, FAN, G, RP, true>(sh.win[l], dx, dy, cur, CAP, nullptr, mid, hi, acc);
      } else {
#pragma unroll 1
        for (int l = i0; l < end; ++l, cur += width)
          if (__builtin_amdgcn_readfirstlane(sh.win[l].n))
            stack_angle<real, FAN, G, RP, true>(sh.win[l], dx, dy, cur, CAP, nullptr, mid, hi, acc);
      }
      which ^= 1;
    }
    if (direct) {
#pragma unroll 1
      for (int l = 0; l < nb; ++l)
        if (__builtin_amdgcn_readfirstlane(sh.win[l].n) == 0)
          stack_angle<real, FAN, G, RP, false>(
              sh.win[l], dx, dy, LdsEntry<real>(), 0,
              [&](int g, int i) {
                return __builtin_bit_cast(Slices<real, ZV>, S[(int64_t)(ab + l) * Nsp + g * quad + i]);
              },
              mid, hi, acc);
    }
#pragma unroll
    for (int r = 0; r < RP; ++r)
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int z = 0; z < ZV; ++z) {
          tot[r][g][z] += acc[r][g][z];
          acc[r][g][z] = 0;
        }
  }
#pragma unroll
  for (int r = 0; r < RP; ++r) {
    const int x = xa + px + 8 * (r & 1), y = ya + py + 8 * (r >> 1);
    if (x >= J.Nx || y >= J.Ny) continue;
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int z = 0; z < ZV; ++z) {
        const int zz = (zb * G + g) * ZV + z;
        if (zz >= J.Nz) continue;
        if (part)
          part[(((int64_t)band * J.Nz + zz) * J.Ny + y) * J.Nx + x] = tot[r][g][z];
        else
          store_back(J, x, y, zz, tot[r][g][z]);
      }
  }
}

// ---------------------------------------------------------------------------
// Forward projection.
// ---------------------------------------------------------------------------
// Image copies of the slice groups: x-fastest entries X[(q Ny + y)(Nx + 1) + x]
// and y-fastest entries Y[(q Nx + x)(Ny + 1) + y]; the last entry of a row is
// zero (reads outside the row take it).

// One ray of a strip in the frame whose rows run along it: the strip's left
// edge crosses row y at column u0 + m y, its right edge at v0 + n y.  Parallel
// beam: a pixel d columns right of the left edge weighs 1 - |A d - 1|.  Fanbeam:
// (1 - |A d / t - 1|) / t with t = t0 + t1 y + t2 d, the pixel's depth over the
// source-detector distance; A, t0, t1 and t2 carry a common power of two that
// makes t at least 1 over the image.
struct StripRay {
  double u0, m, v0, n, A, t0, t1, t2;
};

// One angle of the block: its table entries in double and the power of two
// (0: none, a corner of the image is not in front of the source).
struct FwdAngle {
  double o[6], scale;
  int a;
};

// The frame of a ray: rows along y (x fastest), or flipped, where an edge of its
// strip is flatter than that (gratopy/fanbeam.cl:150-165).
template <typename real>
__device__ __forceinline__ bool strip_flipped(const Job<real> &J, const FwdAngle &r, double s) {
  if (!J.fan) return fabs(r.o[0]) < fabs(r.o[1]);
  auto steep = [&](double d) {
    return fabs(r.o[4] + r.o[0] * d - r.o[2]) < fabs(r.o[5] + r.o[1] * d - r.o[3]);
  };
  const double d = s - (double)J.geo[5];
  return !(steep(d - 1) && steep(d + 1));
}

// Whether both edges of a fan ray's strip run from the source to the rows at its
// image side, the side for which strip_ray tells left from right (in its own
// frame a ray of a wide fan may leave on either side of the source's row).
template <typename real>
__device__ __forceinline__ bool strip_forward(const Job<real> &J, const FwdAngle &r, double s, bool flip) {
  const double yd = flip ? r.o[0] : r.o[1], qy = flip ? r.o[2] : r.o[3], d0 = (flip ? r.o[4] : r.o[5]) - qy;
  const double d = s - (double)J.geo[5];
  return qy * (d0 + yd * (d - 1)) < 0 && qy * (d0 + yd * (d + 1)) < 0;
}

template <typename real>
__device__ __forceinline__ FwdAngle fwd_angle(const Job<real> &J, int a) {
  FwdAngle r;
  r.a = a;
  r.scale = 1;
  for (int i = 0; i < 6; ++i) r.o[i] = J.ofs[8 * (int64_t)a + i];
  if (J.fan) {
    // depth over source-detector distance, linear: least at a corner
    const double R = J.geo[0], ddx = (r.o[4] - r.o[2]) / (R * R), ddy = (r.o[5] - r.o[3]) / (R * R);
    const double t = (double)J.geo[1] / R - ddx * (double)J.geo[3] - ddy * (double)J.geo[4] +
                     fmin(0.0, ddx * (J.Nx - 1)) + fmin(0.0, ddy * (J.Ny - 1));
    r.scale = t > 1e-30 ? ldexp(1.0, max(0, 1 - ilogb(t))) : 0.0;
  }
  return r;
}

template <typename real, bool FAN>
__device__ __forceinline__ StripRay strip_ray(const Job<real> &J, const FwdAngle &g, double s, bool flip) {
  const double *o = g.o;
  StripRay r;
  if constexpr (!FAN) {
    const double X = flip ? o[1] : o[0], Y = flip ? o[0] : o[1], i = 1.0 / X;
    r.m = r.n = -Y * i;
    const double c = (s - o[2]) * i, h = fabs(i);
    r.u0 = c - h;
    r.v0 = c + h;
    r.A = fabs(X);
    r.t0 = r.t1 = r.t2 = 0;
  } else {
    const double R = J.geo[0], dxi = J.geo[2], mid = J.geo[5];
    const double midx = flip ? J.geo[4] : J.geo[3], midy = flip ? J.geo[3] : J.geo[4];
    const double xd = flip ? o[1] : o[0], yd = flip ? o[0] : o[1];
    const double qx = flip ? o[3] : o[2], qy = flip ? o[2] : o[3];
    const double d0x = flip ? o[5] : o[4], d0y = flip ? o[4] : o[5];
    double sl = s - 1, sr = s + 1;
    double pl = (d0x + xd * (sl - mid) - qx) / (d0y + yd * (sl - mid) - qy);
    double pr = (d0x + xd * (sr - mid) - qx) / (d0y + yd * (sr - mid) - qy);
    if (qy * (pr - pl) > 0) {  // the rays run away from the source: rows lie at -qy of it
      const double w = pl;
      pl = pr;
      pr = w;
      sl = s + 1;
    }
    const double ddx = (d0x - qx) / (R * R), ddy = (d0y - qy) / (R * R);
    r.m = pl;
    r.n = pr;
    r.u0 = qx + midx - pl * (midy + qy);
    r.v0 = qx + midx - pr * (midy + qy);
    r.A = g.scale * fabs(xd / (dxi * dxi) + (mid - sl) * ddx);
    r.t0 = g.scale * (ddx * (r.u0 - midx) - ddy * midy + (double)J.geo[1] / R);
    r.t1 = g.scale * (ddx * pl + ddy);
    r.t2 = g.scale * ddx;
  }
  return r;
}

// Column of a strip's left edge along the rows: whole part and fraction.
// Single precision carries 32.32 fixed point, two integer additions a row.
template <typename real>
struct StripColumn;

template <>
struct StripColumn<float> {
  int64_t u, m;
  __device__ __forceinline__ void start(double u0, double slope, int y) {
    const double v = fma(slope, (double)y, u0), f = floor(v);
    u = ((int64_t)(int)f << 32) + (int64_t)(uint32_t)((v - f) * 4294967296.0);
    m = (int64_t)rint(slope * 4294967296.0);
  }
  __device__ __forceinline__ int whole() const { return (int)(u >> 32); }
  // 1 - fraction: distance of the first whole column right of the edge
  __device__ __forceinline__ float first() const { return fma((float)(uint32_t)u, -0x1p-32f, 1.0f); }
  __device__ __forceinline__ void step() { u += m; }
};

template <>
struct StripColumn<double> {
  double u0, m, y;
  __device__ __forceinline__ void start(double u, double slope, int y0) {
    u0 = u;
    m = slope;
    y = y0;
  }
  __device__ __forceinline__ int whole() const { return (int)floor(fma(m, y, u0)); }
  __device__ __forceinline__ double first() const { return 1.0 - Arith<double>::fract(fma(m, y, u0)); }
  __device__ __forceinline__ void step() { y += 1; }
};

constexpr int kFwdAngles = 8;   // angles per block, neighbours in direction
constexpr int kFwdKnot = 16;    // rows per interval of the window table
constexpr int kFwdKnots = 256;  // intervals per table

template <typename real, int G, int CAP>
struct FwdShared {
  Entry<real> buf[2][G * CAP];
  int4 table[kFwdKnots];  // FwdChunk of each interval: first column, pitch, rows per chunk, taps
  FwdAngle angle[kFwdAngles];
  StripRay edge[2 * kFwdAngles];
  int flips, irregular, first, last;
};

// Lane's ray within its wave's 64: a 16-byte LDS read is served in four
// phases of 16 lanes, {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the same of
// the upper half (found by pairing lanes on one bank).  Each phase gets 16
// neighbouring rays, whose entries then lie in different banks while rays are
// at most a column apart.
__device__ __forceinline__ int phase_ray(int lane) {
  const int l = lane & 31;
  int r;
  if (l < 4)
    r = l;
  else if (l < 12)
    r = l + 12;
  else if (l < 16)
    r = l - 8;
  else if (l < 20)
    r = l + 8;
  else if (l < 28)
    r = l - 12;
  else
    r = l;
  return (lane & 32) + r;
}

// Rows [y, y + rows) of one window: image columns from (xw(y) >> 32) + lo on,
// pitch of them, at most `taps` per ray.
struct FwdChunk {
  int y, rows, lo, pitch, taps;
};

// What a lane keeps of its ray, at the next row.
template <typename real>
struct LaneRay {
  StripColumn<real> col;
  real A, t0, t1, t2;
  __device__ __forceinline__ void start(const StripRay &r, int y) {
    col.start(r.u0, r.m, y);
    A = (real)r.A;
    t0 = (real)r.t0;
    t1 = (real)r.t1;
    t2 = (real)r.t2;
  }
};

// Adds the strip rows of one chunk, T columns each (T = 0: chunk.taps): acc +=
// w(x, y) image(x, y).  xw, xm: the window's 32.32 start column and its slant.
template <typename real, bool FAN, int G, int T, typename Lds, int Z>
__device__ __forceinline__ void strip_rows(LaneRay<real> &R, const FwdChunk &c, int64_t xw, int64_t xm,
                                           Lds buf, int plane, real (&acc)[G][Z]) {
  using A = Arith<real>;
  int base = 1 - c.lo;
  real y = (real)c.y;
#pragma unroll 1
  for (int r = 0; r < c.rows; ++r) {
    const Lds p = buf + (R.col.whole() + (base - (int)(xw >> 32)));
    const real d = R.col.first();
    real n = R.A * d, t = FAN ? fma(d, R.t2, fma(y, R.t1, R.t0)) : (real)0;
    auto weight = [&] {
      real w;
      if constexpr (FAN) {
        const real q = A::rcp_positive(t), e = fma(n, q, (real)-1);
        w = A::clamp01(fma(-fabs(e), q, q));
        t += R.t2;
      } else {
        w = A::clamp01((real)1 - fabs(n - (real)1));
      }
      n += R.A;
      return w;
    };
    auto add = [&](real w, int i) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const Slices<real, Z> e = lds_slices<real>(p + g * plane + i);
#pragma unroll
        for (int z = 0; z < Z; ++z) acc[g][z] = fma(w, e.v[z], acc[g][z]);
      }
    };
    if constexpr (T > 0) {
      real w[T];
#pragma unroll
      for (int i = 0; i < T; ++i) w[i] = weight();
#pragma unroll
      for (int i = 0; i < T; ++i) add(w[i], i);
    } else {
#pragma unroll 1
      for (int i = 0; i < c.taps; ++i) add(weight(), i);
    }
    R.col.step();
    base += c.pitch;
    xw += xm;
    y += 1;
  }
}

// The same rows without windows (they do not fit LDS, or the ray leaves the
// block's frame): every pixel of the strip, as pixel(g, y, x) reads group g's
// from memory.
template <typename real, bool FAN, int G, typename Pixel, int Z>
__device__ __forceinline__ void strip_direct(const StripRay &R, int y0, int y1, int Nxx, Pixel pixel,
                                             real (&acc)[G][Z]) {
#pragma unroll 1
  for (int y = y0; y < y1; ++y) {
    const double u = fma(R.m, (double)y, R.u0), v = fma(R.n, (double)y, R.v0);
    // whole columns strictly inside (u, v) and the image; the comparisons keep
    // infinities and NaN away from the conversions
    if (!(u < (double)Nxx && v > -1.0)) continue;
    const int xl = u > -1.0 ? (int)floor(u) + 1 : 0;
    const int xh = v < (double)Nxx ? (int)ceil(v) - 1 : Nxx - 1;
#pragma unroll 1
    for (int x = xl; x <= xh; ++x) {
      const double d = (double)x - u;
      real w;
      if constexpr (FAN) {
        const real q = (real)1 / (real)(R.t0 + R.t1 * y + R.t2 * d);
        w = ((real)1 - fabs(fma((real)(R.A * d), q, (real)-1))) * q;
      } else {
        w = (real)1 - fabs((real)(R.A * d - 1.0));
      }
      w = w > (real)0 ? w : (real)0;
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const auto e = pixel(g, y, x);
#pragma unroll
        for (int z = 0; z < Z; ++z) acc[g][z] = fma(w, e.v[z], acc[g][z]);
      }
    }
  }
}

// Results of one ray in G slice groups: band partials, or the projection with
// its scale and epilogue.
template <typename real, bool FAN, int G>
__device__ __forceinline__ void strip_store(const Job<real> &J, int s, int a, int zb, int band, real *part,
                                            real scale, const real (&sum)[G][kSlices<real>]) {
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int z = 0; z < kSlices<real>; ++z) {
      const int zz = (zb * G + g) * kSlices<real> + z;
      if (zz >= J.Nz) continue;
      const real v = sum[g][z] * scale;
      if (part)
        part[(((int64_t)band * J.Nz + zz) * J.Na + a) * J.Ns + s] = v;
      else if (FAN)
        fan_store(J, s, a, zz, v);
      else
        store_fwd(J, s, a, zz, v * radon_scale(J));
    }
}

// Forward projection of 64 H rays at kFwdAngles angles (neighbours in
// direction: perm lists the angles sorted by it) in G slice groups.  The rays
// walk the rows of their frame together: per chunk of rows the block copies
// the columns that its rays can meet into LDS (slanted windows, the next chunk
// loading while the current one is summed), and every lane adds the T columns
// of each strip row, weights computed once for all slices.  Wave w: rays 64
// (w % H) .. + 63, angles 2 (w / H) and the next.
template <typename real, bool FAN, int G, int H, int CAP>
__device__ __forceinline__ void fwd_stack_block(const Job<real> &J, const int *perm, int rb, int ag, int zb,
                                                int band, int nbands, real *part,
                                                FwdShared<real, G, CAP> &sh) {
  using E = Entry<real>;
  constexpr int ZV = kSlices<real>;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int first = rb * 64 * H, nray = min(64 * H, J.Ns - first);
  const int s_own = first + (wv % H) * 64 + phase_ray(lane), s = min(s_own, J.Ns - 1);
  const double s_mid = first + 0.5 * (nray - 1);
  const int g0 = ag * kFwdAngles, na = min(kFwdAngles, J.Na - g0);
  const int mine = 2 * (wv / H);  // the wave's first angle in the group
  if (tid == 0) sh.flips = 0;
  __syncthreads();
  if (tid < na) {
    const FwdAngle r = fwd_angle(J, perm[g0 + tid]);
    sh.angle[tid] = r;
    if (strip_flipped(J, r, s_mid)) atomicOr(&sh.flips, 1 << tid);
  }
  __syncthreads();
  const int flips = __builtin_amdgcn_readfirstlane(sh.flips);

  // runs of angles with one frame (nearly always the whole group)
  for (int sub = 0, sub_end; sub < na; sub = sub_end) {
    const bool flip = (flips >> sub) & 1;
    sub_end = sub + 1;
    while (sub_end < na && (bool)((flips >> sub_end) & 1) == flip) ++sub_end;
    const int Nxx = flip ? J.Ny : J.Nx, Nyy = flip ? J.Nx : J.Ny;
    const int y0 = (int)((int64_t)Nyy * band / nbands), y1 = (int)((int64_t)Nyy * (band + 1) / nbands);
    const int64_t quad = (int64_t)Nyy * (Nxx + 1);
    const E *img = reinterpret_cast<const E *>(flip ? J.imgY : J.imgX) + (int64_t)zb * G * quad;

    __syncthreads();  // the previous run is done with the tables
    if (tid == 0) {
      sh.irregular = 0;
      sh.first = kFwdKnots;
      sh.last = -1;
    }
    __syncthreads();
    const int nedge = 2 * (sub_end - sub);
    if (tid < nedge) {
      const FwdAngle &g = sh.angle[sub + (tid >> 1)];
      const double se = (tid & 1) ? first + nray - 1 : first;
      const StripRay r = strip_ray<real, FAN>(J, g, se, flip);
      sh.edge[tid] = r;
      bool ok = g.scale > 0 && fabs(r.m) < 4 && fabs(r.n) < 4 && fabs(r.u0) < 1e6 && fabs(r.v0) < 1e6;
      ok = ok && (!FAN || strip_forward(J, g, se, flip));
      if (!ok) atomicOr(&sh.irregular, 1);
    }
    __syncthreads();
    // the windows' common slant: start column (xb + y xm) >> 32
    const StripRay &e0 = sh.edge[0], &e1 = sh.edge[nedge - 1];
    const int64_t xm = (int64_t)rint(0.5 * (e0.m + e1.m) * 4294967296.0);
    const int64_t xb = (int64_t)rint(0.5 * (e0.u0 + e1.u0)) << 32;
    // Window of rows [16 k, 16 k + 16): (first column, pitch, rows per chunk,
    // taps), rows = 0 where no ray meets the image.  Every edge is linear along
    // the rows, so the extremes lie at the interval's ends; it holds all taps of
    // every ray, with one whole column to spare on each side for the rounding.
    auto interval = [&](int k) {
      double lo = 1e30, hi = -1e30, w = 0, xl = 1e30, xr = -1e30;
      for (int end = 0; end < 2; ++end) {
        const int y = (k + end) * kFwdKnot;
        const double c = (double)(xb + y * xm) * (1.0 / 4294967296.0);
        for (int i = 0; i < nedge; ++i) {
          const StripRay &r = sh.edge[i];
          const double u = fma(r.m, (double)y, r.u0), v = fma(r.n, (double)y, r.v0);
          lo = fmin(lo, u - c);
          hi = fmax(hi, u - c);
          xl = fmin(xl, u);
          xr = fmax(xr, v);
          w = fmax(w, v - u);
        }
      }
      const int l = (int)floor(lo) - 1, taps = (int)floor(w + 1e-3) + 1;
      const int pitch = (int)floor(hi) + taps + 2 - l;
      return make_int4(l, pitch, xr > -1 && xl < Nxx ? min(max(CAP / pitch, 1), kFwdKnot) : 0, taps);
    };
    const int k0 = y0 / kFwdKnot, k_end = (y1 + kFwdKnot - 1) / kFwdKnot;
    // the first table, and the check of every interval's width
    auto fill = [&](int kb) {
      if (tid < min(kFwdKnots, k_end - kb)) {
        const int4 t = interval(kb + tid);
        sh.table[tid] = t;
        if (t.z) {
          atomicMin(&sh.first, tid);
          atomicMax(&sh.last, tid);
          if (t.y > CAP) atomicOr(&sh.irregular, 2);
        }
      }
    };
    if (!sh.irregular) {
      for (int k = k0 + kFwdKnots + tid; k < k_end; k += 256 * H) {
        const int4 t = interval(k);
        if (t.z && t.y > CAP) atomicOr(&sh.irregular, 2);
      }
      fill(k0);
    }
    __syncthreads();
    const int irregular = __builtin_amdgcn_readfirstlane(sh.irregular);
    real tot[2][G][ZV];
    bool active[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      active[e] = mine + e >= sub && mine + e < sub_end;
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int z = 0; z < ZV; ++z) tot[e][g][z] = 0;
    }
    // buffers over the first and the last group's copy
    const __amdgpu_buffer_rsrc_t rs0 =
        __builtin_amdgcn_make_buffer_rsrc((void *)img, (short)0, (int)(quad * 16), 0x00020000);
    const __amdgpu_buffer_rsrc_t rs1 = __builtin_amdgcn_make_buffer_rsrc((void *)(img + (G - 1) * quad),
                                                                         (short)0, (int)(quad * 16), 0x00020000);
    for (int kb = irregular ? k_end : k0; kb < k_end; kb += kFwdKnots) {
      if (kb > k0) {
        __syncthreads();
        if (tid == 0) {
          sh.first = kFwdKnots;
          sh.last = -1;
        }
        __syncthreads();
        fill(kb);
        __syncthreads();
      }
      const int c_end = __builtin_amdgcn_readfirstlane(sh.last) + 1;
      int ci = __builtin_amdgcn_readfirstlane(sh.first);
      if (ci >= c_end) continue;
      const int y_end = min((kb + c_end) * kFwdKnot, y1);
      int cy = max((kb + ci) * kFwdKnot, y0);  // next chunk's first row, in interval ci
      auto next = [&]() {
        FwdChunk c{cy, 0, 0, 0, 0};
        if (cy >= y_end) return c;
        const int4 t = sh.table[ci];
        const int ye = min((kb + ci + 1) * kFwdKnot, y1);
        c.lo = __builtin_amdgcn_readfirstlane(t.x);
        c.pitch = __builtin_amdgcn_readfirstlane(t.y);
        c.rows = min(ye - cy, max(__builtin_amdgcn_readfirstlane(t.z), 1));
        c.taps = __builtin_amdgcn_readfirstlane(t.w);
        cy += c.rows;
        ci += cy == ye;
        return c;
      };
      auto stage = [&](const FwdChunk &c, E *dst) {
        // row r of group g is copied by wave (r G + g) % 4H; columns outside the
        // image take the row's zero entry
        for (int it = wv; it < c.rows * G; it += 4 * H) {
          const int r = it / G, g = it % G, y = c.y + r;
          const int x0 = (int)((xb + y * xm) >> 32) + c.lo, row = y * (Nxx + 1);
          E *to = dst + g * CAP + r * c.pitch;
          for (int base = 0; base < c.pitch; base += 64) {
            const int j = base + lane;
            if (j < c.pitch) {
              const int at = (row + (int)min((uint32_t)(x0 + j), (uint32_t)Nxx)) * 16;
              auto *lds = (__attribute__((address_space(3))) void *)(to + base);
              if (G == 1 || g == 0)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs0, lds, 16, at, 0, 0, 0);
              else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rs1, lds, 16, at, 0, 0, 0);
            }
          }
        }
      };
      LaneRay<real> ray[2];
#pragma unroll
      for (int e = 0; e < 2; ++e)
        if (active[e])
          ray[e].start(strip_ray<real, FAN>(J, sh.angle[mine + e], s, flip), cy);
      FwdChunk cur = next();
      int which = 0;
      stage(cur, sh.buf[0]);
      while (cur.rows) {
        __builtin_amdgcn_s_waitcnt(0x0f70);  // this wave's copies have landed
        __syncthreads();                     // everybody's have; the other buffer is free
        const FwdChunk nxt = next();
        if (nxt.rows) stage(nxt, sh.buf[which ^ 1]);
        const LdsEntry<real> buf = (LdsEntry<real>)sh.buf[which];
        const int64_t xw = xb + cur.y * xm;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          if (!active[e]) continue;
          real acc[G][ZV];
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int z = 0; z < ZV; ++z) acc[g][z] = 0;
          switch (cur.taps) {
            case 1:
              strip_rows<real, FAN, G, 1>(ray[e], cur, xw, xm, buf, CAP, acc);
              break;
            case 2:
              strip_rows<real, FAN, G, 2>(ray[e], cur, xw, xm, buf, CAP, acc);
              break;
            case 3:
              strip_rows<real, FAN, G, 3>(ray[e], cur, xw, xm, buf, CAP, acc);
              break;
            case 4:
              strip_rows<real, FAN, G, 4>(ray[e], cur, xw, xm, buf, CAP, acc);
              break;
            default:
              strip_rows<real, FAN, G, 0>(ray[e], cur, xw, xm, buf, CAP, acc);
          }
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int z = 0; z < ZV; ++z) tot[e][g][z] += acc[g][z];
        }
        which ^= 1;
        cur = nxt;
      }
    }
    // Results, and the rays to take without windows: those of an irregular run
    // and, whatever the pixel, those that met a value which is not finite (a tap
    // of zero weight may lie outside the strip).
    bool again[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      again[e] = false;
      if (!active[e] || s_own >= J.Ns) continue;
      real check = 0;
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int z = 0; z < ZV; ++z) check = fma(tot[e][g][z], (real)0, check);
      again[e] = irregular || check != (real)0;
      if (!again[e])
        strip_store<real, FAN, G>(J, s, sh.angle[mine + e].a, zb, band, part, (real)sh.angle[mine + e].scale,
                                  tot[e]);
    }
#pragma unroll 1
    for (int e = 0; e < 2; ++e) {
      if (!(e ? again[1] : again[0])) continue;
      FwdAngle g = sh.angle[mine + e];
      g.scale = 1;
      // rays that leave the block's frame take their own, in every row band alike
      const bool f = irregular & 1 ? strip_flipped(J, g, s) : flip;
      const int nx = f ? J.Ny : J.Nx, ny = f ? J.Nx : J.Ny;
      const int64_t qd = (int64_t)ny * (nx + 1);
      const E *from = reinterpret_cast<const E *>(f ? J.imgY : J.imgX) + (int64_t)zb * G * qd;
      real sum[G][ZV] = {};
      strip_direct<real, FAN>(strip_ray<real, FAN>(J, g, s, f), (int)((int64_t)ny * band / nbands),
                              (int)((int64_t)ny * (band + 1) / nbands), nx,
                              [&](int gr, int y, int x) { return from[gr * qd + (int64_t)y * (nx + 1) + x]; }, sum);
      strip_store<real, FAN, G>(J, s, g.a, zb, band, part, (real)1, sum);
    }
  }
}

}  // namespace gt
