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

template <typename real>
__device__ __forceinline__ Entry<real> lds_entry(LdsEntry<real> p) {
  typedef real vec __attribute__((ext_vector_type(kSlices<real>)));
  return __builtin_bit_cast(Entry<real>, *(const __attribute__((address_space(3))) vec *)p);
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
__device__ __forceinline__ TileWindow<real> tile_window(const Job<real> &J, int a, int xa, int ya,
                                                        int cap) {
  const AngleRec<real> c = J.tab[a];
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
// otherwise row + g quad are the padded sinogram rows in memory, read with the
// coordinate clamped to [0.5, Ns + 2.5].
template <typename real, bool FAN, int G, int RP, bool STAGED>
__device__ __forceinline__ void stack_angle(const TileWindow<real> &W, real dx, real dy,
                                            LdsEntry<real> win, int plane,
                                            const Entry<real> *row, int64_t quad, real mid, real hi,
                                            real (&acc)[RP][G][kSlices<real>]) {
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
    Entry<real> e0[RP], e1[RP];
#pragma unroll
    for (int r = 0; r < RP; ++r) {
      if (STAGED) {
        e0[r] = lds_entry<real>(win + g * plane + ix[r]);
        e1[r] = lds_entry<real>(win + g * plane + ix[r] + 1);
      } else {
        e0[r] = row[g * quad + ix[r]];
        e1[r] = row[g * quad + ix[r] + 1];
      }
    }
#pragma unroll
    for (int r = 0; r < RP; ++r)
#pragma unroll
      for (int z = 0; z < kSlices<real>; ++z)
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
        const TileWindow<real> W = tile_window<real, FAN, T::kX, T::kY>(J, ab + tid, xa, ya, CAP);
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
          stack_angle<real, FAN, G, RP, true>(sh.win[l], dx, dy, cur, CAP, nullptr, 0, mid, hi, acc);
      } else {
#pragma unroll 1
        for (int l = i0; l < end; ++l, cur += width)
          if (__builtin_amdgcn_readfirstlane(sh.win[l].n))
            stack_angle<real, FAN, G, RP, true>(sh.win[l], dx, dy, cur, CAP, nullptr, 0, mid, hi, acc);
      }
      which ^= 1;
    }
    if (direct) {
#pragma unroll 1
      for (int l = 0; l < nb; ++l)
        if (__builtin_amdgcn_readfirstlane(sh.win[l].n) == 0)
          stack_angle<real, FAN, G, RP, false>(sh.win[l], dx, dy, nullptr, 0,
                                                   S + (int64_t)(ab + l) * Nsp, quad, mid,
                                                   hi, acc);
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

}  // namespace gt
