// The FP64 shadow step of the gradient rollout as device code: launched by itself
// (k_shadow_step, cf_adjoint.hip) and beside the tile sort (k_sort_shadow, cf_kernels.hip);
// with the helpers it shares with the adjoint's kernels.
#pragma once

#include "cf_internal.h"

namespace cf {

// fmod(y, L) for L > 0, exactly: for y in [0, 2L) it is y or y - L (the subtraction is exact
// there), else fmod itself.
__device__ __forceinline__ double wrap_d(double y, double L) {
  if (y >= 0.0 && y < 2.0 * L) return y >= L ? y - L : y;
  return fmod(y, L);
}

__device__ __forceinline__ double min_image_d(double d, double L) {
  if (d > L * 0.5) d -= L;
  if (d < -L * 0.5) d += L;
  return d;
}

__device__ __forceinline__ float min_image_f(float d, float L) {
  if (d > L * 0.5f) d -= L;
  if (d < -L * 0.5f) d += L;
  return d;
}

__device__ __forceinline__ int bin_axis_a(float x, float ih, int n) {
  float u = x * ih;
  if (!(u >= 0.0f)) return 0;
  if (u >= (float)n) return n - 1;
  return (int)u;
}

// The FP64 density factor of a frozen count (the oracle's op order).
__device__ __forceinline__ double shadow_fac(const AdjConst& c, int cnt, int prev) {
  const double avg = (double)(cnt + prev) * 0.5;
  const double dens = fmin(avg / c.max_exp, 1.0);
  return 1.0 - (1.0 - c.balance) * dens;
}

// ---- pair kernels: G lanes per particle -----------------------------------------------
//
// One lane per particle would leave most of the GPU idle at a few tens of thousands of
// particles and walk every candidate serially.  Instead the stencil's cells are split
// over G lanes (cell index c = g, g+G, ...) and the lanes' partial sums are reduced in a
// fixed order, so results are deterministic.

constexpr int kAdjG = 8;                       // lanes per particle
constexpr int kAdjBlock = 128;                 // threads per block
constexpr int kAdjPer = kAdjBlock / kAdjG;     // particles per block
constexpr int kAdjVals = 4 + kMaxTypes;        // lx, ly, lz, ratio, table row

// Visit the stencil cells c = first, first + step, ... of the (2r+1)^3 cube around
// (cx, cy, cz) (every cell once on axes with fewer than 2r+1 cells), in a fixed order:
// for_cell_runs passes each cell's slot range, for_cells_split each of its slots.  Cell
// coordinates come from float reciprocals: (c + 1/2) / m is at least 1/(2m) away from an
// integer and m <= 25, far beyond the float error.
template <class Fn>
__device__ __forceinline__ void for_cell_runs(const SimDesc& sd, const uint32_t* start, int cx,
                                              int cy, int cz, int r, int first, int step,
                                              Fn&& fn) {
  const bool gx = sd.nx < 2 * r + 1, gy = sd.ny < 2 * r + 1, gz = sd.nz < 2 * r + 1;
  const int nxo = gx ? sd.nx : 2 * r + 1, nyo = gy ? sd.ny : 2 * r + 1,
            nzo = gz ? sd.nz : 2 * r + 1;
  const int ncell = nxo * nyo * nzo, nxy = nxo * nyo;
  const float inxy = 1.0f / (float)nxy, inx = 1.0f / (float)nxo;
  for (int ci = first; ci < ncell; ci += step) {
    const int iz = (int)(((float)ci + 0.5f) * inxy);
    const int rem = ci - iz * nxy;
    const int iy = (int)(((float)rem + 0.5f) * inx);
    const int ix = rem - iy * nxo;
    int x = gx ? ix : cx + ix - r, y = gy ? iy : cy + iy - r, z = gz ? iz : cz + iz - r;
    if (x < 0) x += sd.nx; else if (x >= sd.nx) x -= sd.nx;
    if (y < 0) y += sd.ny; else if (y >= sd.ny) y -= sd.ny;
    if (z < 0) z += sd.nz; else if (z >= sd.nz) z -= sd.nz;
    const int cc = sd.c0 + x + sd.nx * (y + sd.ny * z);
    fn(start[cc], start[cc + 1]);
  }
}

template <class Fn>
__device__ __forceinline__ void for_cells_split(const SimDesc& sd, const uint32_t* start, int cx,
                                                int cy, int cz, int r, int first, int step,
                                                Fn&& fn) {
  for_cell_runs(sd, start, cx, cy, cz, r, first, step, [&](uint32_t q0, uint32_t q1) {
    for (uint32_t q = q0; q < q1; ++q) fn(q);
  });
}

constexpr int kAdjHits = kPairList;  // also the stride of the force kernel's lists

// The pair kernel's particle context and its FP32 in-range decision, shared by the walk
// kernel and the pair kernel.
struct AdjOwn {
  float4 pi;
  int p, ti, cx, cy, cz;
};

__device__ __forceinline__ AdjOwn adj_own(const AdjArgs& a, const SimDesc& sd, int k, bool active) {
  AdjOwn c;
  c.p = sd.p0 + k;
  c.pi = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  c.ti = -1;
  c.cx = c.cy = c.cz = 0;
  if (active) {
    c.pi = a.pos[c.p];
    c.ti = (int)__float_as_uint(c.pi.w);
    c.cx = bin_axis_a(c.pi.x, sd.ihx, sd.nx);
    c.cy = bin_axis_a(c.pi.y, sd.ihy, sd.ny);
    c.cz = bin_axis_a(c.pi.z, sd.ihz, sd.nz);
  }
  return c;
}

// the forward's FP32 decision (ParticleSimulation.cu:92-112 with the engine's op order)
__device__ __forceinline__ bool adj_in_range(const AdjArgs& a, const SimDesc& sd, const AdjOwn& c,
                                             uint32_t q) {
  if ((int)q == c.p) return false;
  const float4 pj = a.pos[q];
  const int tj = (int)__float_as_uint(pj.w);
  const float fx = min_image_f(pj.x - c.pi.x, sd.Lx), fy = min_image_f(pj.y - c.pi.y, sd.Ly),
              fz = min_image_f(pj.z - c.pi.z, sd.Lz);
  const float s2f = fmaf(fz, fz, fmaf(fy, fy, fx * fx));
  return s2f + 1e-4f < a.thr[c.ti * a.c.T + tj];
}

// The shadow step of the particle of thread `thread` of the launch (kAdjG lanes each; a
// particle's lanes lie in one wave).
__device__ __forceinline__ void shadow_block(const AdjArgs& a, int thread) {
  constexpr int G = kAdjG;
  const SimDesc sd = a.sims[0];
  const int k = thread / G, g = thread % G;
  const bool active = k < sd.n;
  const AdjOwn c = adj_own(a, sd, k, active);
  const int T = a.c.T;
  double fx = 0.0, fy = 0.0, fz = 0.0;
  int cnt = 0;
  uint32_t idi = 0;
  double4 xi = make_double4(0.0, 0.0, 0.0, 0.0);
  const double R = a.c.radius, rho = a.c.ratio;
  const double effi = active ? R * (1.0 + a.c.rbt[c.ti] * rho) : 0.0;
  // the FP64 force term of one in-range pair (the oracle's op order), partner type tj at
  // shadow position xj
  auto pair = [&](int tj, const double4& xj) {
    const double dx = min_image_d(xj.x - xi.x, sd.Lx);
    const double dy = min_image_d(xj.y - xi.y, sd.Ly);
    const double dz = min_image_d(xj.z - xi.z, sd.Lz);
    const double dist = sqrt(dx * dx + dy * dy + dz * dz + (double)1e-4f);
    const double eff = (effi + R * (1.0 + a.c.rbt[tj] * rho)) * 0.5;
    const double r = dist / eff;
    const double net = (a.c.rep * exp(-a.c.k * r * r) - a.c.att * r) * a.c.table[c.ti * T + tj];
    fx += dx / dist * net;
    fy += dy / dist * net;
    fz += dz / dist * net;
  };
  int prev = 0;
  double4 vi = make_double4(0.0, 0.0, 0.0, 0.0);
  if (active) {
    idi = a.id[c.p];
    xi = a.x64[idi];
    if (g == 0) {  // the integration's inputs, loaded before the pairs are summed
      prev = __float_as_int(a.vel[c.p].w);
      vi = a.v64[idi];
    }
    // the lane's first two list entries beside the list's length, and below the next trip's
    // beside this one's pairs (entries past the length are never used)
    static_assert(2 * G <= kAdjHits, "two entries per lane");
    const uint32_t* lst = a.hits + (long)k * kAdjHits;
    uint32_t nh = 0u, qa = 0u, qb = 0u;
    if (a.hits) {
      nh = a.nhits[k];
      qa = lst[g];
      qb = lst[g + G];
    }
    if (a.hits && nh <= (uint32_t)kAdjHits) {
      if (g == 0) cnt = (int)nh;
      // the lane's entries two at a time, each stage's loads issued together (list entry,
      // then type and index, then shadow position); pairs summed in entry order
#pragma nounroll
      for (uint32_t e = g; e < nh; e += 2 * G) {
        const bool two = e + G < nh;
        const uint32_t q0 = qa, q1 = two ? qb : q0;
        qa = lst[min(e + 2 * G, (uint32_t)kAdjHits - 1u)];
        qb = lst[min(e + 3 * G, (uint32_t)kAdjHits - 1u)];
        const int t0 = (int)__float_as_uint(a.pos[q0].w), t1 = (int)__float_as_uint(a.pos[q1].w);
        const uint32_t j0 = a.id[q0], j1 = a.id[q1];
        const double4 x0 = a.x64[j0], x1 = a.x64[j1];
        pair(t0, x0);
        if (two) pair(t1, x1);
      }
    } else {
      for_cells_split(sd, a.start, c.cx, c.cy, c.cz, sd.reach, g, G, [&](uint32_t q) {
        if (!adj_in_range(a, sd, c, q)) return;
        ++cnt;
        pair((int)__float_as_uint(a.pos[q].w), a.x64[a.id[q]]);
      });
    }
  }
#pragma unroll
  for (int m = G / 2; m > 0; m >>= 1) {
    fx += __shfl_xor(fx, m, 64);
    fy += __shfl_xor(fy, m, 64);
    fz += __shfl_xor(fz, m, 64);
    cnt += __shfl_xor(cnt, m, 64);
  }
  if (!active || g != 0) return;
  const double m = a.c.fm * shadow_fac(a.c, cnt, prev) * a.c.dt;
  const double vx = vi.x * a.c.friction + fx * m;
  const double vy = vi.y * a.c.friction + fy * m;
  const double vz = vi.z * a.c.friction + fz * m;
  // the w of the state carry its counts: this step's (velocity) and the one before (position)
  a.v64_next[idi] = make_double4(vx, vy, vz, (double)cnt);
  a.x64_next[idi] = make_double4(wrap_d(xi.x + vx * a.c.dt + (double)sd.Lx, (double)sd.Lx),
                                 wrap_d(xi.y + vy * a.c.dt + (double)sd.Ly, (double)sd.Ly),
                                 wrap_d(xi.z + vz * a.c.dt + (double)sd.Lz, (double)sd.Lz),
                                 (double)prev);
}

}  // namespace cf
