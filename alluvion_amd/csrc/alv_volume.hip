// alv_volume.hip -- volume maps (update_volume_field, runner.hpp:1616-1694):
// at every node of a boundary's map, the Peirce product rule over the ball of
// radius h around the node (60 x 30 x 15 = 27,000 points) of the boundary's
// indicator, smoothed by the kernel: 1 where sign * distance <= 0,
// W(sign * distance) / W(0) outside, 0 from h on.
//
// A node whose whole ball lies farther than h outside the boundary sums exact
// zeros, and one whose ball lies inside sums the weights alone, so only the
// nodes between run the quadrature: a first pass writes the two constant
// classes and lists the rest, cell by cell in 4 x 4 x 4 blocks of cells, so
// that the 64 nodes of a wave lie within a few cells of each other.  The
// quadrature's points and weights are uniform over a wave and come from one
// table through scalar loads.  Every node's terms are added in the rule's
// order by one lane, so the sums are those of the plain triple loop, bit for
// bit, whichever kernel evaluates the terms.
//
// Bound by VALU issue: about 23 (sphere) to 55 (shell) instructions per point
// for the distance and 14 for the kernel where it runs.  Measured on an
// MI355X: a 128^3 sphere map (14.9 M nodes, 42 % listed) 548 -> 111 ms, a
// sampled 32^3 box map 240 -> 42 ms (a 128-byte line of nodal values per cell
// where the node arrays took 32 scattered loads per point; still half on the
// loads' line lookups), 12^3 maps 9 -> 0.9 ms (sampled 5 ms).
#include <float.h>
#include <hip/hip_runtime.h>

#include <algorithm>

#include "alv_device.hpp"
#include "alv_kernels.hpp"

namespace alv {
namespace {

constexpr float kPiF = 3.14159265358979323846f;
constexpr unsigned kRays = 60u * 30u, kRadii = 15u, kUnit = 5u;
constexpr unsigned kBallPoints = kRays * kRadii;
static_assert(kRadii % kUnit == 0u, "a ray is a whole number of units");
// Lebesgue constant of the 32-node element, max over a cell of sum |N_j|
// (5.75, reached at the centre of the cell), rounded up
constexpr float kLebesgue = 5.76f;

// Peirce constants are packed as cosphi[30], sinphi[30], b[30], r[15], c[15].
// grid_form: the weights' product as the distance-map variant forms it.
__device__ inline float ball_weight(const float* pc, unsigned j, unsigned k, int grid_form) {
  const float kb = pc[60 + j], kc = pc[105 + k];
  if (grid_form) return (2.0f * kPiF / 60.0f * kb) * kc;
  return 2.0f * kPiF * kb * kc / 60.0f;
}

// the points of the rule on the ball of radius h, (q, weight), in its order
__global__ __launch_bounds__(256) void k_ball_points(float h, const float* __restrict__ pc,
                                                     int grid_form, float4* __restrict__ pts) {
  const unsigned t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= kBallPoints) return;
  const unsigned i = t / (30u * kRadii), j = t / kRadii % 30u, k = t % kRadii;
  const float theta = 2.0f * kPiF * float(i + 1) / 60.0f;
  const float ct = cosf(theta), st = sinf(theta);
  const vec3 u = mk(pc[30 + j] * ct, pc[30 + j] * st, pc[j]);
  pts[t] = f4((h * pc[90 + k]) * u, ball_weight(pc, j, k, grid_form));
}

// ---------------------------------------------------------------------------
// Node classes
// ---------------------------------------------------------------------------
// Thread order of the class passes: seven threads per cell corner (i, j, k),
// its corner node and the two nodes of the x-, y- and z-edge that start
// there, over 4 x 4 x 4 blocks of corners.
inline size_t class_threads(const GridGeomDev& g) {
  size_t n = 7u * 64u;
  for (int a = 0; a < 3; ++a) n *= (g.res[a] + 1u + 3u) / 4u;
  return n;
}
__device__ inline bool class_node(const GridGeomDev& g, size_t t, unsigned ijk[3], unsigned& l) {
  const unsigned s = unsigned(t % 7u);
  size_t c = t / 7u;
  const unsigned in = unsigned(c % 64u);
  c /= 64u;
  const unsigned rx = g.res[0], ry = g.res[1], rz = g.res[2];
  const unsigned bx = (rx + 4u) / 4u, by = (ry + 4u) / 4u;
  const unsigned i = 4u * unsigned(c % bx) + (in & 3u);
  const unsigned j = 4u * unsigned(c / bx % by) + ((in >> 2) & 3u);
  const unsigned k = 4u * unsigned(c / bx / by) + (in >> 4);
  ijk[0] = i;
  ijk[1] = j;
  ijk[2] = k;
  if (i > rx || j > ry || k > rz) return false;
  unsigned base = (rx + 1) * (ry + 1) * (rz + 1);
  if (s == 0u) {
    l = (k * (ry + 1) + j) * (rx + 1) + i;
    return true;
  }
  if (s <= 2u) {
    l = base + 2u * ((k * (ry + 1) + j) * rx + i) + (s - 1u);
    return i < rx;
  }
  base += 2u * (rx * (ry + 1) * (rz + 1));
  if (s <= 4u) {
    l = base + 2u * ((i * (rz + 1) + k) * ry + j) + (s - 3u);
    return j < ry;
  }
  base += 2u * ((rx + 1) * ry * (rz + 1));
  l = base + 2u * ((j * (rx + 1) + i) * rz + k) + (s - 5u);
  return k < rz;
}

// Writes a constant node, or appends it to the list (one atomic per wave,
// the wave's nodes staying together and in order).
__device__ inline void put_class(bool live, bool out, bool in, unsigned l, float full, float* vol,
                                 unsigned* list, unsigned* count) {
  if (live && (out || in)) vol[l] = out ? 0.0f : full;
  const bool near = live && !out && !in;
  const unsigned long long m = __ballot(near);
  if (m == 0ull) return;
  const unsigned lane = threadIdx.x & 63u;
  unsigned base = 0;
  if (lane == unsigned(__builtin_ctzll(m))) base = atomicAdd(count, unsigned(__popcll(m)));
  base = __shfl(int(base), __builtin_ctzll(m), 64);
  if (near) list[base + unsigned(__popcll(m & ((1ull << lane) - 1ull)))] = l;
}

// An analytic distance changes by at most the length moved, so the distance
// at the node bounds it over the ball.  `reach` is the ball's radius with a
// margin for the rounding of coordinates and distances, times |sign|.
__global__ __launch_bounds__(256) void k_class_analytic(SimParams p, BoundaryDev B, float reach,
                                                        float full_sum, float* __restrict__ vol,
                                                        unsigned* __restrict__ list,
                                                        unsigned* __restrict__ count) {
  const size_t t = size_t(blockIdx.x) * kBlock + threadIdx.x;
  unsigned ijk[3], l = 0;
  const bool live = class_node(B.geom, t, ijk, l);
  float d = 0.0f;
  if (live) d = sdf_eval(B, node_position(B.geom, l)) * B.sign;
  put_class(live, d > p.h + reach, d < -reach, l, full_sum * p.h2 * p.h, vol, list, count);
}

// A distance map's cells: the 32 nodal values in one 128-byte line (the order
// of grid_cell_nodes), and bounds of sign times the interpolated distance.
// The element reproduces linear functions, so the interpolant is the linear
// part L through the corners plus at most kLebesgue times the largest nodal
// difference from L; the margin covers the rounding of the interpolation.
// A cell with a value that is not finite (or beyond 1e30) has no bounds.
__global__ __launch_bounds__(256) void k_map_cells(GridGeomDev g, const float* __restrict__ dist,
                                                   float sign, float h, float* __restrict__ cells,
                                                   float2* __restrict__ bounds) {
  const unsigned c = blockIdx.x * kBlock + threadIdx.x;
  const unsigned rx = g.res[0], ry = g.res[1], rz = g.res[2];
  if (c >= rx * ry * rz) return;
  const int ip[3] = {int(c % rx), int(c / rx % ry), int(c / (rx * ry))};
  unsigned id[32];
  grid_cell_nodes(g.res, ip, id);
  float v[32];
  float big = 0.0f;
  bool bad = false;
#pragma unroll
  for (int n = 0; n < 32; ++n) {
    v[n] = dist[id[n]];
    bad |= !(fabsf(v[n]) < 1e30f);
    big = fmaxf(big, fabsf(v[n]));
  }
  float4* out = reinterpret_cast<float4*>(cells + size_t(c) * 32u);
#pragma unroll
  for (int n = 0; n < 8; ++n) out[n] = make_float4(v[4 * n], v[4 * n + 1], v[4 * n + 2], v[4 * n + 3]);
  float m = 0.0f, gx = 0.0f, gy = 0.0f, gz = 0.0f;
#pragma unroll
  for (int n = 0; n < 8; ++n) {
    m += v[n];
    gx += (n & 1) ? v[n] : -v[n];
    gy += (n & 2) ? v[n] : -v[n];
    gz += (n & 4) ? v[n] : -v[n];
  }
  m *= 0.125f;
  gx *= 0.125f;
  gy *= 0.125f;
  gz *= 0.125f;
  float r = 0.0f;
#pragma unroll
  for (int n = 0; n < 32; ++n) {
    float x, y, z;  // the node's local coordinates (grid_cell_nodes)
    if (n < 8) {
      x = (n & 1) ? 1.0f : -1.0f;
      y = (n & 2) ? 1.0f : -1.0f;
      z = (n & 4) ? 1.0f : -1.0f;
    } else {
      const int e = (n & 7) >> 1;
      const float u = (n & 1) ? 1.0f / 3.0f : -1.0f / 3.0f;
      const float lo = (e & 1) ? 1.0f : -1.0f, hi = (e >> 1) ? 1.0f : -1.0f;
      if (n < 16) {
        x = u, y = hi, z = lo;
      } else if (n < 24) {
        x = lo, y = u, z = hi;
      } else {
        x = hi, y = lo, z = u;
      }
    }
    r = fmaxf(r, fabsf(v[n] - (m + gx * x + gy * y + gz * z)));
  }
  const float w = fabsf(gx) + fabsf(gy) + fabsf(gz) + kLebesgue * r + 1e-4f * (big + h);
  const float a = (m - w) * sign, b = (m + w) * sign;
  bounds[c] = bad ? make_float2(-FLT_MAX, FLT_MAX) : make_float2(fminf(a, b), fmaxf(a, b));
}
// the bounds over the 2 w + 1 cells along one axis (three passes: over the
// box of cells that the ball of any node of the cell can reach)
__global__ __launch_bounds__(256) void k_spread_bounds(GridGeomDev g, int axis, unsigned w,
                                                       const float2* __restrict__ in,
                                                       float2* __restrict__ out) {
  const unsigned c = blockIdx.x * kBlock + threadIdx.x;
  const unsigned rx = g.res[0], ry = g.res[1], rz = g.res[2];
  if (c >= rx * ry * rz) return;
  const unsigned at = axis == 0 ? c % rx : (axis == 1 ? c / rx % ry : c / (rx * ry));
  const unsigned stride = axis == 0 ? 1u : (axis == 1 ? rx : rx * ry);
  const unsigned a = at - min(at, w), b = min(at + w, g.res[axis] - 1u);
  float lo = FLT_MAX, hi = -FLT_MAX;
  for (unsigned k = a; k <= b; ++k) {
    const float2 v = in[c + k * stride - at * stride];
    lo = fminf(lo, v.x);
    hi = fmaxf(hi, v.y);
  }
  out[c] = make_float2(lo, hi);
}
// Points off the map have distance FLT_MAX, which is outside (a zero term)
// for a positive sign and inside (the weight alone) for a negative one; both
// agree with the class of the cells around only in that combination, which
// is the one the bounds of a class and the sign give: an "out" node of a
// negative sign, or an "in" node of a positive one, is a class only when its
// whole ball lies on the map.
__global__ __launch_bounds__(256) void k_class_grid(SimParams p, GridGeomDev g, float sign,
                                                    float reach, float full_sum,
                                                    const float2* __restrict__ bounds,
                                                    float* __restrict__ vol,
                                                    unsigned* __restrict__ list,
                                                    unsigned* __restrict__ count) {
  const size_t t = size_t(blockIdx.x) * kBlock + threadIdx.x;
  unsigned ijk[3], l = 0;
  const bool live = class_node(g, t, ijk, l);
  bool out = false, in = false;
  if (live) {
    const unsigned rx = g.res[0], ry = g.res[1], rz = g.res[2];
    const float2 b = bounds[(min(ijk[2], rz - 1u) * ry + min(ijk[1], ry - 1u)) * rx +
                            min(ijk[0], rx - 1u)];
    const vec3 x = node_position(g, l);
    const bool on_map = x.x - reach > g.dmin[0] && x.y - reach > g.dmin[1] &&
                        x.z - reach > g.dmin[2] && x.x + reach < g.dmax[0] &&
                        x.y + reach < g.dmax[1] && x.z + reach < g.dmax[2];
    out = b.x > p.h && (on_map || sign > 0.0f);
    in = b.y <= 0.0f && (on_map || sign < 0.0f);
  }
  put_class(live, out, in, l, full_sum * p.h2 * p.h, vol, list, count);
}

// ---------------------------------------------------------------------------
// Quadrature of the listed nodes
// ---------------------------------------------------------------------------
// sdf_eval with the refined square root (the same correctly rounded value)
__device__ inline float box_dist_rn(vec3 x, const float half[3]) {
  const vec3 diff = mk(fabsf(x.x) - half[0], fabsf(x.y) - half[1], fabsf(x.z) - half[2]);
  const vec3 cl = mk(fmaxf(diff.x, 0.0f), fmaxf(diff.y, 0.0f), fmaxf(diff.z, 0.0f));
  return sqrt_rn(length_sqr(cl)) + fminf(fmaxf(diff.x, fmaxf(diff.y, diff.z)), 0.0f);
}
template <int Type>
struct AnalyticDist {
  BoundaryDev B;
  __device__ float operator()(vec3 x) const {
    if (Type == ALV_DIST_BOX) return (box_dist_rn(x, B.half) - B.outset) * B.sign;
    if (Type == ALV_DIST_BOX_SHELL)
      return fmaxf(box_dist_rn(x, B.half_outer) - B.outset, -(box_dist_rn(x, B.half) - B.outset)) *
             B.sign;
    return (sqrt_rn(length_sqr(x)) - B.radius) * B.sign;
  }
  __device__ vec3 node(unsigned l) const { return node_position(B.geom, l); }
  // |change of the distance| per length moved, and the rounding margin
  __device__ float slope() const { return fabsf(B.sign); }
};
struct MapDist {
  GridGeomDev g;
  const float* cells;
  float sign;
  __device__ float operator()(vec3 x) const {
    int ip[3];
    vec3 xi;
    if (!grid_resolve(g, x, ip, xi)) return FLT_MAX * sign;
    const float4* src = reinterpret_cast<const float4*>(
        cells + size_t((unsigned(ip[2]) * g.res[1] + unsigned(ip[1])) * g.res[0] + unsigned(ip[0])) * 32u);
    float v[32];
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      const float4 q = src[n];
      v[4 * n] = q.x;
      v[4 * n + 1] = q.y;
      v[4 * n + 2] = q.z;
      v[4 * n + 3] = q.w;
    }
    constexpr unsigned id[32] = {0,  1,  2,  3,  4,  5,  6,  7,  8,  9,  10, 11, 12, 13, 14, 15,
                                 16, 17, 18, 19, 20, 21, 22, 23, 24, 25, 26, 27, 28, 29, 30, 31};
    return grid_interpolate(v, id, xi) * sign;
  }
  __device__ vec3 node(unsigned l) const { return node_position(g, l); }
  // nothing is known between the nodes: no radius is skipped
  __device__ float slope() const { return FLT_MAX; }
};

// The terms of kUnit consecutive points at node x.  The kernel runs only when
// some lane of the wave has a point in its support; W_dist's expressions.
template <class D>
__device__ inline void unit_terms(const D& dist, vec3 x, const float4* __restrict__ t,
                                  const SimParams& p, float inv_w0, float (&term)[kUnit]) {
  float dm[kUnit];
  bool act = false;
#pragma unroll
  for (unsigned u = 0; u < kUnit; ++u) {
    dm[u] = dist(x + mk(t[u].x, t[u].y, t[u].z));
    act |= dm[u] > 0.0f && dm[u] < p.h * 1.00001f;
  }
  if (__ballot(act) == 0ull) {
#pragma unroll
    for (unsigned u = 0; u < kUnit; ++u) term[u] = dm[u] <= 0.0f ? t[u].w : 0.0f;
    return;
  }
#pragma unroll
  for (unsigned u = 0; u < kUnit; ++u) {
    const float q = div_known(dm[u], p.h, p.inv_h);
    const float conj = 1.0f - q;
    const float inner = (6.0f * q - 6.0f) * q * q + 1.0f;
    const float outer = 2.0f * conj * conj * conj;
    float g = div_known((q <= 0.5f ? inner : (q <= 1.0f ? outer : 0.0f)) * p.k, p.w0, inv_w0);
    asm volatile("" : "+v"(g));  // a select, not a branch per point
    term[u] = t[u].w * (dm[u] <= 0.0f ? 1.0f : g);
  }
}

// Leading radii of every ray whose points are all outside the support (skip)
// or all inside the boundary (add the weights) for every node of the wave:
// from the distances d at the nodes and the radii.  Uniform over the wave.
__device__ inline void wave_trivial(float d, float slope, const float* pc, const SimParams& p,
                                    float margin, int& units, bool& inside) {
  float lo = d, hi = d;
  for (int o = 32; o > 0; o >>= 1) {
    lo = fminf(lo, __shfl_xor(lo, o, 64));
    hi = fmaxf(hi, __shfl_xor(hi, o, 64));
  }
  int n_out = 0, n_in = 0;
  if (slope < FLT_MAX && lo == lo && hi == hi) {
    for (int k = 0; k < int(kRadii / kUnit); ++k) {
      const float r = slope * (p.h * pc[90 + k * kUnit + kUnit - 1] + margin);
      n_out += lo - r > p.h ? 1 : 0;
      n_in += hi + r < 0.0f ? 1 : 0;
    }
  }
  units = __builtin_amdgcn_readfirstlane(max(n_out, n_in));
  inside = __builtin_amdgcn_readfirstlane(n_in) > 0;
}

// One node per lane, a wave's nodes being neighbours in the list.
template <class D>
__global__ __launch_bounds__(256) void k_ball_sums(SimParams p, D dist, float margin,
                                                   const float4* __restrict__ pts,
                                                   const float* __restrict__ pc,
                                                   const unsigned* __restrict__ list,
                                                   const unsigned* __restrict__ count,
                                                   unsigned least, size_t first,
                                                   float* __restrict__ vol) {
  const unsigned n = *count;
  const size_t at = first + size_t(blockIdx.x) * kBlock + threadIdx.x;
  if (n <= least || at - (threadIdx.x & 63u) >= n) return;  // whole waves
  const unsigned l = list[min(at, size_t(n) - 1u)];
  const vec3 x = dist.node(l);
  int skip;
  bool inside;
  wave_trivial(dist(x), dist.slope(), pc, p, margin, skip, inside);
  const float inv_w0 = 1.0f / p.w0;
  float sum = 0.0f;
  for (unsigned ray = 0; ray < kRays; ++ray) {
    const float4* t = pts + ray * kRadii;
    if (inside)
      for (int k = 0; k < skip * int(kUnit); ++k) sum += t[k].w;
    for (int k = skip; k < int(kRadii / kUnit); ++k) {
      float term[kUnit];
      unit_terms(dist, x, t + k * kUnit, p, inv_w0, term);
#pragma unroll
      for (unsigned u = 0; u < kUnit; ++u) sum += term[u];
    }
  }
  if (at < n) vol[l] = sum * p.h2 * p.h;
}

// Few nodes: 64 nodes per block of 16 waves.  Waves 1 to 15 evaluate the
// terms of one unit each (five rays a round) into LDS, wave 0 adds the
// previous round's terms in order meanwhile.  The instance for distance maps
// spills five registers at its bound of 64 and is the faster for it: 42 ms
// against 43 for a sampled 32^3 map.
constexpr unsigned kTeam = 16;
constexpr unsigned kRoundRays = (kTeam - 1u) * kUnit / kRadii;
static_assert((kTeam - 1u) * kUnit % kRadii == 0u && kRays % kRoundRays == 0u, "whole rays");
template <class D>
__global__ __launch_bounds__(kTeam * 64, 8) void k_ball_sums_team(
    SimParams p, D dist, float margin, const float4* __restrict__ pts,
    const float* __restrict__ pc, const unsigned* __restrict__ list,
    const unsigned* __restrict__ count, unsigned most, float* __restrict__ vol) {
  constexpr unsigned kRound = kRoundRays * kRadii;
  __shared__ float terms[2][kRound][64];
  const unsigned n = *count;
  if (n > most) return;
  const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const unsigned at = blockIdx.x * 64u + lane;
  if (blockIdx.x * 64u >= n) return;  // the whole block
  const unsigned l = list[min(at, n - 1u)];
  const vec3 x = dist.node(l);
  int skip;
  bool inside;
  wave_trivial(dist(x), dist.slope(), pc, p, margin, skip, inside);
  const float inv_w0 = 1.0f / p.w0;
  const unsigned unit = __builtin_amdgcn_readfirstlane(wave) - 1u;
  const unsigned ray_in = unit / (kRadii / kUnit), k_in = unit % (kRadii / kUnit);
  float sum = 0.0f;
  for (unsigned round = 0; round <= kRays / kRoundRays; ++round) {
    if (wave == 0u) {
      if (round > 0u) {
        const float(*src)[64] = terms[(round - 1u) & 1u];
        const float4* t = pts + (round - 1u) * kRound;
        for (unsigned r = 0; r < kRoundRays; ++r) {
          for (unsigned k = 0; k < kRadii / kUnit; ++k) {
            const unsigned b = r * kRadii + k * kUnit;
            if (int(k) < skip) {
              if (inside)
                for (unsigned u = 0; u < kUnit; ++u) sum += t[b + u].w;
            } else {
#pragma unroll
              for (unsigned u = 0; u < kUnit; ++u) sum += src[b + u][lane];
            }
          }
        }
      }
    } else if (round < kRays / kRoundRays && int(k_in) >= skip) {
      float term[kUnit];
      const unsigned b = ray_in * kRadii + k_in * kUnit;
      unit_terms(dist, x, pts + round * kRound + b, p, inv_w0, term);
#pragma unroll
      for (unsigned u = 0; u < kUnit; ++u) terms[round & 1u][b + u][lane] = term[u];
    }
    __syncthreads();
  }
  if (wave == 0u && at < n) vol[l] = sum * p.h2 * p.h;
}

// Up to this many listed nodes run as teams: a wave per 64 nodes would leave
// the chip's 1,024 SIMDs with fewer than eight waves each and a last round
// that is nearly empty.  About 340,000 listed nodes (48^3 cells) take 7.8-9.1
// ms as teams and 9.4-10.2 ms as waves; beyond, the team's LDS round trip
// costs as much as the rounds save.
constexpr unsigned kTeamNodes = 1u << 19;
constexpr size_t kSlice = size_t(1) << 24;  // listed nodes per launch

template <class D>
void launch_ball_sums(const SimParams& p, const D& dist, float margin, const float4* pts,
                      const float* pc, const unsigned* list, const unsigned* count, size_t nodes,
                      float* vol, hipStream_t s) {
  // the number of listed nodes stays on the device: both kernels start and
  // the one it is not for returns at once
  const unsigned teams = unsigned((std::min(nodes, size_t(kTeamNodes)) + 63u) / 64u);
  hipLaunchKernelGGL(k_ball_sums_team<D>, dim3(teams), dim3(kTeam * 64u), 0, s, p, dist, margin,
                     pts, pc, list, count, kTeamNodes, vol);
  for (size_t b = 0; nodes > kTeamNodes && b < nodes; b += kSlice)
    hipLaunchKernelGGL(k_ball_sums<D>, dim3(unsigned((std::min(kSlice, nodes - b) + kBlock - 1) / kBlock)),
                       dim3(kBlock), 0, s, p, dist, margin, pts, pc, list, count, kTeamNodes, b, vol);
}

// The sum of all weights in the rule's order: what a node inside adds up.
float full_sum(const float* table, bool grid_form) {
  float sum = 0.0f;
  const float wi = 2.0f * kPiF / 60.0f;
  for (unsigned i = 0; i < 60; ++i)
    for (unsigned j = 0; j < 30; ++j)
      for (unsigned k = 0; k < kRadii; ++k) {
        const float kb = table[60 + j], kc = table[105 + k];
        sum += grid_form ? (wi * kb) * kc : 2.0f * kPiF * kb * kc / 60.0f;
      }
  return sum;
}

// Workspace: the points, the counter and the list; for distance maps also the
// cells and two arrays of bounds.
constexpr size_t align256(size_t n) { return (n + 255u) / 256u * 256u; }
constexpr size_t kPtsBytes = align256(kBallPoints * sizeof(float4));
size_t list_bytes(const GridGeomDev& g) { return align256(size_t(g.num_nodes) * sizeof(unsigned)); }
size_t num_cells(const GridGeomDev& g) { return size_t(g.res[0]) * g.res[1] * g.res[2]; }

// the largest coordinate (or extent) that enters the distances
float extent(const GridGeomDev& g) {
  float m = 0.0f;
  for (int a = 0; a < 3; ++a) m = std::max(m, std::max(fabsf(g.dmin[a]), fabsf(g.dmax[a])));
  return m;
}
}  // namespace

size_t volume_field_workspace(const GridGeomDev& g, bool distance_map) {
  size_t n = kPtsBytes + 256u + list_bytes(g);
  if (distance_map) n += num_cells(g) * 128u + 2u * align256(num_cells(g) * sizeof(float2));
  return n;
}

void launch_volume_field_analytic(const SimParams& p, const BoundaryDev& b, float* volume,
                                  const float* peirce, const float* peirce_host, void* workspace,
                                  hipStream_t s) {
  if (b.geom.num_nodes == 0) return;
  char* ws = static_cast<char*>(workspace);
  float4* pts = reinterpret_cast<float4*>(ws);
  unsigned* count = reinterpret_cast<unsigned*>(ws + kPtsBytes);
  unsigned* list = reinterpret_cast<unsigned*>(ws + kPtsBytes + 256u);
  launch_fill_u32(count, 0u, 1, s);
  hipLaunchKernelGGL(k_ball_points, dim3(grid_for(kBallPoints)), dim3(kBlock), 0, s, p.h, peirce, 0,
                     pts);
  float m = extent(b.geom) + std::max(fabsf(b.radius), fabsf(b.outset));
  for (int a = 0; a < 3; ++a) m = std::max(m, std::max(fabsf(b.half[a]), fabsf(b.half_outer[a])));
  // rounding of the coordinates and the distance: a few 2^-24 of m each
  const float margin = 1e-3f * p.h + 1e-5f * m;
  hipLaunchKernelGGL(k_class_analytic, dim3(unsigned((class_threads(b.geom) + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, s, p, b, fabsf(b.sign) * (p.h + margin),
                     full_sum(peirce_host, false), volume, list, count);
  const size_t n = b.geom.num_nodes;
  if (b.type == ALV_DIST_BOX)
    launch_ball_sums(p, AnalyticDist<ALV_DIST_BOX>{b}, margin, pts, peirce, list, count, n, volume, s);
  else if (b.type == ALV_DIST_BOX_SHELL)
    launch_ball_sums(p, AnalyticDist<ALV_DIST_BOX_SHELL>{b}, margin, pts, peirce, list, count, n,
                     volume, s);
  else
    launch_ball_sums(p, AnalyticDist<ALV_DIST_SPHERE>{b}, margin, pts, peirce, list, count, n, volume,
                     s);
}

void launch_volume_field_grid(const SimParams& p, const GridGeomDev& g, const float* distance,
                              float* volume, float sign, const float* peirce,
                              const float* peirce_host, void* workspace, hipStream_t s) {
  if (g.num_nodes == 0) return;
  char* ws = static_cast<char*>(workspace);
  float4* pts = reinterpret_cast<float4*>(ws);
  unsigned* count = reinterpret_cast<unsigned*>(ws + kPtsBytes);
  unsigned* list = reinterpret_cast<unsigned*>(ws + kPtsBytes + 256u);
  float* cells = reinterpret_cast<float*>(ws + kPtsBytes + 256u + list_bytes(g));
  const size_t nc = num_cells(g);
  float2* b0 = reinterpret_cast<float2*>(reinterpret_cast<char*>(cells) + nc * 128u);
  float2* b1 = reinterpret_cast<float2*>(reinterpret_cast<char*>(b0) + align256(nc * sizeof(float2)));
  launch_fill_u32(count, 0u, 1, s);
  hipLaunchKernelGGL(k_ball_points, dim3(grid_for(kBallPoints)), dim3(kBlock), 0, s, p.h, peirce, 1,
                     pts);
  const dim3 cgrid(unsigned((nc + kBlock - 1) / kBlock));
  hipLaunchKernelGGL(k_map_cells, cgrid, dim3(kBlock), 0, s, g, distance, sign, p.h, cells, b0);
  const float reach = p.h * 1.001f + 1e-5f * extent(g);
  for (int a = 0; a < 3; ++a) {
    // cells that a ball can reach from any node of a cell, and one for the
    // rounding of the cell search
    const float w = std::min(reach / g.cs[a], float(g.res[a]));
    hipLaunchKernelGGL(k_spread_bounds, cgrid, dim3(kBlock), 0, s, g, a,
                       w >= 0.0f ? unsigned(w) + 1u : g.res[a], a == 1 ? b1 : b0, a == 1 ? b0 : b1);
  }
  hipLaunchKernelGGL(k_class_grid, dim3(unsigned((class_threads(g) + kBlock - 1) / kBlock)),
                     dim3(kBlock), 0, s, p, g, sign, reach, full_sum(peirce_host, true), b1, volume,
                     list, count);
  launch_ball_sums(p, MapDist{g, cells, sign}, 0.0f, pts, peirce, list, count, g.num_nodes, volume,
                   s);
}

}  // namespace alv
