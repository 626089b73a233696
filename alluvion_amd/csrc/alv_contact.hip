// alv_contact.hip -- rigid-body contact detection (reference runner.hpp:3833-
// 3914 `collision_test`, analytic-distance variant; pile.hpp:826-904
// `find_contacts`).
//
// Every collision vertex of body i is tested against the signed distance of
// body j (box or sphere, in j's frame).  The reference appends contacts with
// an atomic counter, so their order -- and the result of the sequential
// Gauss-Seidel contact solve that follows -- depends on thread timing.  Here
// the candidates are numbered (pair in (i, j) order, then vertex), one pass
// over all of them leaves a bit per candidate, and a second one places each
// hit at the number of bits before its own, so contacts come out in that
// order on every run.  Few candidates are tested and placed by one block.
#include <hip/hip_runtime.h>

#include "alv_contact.hpp"
#include "alv_device.hpp"

namespace alv {
namespace {

constexpr unsigned kContactThreads = 256;
constexpr unsigned kContactWaves = kContactThreads / 64;
// Candidates that one block tests and numbers by itself, in one launch: a whole
// find_contacts of 24 takes 55 us and 57 with the two passes, of 768 62 and 64,
// of 1,024 both 68; a second round of 1,024 takes one block 8 us more.
constexpr unsigned kFewCandidates = 1024;

// R diag(v) R^T for the rotation of q, stored as diagonal and (01, 02, 12)
// off-diagonal (runner.hpp:178-199).
__device__ inline void congruent_matrix(vec3 v, float4 q, vec3* diag, vec3* off) {
  const float m00 = 1 - 2 * (q.y * q.y + q.z * q.z), m01 = 2 * (q.x * q.y - q.z * q.w),
              m02 = 2 * (q.x * q.z + q.y * q.w);
  const float m10 = 2 * (q.x * q.y + q.z * q.w), m11 = 1 - 2 * (q.x * q.x + q.z * q.z),
              m12 = 2 * (q.y * q.z - q.x * q.w);
  const float m20 = 2 * (q.x * q.z - q.y * q.w), m21 = 2 * (q.y * q.z + q.x * q.w),
              m22 = 1 - 2 * (q.x * q.x + q.y * q.y);
  *diag = mk(v.x * m00 * m00 + v.y * m01 * m01 + v.z * m02 * m02,
             v.x * m10 * m10 + v.y * m11 * m11 + v.z * m12 * m12,
             v.x * m20 * m20 + v.y * m21 * m21 + v.z * m22 * m22);
  *off = mk(v.x * m00 * m10 + v.y * m01 * m11 + v.z * m02 * m12,
            v.x * m00 * m20 + v.y * m01 * m21 + v.z * m02 * m22,
            v.x * m10 * m20 + v.y * m11 * m21 + v.z * m12 * m22);
}

// Impulse response matrix K = I/m - [r]x I_w^-1 [r]x of one body at lever
// arm r (runner.hpp:265-288); zero for a body of zero mass.
__device__ inline void contact_k(vec3 r, float mass, vec3 d, vec3 o, vec3* kd, vec3* ko) {
  *kd = mk(0.f, 0.f, 0.f);
  *ko = mk(0.f, 0.f, 0.f);
  if (mass == 0.f) return;
  const float im = 1 / mass;
  *kd = mk(r.z * r.z * d.y - r.y * r.z * o.z * 2 + r.y * r.y * d.z + im,
           r.z * r.z * d.x - r.x * r.z * o.y * 2 + r.x * r.x * d.z + im,
           r.y * r.y * d.x - r.x * r.y * o.x * 2 + r.x * r.x * d.y + im);
  *ko = mk(-r.z * r.z * o.x + r.x * r.z * o.z + r.y * r.z * o.y - r.x * r.y * d.z,
           r.y * r.z * o.x - r.x * r.z * d.y - r.y * r.y * o.y + r.x * r.y * o.z,
           -(r.y * r.z * d.x) + r.x * r.z * o.x + r.x * r.y * o.y - r.x * r.x * o.z);
}

__device__ inline vec3 sym_apply(vec3 v, vec3 d, vec3 o) {
  return mk(v.x * d.x + v.y * o.x + v.z * o.y, v.x * o.x + v.y * d.y + v.z * o.z,
            v.x * o.y + v.y * o.z + v.z * d.z);
}

__device__ inline void put3(float* dst, vec3 v) {
  dst[0] = v.x;
  dst[1] = v.y;
  dst[2] = v.z;
}

// Tests vertex `vert` of body i against body j: whether it is inside body j
// (dist < 0) and, with `Record`, the record of one that is.  World vertices
// (pellets, collision_test_with_pellets, runner.hpp:3627-3727) are already
// placed; body-frame vertices are placed with body i's kinematics.  `inertia`
// holds [B][3] principal inertia, then [B][2] (restitution, friction).
template <bool Record>
__device__ bool test_vertex(unsigned i, unsigned j, unsigned flags, unsigned nb,
                            const BoundaryDev* bodies, const float* inertia, const float* verts,
                            unsigned vert, float tolerance, alv_contact* out) {
  const BoundaryDev& Bi = bodies[i];
  const BoundaryDev& Bj = bodies[j];
  if ((flags & kJobSkip) && (i == j || (Bi.mass == 0.f && Bj.mass == 0.f))) return false;
  const float4 qi = make_float4(Bi.q[0], Bi.q[1], Bi.q[2], Bi.q[3]);
  const float4 qj = make_float4(Bj.q[0], Bj.q[1], Bj.q[2], Bj.q[3]);
  const vec3 xi = mk(Bi.x[0], Bi.x[1], Bi.x[2]), xj = mk(Bj.x[0], Bj.x[1], Bj.x[2]);
  const vec3 vx = mk(verts[3 * vert], verts[3 * vert + 1], verts[3 * vert + 2]);
  const vec3 cp_i = (flags & kJobWorld) ? vx : rotate(vx, qi) + xi;
  const vec3 wrt_j = rotate(cp_i - xj, conjugate(qj));
  float dist;
  vec3 n;
  if (Bj.type == ALV_DIST_MAP) {
    // collision_find_dist_normal (runner.hpp:1794-1825): outside the map
    // only the sign is known (no contact for a positive sign)
    dist = Bj.sign;
    n = mk(0.f, 0.f, 0.f);
    int ip[3];
    vec3 inner;
    if (grid_resolve(Bj.geom, wrt_j, ip, inner)) {
      vec3 g;
      float unused;
      dist = Bj.sign * grid_map_eval<false>(Bj.distance, nullptr, Bj.geom.res, ip, inner,
                                            Bj.geom.cs, g, unused) -
             tolerance;
      n = g * Bj.sign;
    }
  } else {
    dist = sdf_eval(Bj, wrt_j) * Bj.sign - tolerance;
    n = sdf_gradient(Bj, wrt_j, 1e-3f) * Bj.sign;
  }
  if (!(dist < 0)) return false;
  if (!Record) return true;
  n = n * (1.0f / sqrtf(length_sqr(n)));
  const vec3 cp_j = rotate(wrt_j - dist * n, qj) + xj;
  const vec3 nw = rotate(n, qj);
  const vec3 r_i = cp_i - xi, r_j = cp_j - xj;
  const vec3 u_i = mk(Bi.v[0], Bi.v[1], Bi.v[2]) + cross(mk(Bi.omega[0], Bi.omega[1], Bi.omega[2]), r_i);
  const vec3 u_j = mk(Bj.v[0], Bj.v[1], Bj.v[2]) + cross(mk(Bj.omega[0], Bj.omega[1], Bj.omega[2]), r_j);
  const vec3 u_rel = u_i - u_j;
  const float u_rel_n = dot(nw, u_rel);
  vec3 t = u_rel - u_rel_n * nw;
  if (length_sqr(t) > 1e-6f) t = t * (1.0f / sqrtf(length_sqr(t)));
  const float* Ii = inertia + 3 * i;
  const float* Ij = inertia + 3 * j;
  const float* rf = inertia + 3 * nb;
  vec3 di, oi, dj, oj;
  congruent_matrix(mk(1 / Ii[0], 1 / Ii[1], 1 / Ii[2]), qi, &di, &oi);
  congruent_matrix(mk(1 / Ij[0], 1 / Ij[1], 1 / Ij[2]), qj, &dj, &oj);
  vec3 kdi, koi, kdj, koj;
  contact_k(r_i, Bi.mass, di, oi, &kdi, &koi);
  contact_k(r_j, Bj.mass, dj, oj, &kdj, &koj);
  const vec3 kd = kdi + kdj, ko = koi + koj;
  out->i = i;
  out->j = j;
  put3(out->cp_i, cp_i);
  put3(out->cp_j, cp_j);
  put3(out->n, nw);
  put3(out->t, t);
  put3(out->iiwi_diag, di);
  put3(out->iiwi_off_diag, oi);
  put3(out->iiwj_diag, dj);
  put3(out->iiwj_off_diag, oj);
  out->friction = rf[2 * i + 1] + rf[2 * j + 1];
  out->nkninv = 1 / dot(nw, sym_apply(nw, kd, ko));
  out->pmax = 1 / dot(t, sym_apply(t, kd, ko)) * dot(u_rel, t);
  out->goalu = u_rel_n < 0 ? -(rf[2 * i] * rf[2 * j]) * u_rel_n : 0.0f;
  out->impulse_sum = 0;
  return true;
}

// Candidate c: the last job whose first candidate is not past it.
template <bool Record>
__device__ bool test_candidate(unsigned c, const ContactJob* jobs, unsigned num_jobs, unsigned nb,
                               const BoundaryDev* bodies, const float* inertia,
                               const float* verts, float tolerance, alv_contact* out) {
  unsigned lo = 0, hi = num_jobs;
  while (hi - lo > 1) {
    const unsigned mid = (lo + hi) / 2;
    if (jobs[mid].cbase <= c)
      lo = mid;
    else
      hi = mid;
  }
  const ContactJob J = jobs[lo];
  const unsigned local = c - J.cbase;
  return test_vertex<Record>(J.i, J.j + local % J.nj, J.flags, nb, bodies, inertia, verts,
                             J.vbase + local / J.nj, tolerance, out);
}

// Few candidates: one block, the hits numbered by a scan over its waves.
__global__ __launch_bounds__(kFewCandidates) void k_collision_few(
    const ContactJob* jobs, unsigned num_jobs, unsigned num_candidates, unsigned nb,
    const BoundaryDev* bodies, const float* inertia, const float* verts, float tolerance,
    unsigned max_contacts, alv_contact* contacts, unsigned* count) {
  __shared__ unsigned wave_sum[kFewCandidates / 64];
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  alv_contact rec;
  const bool hit = threadIdx.x < num_candidates &&
                   test_candidate<true>(threadIdx.x, jobs, num_jobs, nb, bodies, inertia, verts,
                                        tolerance, &rec);
  const unsigned long long mask = __ballot(hit);
  if (lane == 0) wave_sum[wave] = unsigned(__popcll(mask));
  __syncthreads();
  unsigned slot = 0;
  for (unsigned w = 0; w < wave; ++w) slot += wave_sum[w];
  if (threadIdx.x == blockDim.x - 1) count[0] = slot + wave_sum[wave];
  slot += unsigned(__popcll(mask & ((1ull << lane) - 1ull)));
  if (hit && slot < max_contacts) contacts[slot] = rec;
}

// One candidate per thread; hits[w]: the candidates 64 w ... that are inside.
// Bound by the latency of a candidate's chain of loads (job, bodies, vertex),
// which one workgroup walking the list paid once per 1,024 candidates: 45,000
// took 90 us; this pass takes 4 and the records 7.
__global__ __launch_bounds__(kContactThreads) void k_collision_hits(
    const ContactJob* jobs, unsigned num_jobs, unsigned num_candidates, unsigned nb,
    const BoundaryDev* bodies, const float* inertia, const float* verts, float tolerance,
    unsigned long long* hits) {
  const unsigned c = blockIdx.x * kContactThreads + threadIdx.x;
  const bool hit = c < num_candidates && test_candidate<false>(c, jobs, num_jobs, nb, bodies,
                                                               inertia, verts, tolerance, nullptr);
  const unsigned long long mask = __ballot(hit);
  if ((threadIdx.x & 63) == 0) hits[c / 64] = mask;
}

// A contact's slot is the number of hits before it: each block counts the
// bits before its own (8 bytes per 64 candidates, from L2); a block without
// hits does nothing but the last one, which leaves the total.
__global__ __launch_bounds__(kContactThreads) void k_collision_records(
    const ContactJob* jobs, unsigned num_jobs, unsigned num_candidates, unsigned nb,
    const BoundaryDev* bodies, const float* inertia, const float* verts, float tolerance,
    const unsigned long long* hits, unsigned max_contacts, alv_contact* contacts,
    unsigned* count) {
  __shared__ unsigned wave_sum[kContactWaves];
  const unsigned first = blockIdx.x * kContactWaves;  // the block's first word
  const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool last = blockIdx.x + 1 == gridDim.x;
  unsigned long long own = 0;
  for (unsigned w = 0; w < kContactWaves; ++w) own |= hits[first + w];
  if (own == 0 && !last) return;
  unsigned before = 0;
  for (unsigned w = threadIdx.x; w < first; w += kContactThreads) before += __popcll(hits[w]);
  for (int m = 32; m > 0; m >>= 1) before += __shfl_xor(before, m);
  if (lane == 0) wave_sum[wave] = before;
  __syncthreads();
  before = 0;
  for (unsigned w = 0; w < kContactWaves; ++w) before += wave_sum[w];
  for (unsigned w = 0; w < wave; ++w) before += __popcll(hits[first + w]);
  const unsigned long long mask = hits[first + wave];
  const unsigned slot = before + __popcll(mask & ((1ull << lane) - 1ull));
  if (((mask >> lane) & 1ull) && slot < max_contacts) {
    alv_contact rec;
    test_candidate<true>(blockIdx.x * kContactThreads + threadIdx.x, jobs, num_jobs, nb, bodies,
                         inertia, verts, tolerance, &rec);
    contacts[slot] = rec;
  }
  if (last && threadIdx.x == kContactThreads - 1) count[0] = before + __popcll(mask);
}

}  // namespace

size_t collision_hit_words(unsigned num_candidates) {
  return (size_t(num_candidates) + kContactThreads - 1) / kContactThreads * kContactWaves;
}

void launch_collision(const ContactJob* jobs, unsigned num_jobs, unsigned num_candidates,
                      unsigned nb, const BoundaryDev* bodies, const float* inertia,
                      const float* verts, float tolerance, unsigned max_contacts,
                      unsigned long long* hits, alv_contact* contacts, unsigned* count,
                      hipStream_t s) {
  if (num_candidates <= kFewCandidates) {
    hipLaunchKernelGGL(k_collision_few, dim3(1), dim3((num_candidates + 63u) / 64u * 64u), 0, s, jobs,
                       num_jobs, num_candidates, nb, bodies, inertia, verts, tolerance, max_contacts,
                       contacts, count);
    return;
  }
  const dim3 blocks(unsigned(collision_hit_words(num_candidates) / kContactWaves));
  hipLaunchKernelGGL(k_collision_hits, blocks, dim3(kContactThreads), 0, s, jobs, num_jobs,
                     num_candidates, nb, bodies, inertia, verts, tolerance, hits);
  hipLaunchKernelGGL(k_collision_records, blocks, dim3(kContactThreads), 0, s, jobs, num_jobs,
                     num_candidates, nb, bodies, inertia, verts, tolerance, hits, max_contacts,
                     contacts, count);
}

}  // namespace alv
