// kernels.hip -- CDNA4 (gfx950) kernels of the exact collision-check path.
//
//   fk_points / fk_edges : forward kinematics, one lane per configuration,
//                          frames kept in VGPRs and written once to HBM.
//                          fk_edges also marks, per group of 64 samples, the
//                          pairs that bounds over the group leave open.
//   sva                  : persistent separating-vector kernel; a wave walks
//                          pairs over 64 items with a bound test (pair operands
//                          in scalar registers) and puts what that leaves
//                          open into a ring in LDS, whose pairs its lanes then
//                          take one each through the Chung-Wang test (the
//                          scene's vertices and adjacency in LDS).
//   edge_prologue/compact: edge sample counts, and per-window compaction of
//                          the samples of still-open edges.
//
// Arithmetic follows the reference's host path operation by operation:
// the file is compiled with -ffp-contract=off (no FMA contraction), IEEE
// division and sqrt, denormals kept.  Comparisons keep the reference's
// direction so NaN behaves as it does there.
#include <hip/hip_runtime.h>

#include <cmath>

#include "glibc_trig.h"
#include "runtime.h"

namespace gprm {

namespace {

// ----------------------------------------------------------------------------
// geometry (prm/src/lib/collision4/geo4.h)
// ----------------------------------------------------------------------------
struct V3 {
  float x, y, z;
};
struct V2 {
  float x, y;
};
// trafo4 (geo4.h:22-24): columns 0..3, rows x,y,z.
struct T12 {
  float m[12];  // col c, row r at m[3*c + r]
};

__device__ __forceinline__ V3 v3(float4 a) { return V3{a.x, a.y, a.z}; }

// Pointers that a kernel loads from memory (the multi-scene task tables) are
// generic to the compiler, and their accesses flat ones, which wait for LDS
// and global memory together.  The kernels' hot accesses name the address
// space instead.
#define GAS __attribute__((address_space(1)))
typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ V3 v3(f32x4 a) { return V3{a.x, a.y, a.z}; }

// sprod (geo4.h:130-132)
__device__ __forceinline__ float dot3(const V3& u, const V3& v) {
  return (u.x * v.x + u.y * v.y) + u.z * v.z;
}
// normalize(float4&) (geo4.h:165-171)
__device__ __forceinline__ float normalize3(V3& u) {
  float norm = __builtin_sqrtf((u.x * u.x + u.y * u.y) + u.z * u.z);
  float factor = 1.0f / norm;
  if (factor == __builtin_inff()) factor = 0.0f;
  u.x *= factor;
  u.y *= factor;
  u.z *= factor;
  return norm;
}
// normalize(float2&) (geo4.h:80-83), no zero guard
__device__ __forceinline__ void normalize2(V2& u) {
  float factor = 1.0f / __builtin_sqrtf(u.x * u.x + u.y * u.y);
  u.x *= factor;
  u.y *= factor;
}
// cross2 (geo4.h:66-68)
__device__ __forceinline__ float cross2(const V2& v, const V2& w) { return v.x * w.y - v.y * w.x; }

// trafo4::apply(u, Tu) (geo4.h:215-221)
__device__ __forceinline__ V3 t_apply(const T12& t, const V3& u) {
  const float* c = t.m;
  V3 r;
  r.x = ((c[0] * u.x + c[3] * u.y) + c[6] * u.z) + c[9];
  r.y = ((c[1] * u.x + c[4] * u.y) + c[7] * u.z) + c[10];
  r.z = ((c[2] * u.x + c[5] * u.y) + c[8] * u.z) + c[11];
  return r;
}
// trafo4::apply_rot(u) (geo4.h:223-230)
__device__ __forceinline__ V3 t_apply_rot(const T12& t, const V3& u) {
  const float* c = t.m;
  V3 r;
  r.x = (c[0] * u.x + c[3] * u.y) + c[6] * u.z;
  r.y = (c[1] * u.x + c[4] * u.y) + c[7] * u.z;
  r.z = (c[2] * u.x + c[5] * u.y) + c[8] * u.z;
  return r;
}
// trafo4::apply_rot_inv(u, Rtu) (geo4.h:249-255)
__device__ __forceinline__ V3 t_apply_rot_inv(const T12& t, const V3& u) {
  const float* c = t.m;
  V3 r;
  r.x = (c[0] * u.x + c[1] * u.y) + c[2] * u.z;
  r.y = (c[3] * u.x + c[4] * u.y) + c[5] * u.z;
  r.z = (c[6] * u.x + c[7] * u.y) + c[8] * u.z;
  return r;
}
// trafo4::set(a, alpha, q, d) (geo4.h:194-203), with ca = cos(alpha) and
// sa = sin(alpha) given (the twist is constant per joint; DevRobot holds them)
__device__ __forceinline__ T12 t_set_cs(float a, float ca, float sa, float q, float d) {
  float cq = gprm_trig::cosf_ref(q), sq = gprm_trig::sinf_ref(q);
  T12 t;
  t.m[0] = cq;      t.m[3] = -sq;     t.m[6] = 0.0f;  t.m[9] = a;
  t.m[1] = sq * ca; t.m[4] = cq * ca; t.m[7] = -sa;   t.m[10] = -sa * d;
  t.m[2] = sq * sa; t.m[5] = cq * sa; t.m[8] = ca;    t.m[11] = ca * d;
  return t;
}
// this = T * this (trafo4::lapply, geo4.h:272-279)
__device__ __forceinline__ T12 t_lapply(const T12& self, const T12& T) {
  T12 r;
  for (int c = 0; c < 3; ++c) {
    V3 col = t_apply_rot(T, V3{self.m[3 * c], self.m[3 * c + 1], self.m[3 * c + 2]});
    r.m[3 * c] = col.x; r.m[3 * c + 1] = col.y; r.m[3 * c + 2] = col.z;
  }
  V3 col = t_apply(T, V3{self.m[9], self.m[10], self.m[11]});
  r.m[9] = col.x; r.m[10] = col.y; r.m[11] = col.z;
  return r;
}

// Kinematics<ndof>::calculate (kinematics.h:27-37); frames 1..ndof of item
// to the frame array, link-major and quad-planar: float4 j (0..2) of link
// frame i of item at out4[(3 i + j) stride + item], so each quad of one link
// is a contiguous array over the items.
// T0 = set(0, 0, 0, 0) (kinematics.h:27-37; trafo4::set, geo4.h:32-47),
// from cos/sin(0) held in rb
__device__ __forceinline__ T12 t_base(const DevRobot& rb) {
  const float cq = rb.c0, sq = rb.s0, ca = rb.c0, sa = rb.s0, a = 0.0f, d = 0.0f;
  T12 T;
  T.m[0] = cq;      T.m[3] = -sq;     T.m[6] = 0.0f;  T.m[9] = a;
  T.m[1] = sq * ca; T.m[4] = cq * ca; T.m[7] = -sa;   T.m[10] = -sa * d;
  T.m[2] = sq * sa; T.m[5] = cq * sa; T.m[8] = ca;    T.m[11] = ca * d;
  return T;
}

// each(i, T): called with every link frame i (1..ndof) as it is formed.
template <int NDOF, class F>
__device__ __forceinline__ void fk_store(const DevRobot& rb, const float* q, float* __restrict__ out, int item,
                                         long long stride, F each) {
  const int nd = NDOF > 0 ? NDOF : rb.ndof;
  T12 T = t_base(rb);
#pragma unroll
  for (int i = 0; i < (NDOF > 0 ? NDOF : kMaxDofDev); ++i) {
    if (NDOF == 0 && i >= nd) break;
    float qset = rb.q[i], dset = rb.d[i];
    if (rb.types[i] == 0) qset = q[i];
    else dset = q[i];
    T12 A = t_set_cs(rb.a[i], rb.ca[i], rb.sa[i], qset, dset);
    T = t_lapply(A, T);
    // quad-planar: the lanes of a wave store each quad of 64 consecutive
    // items as one contiguous 1 KB span
    float4* o = reinterpret_cast<float4*>(out) + (size_t)i * 3 * stride + item;
    o[0] = make_float4(T.m[0], T.m[1], T.m[2], T.m[3]);
    o[stride] = make_float4(T.m[4], T.m[5], T.m[6], T.m[7]);
    o[2 * stride] = make_float4(T.m[8], T.m[9], T.m[10], T.m[11]);
    each(i + 1, T);
  }
}

// Frame of link sys (1..ndof) of item from the frame array: link-major and
// quad-planar, float4 j (0..2) of link s of item i at
// frames4[((s - 1) 3 + j) stride + i].
__device__ __forceinline__ T12 load_frame(const float* __restrict__ frames, int item, long long stride, int sys) {
  const GAS f32x4* f = (const GAS f32x4*)frames + (size_t)(sys - 1) * 3 * stride + item;
  const f32x4 a = f[0], b = f[stride], c = f[2 * stride];
  T12 t;
  t.m[0] = a.x; t.m[1] = a.y; t.m[2] = a.z;  t.m[3] = a.w;
  t.m[4] = b.x; t.m[5] = b.y; t.m[6] = b.z;  t.m[7] = b.w;
  t.m[8] = c.x; t.m[9] = c.y; t.m[10] = c.z; t.m[11] = c.w;
  return t;
}

// `norm < collision_eps` and `dp >= -collision_eps` compare a float with the
// double 1e-6 (collision4.h:20,242,296).  float(1e-6) = 0x1.0c6f7ap-20 lies
// below 1e-6, so both become exact float comparisons with it.
constexpr float kEpsBelow = 0x1.0c6f7ap-20f;

// ---- bound arithmetic ------------------------------------------------------
// The bound tests' own products: they only have to stay inside the tests'
// margins, so they use fused multiply-adds.
__device__ __forceinline__ float b_dot(const V3& u, const V3& v) {
  return __builtin_fmaf(u.z, v.z, __builtin_fmaf(u.y, v.y, u.x * v.x));
}
__device__ __forceinline__ V3 b_apply(const T12& t, const V3& u) {
  const float* c = t.m;
  V3 r;
  r.x = __builtin_fmaf(c[6], u.z, __builtin_fmaf(c[3], u.y, __builtin_fmaf(c[0], u.x, c[9])));
  r.y = __builtin_fmaf(c[7], u.z, __builtin_fmaf(c[4], u.y, __builtin_fmaf(c[1], u.x, c[10])));
  r.z = __builtin_fmaf(c[8], u.z, __builtin_fmaf(c[5], u.y, __builtin_fmaf(c[2], u.x, c[11])));
  return r;
}
// A bounding sphere's radius with the bound tests' margins in it: r (1 +
// 2^-8) + 2^-9 (|c|_1 + r), c its centre in the world frame.
__device__ __forceinline__ float bound_radius(const V3& c, float r) {
  return __builtin_fmaf(r, 1.0f + 0x1p-8f, 0x1p-9f * ((fabsf(c.x) + fabsf(c.y)) + (fabsf(c.z) + r)));
}

// ---- pair masks ------------------------------------------------------------
// Which pairs does a group of 64 items (a wave) have to test at all?  For
// most pairs the bound test of the separating-vector kernel passes with room
// to spare on every item of the group, above all where the items are adjacent
// samples of an edge, whose links hardly move: on the 6-DOF roadmap's 64
// consecutive samples about 9 of 10 pairs.  The kinematics kernel, which has
// the frames in registers, decides those pairs for the whole group:
//   - per row of 16 lanes and moving polytope, the centre c and the start
//     vertex v at the row's middle item, and the largest distances mc, mv of
//     the other items' from them (row reductions);
//   - then lane l takes pair l, l + 64, ...: with D0 = vQ - vP, E0 = cQ - cP
//     of the middle items, every item's D and E lie within mv = mvP + mvQ and
//     mc = mcP + mcQ of them, so
//       D.E - (rP + rQ)|D| >= D0.E0 - mv|E0| - mc|D0| - mv mc - R (|D0| + mv),
//     R the radii with the bound test's margins.  Where that is positive (and
//     |D0| - mv > 1e-4) on all four rows, the bound test's sphere comparison
//     would pass for every item, and the pair is left out of the group's mask.
// It costs a wave about 700 instructions per group where the bound tests it
// saves are about 100 pairs of 30 to 55 each on that scene.
// With the windows of adjacent samples: the 6-DOF roadmap's edges 3.16 ->
// 2.51 ms, 20,011 local 7-DOF edges 782 -> 650 us.
struct CullTab {
  f32x4* ab;  // entry e: ab[2 e] = (centre, mc), ab[2 e + 1] = (start vertex, mv)
  float* r;   // entry e: R
  int nworld, nmov;
  int wave0;  // this wave's first entry: row k's moving polytope m at wave0 + k nmov + m
};

__device__ __forceinline__ const __attribute__((address_space(4))) f32x4* cull_polys(const SceneImg& img) {
  return (const __attribute__((address_space(4))) f32x4*)(reinterpret_cast<unsigned long long>(img.blob) +
                                                          (unsigned long long)img.off_cull);
}

// Tables of a block in its dynamic LDS, the polytopes at rest filled in.
// Every thread of the block calls it.
__device__ __forceinline__ CullTab cull_stage(const SceneImg& img, int4* lds) {
  CullTab t;
  const int entries = img.nworld + (int)(blockDim.x >> 6) * 4 * img.nmov;
  t.ab = reinterpret_cast<f32x4*>(lds);
  t.r = reinterpret_cast<float*>(t.ab + 2 * entries);
  t.nworld = img.nworld;
  t.nmov = img.nmov;
  t.wave0 = img.nworld + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) * 4 * img.nmov;
  const GAS f32x4* src = (const GAS f32x4*)(reinterpret_cast<const char*>(img.blob) + img.off_cull);
  for (int i = threadIdx.x; i < img.nworld; i += blockDim.x) {
    f32x4 c = src[2 * i];
    t.r[i] = c.w;
    c.w = 0.0f;
    t.ab[2 * i] = c;
    t.ab[2 * i + 1] = src[2 * i + 1];
  }
  __syncthreads();
  return t;
}

// x of the row's lane 8 (DPP row_newbcast), in all 16 lanes of the row.
__device__ __forceinline__ float row_middle(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x150 + 8, 0xf, 0xf, false));
}
// The largest x of the row (x >= 0), in all its lanes (DPP row_ror).
__device__ __forceinline__ float row_max(float x) {
  x = fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, false)));
  x = fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x124, 0xf, 0xf, false)));
  x = fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x122, 0xf, 0xf, false)));
  x = fmaxf(x, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x121, 0xf, 0xf, false)));
  return x;
}
// How far the row's items lie from its middle one, at most: a NaN counts as
// infinitely far; enlarged against the rounding of the positions (2^-16 of
// their magnitude) and of the distance itself.
__device__ __forceinline__ float row_reach(const V3& x, const V3& x0, float mag) {
  const V3 d{x.x - x0.x, x.y - x0.y, x.z - x0.z};
  float d2 = b_dot(d, d);
  d2 = d2 < __builtin_inff() ? d2 : __builtin_inff();
  return __builtin_fmaf(__builtin_amdgcn_sqrtf(row_max(d2)), 1.0f + 0x1p-10f, 0x1p-16f * mag);
}

// The rows' entries of link l's polytopes; every lane of the wave has a valid
// item's frame T of that link.
__device__ __forceinline__ void cull_link(const SceneImg& img, const CullTab& t, int l, const T12& T) {
  const int lane = threadIdx.x & 63;
  for (int m = img.mov_off[l]; m < img.mov_off[l + 1]; ++m) {
    const f32x4 c4 = cull_polys(img)[2 * (img.nworld + m)], v4 = cull_polys(img)[2 * (img.nworld + m) + 1];
    const V3 c = b_apply(T, v3(c4)), v = b_apply(T, v3(v4));
    const V3 c0{row_middle(c.x), row_middle(c.y), row_middle(c.z)};
    const V3 v0{row_middle(v.x), row_middle(v.y), row_middle(v.z)};
    const float mag = (fabsf(c0.x) + fabsf(c0.y)) + (fabsf(c0.z) + c4.w);
    const float mc = row_reach(c, c0, mag), mv = row_reach(v, v0, mag);
    if ((lane & 15) == 0) {
      const int e = t.wave0 + (lane >> 4) * t.nmov + m;
      t.ab[2 * e] = f32x4{c0.x, c0.y, c0.z, mc};
      t.ab[2 * e + 1] = f32x4{v0.x, v0.y, v0.z, mv};
      t.r[e] = __builtin_fmaf(c4.w, 1.0f + 0x1p-8f, 0x1p-9f * (mag + 2.0f * mc));
    }
  }
}

// The group's mask words, after cull_link of every link.
__device__ __forceinline__ void cull_pairs(const SceneImg& img, const CullTab& t, unsigned long long* __restrict__ mask,
                                           int group) {
  const int lane = threadIdx.x & 63;
  // the entries were written by other lanes of this wave
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  const GAS int* cpairs = (const GAS int*)(reinterpret_cast<const char*>(img.blob) + img.off_cpairs);
  const int nw = (img.M + 63) >> 6;
  for (int w = 0; w < nw; ++w) {
    const int pair = 64 * w + lane;
    const int cp = cpairs[pair < img.M ? pair : 0];
    const int p = cp & 0xffff, q = (int)((unsigned)cp >> 16);
    const int pe = p < t.nworld ? p : t.wave0 + (p - t.nworld), ps = p < t.nworld ? 0 : t.nmov;
    const int qe = q < t.nworld ? q : t.wave0 + (q - t.nworld), qs = q < t.nworld ? 0 : t.nmov;
    bool far = true;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int ip = pe + k * ps, iq = qe + k * qs;
      const f32x4 pc = t.ab[2 * ip], pv = t.ab[2 * ip + 1], qc = t.ab[2 * iq], qv = t.ab[2 * iq + 1];
      const V3 E{qc.x - pc.x, qc.y - pc.y, qc.z - pc.z}, D{qv.x - pv.x, qv.y - pv.y, qv.z - pv.z};
      const float mc = qc.w + pc.w, mv = qv.w + pv.w, R = t.r[ip] + t.r[iq];
      const float ne = __builtin_amdgcn_sqrtf(b_dot(E, E)), nd = __builtin_amdgcn_sqrtf(b_dot(D, D));
      float lhs = b_dot(D, E);
      lhs = __builtin_fmaf(-mv, ne, lhs);
      lhs = __builtin_fmaf(-mc, nd + mv, lhs);
      far = far & (lhs > R * (nd + mv)) & (nd - mv > 1e-4f);
    }
    const unsigned long long m = __ballot((pair < img.M) & !far);
    if (lane == 0) mask[(size_t)group * nw + w] = m;
  }
}

// ----------------------------------------------------------------------------
// kinematics kernels
// ----------------------------------------------------------------------------
// Point mode result word of one configuration: ((pair+1) << 4) | (code+1)
// of the first colliding pair in CRS order (updated by atomicMin), kWordFree
// while none is known; out of bounds is (0 << 4) | (1+1).
constexpr int kWordFree = 0x7fffffff;
constexpr int kWordOutOfBounds = 2;

template <int NDOF>
__global__ void __launch_bounds__(kFkBlock)
    fk_points_kernel(DevRobot rb, const float* __restrict__ q, long long offset, int n,
                     float* __restrict__ frames, long long fstride, int* __restrict__ word, int check_bounds,
                     unsigned* __restrict__ zero_counter, const unsigned char* __restrict__ skip,
                     int* __restrict__ group_done) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  // the separating-vector launch that follows claims units from these counters
  // and counts completed units per group of 64 items in group_done
  if (zero_counter != nullptr && i < kSvaQueues) zero_counter[i * kSvaQueueStride] = 0u;
  if (group_done != nullptr && (i & 63) == 0 && i < n) group_done[i >> 6] = 0;
  if (i >= n) return;
  const int nd = NDOF > 0 ? NDOF : rb.ndof;
  float qq[kMaxDofDev];
#pragma unroll
  for (int j = 0; j < (NDOF > 0 ? NDOF : kMaxDofDev); ++j)
    if (NDOF > 0 || j < nd) qq[j] = q[i + offset * j];
  if (skip != nullptr && skip[i]) {
    word[i] = kWordOutOfBounds;
  } else if (check_bounds) {
    // check_boundaries(q) (robotconfigspace.cpp:795-802)
    int st = 0;
    for (int j = 0; j < nd; ++j)
      if (qq[j] < rb.mins[j] || qq[j] > rb.maxs[j]) { st = 1; break; }
    word[i] = st ? kWordOutOfBounds : kWordFree;
  } else {
    word[i] = kWordFree;
  }
  fk_store<NDOF>(rb, qq, frames, i, fstride, [](int, const T12&) {});
}

// The frames of n configurations as Kinematics<ndof>::calculate leaves its
// trafos (kinematics.h:28-37): the base frame and the link frames the
// kinematics kernel stored, unpacked to out[(i (ndof + 1) + s) 12 + m] with
// m = 3 column + row (trafo4's four columns of x, y, z).
__global__ void __launch_bounds__(256)
    frames_unpack_kernel(DevRobot rb, const float* __restrict__ frames, long long fstride, int n,
                         float* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  float* o = out + (size_t)i * (rb.ndof + 1) * 12;
  const T12 T0 = t_base(rb);
  for (int m = 0; m < 12; ++m) o[m] = T0.m[m];
  for (int s = 1; s <= rb.ndof; ++s) {
    const T12 t = load_frame(frames, i, fstride, s);
    for (int m = 0; m < 12; ++m) o[12 * s + m] = t.m[m];
  }
}

// codes[i] from the point mode result word.
__global__ void finalize_points_kernel(const int* __restrict__ word, int* __restrict__ codes, int n) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int w = word[i];
  codes[i] = w == kWordFree ? 0 : (w & 15) - 1;
}

// Frames of item i of an edge round to slot `slot`: sample item_pos[i] of its
// edge, interpolated as robotconfigspace.cpp:406-420 does (c1 = s/(T-1),
// c2 = 1 - c1, q = c1 qs + c2 qe), then the kinematics.
template <int NDOF, class F>
__device__ __forceinline__ void fk_edge_item(const DevRobot& rb, const EdgeArgs& ea, const int* __restrict__ item_edge,
                                             const int* __restrict__ item_pos, int i, int slot,
                                             float* __restrict__ frames, long long fstride, F each) {
  const int nd = NDOF > 0 ? NDOF : rb.ndof;
  const int e = item_edge[i] & ~kItemPad;
  const int s = item_pos[i];
  const int T = ea.testnum[e];
  float c1, c2;
  if (T > 0) {
    c1 = (float)s / (float)(T - 1);
    c2 = 1.0f - c1;
  } else {
    c1 = 1.0f;
    c2 = 0.0f;
  }
  float qq[kMaxDofDev];
#pragma unroll
  for (int j = 0; j < (NDOF > 0 ? NDOF : kMaxDofDev); ++j)
    if (NDOF > 0 || j < nd) qq[j] = c1 * ea.qs[e + ea.offset * j] + c2 * ea.qe[e + ea.offset * j];
  fk_store<NDOF>(rb, qq, frames, slot, fstride, each);
}

// Kinematics (and pair masks) of items [0, n), the grid striding over them
// in whole groups of 64; the last group's lanes past the end take the last
// item (in bounds: the planes hold whole groups), so that the wave's
// reductions see valid items only.
template <int NDOF>
__device__ __forceinline__ void fk_edge_items(const DevRobot& rb, const EdgeArgs& ea, const int* __restrict__ item_edge,
                                              const int* __restrict__ item_pos, int n, int first, int step,
                                              float* __restrict__ frames, long long fstride, const SceneImg& img,
                                              unsigned long long* __restrict__ mask, int4* smem) {
  CullTab tab{};
  if (mask != nullptr) tab = cull_stage(img, smem);
  for (int slot = first; (slot & ~63) < n; slot += step) {
    const int i = slot < n ? slot : n - 1;
    if (mask == nullptr) {
      fk_edge_item<NDOF>(rb, ea, item_edge, item_pos, i, slot, frames, fstride, [](int, const T12&) {});
    } else {
      fk_edge_item<NDOF>(rb, ea, item_edge, item_pos, i, slot, frames, fstride,
                         [&](int l, const T12& T) { cull_link(img, tab, l, T); });
      cull_pairs(img, tab, mask, slot >> 6);
    }
  }
}

template <int NDOF>
__global__ void __launch_bounds__(kFkBlock)
    fk_edges_kernel(DevRobot rb, EdgeArgs ea, const int* __restrict__ item_edge,
                    const int* __restrict__ item_pos, const int* __restrict__ nitems_dev, int cap,
                    float* __restrict__ frames, long long fstride, SceneImg img,
                    unsigned long long* __restrict__ mask) {
  extern __shared__ int4 smem[];
  int n = *nitems_dev;
  if (n > cap) n = cap;
  fk_edge_items<NDOF>(rb, ea, item_edge, item_pos, n, blockIdx.x * blockDim.x + threadIdx.x, gridDim.x * blockDim.x,
                      frames, fstride, img, mask, smem);
}

// testnum (robotconfigspace.cpp:660-673).
template <int BLOCK>
__device__ __forceinline__ void edge_prologue_one(int ndof, float dq, const EdgeArgs& ea, int k,
                                                  int* __restrict__ testnum,
                                                  int* __restrict__ max_testnum,
                                                  unsigned long long* __restrict__ total, bool only = false) {
  int T = 0;
  if (k < ea.nedges && ea.skip != nullptr && ea.skip[k]) {
    testnum[k] = 0;
    ea.edge_res[k] = kEdgeSkipped;
  } else if (k < ea.nedges) {
    float norm = 0.0f;
    for (int i = 0; i < ndof; ++i) {
      float diff = ea.qe[k + ea.offset * i] - ea.qs[k + ea.offset * i];
      norm += diff * diff;
    }
    norm = __builtin_sqrtf(norm);
    // an undefined length (NaN) is one sample, an infinite one none
    const float steps = norm / dq;
    T = steps >= 0x1p31f ? 0 : steps == steps ? (int)steps + 1 : 1;
    testnum[k] = T;
    ea.edge_res[k] = 0;
  }
  // One atomic pair per block: same-address atomics from all CUs serialise
  // at the memory side (about 15 ns each), and one pair per wave took 45 us
  // for 100k edges.  Every thread of the block calls this function (threads
  // past the edges bring T = 0).
  __shared__ int s_max[BLOCK / 64];
  __shared__ unsigned long long s_sum[BLOCK / 64];
  int tmax = T;
  unsigned long long tsum = (unsigned long long)T;
  for (int d = 32; d >= 1; d >>= 1) {
    tmax = max(tmax, __shfl_xor(tmax, d, 64));
    tsum += __shfl_xor(tsum, d, 64);
  }
  if ((threadIdx.x & 63) == 0) {
    s_max[threadIdx.x >> 6] = tmax;
    s_sum[threadIdx.x >> 6] = tsum;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < BLOCK / 64; ++w) {
      tmax = max(tmax, s_max[w]);
      tsum += s_sum[w];
    }
    if (only) {
      *max_testnum = tmax;
      *total = tsum;
    } else if (tmax > 0) {
      atomicMax(max_testnum, tmax);
      atomicAdd(total, tsum);
    }
  }
}

// The block that finishes last leaves the totals in pinned memory, so that the
// host waits for this launch and nothing more.  (With an event, a copy on a
// second stream and a wait for that, calls of short edges, which are one round,
// took 108-138 us where 75-105 are enough: 32 edges of 0.08 rad on the 4-DOF
// scene 113 and 81 us.)
__global__ void __launch_bounds__(kPrologueBlock)
    edge_prologue_kernel(int ndof, float dq, EdgeArgs ea, int* __restrict__ testnum, int* max_testnum,
                         unsigned long long* total, unsigned* blocks, EdgePinned* host) {
  const bool only = gridDim.x == 1;
  edge_prologue_one<kPrologueBlock>(ndof, dq, ea, blockIdx.x * kPrologueBlock + threadIdx.x, testnum, max_testnum,
                                    total, only);
  if (host == nullptr || threadIdx.x != 0) return;
  if (!only) {
    __threadfence();
    if (atomicAdd(blocks, 1u) != gridDim.x - 1) return;
    __threadfence();
  }
  host->maxT = only ? *max_testnum : atomicMax(max_testnum, 0);
  host->total = only ? *total : atomicAdd(total, 0ull);
}

// Items for ranks [r0, r1) in the window [l0, l1) of every open edge, an edge's
// samples in ascending order on consecutive slots.  Runs of more than kRunShort
// samples start at a multiple of 16 and are padded to one (edge_run_slots);
// the block's short runs follow them packed, padded together.  Padding items
// repeat a sample, so that the rows' pair masks see valid items only, and are
// marked (kItemPad): the separating-vector kernel leaves them out.
// One atomic per block reserves the block's slots (same-address atomics
// serialise at the memory side; one per wave took 23 us for 100k edges);
// each lane's slots follow by prefix count.  Every thread of the block calls
// it; threads with e >= e1 contribute nothing.
template <int BLOCK>
__device__ __forceinline__ void edge_compact_one(const EdgeArgs& ea, int e, int e1, int l0, int l1, int r0, int r1,
                                                 int* __restrict__ item_edge, int* __restrict__ item_pos, int cap,
                                                 int* __restrict__ nitems, int* __restrict__ nsamples,
                                                 int* __restrict__ overflow) {
  int a = 1, b = 0, cnt = 0;
  if (e < e1 && __hip_atomic_load(&ea.edge_res[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0)
    edge_window(ea.testnum[e], l0, l1, &a, &b, &cnt);
  cnt = max(min(cnt, r1) - r0, 0);
  const bool is_short = cnt <= kRunShort;
  // prefix sums of the long runs' slots, the short runs' and the samples
  int lng = is_short ? 0 : (int)edge_run_slots(cnt), shr = is_short ? cnt : 0, smp = cnt;
  const int slots = lng;
  const int lane = threadIdx.x & 63;
  for (int d = 1; d < 64; d <<= 1) {
    const int u = __shfl_up(lng, d, 64), v = __shfl_up(shr, d, 64), x = __shfl_up(smp, d, 64);
    if (lane >= d) {
      lng += u;
      shr += v;
      smp += x;
    }
  }
  __shared__ int s_long[BLOCK / 64], s_short[BLOCK / 64], s_smp[BLOCK / 64];
  __shared__ int s_base, s_short0, s_shorts;
  const int w = threadIdx.x >> 6;
  if (lane == 63) {
    s_long[w] = lng;
    s_short[w] = shr;
    s_smp[w] = smp;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    int sl = 0, ss = 0, sn = 0;
    for (int i = 0; i < BLOCK / 64; ++i) {
      const int u = s_long[i], v = s_short[i];
      s_long[i] = sl;
      s_short[i] = ss;
      sl += u;
      ss += v;
      sn += s_smp[i];
    }
    const int total = sl + (ss + 15) / 16 * 16;
    s_base = total > 0 ? atomicAdd(nitems, total) : 0;
    s_short0 = sl;
    s_shorts = ss;
    if (nsamples != nullptr && sn > 0) atomicAdd(nsamples, sn);
    if (overflow != nullptr && s_base > cap - total) *overflow = 1;
  }
  __syncthreads();
  // first slot of the lane's run, and the end of its padding: the block's
  // last short run pads for all of them
  const int o = s_base + (is_short ? s_short0 + s_short[w] + shr - cnt : s_long[w] + lng - slots);
  int fill = is_short ? cnt : slots;
  if (is_short && cnt > 0 && s_short[w] + shr == s_shorts) fill += (s_shorts + 15) / 16 * 16 - s_shorts;
  // Four runs at a time, one to each row of 16 lanes, so that every store
  // instruction covers four spans of consecutive slots.
  unsigned long long runs = __ballot(cnt > 0);
  const int row = lane >> 4, col = lane & 15;
  while (runs) {
    int src = -1;
    for (int k = 0; k < 4 && runs; ++k) {
      const int t = __builtin_ctzll(runs);
      runs &= runs - 1;
      if (k == row) src = t;
    }
    const int from = src < 0 ? 0 : src;
    const int c = __shfl(cnt, from, 64), f = __shfl(fill, from, 64), os = __shfl(o, from, 64), es = __shfl(e, from, 64);
    const int as = __shfl(a, from, 64), bs = __shfl(b, from, 64);
    if (src < 0) continue;
    for (int t = col; t < f && os + t < cap; t += 16) {
      item_edge[os + t] = t < c ? es : es | kItemPad;
      item_pos[os + t] = edge_window_sample(as, bs, r0 + (t < c ? t : c - 1));
    }
  }
}

__global__ void __launch_bounds__(kCompactBlock)
    edge_compact_kernel(EdgeArgs ea, EdgeLaunch p, int* __restrict__ item_edge, int* __restrict__ item_pos,
                        int* __restrict__ nitems, int* __restrict__ nsamples, unsigned* __restrict__ zero_queues,
                        int slice, int* __restrict__ overflow) {
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < kSvaQueues) zero_queues[threadIdx.x * kSvaQueueStride] = 0u;
  const int r0 = p.r0 + (int)blockIdx.y * slice;
  edge_compact_one<kCompactBlock>(ea, p.e0 + blockIdx.x * kCompactBlock + threadIdx.x, p.e1, p.l0, p.l1, r0,
                                  r0 + min(slice, p.r1 - r0), item_edge, item_pos, p.cap, nitems, nsamples,
                                  overflow);
}

// Multi-scene edge calls: one task per scene (prologue) or per scene part of
// a launch step (compaction, kinematics); block b of a grid belongs to the
// last task whose first block (block0 for the prologue and the compaction,
// fblock0 for the kinematics) is <= b.
template <bool FK>
__device__ __forceinline__ const EdgeTask& edge_task_of(const EdgeTask* __restrict__ tasks, int ntasks) {
  int lo = 0, hi = ntasks - 1;
  const int b = blockIdx.x;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if ((FK ? tasks[mid].fblock0 : tasks[mid].block0) <= b) lo = mid;
    else hi = mid - 1;
  }
  return tasks[lo];
}

__global__ void __launch_bounds__(256) edge_prologue_multi_kernel(const EdgeTask* __restrict__ tasks, int ntasks) {
  const EdgeTask& T = edge_task_of<false>(tasks, ntasks);
  edge_prologue_one<256>(T.rb.ndof, T.dq, T.ea, (blockIdx.x - T.block0) * 256 + threadIdx.x, T.testnum,
                         T.max_testnum, T.total);
}

__global__ void __launch_bounds__(kCompactBlockMulti)
    edge_compact_multi_kernel(const EdgeTask* __restrict__ tasks, int ntasks) {
  const EdgeTask& T = edge_task_of<false>(tasks, ntasks);
  const int xblocks = (T.e1 - T.e0 + kCompactBlockMulti - 1) / kCompactBlockMulti;
  const int y = (int)(blockIdx.x - T.block0) / xblocks, x = (int)(blockIdx.x - T.block0) - y * xblocks;
  const int r0 = T.r0 + y * T.slice;
  edge_compact_one<kCompactBlockMulti>(T.ea, T.e0 + x * kCompactBlockMulti + threadIdx.x, T.e1, T.l0, T.l1, r0,
                                       r0 + min(T.slice, T.r1 - r0), T.item_edge, T.item_pos, T.cap, T.nitems,
                                       nullptr, nullptr);
}

template <int NDOF>
__global__ void __launch_bounds__(kFkBlock) fk_edges_multi_kernel(const EdgeTask* __restrict__ tasks, int ntasks) {
  extern __shared__ int4 smem[];
  const EdgeTask& T = edge_task_of<true>(tasks, ntasks);
  int n = *T.nitems;
  if (n > T.cap) n = T.cap;
  // one pass: the task's blocks cover its capacity
  fk_edge_items<NDOF>(T.rb, T.ea, T.item_edge, T.item_pos, n, (blockIdx.x - T.fblock0) * kFkBlock + threadIdx.x,
                      0x40000000, T.frames, (long long)T.cap, T.img, T.mask, smem);
}

// ---- cell index for the radius search -------------------------------------
// Nodes are binned by their first g.dims coordinates into cells at least D
// wide, so every node within D of a query lies in the 3^dims cells around the
// query's own cell.  The index is a counting sort: per-cell counts, their
// exclusive scan, and a scatter of the coordinates (SoA, stride n) and node
// ids into cell order.


__global__ void grid_count_kernel(CellGrid g, const float* __restrict__ nodes, int n, long long noff,
                                  int* __restrict__ cell_id, int* __restrict__ counts) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= n) return;
  int c = 0;
  for (int d = g.dims - 1; d >= 0; --d) c = c * g.cells[d] + grid_coord(g, d, nodes[l + noff * d]);
  cell_id[l] = c;
  atomicAdd(&counts[c], 1);
}

// Exclusive scan of counts[0, ncells) into starts and cursor (one block of 1024).
__global__ void __launch_bounds__(1024) grid_scan_kernel(const int* __restrict__ counts, int* __restrict__ starts,
                                                         int* __restrict__ cursor, int ncells) {
  __shared__ int part[1024];
  const int t = threadIdx.x;
  const int per = (ncells + 1023) / 1024;
  const int c0 = min(ncells, t * per), c1 = min(ncells, c0 + per);
  int sum = 0;
  for (int c = c0; c < c1; ++c) sum += counts[c];
  part[t] = sum;
  __syncthreads();
  for (int o = 1; o < 1024; o <<= 1) {  // inclusive Hillis-Steele scan of the partial sums
    const int v = t >= o ? part[t - o] : 0;
    __syncthreads();
    part[t] += v;
    __syncthreads();
  }
  int run = part[t] - sum;
  for (int c = c0; c < c1; ++c) {
    starts[c] = run;
    cursor[c] = run;
    run += counts[c];
  }
}

__global__ void grid_scatter_kernel(int ndof, const float* __restrict__ nodes, int n, long long noff,
                                    const int* __restrict__ cell_id, int* __restrict__ cursor,
                                    float* __restrict__ sorted, int* __restrict__ sid) {
  const int l = blockIdx.x * blockDim.x + threadIdx.x;
  if (l >= n) return;
  const int pos = atomicAdd(&cursor[cell_id[l]], 1);
  for (int i = 0; i < ndof; ++i) sorted[pos + (size_t)n * i] = nodes[l + noff * i];
  sid[pos] = l;
}

constexpr int pow3(int d) { return d == 0 ? 1 : 3 * pow3(d - 1); }
constexpr int kNeighbourCells = pow3(kGridDims);
static_assert(kNeighbourCells <= 256, "one thread per neighbour cell in a 256-thread block");

// Radius search over the cell index (get_near_vertices,
// prm/src/lib/prm/prmsolver.cpp:2532-2574): one block per query; the nodes
// of the (up to 3^kGridDims) neighbouring cells form one index range that the
// block's threads stride through.  |q_l - query_j|^2 < D^2 in float with the
// reference's summation order.
//
// Two passes: WRITE 0 counts each query's matches, a scan gives each query its
// place in the output, and WRITE 1 finds the matches again and writes them
// there, in node order if they fit the stage (kNearStage), so that the pairs
// come out sorted by (query, node).  Appending with one atomic per wave took
// 426 us for 20,000 queries among as many nodes (50,000 atomics on one
// address); the two passes and the scan take 65 + 72 + 31.
constexpr int kNearStage = 1024;
template <int WRITE>
__global__ void __launch_bounds__(256)
    near_grid_kernel(int ndof, const float* __restrict__ queries, int nq, long long qoff, CellGrid g,
                     const int* __restrict__ starts, const int* __restrict__ counts, const float* __restrict__ sorted,
                     const int* __restrict__ sid, int n, float D2, int* __restrict__ qcount,
                     const long long* __restrict__ qstart, int* __restrict__ out_q, int* __restrict__ out_node,
                     float* __restrict__ out_d2, int cap) {
  constexpr int NK = kNeighbourCells;
  __shared__ int s_start[NK], s_pre[256 + 1], s_wave[4], s_found;
  __shared__ int s_node[WRITE ? kNearStage : 1];
  __shared__ float s_d2[WRITE ? kNearStage : 1];
  const int j = blockIdx.x;
  if (j >= nq) return;
  const int matches = WRITE ? qcount[j] : 0;
  if (WRITE && matches == 0) return;
  float qr[kMaxDofDev];
  for (int i = 0; i < ndof; ++i) qr[i] = queries[j + qoff * i];
  int here = 0;
  if (threadIdx.x < NK) {
    // neighbour k: offset digit[d] - 1 in grid dimension d; a dimension
    // without grid (d >= dims) takes only offset 0; a cell whose faces lie
    // D or more from the query is skipped (cell_gap2)
    int digit[kGridDims];
    for (int d = 0, rem = threadIdx.x; d < kGridDims; ++d, rem /= 3) digit[d] = rem % 3;
    int c = 0;
    bool ok = true;
    float lb = 0.0f;
    for (int d = kGridDims - 1; d >= 0; --d) {
      if (d >= g.dims) {
        if (digit[d] != 1) ok = false;
        continue;
      }
      const int x = grid_coord(g, d, qr[d]) + digit[d] - 1;
      if (x < 0 || x >= g.cells[d]) ok = false;
      c = c * g.cells[d] + x;
      lb += cell_gap2(g, d, qr[d], digit[d]);
    }
    if (lb >= D2) ok = false;
    s_start[threadIdx.x] = ok ? starts[c] : 0;
    here = ok ? counts[c] : 0;
  }
  // s_pre: the cells' exclusive prefix sums
  const int lane = threadIdx.x & 63;
  for (int d = 1; d < 64; d <<= 1) {
    const int v = __shfl_up(here, d, 64);
    if (lane >= d) here += v;
  }
  if (lane == 63) s_wave[threadIdx.x >> 6] = here;
  if (threadIdx.x == 0) {
    s_pre[0] = 0;
    s_found = 0;
  }
  __syncthreads();
  for (int w = 0; w < (int)(threadIdx.x >> 6); ++w) here += s_wave[w];
  s_pre[threadIdx.x + 1] = here;
  __syncthreads();
  const int total = s_pre[NK];
  const long long place = WRITE ? qstart[j] : 0;
  const bool staged = WRITE && matches <= kNearStage;
  int mine = 0;
  for (int base = 0; base < total; base += blockDim.x) {
    const int idx = base + threadIdx.x;
    float normsq = 0.0f;
    bool hit = false;
    int node = 0;
    if (idx < total) {
      // the neighbour cell holding idx: last k with s_pre[k] <= idx
      int k = 0;
      for (int step = 128; step > 0; step >>= 1)
        if (k + step < NK && s_pre[k + step] <= idx) k += step;
      const int pos = s_start[k] + (idx - s_pre[k]);
      node_dist2<1>(sorted, (size_t)n, &pos, ndof, qr, &normsq);
      hit = normsq < D2;
      if (WRITE) node = sid[pos];
    }
    if (!WRITE) {
      mine += hit ? 1 : 0;
      continue;
    }
    if (hit) {
      const int o = atomicAdd(&s_found, 1);  // in LDS; the compiler adds once per wave
      if (staged) {
        s_node[o] = node;
        s_d2[o] = normsq;
      } else if (place + o < cap) {
        out_q[place + o] = j;
        out_node[place + o] = node;
        out_d2[place + o] = normsq;
      }
    }
  }
  if (!WRITE) {
    for (int d = 32; d > 0; d >>= 1) mine += __shfl_xor(mine, d, 64);
    if (lane == 0 && mine > 0) atomicAdd(&s_found, mine);
    __syncthreads();
    if (threadIdx.x == 0) qcount[j] = s_found;
  } else if (staged) {
    // each match to its rank among the query's nodes
    __syncthreads();
    for (int t = threadIdx.x; t < matches; t += blockDim.x) {
      const int node = s_node[t];
      int rank = 0;
      for (int u = 0; u < matches; ++u) rank += s_node[u] < node ? 1 : 0;
      if (place + rank < cap) {
        out_q[place + rank] = j;
        out_node[place + rank] = node;
        out_d2[place + rank] = s_d2[t];
      }
    }
  }
}

// Exclusive scan of the queries' match counts, *total their sum (one block).
__global__ void __launch_bounds__(1024)
    near_scan_kernel(const int* __restrict__ qcount, int nq, long long* __restrict__ qstart,
                     long long* __restrict__ total) {
  __shared__ long long s_wave[16];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  long long base = 0;
  for (int j0 = 0; j0 < nq; j0 += 1024) {
    const int j = j0 + (int)threadIdx.x;
    const long long own = j < nq ? qcount[j] : 0;
    long long incl = own;
    for (int d = 1; d < 64; d <<= 1) {
      const long long v = __shfl_up(incl, d, 64);
      if (lane >= d) incl += v;
    }
    if (lane == 63) s_wave[w] = incl;
    __syncthreads();
    long long before = 0, all = 0;
    for (int i = 0; i < 16; ++i) {
      before += i < w ? s_wave[i] : 0;
      all += s_wave[i];
    }
    if (j < nq) qstart[j] = base + before + incl - own;
    base += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) *total = base;
}

__global__ void fill_i32_kernel(int* p, int v, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}
__global__ void fill_u32_kernel(unsigned int* p, unsigned int v, long long n) {
  for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
    p[i] = v;
}

// ----------------------------------------------------------------------------
// separating-vector kernel
// ----------------------------------------------------------------------------

// Scene image as staged in LDS (layout documented at SceneImg).
struct Lds {
  const float4* verts;          // (x, y, z, info bits): info = row offset << 8 | degree
  const int4* pairs;            // (vbP | vbQ << 16, sysP | sysQ << 8, CRS index, kP | kQ << 16)
  const int2* hulls;            // per polytope: vertex count, certificate factor (support)
  const unsigned short* adj;    // rows of 4k neighbour ids, padded with the row's own vertex
};

// A lane's iteration history R[k] (x, y, z) and combs[k] (w: p | q << 16);
// only iterations that do not separate touch it.  The first n entries are in
// LDS (as many as fit beside the launch's resident blocks, history_entries),
// the others in global memory, where a wave's kMaxIter entries are one 10 KB
// block.
// Lanes are adjacent in both.  Every iteration reads all entries before it,
// two at a time: in memory, with entry k of all lanes of the launch together,
// each read was a trip to the L2 and often to another page.  (3,001 points of
// the 7-DOF scene 76 -> 72 us, of which 1 by the blocks; 16 scenes 1.81 -> 1.73
// ms, the 6-DOF roadmap's edges 2.11 -> 2.02 ms.)
constexpr int kHistStride = 64;
struct History {
  f32x4* l;  // LDS, entries ls apart
  int n, ls;
  GAS f32x4* g;  // global memory, entries kHistStride apart
};
__device__ __forceinline__ History lane_history(float4* hist, unsigned thread, f32x4* lds, int n, int ls) {
  return History{lds, n, ls,
                 (GAS f32x4*)hist + (size_t)(thread >> 6) * (size_t)(kMaxIter * kHistStride) + (thread & 63)};
}

__device__ __forceinline__ int info_of(const float4& r) { return __float_as_int(r.w); }

// support_vertex_searcher::search_support_vertex (collision4.h:66-103):
// first improvement over the stored neighbour order, restart at the new
// vertex.  A vertex's neighbours are read 4 at a time with independent loads;
// the first of them (in stored order) whose value exceeds the current maximum
// is the sequential scan's move, found as the lowest set bit of a compare
// mask.  The new maximum is recomputed from the same operands, so it is the
// same float the scan would keep.
__device__ __forceinline__ int climb(const Lds& L, int p, const V3& dir) {
  float4 rec = L.verts[p];
  float mx = dot3(v3(rec), dir);
  int info = info_of(rec);
  int c = 0;
  for (;;) {
    const int off = info >> 8, cnt = info & 255;
    if (c >= cnt) break;
    const uint2 ids = *reinterpret_cast<const uint2*>(L.adj + off + c);
    const float4 r0 = L.verts[ids.x & 0xffff], r1 = L.verts[ids.x >> 16];
    const float4 r2 = L.verts[ids.y & 0xffff], r3 = L.verts[ids.y >> 16];
    // padding entries are the vertex itself: same operands, same value, never > mx
    unsigned bits = (dot3(v3(r0), dir) > mx) ? 1u : 0u;
    bits |= (dot3(v3(r1), dir) > mx) ? 2u : 0u;
    bits |= (dot3(v3(r2), dir) > mx) ? 4u : 0u;
    bits |= (dot3(v3(r3), dir) > mx) ? 8u : 0u;
    if (bits) {
      const unsigned long long packed = ((unsigned long long)ids.y << 32) | ids.x;
      p = (int)((packed >> (16 * __builtin_ctz(bits))) & 0xffff);
      rec = L.verts[p];
      mx = dot3(v3(rec), dir);
      info = info_of(rec);
      c = 0;
    } else {
      c += 4;
    }
  }
  return p;
}

// The vertex that climb(L, p, dir) ends at, for the polytope k whose vertices
// start at v0.  The climb is a chain of dependent reads and takes as many
// steps as the wave's slowest lane; instead the lanes read all vertices of
// their polytope, which depend on nothing, and keep the largest product and
// the next one.  Where they are further apart than the certificate asks
// (support_factor_kernel: then the climb, from any start and in
// its own rounding, ends at the largest), that vertex is the answer; else the
// climb runs.  The scan's products only have to stay inside the certificate.
// 9 vector instructions a vertex against about 65 a climb step (4M points of
// the 7-DOF scene 3.57 -> 3.33 ms, 65,536 points of the 4-DOF scene 71.5 ->
// 67.9 us, one configuration's call 34 -> 31 us).
__device__ __forceinline__ int support(const Lds& L, int k, int v0, int p, const V3& dir) {
  const int2 hull = L.hulls[k];
  float best = -__builtin_inff(), second = -__builtin_inff();
  int at = 0, i = 0;
  const float4* v = L.verts + v0;
  auto take = [&](const float4& r, int j) {
    const float d = b_dot(v3(r), dir);
    second = __builtin_amdgcn_fmed3f(second, best, d);
    at = d > best ? j : at;
    best = fmaxf(best, d);
  };
  for (; i + 4 <= hull.x; i += 4) {
    const float4 r0 = v[i], r1 = v[i + 1], r2 = v[i + 2], r3 = v[i + 3];
    take(r0, i);
    take(r1, i + 1);
    take(r2, i + 2);
    take(r3, i + 3);
  }
  for (; i < hull.x; ++i) take(v[i], i);
  const float need = __int_as_float(hull.y) * ((fabsf(dir.x) + fabsf(dir.y)) + fabsf(dir.z)) + 1e-30f;
  // (false for a NaN, too; need < 1e20 keeps the products far from overflow)
  if ((best - second > need) & (need < 1e20f)) return v0 + at;
  return climb(L, p, dir);
}

// Certificate factors of the polytopes' support scans (support):
// with w the vertex whose product with a direction d is largest, by more than
// factor |d|_1 above every other vertex's, the hill climb in floats ends at w
// from any start; inf if that cannot be promised, or if the climb is the
// cheaper way (more vertices than kScanVertices).
//   The polytope lies in the cone of the stored neighbours' edges e_i at each
// vertex u: w - u = sum l_i e_i, l_i >= 0.  So (w - u).d <= (sum l_i) max e_i.d,
// and u has a neighbour better by (w - u).d / L, L the largest sum l_i over
// all u and w.  The climb's products err by at most g = 3.1 2^-24 vmax |d|_1
// each, the scan's too: it suffices that the scan's margin exceeds
// (2 L + 2) g.  The coefficients are checked here from the stored adjacency,
// so a row that misses edges has no factor.
//   Faces of more than three vertices are not quite plane in floats, so a
// vertex of a face may lie outside the cone by a rounding error.  A negative
// coefficient -m adds at most m |e_i.d| <= 2 m vmax |d|_1, and counts as
// m kScanOutside of sum l_i.  (Refusing any negative one left most boxes to the
// climb: 65,536 points of the 4-DOF scene 66 against 62.5 us so.)
//   A block computes one polytope's factor, 32 lanes a vertex u's part of it:
// each lane inverts one cone (e_i, e_j, e_k) at a time, kCertCones of them go
// to LDS, and every lane tries them for its own vertex w, until all w have a
// sum of at most 4, which need not be bettered.  On the host, pair after pair,
// the 256 polytopes of 32 vertices of a large scene took 21 ms of its set-up,
// 0.04 so (set-up in all 21.2 -> 0.25 ms; 0.13 -> 0.06 for the 7-DOF scene's 39
// polytopes; 23 -> 29 us for the 4-DOF scene's 12, of which 10 are the launch).
constexpr int kScanVertices = 32, kScanDegree = 16, kCertCones = 16, kCertBlock = 32 * kScanVertices;
constexpr double kScanOutside = 5e6;  // 2 vmax |d|_1 over the 2 g (g = 3.41 2^-24 vmax |d|_1) of one l_i, and some
__global__ void __launch_bounds__(kCertBlock) support_factor_kernel(SceneImg img, char* __restrict__ blob) {
  __shared__ double s_v[kScanVertices][3], s_e[kScanVertices][kScanDegree][3], s_len[kScanVertices][kScanDegree];
  __shared__ double s_cone[kScanVertices][kCertCones][9];
  __shared__ int s_nb[kScanVertices][kScanDegree], s_deg[kScanVertices];
  __shared__ unsigned long long s_L;  // the bits of L >= 0, which order as the values do
  __shared__ int s_none;
  int2* const hull = reinterpret_cast<int2*>(blob + img.off_hulls) + blockIdx.x;
  const float4* const verts = reinterpret_cast<const float4*>(blob + img.off_verts);
  const unsigned short* const adj = reinterpret_cast<const unsigned short*>(blob + img.off_adj);
  const int n = hull->x, v0 = hull->y;
  const int u = threadIdx.x >> 5, w = threadIdx.x & 31;
  if (threadIdx.x == 0) {
    s_L = 0ull;
    s_none = n > kScanVertices ? 1 : 0;
  }
  __syncthreads();
  if (u == 0 && n <= kScanVertices && w < n) {
    const float4 r = verts[v0 + w];
    s_v[w][0] = r.x;
    s_v[w][1] = r.y;
    s_v[w][2] = r.z;
    s_deg[w] = info_of(r) & 255;
    if (s_deg[w] > kScanDegree) s_none = 1;
  }
  __syncthreads();
  const int count = s_none ? 0 : n;
  const int deg = u < count ? s_deg[u] : 0;
  if (w < deg) {
    const int to = adj[(info_of(verts[v0 + u]) >> 8) + w] - v0;
    s_nb[u][w] = to;
    double* const e = s_e[u][w];
    for (int a = 0; a < 3; ++a) e[a] = s_v[to][a] - s_v[u][a];
    s_len[u][w] = __builtin_sqrt(e[0] * e[0] + e[1] * e[1] + e[2] * e[2]);
  }
  __syncthreads();
  if (u < count) {
    const bool asked = w < count && w != u;
    double x[3] = {0.0, 0.0, 0.0}, best = asked ? 1e300 : 0.0;
    if (asked)
      for (int a = 0; a < 3; ++a) x[a] = s_v[w][a] - s_v[u][a];
    for (int i = 0; i < deg; ++i)  // a neighbour: its own edge
      if (asked && s_nb[u][i] == w) best = 1.0;
    const int triples = deg * (deg - 1) * (deg - 2) / 6;
    const unsigned long long half = 0xffffffffull << (threadIdx.x & 32);
    for (int t0 = 0; t0 < triples && (__ballot(best > 4.0) & half) != 0ull; t0 += kCertCones) {
      const int t = t0 + w;
      if (w < kCertCones) {
        double* const m = s_cone[u][w];
        m[0] = __builtin_nan("");  // no cone: every comparison with it is false
        if (t < triples) {
          int i = 0, j, k = t;  // triple t: i < j < k
          for (int c; k >= (c = (deg - 1 - i) * (deg - 2 - i) / 2); ++i) k -= c;
          for (j = i + 1; k >= deg - 1 - j; ++j) k -= deg - 1 - j;
          k += j + 1;
          const double *ei = s_e[u][i], *ej = s_e[u][j], *f = s_e[u][k];
          const double c[3] = {ei[1] * ej[2] - ei[2] * ej[1], ei[2] * ej[0] - ei[0] * ej[2],
                               ei[0] * ej[1] - ei[1] * ej[0]};
          const double det = c[0] * f[0] + c[1] * f[1] + c[2] * f[2];
          if (fabs(det) > 1e-5 * s_len[u][i] * s_len[u][j] * s_len[u][k]) {
            const double inv = 1.0 / det;
            m[0] = (ej[1] * f[2] - ej[2] * f[1]) * inv;
            m[1] = (ej[2] * f[0] - ej[0] * f[2]) * inv;
            m[2] = (ej[0] * f[1] - ej[1] * f[0]) * inv;
            m[3] = (f[1] * ei[2] - f[2] * ei[1]) * inv;
            m[4] = (f[2] * ei[0] - f[0] * ei[2]) * inv;
            m[5] = (f[0] * ei[1] - f[1] * ei[0]) * inv;
            for (int a = 0; a < 3; ++a) m[6 + a] = c[a] * inv;
          }
        }
      }
      // the cones were written by other lanes of this wave
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
      __builtin_amdgcn_wave_barrier();
      for (int s = 0; s < kCertCones; ++s) {
        const double* const m = s_cone[u][s];
        double sum = 0.0;
        for (int r = 0; r < 9; r += 3) {
          const double l = m[r] * x[0] + m[r + 1] * x[1] + m[r + 2] * x[2];
          sum += l > 0.0 ? l : -kScanOutside * l;
        }
        if (sum < best) best = sum;
      }
      __builtin_amdgcn_wave_barrier();  // before the next cones
    }
    if (best > 1e6) s_none = 1;
    else atomicMax(&s_L, (unsigned long long)__double_as_longlong(best));
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  double vmax = 0.0;
  for (int i = 0; i < count; ++i)
    for (int a = 0; a < 3; ++a) vmax = fmax(vmax, fabs(s_v[i][a]));
  // the products' errors, and 1e-8 vmax for the coefficients' own
  const double L = __longlong_as_double((long long)s_L);
  const float f = (float)(((2.0 * L + 2.0) * 3.41 * 0x1p-24 + 1e-8) * vmax * (1.0 + 1e-6));
  const bool ok = s_none == 0 && f < __builtin_inff();
  *hull = make_int2(ok ? n : 0, __float_as_int(ok ? f : __builtin_inff()));
}

// orthtrafo23 (collision4.h:111-134)
struct Orth {
  float M0, M1, M2, M3, M4, M5;
};
__device__ __forceinline__ V2 mult23(const Orth& o, const V3& x) {
  return V2{(o.M0 * x.x + o.M1 * x.y) + o.M2 * x.z, (o.M3 * x.x + o.M4 * x.y) + o.M5 * x.z};
}

// Iteration that did not separate (collision4.h:301-323): repetition test,
// w update, half plane (find_half_plane, collision4.h:136-223), reflection.
// Returns a nonzero code when the pair is decided (l+1: no half plane), else
// 0.  Taken by few iterations, but it sets the latency of a full test: the
// history R[0..k-1] lives in memory, so it is read in one pass with
// kHistBatch loads in flight, and the repetition test and the half-plane scan run
// together on each entry.  The scan's outcome counts only when no (p,q)
// repeats, as in the reference, where the repetition test comes first; the
// scan stops changing ra/rb where find_half_plane returns false.
constexpr int kHistBatch = 2;  // history loads in flight (four spill registers at five waves per SIMD)
__device__ __forceinline__ int sva_slow(const History& H, int& k, int l, int pq, const V3& r,
                                        float dp, V3& S, V3& w) {
  const f32x4 mine{r.x, r.y, r.z, __int_as_float(pq)};
  if (k < H.n) H.l[k * H.ls] = mine;
  else H.g[k * kHistStride] = mine;
  // find_half_plane returns at once (w unchanged) when w.r > 0
  const bool scan = k >= 2 && !(dot3(w, r) > 0);
  Orth o{};
  if (scan) {
    // orthtrafo23 M(rk)
    float x = r.x, y = r.y, z = r.z;
    float d2 = x * x + y * y;
    float d = __builtin_sqrtf(d2);
    o.M0 = x * z / d; o.M1 = y * z / d; o.M2 = -d;
    o.M3 = -y / d;    o.M4 = x / d;     o.M5 = 0.0f;
  }
  bool rep = false, fail = false;
  V3 r0{0.0f, 0.0f, 0.0f};
  V2 ra{0.0f, 0.0f}, rb{0.0f, 0.0f};
  for (int j0 = 0; j0 < k; j0 += kHistBatch) {
    f32x4 e[kHistBatch];
#pragma unroll
    for (int u = 0; u < kHistBatch; ++u) {
      e[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
      if (j0 + u >= k) continue;
      if (j0 + u < H.n) e[u] = H.l[(j0 + u) * H.ls];
      else e[u] = H.g[(j0 + u) * kHistStride];
    }
#pragma unroll
    for (int u = 0; u < kHistBatch; ++u) {
      const int j = j0 + u;
      if (j >= k) break;
      rep = rep || __float_as_int(e[u].w) == pq;
      if (j == 0) r0 = v3(e[u]);
      if (!scan || fail) continue;
      const V2 T = mult23(o, v3(e[u]));
      if (j == 0) {
        ra = T;
      } else if (j == 1) {
        rb = T;
        if (cross2(ra, rb) < 0) {
          rb = ra;
          ra = T;
        }
      } else {
        const float rbcross = cross2(rb, T);
        if (cross2(ra, T) > 0) {
          if (rbcross > 0) rb = T;
        } else {
          if (rbcross < 0) ra = T;
          else fail = true;
        }
      }
    }
  }
  if (rep) {
    S = w;  // (p,q) seen before
    return 0;
  }
  if (k == 1) {
    w = V3{r0.x + r.x, r0.y + r.y, r0.z + r.z};
    normalize3(w);
  }
  if (scan) {
    if (fail) return l + 1;
    normalize2(ra);
    normalize2(rb);
    V2 T{ra.x + rb.x, ra.y + rb.y};
    normalize2(T);
    w.x = o.M0 * T.x + o.M3 * T.y;
    w.y = o.M1 * T.x + o.M4 * T.y;
    w.z = o.M2 * T.x + o.M5 * T.y;
  }
  float b = -2.0f * dp;
  S.x = S.x + b * r.x;
  S.y = S.y + b * r.y;
  S.z = S.z + b * r.z;
  ++k;
  return 0;
}

// Work counters of one lane of the separating-vector loop.
struct SvaCounts {
  unsigned sep = 0, col = 0, dropped = 0, units = 0, iter = 0, bound = 0;
  unsigned claimed = 0;  // units this lane claimed (all finished when the loop returns)
};

// Copy a scene image into LDS (every thread of the block takes part; the
// caller synchronises before reading it).
template <int BLOCK>
__device__ __forceinline__ Lds stage_scene(const SceneImg& img, int4* smem) {
  const int n16 = img.bytes >> 4;
  for (int i = threadIdx.x; i < n16; i += BLOCK) smem[i] = img.blob[i];
  const char* base = reinterpret_cast<const char*>(smem);
  Lds L;
  L.verts = reinterpret_cast<const float4*>(base + img.off_verts);
  L.pairs = reinterpret_cast<const int4*>(base + img.off_pairs);
  L.adj = reinterpret_cast<const unsigned short*>(base + img.off_adj);
  L.hulls = reinterpret_cast<const int2*>(base + img.off_hulls);
  return L;
}

// The scene read where it lies in the global image (scenes beyond LDS): the
// same layout, through the caches.
__device__ __forceinline__ Lds scene_global(const SceneImg& img) {
  const char* base = reinterpret_cast<const char*>(img.blob);
  Lds L;
  L.verts = reinterpret_cast<const float4*>(base + img.off_verts);
  L.pairs = reinterpret_cast<const int4*>(base + img.off_pairs);
  L.adj = reinterpret_cast<const unsigned short*>(base + img.off_adj);
  L.hulls = reinterpret_cast<const int2*>(base + img.off_hulls);
  return L;
}

// The records of a (wave-uniform) pair and polytope: scalar loads, constant
// for the launch.
typedef int i32x2 __attribute__((ext_vector_type(2)));
typedef int i32x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ i32x2 load_pairrec(const SceneImg& img, int pair) {
  const unsigned long long p = reinterpret_cast<unsigned long long>(img.blob) + (unsigned long long)img.off_pairrecs +
                               8ull * (unsigned)pair;
  return *(const __attribute__((address_space(4))) i32x2*)p;
}
__device__ __forceinline__ i32x16 load_polyrec(const SceneImg& img, int poly) {
  const unsigned long long p = reinterpret_cast<unsigned long long>(img.blob) + (unsigned long long)img.off_polyrecs +
                               sizeof(PolyRec) * (unsigned)poly;
  return *(const __attribute__((address_space(4))) i32x16*)p;
}
__device__ __forceinline__ V3 rec_v3(const i32x16& r, int at) {
  return V3{__int_as_float(r[at]), __int_as_float(r[at + 1]), __int_as_float(r[at + 2])};
}

// Deferred pair tests of one wave: a ring of CAP = sva_ring_cap(BLOCK)
// entries in LDS, (item, pair) in ent and the item's edge (edge mode) in
// edge.  Phase B starts as soon as CAP - 64 entries wait, so the ring never
// holds more than CAP - 1.
struct Ring {
  int2* ent;
  int* edge;
};
template <int BLOCK>
__device__ __forceinline__ Ring wave_ring(int4* smem) {
  constexpr int CAP = sva_ring_cap(BLOCK);
  int2* const ent = reinterpret_cast<int2*>(smem);
  int* const edge = reinterpret_cast<int*>(ent + (BLOCK / 64) * CAP);
  const int w = threadIdx.x >> 6;
  return Ring{ent + w * CAP, edge + w * CAP};
}

// Work units of a separating-vector launch: (chunk of pairs_per_unit pairs,
// group of 64 consecutive items), numbered chunk-major.
__device__ __forceinline__ unsigned sva_unit_count(const SvaArgs& A, int nitems) {
  return (unsigned)((nitems + 63) >> 6) * (unsigned)A.units_per_item;
}

// The rings of a block's waves as one queue (the last drain): wave w's waiting
// entries, moved to the start of its ring, are numbered from first[w]; next
// is the first number not taken yet.  It lies in the last 64 slots of the
// block's first ring, which are free then (a ring with more than CAP - 65
// entries would have been drained), so it needs no LDS of its own.
template <int WAVES>
struct Pool {
  unsigned first[WAVES + 1], next;
};
static_assert(sizeof(Pool<16>) <= 63 * sizeof(int2), "fits the free slots before the last");

// Phase B of sva_units: every lane takes a deferred pair from the wave's
// ring and runs the full separating-vector test (collision4.h:227-332) until
// the ring is empty.  The gate is re-read when a pair is taken.  POOLED: the
// pairs come from the block's pool instead.
template <int EDGE, int CAP, int WAVES, bool POOLED>
__device__ __forceinline__ void sva_drain(const SvaArgs& A, const Lds& L, const Ring& R,
                                          const History& H, unsigned& d_head, unsigned d_tail,
                                          Pool<WAVES>* pool, unsigned& n_sep, unsigned& n_col, unsigned& n_dropped, unsigned& n_iter) {
  const int lane = threadIdx.x & 63;
  const unsigned long long lt_mask = (1ull << lane) - 1ull;
  // the ring's entries were written by other lanes of this wave
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  bool busy = false;
  T12 tp, tq;
#pragma unroll
  for (int i = 0; i < 12; ++i) tp.m[i] = tq.m[i] = 0.0f;
  int bitem = 0, bedge = 0, crs = 0, k = 0, l = 0, p = 0, q = 0, vbP = 0, vbQ = 0, polys = 0;
  bool sysP0 = true, sysQ0 = true;
  V3 S{0, 0, 0}, w{0, 0, 0};
  for (;;) {
    const unsigned long long wm = __ballot(!busy);
    const unsigned want = (unsigned)__popcll(wm);
    if (POOLED && d_head != d_tail && wm != 0ull) {
      // d_head: the first number the wave may take, d_tail: the pool's end
      unsigned at = 0;
      if (lane == 0) at = atomicAdd(&pool->next, want);
      at = __builtin_amdgcn_readfirstlane(at);
      d_head = at < d_tail ? at : d_tail;
    }
    const unsigned avail = d_tail - d_head;
    const unsigned take = want < avail ? want : avail;
    if (!busy && (unsigned)__popcll(wm & lt_mask) < take) {
      unsigned slot = d_head + (unsigned)__popcll(wm & lt_mask);
      if (POOLED) {
        // the ring that holds it (R is the block's first ring)
        int w = 0;
        for (int step = WAVES / 2; step > 0; step /= 2)
          if (pool->first[w + step] <= slot) w += step;
        slot = w * CAP + (slot - pool->first[w]);
      } else {
        slot &= CAP - 1;
      }
      const int2 e = R.ent[slot];
      bitem = e.x;
      const int4 pd = L.pairs[e.y];
      crs = pd.z;
      polys = pd.w;
      // the gate and the frames are loaded together (one memory round
      // trip); the frames of a pair that turns out dropped are not used
      int gv;
      if (EDGE) {
        bedge = R.edge[slot];
        gv = __hip_atomic_load((GAS int*)A.edge_res + bedge, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      } else {
        gv = __hip_atomic_load((GAS int*)A.word + bitem, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      vbP = pd.x & 0xffff;
      vbQ = (int)((unsigned)pd.x >> 16);
      const int sP = pd.y & 255, sQ = pd.y >> 8;
      sysP0 = sP == 0;
      sysQ0 = sQ == 0;
      if (!sysP0) tp = load_frame(A.frames, bitem, A.fstride, sP);
      if (!sysQ0) tq = load_frame(A.frames, bitem, A.fstride, sQ);
      const bool drop = EDGE ? gv != 0 : (gv >> 4) <= crs;
      if (drop) {
        ++n_dropped;
      } else {
        // start of the pair (collision4.h:228-244)
        const V3 vq = v3(L.verts[vbQ]), vp = v3(L.verts[vbP]);
        const V3 Pq = sysQ0 ? vq : t_apply(tq, vq);
        const V3 Pp = sysP0 ? vp : t_apply(tp, vp);
        S = V3{Pq.x - Pp.x, Pq.y - Pp.y, Pq.z - Pp.z};
        const float norm = normalize3(S);
        if (norm <= kEpsBelow) S.x = 1.0f;
        p = vbP;
        q = vbQ;
        k = 0;
        l = 0;
        w = V3{0.0f, 0.0f, 0.0f};
        busy = true;
      }
    }
    if (!POOLED) d_head += take;
    if (__ballot(busy) == 0ull) {
      if (d_head == d_tail) break;
      continue;
    }
    if (!busy) continue;
    ++n_iter;

    // ---- one iteration (collision4.h:266-300) ------------------------------
    V3 Sp = sysP0 ? S : t_apply_rot_inv(tp, S);
    V3 Sn{-S.x, -S.y, -S.z};
    V3 Sq = sysQ0 ? Sn : t_apply_rot_inv(tq, Sn);
    p = support(L, polys & 0xffff, vbP, p, Sp);
    q = support(L, (int)((unsigned)polys >> 16), vbQ, q, Sq);
    V3 vp = v3(L.verts[p]), vq = v3(L.verts[q]);
    V3 p0 = sysP0 ? vp : t_apply(tp, vp);
    V3 q0 = sysQ0 ? vq : t_apply(tq, vq);
    V3 r{q0.x - p0.x, q0.y - p0.y, q0.z - p0.z};
    normalize3(r);
    float dp = dot3(S, r);

    bool fin = false;
    int code = 0;
    if (dp >= -kEpsBelow) {
      fin = true;
    } else {
      code = sva_slow(H, k, l, (p - vbP) | ((q - vbQ) << 16), r, dp, S, w);
      if (code != 0) {
        fin = true;
      } else if (++l >= kMaxIter) {
        fin = true;
        code = -1;
      }
    }
    if (fin) {
      if (code != 0) {
        ++n_col;
        if (EDGE) {
          __hip_atomic_store((GAS int*)A.edge_res + bedge, code, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
          __hip_atomic_fetch_min((GAS int*)A.word + bitem, ((crs + 1) << 4) | (code + 1), __ATOMIC_RELAXED,
                                 __HIP_MEMORY_SCOPE_AGENT);
        }
      } else {
        ++n_sep;
      }
      busy = false;
    }
  }
}

// Units of one scene (its image in L) until its queue is exhausted, every
// deferred pair included.  A wave claims a unit (one chunk of pairs, 64
// consecutive items: lane l takes item 64 g + l) and walks the chunk's pairs
// in step, so the pair record, the frame changes and the caches below are
// the same in every lane.  Work alternates between two wave-wide phases:
//   A. for each pair every lane starts the pair on its item (gate, frames,
//      the start direction) and applies the bound test, which decides most
//      pairs; a pair it does not decide is appended to the wave's ring;
//   B. once 64 pairs wait (and at the end), every lane takes deferred pairs
//      and runs the full test until the ring is empty (sva_drain).
// H: this lane's iteration history; R: the wave's ring.  Waves
// run independently until the queue is exhausted; with POOL the last drain is
// the block's (every thread calls).  cnt.claimed counts the wave's units (the
// same in every lane), all finished on return.
template <int EDGE, int CAP, int WAVES, bool POOL>
__device__ __forceinline__ void sva_units(const SvaArgs& A, const Lds& L, const Ring& R,
                                          const History& H, SvaCounts& cnt) {
  const int lane = threadIdx.x & 63;
  const unsigned long long lt_mask = (1ull << lane) - 1ull;
  // the same in every lane, as are the unit indices derived from it: said by
  // readfirstlane, so that the pair loop and the records stay scalar also
  // where the arguments were loaded from memory
  const int nitems =
      __builtin_amdgcn_readfirstlane(A.nitems >= 0 ? A.nitems : (int)min((long long)*A.nitems_dev, A.fstride));
  const int M = A.img.M;
  const int PC = A.pairs_per_unit;
  const unsigned ngroups = (unsigned)((nitems + 63) >> 6);
  const unsigned nunits = sva_unit_count(A, nitems);

  unsigned d_head = 0, d_tail = 0;  // the ring's cursors (the same in every lane)
  unsigned n_sep = 0, n_col = 0, n_dropped = 0, n_units = 0, n_iter = 0, n_claimed = 0;
  unsigned s_dropped = 0, s_bound = 0;  // the wave's, in scalar registers

  // Point mode with the codes written here: a unit is complete once the
  // ring holds none of its deferred pairs, which is certain whenever the
  // ring is empty.  Units whose pairs are all walked wait in a per-wave list
  // (the ring's edge array, unused in point mode) until the ring next
  // empties; then each adds one to its group's counter, and the wave that
  // brings a group to units_per_item writes that group's 64 codes.  No wave
  // waits for another.
  const bool fuse = !EDGE && A.group_done != nullptr;
  unsigned n_pend = 0;  // the same in every lane
  auto complete_pending = [&]() {
    for (unsigned k = 0; k < n_pend; ++k) {
      const unsigned cu = (unsigned)R.edge[k];
      const unsigned g = cu % ngroups;
      int old = 0;
      // Words and counters are only touched by agent-scope atomics, which
      // are coherent across the XCDs' L2s; what matters is that this wave's
      // word updates (any lane) have completed before its count, which
      // waiting for all its outstanding memory operations gives.  (An
      // agent-scope release or acquire fence would also write back or
      // invalidate the XCD's whole L2, per wave: it made the launch three
      // times slower.)
      __builtin_amdgcn_s_waitcnt(0);
      if (lane == 0)
        old = __hip_atomic_fetch_add((GAS int*)A.group_done + g, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      old = __shfl(old, 0, 64);
      if (old == A.units_per_item - 1) {
        // every unit of the group has finished: the words are final (the
        // loads below are issued after the count came back)
        const int it = (int)(g << 6) + lane;
        if (it < nitems) {
          const int w = __hip_atomic_load((GAS int*)A.word + it, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          ((GAS int*)A.codes)[it] = w == 0x7fffffff ? 0 : (w & 15) - 1;
        }
      }
    }
    n_pend = 0;
    // the list's entries were read by every lane before lane 0 refills it
    __builtin_amdgcn_wave_barrier();
  };

  // Work distribution.  Claims on one counter serialise at the memory side
  // (about 15 ns each), so a launch of small units must not claim them one by
  // one from one counter: with static_first, wave w takes units w, w + nwaves,
  // ... for three quarters of the full rounds (all of them when there are
  // less than four rounds), and the rest is dealt out to kSvaQueues queues,
  // unit k of it to queue k mod kSvaQueues, each with a counter of its own
  // from which every kSvaQueues-th wave claims guided chunks of max(1, left /
  // (2 x the queue's waves)).  The queues hold alike work, so no wave steals
  // from another's.  (One counter for all: 2.51 against 2.11 ms for the 6-DOF
  // roadmap, 650 against 468 us for 20,011 local 7-DOF edges, 311 against 191 us
  // for 2,048 local 4-DOF ones; one round of static units, half or all of
  // them: 2.24, 2.14, 2.31 ms for the roadmap, 3.49, 3.35, 3.68 against 3.32 ms
  // for 4M points of the 7-DOF scene.)  Without static_first (the multi-scene kernel, where
  // blocks rotate over the scenes) one queue holds everything.  Once fewer
  // units than waves may remain, a wave reads the counter before claiming, so
  // that waves finding the queue drained leave without an atomic.
  const unsigned nwaves = (gridDim.x * blockDim.x) >> 6;
  // wave-uniform values held in scalar registers: the unit index, and from
  // it the pair loop, the pair records and the cache tags below
  const unsigned wave = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  unsigned nstatic = 0, nq = 1, q = 0;
  if (A.static_first) {
    const unsigned rounds = nunits / nwaves;
    nstatic = rounds < 4 ? nunits : rounds * 3 / 4 * nwaves;
    nq = kSvaQueues;
    q = wave % kSvaQueues;
  }
  // the queue's units and waves, and its counter
  const unsigned qunits = nunits - nstatic > q ? (nunits - nstatic - q + nq - 1) / nq : 0u;
  const unsigned qwaves = nwaves / nq > 0 ? nwaves / nq : 1u;
  GAS unsigned* const counter = (GAS unsigned*)A.counter + q * kSvaQueueStride;
  unsigned su = wave;          // next static unit
  unsigned cur = 0, cend = 0;  // the queue's units [cur, cend) are claimed
  unsigned seen = 0;           // the counter as last observed by this wave
  for (;;) {
    unsigned u;
    if (su < nstatic) {
      u = su;
      su += nwaves;
    } else if (cur < cend) {
      u = nstatic + q + nq * cur++;
    } else {
      const unsigned left = qunits > seen ? qunits - seen : 0u;
      if (left == 0) break;
      const unsigned k = left / (2 * qwaves) > 1 ? left / (2 * qwaves) : 1u;
      unsigned b = 0xffffffffu;
      if (lane == 0) {
        bool go = true;
        if (left < qwaves) go = __hip_atomic_load(counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < qunits;
        if (go) b = __hip_atomic_fetch_add(counter, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      b = __builtin_amdgcn_readfirstlane(b);
      if (b == 0xffffffffu || b >= qunits) break;
      seen = b + k;
      cur = b;
      cend = b + k < qunits ? b + k : qunits;
      u = nstatic + q + nq * cur++;
    }
    ++n_claimed;
    const unsigned ch = u / ngroups;
    const int item = (int)((u - ch * ngroups) << 6) + lane;
    bool active = item < nitems;
    const int p0 = (int)ch * PC, p1 = min(M, p0 + PC);
    // early exit: in edge mode once any sample of the edge is blocked; in
    // point mode for pairs after (in CRS order) a pair known to collide,
    // since the reference returns the first colliding pair's code.
    int edge = 0, gate = 0x7fffffff;
    bool open_item = active;
    if (EDGE && active) {
      edge = ((const GAS int*)A.item_edge)[item];
      active = open_item = edge >= 0;  // no padding
    }
    if (active) {
      if (EDGE) {
        open_item = __hip_atomic_load((GAS int*)A.edge_res + edge, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;
      } else {
        gate = __hip_atomic_load((GAS int*)A.word + item, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >> 4;
      }
    }
    // the lanes whose item is in the launch, and those of them that are open
    const unsigned long long act = __ballot(active), opn = EDGE ? __ballot(open_item) : act;
    // The chunk's pairs in order: all of them in point mode (random
    // configurations leave few pairs out of a mask; walking the masks' bits
    // alone cost 3.55 against 3.33 ms for 4M points of the 7-DOF scene), in
    // edge mode those that the group's mask leaves; the others are decided by
    // the bounds for every item (cull_pairs).
    const unsigned long long mrow =
        reinterpret_cast<unsigned long long>(A.mask) + 8ull * (u - ch * ngroups) * (unsigned)((M + 63) >> 6);
    const int wl = (p1 - 1) >> 6;
    int w = (p0 >> 6) - 1;
    unsigned long long bits = 0ull;
    auto next_pair = [&]() {
      while (bits == 0ull) {
        if (w >= wl) return -1;
        ++w;
        // a scalar load: the masks are constant during the launch
        bits = A.mask == nullptr ? ~0ull : ((const __attribute__((address_space(4))) unsigned long long*)mrow)[w];
        if (w == p0 >> 6) bits &= ~0ull << (p0 & 63);
        if (w == wl) bits &= ~0ull >> (63 - ((p1 - 1) & 63));
      }
      const int p = 64 * w + __builtin_ctzll(bits);
      bits &= bits - 1;
      return p;
    };
    // The unit's pairs run in segments that end where the ring is drained.
    // The caches are local to a segment, so nothing of them is live across
    // a drain, which has registers of its own.
    int left = EDGE ? p1 - p0 : 0;  // pairs not walked
    int cur_pair = EDGE ? -1 : p0, nxt_pair = EDGE ? -1 : p0 + 1;
    if (EDGE && opn != 0ull) {
      cur_pair = next_pair();
      nxt_pair = next_pair();
    }
    while (EDGE ? cur_pair >= 0 : cur_pair < p1) {
      // wave-uniform cache: Q's world bounds for polytope ckQ and its start
      // vertex
      int ckQ = -1;
      V3 cQw{0, 0, 0}, PqW{0, 0, 0};
      // Q's box axes in the world frame, times its half extents
      V3 aQ0{0, 0, 0}, aQ1{0, 0, 0}, aQ2{0, 0, 0};
      float RQ = 0.0f, rQ = 0.0f;
      // the pair's operands are in scalar registers, loaded a pair ahead (its
      // record two pairs ahead), so they cost no vector instruction.  LDS
      // reads moved to scalar registers, selects between the frames, lane
      // counters and unfused products had made 110 vector instructions a
      // pair; now it is about 30, and 25 more where the boxes are needed
      // (4.28 -> 3.57 ms for 4M configurations of the 7-DOF scene, 3.83 ->
      // 3.26 ms for the 6-DOF roadmap's edges).
      i32x2 pr1 = load_pairrec(A.img, cur_pair), pr2 = load_pairrec(A.img, EDGE ? max(nxt_pair, 0) : min(nxt_pair, M - 1));
      i32x16 poly1 = load_polyrec(A.img, pr1[0] & 0xffff);
      bool full = false;
      do {
        const i32x2 pr = pr1;
        const i32x16 cur = poly1;
        const int pair = cur_pair;
        if (EDGE) --left;
        pr1 = pr2;
        poly1 = load_polyrec(A.img, pr1[0] & 0xffff);
        cur_pair = nxt_pair;
        nxt_pair = EDGE ? next_pair() : nxt_pair + 1;
        pr2 = load_pairrec(A.img, EDGE ? max(nxt_pair, 0) : min(nxt_pair, M - 1));
        const int crs = pr[1], kQ = (int)((unsigned)pr[0] >> 16);
        // Frames are loaded by every lane: an inactive lane's item is below
        // the plane stride (the item count rounded up to 64), and what it
        // computes from them is masked out below.
        if (kQ != ckQ) {
          const i32x16 rq = load_polyrec(A.img, kQ);
          const V3 hq = rec_v3(rq, 8);
          rQ = __int_as_float(rq[7]);
          if (rq[11] == 0) {
            PqW = rec_v3(rq, 0);
            cQw = rec_v3(rq, 4);
            aQ0 = V3{hq.x, 0.0f, 0.0f};
            aQ1 = V3{0.0f, hq.y, 0.0f};
            aQ2 = V3{0.0f, 0.0f, hq.z};
          } else {
            const T12 tq = load_frame(A.frames, item, A.fstride, rq[11]);
            PqW = b_apply(tq, rec_v3(rq, 0));
            cQw = b_apply(tq, rec_v3(rq, 4));
            aQ0 = V3{tq.m[0] * hq.x, tq.m[1] * hq.x, tq.m[2] * hq.x};
            aQ1 = V3{tq.m[3] * hq.y, tq.m[4] * hq.y, tq.m[5] * hq.y};
            aQ2 = V3{tq.m[6] * hq.z, tq.m[7] * hq.z, tq.m[8] * hq.z};
          }
          RQ = bound_radius(cQw, rQ);
          ckQ = kQ;
        }
        // Every lane evaluates the bound test (a SIMD runs the whole wave
        // anyway); the lane's conditions (its item open, its pair not
        // dropped by the gate) are applied to the result.
        const unsigned long long test = EDGE ? opn : act & __ballot(gate > crs);
        // Start of the pair (collision4.h:228-244) and the bound decision
        // of iteration 0: iteration 0 returns 0 whenever
        // S.normalize(q0 - p0) >= -1e-6 for the support vertices p0, q0
        // the climbs find, S = normalize(D) with D the difference of the
        // two start vertices.  If the bounds show S.(q - p) > 0
        // with a wide margin for every vertex p of P and q of Q, that holds
        // whichever vertices the climbs would pick, so the pair test ends
        // here exactly as the reference's does (code 0, one
        // iteration).  The margin, 2^-10 of the magnitudes involved,
        // exceeds the rounding error of every quantity in the test and in
        // the reference's iteration by orders of magnitude.  Both sides of
        // the test scale with |S|, so it runs on D itself: the reference's
        // S differs from D/|D| by a relative 1e-7, far inside the margin.
        // The test also requires |D|_2 > 1e-5, which stays clear of the
        // reference's override of S for |D| <= 1e-6; a NaN D never passes
        // (such pairs are deferred to the exact test).  Nothing here has to
        // be the reference's float, so it may use fused multiply-adds.
        // First the bounding spheres: every vertex lies within r of its
        // polytope's centre c, so S.(q - p) >= S.(cQ - cP) - (rP + rQ)|S|.
        // That costs a few operations and decides most pairs; the boxes'
        // support extents along S (sum_a |S.axis_a| h_a, axes the frame's
        // rotation columns) are tighter and are computed only when some
        // lane's pair the spheres leave open.  The margin is 2^-10 of |S|_1
        // times the magnitudes |c|_1 + r per side; for the spheres it is part
        // of the radii (bound_radius: |S|_1 <= sqrt(3) |S|_2 and 2^-9 >
        // sqrt(3) 2^-10), and the comparison is made on squares (no square
        // root), the radii inflated by 2^-8 against their rounding.
        const V3 vp = rec_v3(cur, 0), cP = rec_v3(cur, 4), hP = rec_v3(cur, 8);
        const float rbP = __int_as_float(cur[3]), rP = __int_as_float(cur[7]);
        const int sP = cur[11];
        // the lanes of `test` that the bounds decide; P's half extents along
        // S come from boxP
        auto decided = [&](const V3& S, const V3& E, float rad, auto boxP) {
          const float dc = b_dot(S, E), ss = b_dot(S, S);
          const unsigned long long cand = __ballot(ss > 1e-10f) & __ballot(dc > 0.0f) & test;
          unsigned long long sep = __ballot(dc * dc > (rad * rad) * ss) & cand;
          if (cand != sep) {
            const float boxQ = (fabsf(b_dot(S, aQ0)) + fabsf(b_dot(S, aQ1))) + fabsf(b_dot(S, aQ2));
            // |cP|_1 <= |cQ|_1 + |E|_1
            const float magQ = (fabsf(cQw.x) + fabsf(cQw.y)) + fabsf(cQw.z);
            const float magE = (fabsf(E.x) + fabsf(E.y)) + fabsf(E.z);
            const float mag = (magQ + magQ) + (magE + (rQ + rP));
            const float thr = 0x1p-10f * mag * (fabsf(S.x) + fabsf(S.y) + fabsf(S.z));
            sep |= __ballot(dc - boxQ - boxP() > thr) & cand;
          }
          return sep;
        };
        unsigned long long sep;
        if (sP == 0) {
          const V3 S{PqW.x - vp.x, PqW.y - vp.y, PqW.z - vp.z};
          const V3 E{cQw.x - cP.x, cQw.y - cP.y, cQw.z - cP.z};
          sep = decided(S, E, RQ + rbP,
                        [&]() { return (fabsf(S.x) * hP.x + fabsf(S.y) * hP.y) + fabsf(S.z) * hP.z; });
        } else {
          // P's frame is loaded for the pair and not kept: a kept one would
          // have to be copied around every pair of a polytope at rest, and
          // few of a scene's pairs have both polytopes on links
          const T12 tp = load_frame(A.frames, item, A.fstride, sP);
          const V3 Pp = b_apply(tp, vp), cw = b_apply(tp, cP);
          const V3 S{PqW.x - Pp.x, PqW.y - Pp.y, PqW.z - Pp.z};
          const V3 E{cQw.x - cw.x, cQw.y - cw.y, cQw.z - cw.z};
          sep = decided(S, E, RQ + bound_radius(cw, rP), [&]() {
            const V3 sp = t_apply_rot_inv(tp, S);
            return (fabsf(sp.x) * hP.x + fabsf(sp.y) * hP.y) + fabsf(sp.z) * hP.z;
          });
        }
        s_dropped += (unsigned)__popcll(act & ~test);
        s_bound += (unsigned)__popcll(sep);
        // append the undecided pairs to the ring; drain it once CAP - 64 wait
        const unsigned long long dm = test & ~sep;
        if (dm != 0ull) {
          if ((dm >> lane) & 1ull) {
            const unsigned slot = (d_tail + (unsigned)__popcll(dm & lt_mask)) & (CAP - 1);
            R.ent[slot] = make_int2(item, pair);
            if (EDGE) R.edge[slot] = edge;
          }
          d_tail += (unsigned)__popcll(dm);
          full = d_tail - d_head >= CAP - 64;
        }
      } while ((EDGE ? cur_pair >= 0 : cur_pair < p1) && !full);
      if (full) {
        sva_drain<EDGE, CAP, WAVES, false>(A, L, R, H, d_head, d_tail, nullptr, n_sep, n_col, n_dropped, n_iter);
        if (fuse) complete_pending();  // the units before this one
      }
    }
    // the pairs the mask left out: separated where the item is open
    if (EDGE) {
      s_bound += (unsigned)left * (unsigned)__popcll(opn);
      s_dropped += (unsigned)left * (unsigned)__popcll(act & ~opn);
    }
    ++n_units;
    if (fuse) {
      if (lane == 0) R.edge[n_pend] = (int)u;
      __builtin_amdgcn_wave_barrier();
      ++n_pend;
      if (d_tail == d_head) {
        complete_pending();
      } else if (n_pend == (unsigned)CAP) {
        sva_drain<EDGE, CAP, WAVES, false>(A, L, R, H, d_head, d_tail, nullptr, n_sep, n_col, n_dropped, n_iter);
        complete_pending();
      }
    }
  }
  // The multi-scene kernel's blocks go on to the next scene together: there,
  // what waits in the block's rings at a scene's end is one queue for all of
  // its waves (16 scenes of 1k-64k configurations: 1.78-1.82 against 2.00 ms).
  // A single scene's launch gains nothing from it (65,536 points of the 4-DOF
  // scene: 72 against 70 us).
  if (!POOL) {
    if (d_tail != d_head)
      sva_drain<EDGE, CAP, WAVES, false>(A, L, R, H, d_head, d_tail, nullptr, n_sep, n_col, n_dropped, n_iter);
  } else {
    const int w = threadIdx.x >> 6;
    const Ring B{R.ent - w * CAP, R.edge - w * CAP};
    Pool<WAVES>* const pool = reinterpret_cast<Pool<WAVES>*>(B.ent + CAP - 64);
    const unsigned count = d_tail - d_head;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    int2 ent[CAP / 64 - 1];
    int edg[CAP / 64 - 1];
#pragma unroll
    for (int k = 0; k < CAP / 64 - 1; ++k) {
      const unsigned slot = (d_head + 64 * k + lane) & (CAP - 1);
      ent[k] = R.ent[slot];
      edg[k] = EDGE ? R.edge[slot] : 0;
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < CAP / 64 - 1; ++k)
      if (64u * k + lane < count) {
        R.ent[64 * k + lane] = ent[k];
        if (EDGE) R.edge[64 * k + lane] = edg[k];
      }
    // each wave leaves its count in the last slot of its own ring (other
    // waves may still be using theirs)
    if (lane == 0) R.ent[CAP - 1].x = (int)count;
    __syncthreads();
    if (threadIdx.x == 0) {
      unsigned sum = 0;
      for (int i = 0; i < WAVES; ++i) {
        pool->first[i] = sum;
        sum += (unsigned)B.ent[i * CAP + CAP - 1].x;
      }
      pool->first[WAVES] = sum;
      pool->next = 0;
    }
    __syncthreads();
    unsigned first = 0, end = __builtin_amdgcn_readfirstlane(pool->first[WAVES]);
    if (end != 0)
      sva_drain<EDGE, CAP, WAVES, true>(A, L, B, H, first, end, pool, n_sep, n_col, n_dropped, n_iter);
    // the pool is read no more after this, and the wave's result words have landed
    // (their groups' counts follow)
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }
  if (fuse) complete_pending();

  if (lane == 0) {
    n_sep += s_bound;
    n_dropped += s_dropped;
    cnt.bound += s_bound;
  }
  cnt.sep += n_sep;
  cnt.col += n_col;
  cnt.dropped += n_dropped;
  cnt.units += n_units;
  cnt.iter += n_iter;
  cnt.claimed += n_claimed;
}

// Per-block sums of the lane counters through LDS, one atomic per counter.
// Every thread of the block calls it; the LDS scene is not read afterwards.
template <int BLOCK>
__device__ __forceinline__ void add_tally(const SvaCounts& c, int4* smem, unsigned long long* tally) {
  __syncthreads();
  unsigned* t = reinterpret_cast<unsigned*>(smem);
  const int tid = threadIdx.x;
  if (tid < kTallyCount) t[tid] = 0u;
  __syncthreads();
  atomicAdd(&t[0], c.sep);
  atomicAdd(&t[1], c.col);
  atomicAdd(&t[2], c.dropped);
  atomicAdd(&t[3], c.units);
  atomicAdd(&t[4], c.iter);
  atomicAdd(&t[5], c.bound);
  __syncthreads();
  if (tid < kTallyCount)
    atomicAdd(&tally[(blockIdx.x % kTallySlots) * kTallyCount + tid], (unsigned long long)t[tid]);
}

// WAVES: occupancy target in waves per SIMD; the compiler keeps the register
// budget at 512/WAVES VGPRs (5 waves: 96 VGPRs; the edge-mode build spills
// two dwords).
// GS: the scene is read from the global image instead of an LDS copy (for
// scenes whose image does not fit).
template <int EDGE, int BLOCK, int WAVES, int GS>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(WAVES, 8))) sva_kernel(SvaArgs A) {
  extern __shared__ int4 smem[];
  // dynamic LDS: the waves' deferral rings (sva_ring_bytes), the lanes'
  // first history entries, then the scene image (unless GS)
  f32x4* const lh = reinterpret_cast<f32x4*>(smem + sva_ring_bytes(BLOCK) / 16);
  const Lds L = GS ? scene_global(A.img)
                   : stage_scene<BLOCK>(A.img, reinterpret_cast<int4*>(lh + (size_t)A.lds_hist * BLOCK));
  const Ring R = wave_ring<BLOCK>(smem);
  __syncthreads();
  const History H = lane_history(A.hist, blockIdx.x * BLOCK + threadIdx.x, lh + threadIdx.x, A.lds_hist, BLOCK);
  SvaCounts c;
  sva_units<EDGE, sva_ring_cap(BLOCK), BLOCK / 64, false>(A, L, R, H, c);
  if (A.tally != nullptr) add_tally<BLOCK>(c, smem, A.tally);
}

// Many scenes in one persistent launch.  Blocks start on different scenes
// (block b on scene b mod ntasks) and visit every scene once in rotation:
// a block whose next scene still has unclaimed units stages that scene's
// image into LDS and runs its units; one that finds the queue drained skips
// it.  When a wave leaves a scene, every unit it claimed there is finished;
// the wave whose count completes the scene's total stamps the device clock.
template <int EDGE, int BLOCK, int WAVES>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(WAVES, 8)))
    sva_multi_kernel(const SceneTask* __restrict__ tasks, int ntasks, unsigned long long* t_start,
                     unsigned long long* tally, int lds_hist) {
  extern __shared__ int4 smem[];
  __shared__ int s_live;
  if (threadIdx.x == 0) atomicMin(t_start, (unsigned long long)wall_clock64());
  f32x4* const lh = reinterpret_cast<f32x4*>(smem + sva_ring_bytes(BLOCK) / 16);
  const History H =
      lane_history(tasks[0].a.hist, blockIdx.x * BLOCK + threadIdx.x, lh + threadIdx.x, lds_hist, BLOCK);
  // dynamic LDS as in sva_kernel: rings, history, scene image
  const Ring R = wave_ring<BLOCK>(smem);
  SvaCounts c;
  for (int r = 0; r < ntasks; ++r) {
    const int t = (int)((blockIdx.x + (unsigned)r) % (unsigned)ntasks);
    const SvaArgs A = tasks[t].a;
    const int ni = A.nitems >= 0 ? A.nitems : (int)min((long long)*A.nitems_dev, A.fstride);
    const unsigned nunits = sva_unit_count(A, ni);
    if (threadIdx.x == 0)
      s_live = __hip_atomic_load(A.counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < nunits ? 1 : 0;
    __syncthreads();
    if (s_live) {
      const Lds L = stage_scene<BLOCK>(A.img, reinterpret_cast<int4*>(lh + (size_t)lds_hist * BLOCK));
      __syncthreads();
      const unsigned before = c.claimed;
      sva_units<EDGE, sva_ring_cap(BLOCK), BLOCK / 64, true>(A, L, R, H, c);
      const unsigned mine = c.claimed - before;  // the wave's units (the same in every lane)
      if ((threadIdx.x & 63) == 0 && mine > 0) {
        const unsigned old = atomicAdd(tasks[t].done, mine);
        if (old + mine == nunits) tasks[t].t_done[0] = (unsigned long long)wall_clock64();
      }
    }
    __syncthreads();  // s_live and the LDS image are reused by the next scene
  }
  if (tally != nullptr) add_tally<BLOCK>(c, smem, tally);
}

// ---- small point-check calls ------------------------------------------------
// One block per configuration of a call of at most kSmallMax: the
// configurations come as kernel arguments and the codes go straight to
// (pinned host) memory, so a call is one launch and one synchronisation.
// The first wave computes the frames into LDS; the threads then run the full
// separating-vector test on the pairs t, t + BLOCK, ... (no bound test: it
// only shortcuts pair tests that end separated), skipping pairs later in
// CRS order than a collision already found, and the block keeps the first
// colliding pair's code, as the batched kernels do.

// Frames 1..ndof of one configuration (kinematics.h:27-37), the same
// operations as fk_store, by the block's first wave: lane i the joint's own
// transformation into out[i] (its sine and cosine are the long part; with one
// lane computing all in turn a call on the 4-DOF scene took 30.4 us, 29.4 so),
// then lane 0 the chain.
__device__ void fk_frames(const DevRobot& rb, const float* q, T12* out) {
  const int lane = threadIdx.x;
  if (lane < rb.ndof) {
    const bool turns = rb.types[lane] == 0;
    out[lane] = t_set_cs(rb.a[lane], rb.ca[lane], rb.sa[lane], turns ? q[lane] : rb.q[lane],
                         turns ? rb.d[lane] : q[lane]);
  }
  // the entries were written by other lanes of this wave
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
  if (lane == 0) {
    T12 T = t_base(rb);
    for (int i = 0; i < rb.ndof; ++i) {
      T = t_lapply(out[i], T);
      out[i] = T;
    }
  }
}

// The full separating-vector test of one pair (collision4.h:227-332), as
// sva_drain runs it per lane; H: this lane's iteration history.
__device__ int sva_pair_full(const Lds& L, const T12& tp, const T12& tq, bool sysP0, bool sysQ0, int vbP, int vbQ,
                             int kP, int kQ, const History& H) {
  const V3 vq0 = v3(L.verts[vbQ]), vp0 = v3(L.verts[vbP]);
  const V3 Pq = sysQ0 ? vq0 : t_apply(tq, vq0);
  const V3 Pp = sysP0 ? vp0 : t_apply(tp, vp0);
  V3 S{Pq.x - Pp.x, Pq.y - Pp.y, Pq.z - Pp.z};
  const float norm = normalize3(S);
  if (norm <= kEpsBelow) S.x = 1.0f;
  int p = vbP, q = vbQ, k = 0;
  V3 w{0.0f, 0.0f, 0.0f};
  for (int l = 0;;) {
    const V3 Sp = sysP0 ? S : t_apply_rot_inv(tp, S);
    const V3 Sn{-S.x, -S.y, -S.z};
    const V3 Sq = sysQ0 ? Sn : t_apply_rot_inv(tq, Sn);
    p = support(L, kP, vbP, p, Sp);
    q = support(L, kQ, vbQ, q, Sq);
    const V3 vp = v3(L.verts[p]), vq = v3(L.verts[q]);
    const V3 p0 = sysP0 ? vp : t_apply(tp, vp);
    const V3 q0 = sysQ0 ? vq : t_apply(tq, vq);
    V3 r{q0.x - p0.x, q0.y - p0.y, q0.z - p0.z};
    normalize3(r);
    const float dp = dot3(S, r);
    if (dp >= -kEpsBelow) return 0;
    const int code = sva_slow(H, k, l, (p - vbP) | ((q - vbQ) << 16), r, dp, S, w);
    if (code != 0) return code;
    if (++l >= kMaxIter) return -1;
  }
}

template <int BLOCK>
__global__ void __launch_bounds__(BLOCK) point_small_kernel(SceneImg img, DevRobot rb, SmallPoints qs, int* out) {
  extern __shared__ int4 smem[];
  // dynamic LDS: the scene image, the frames, the lanes' iteration history
  const Lds L = stage_scene<BLOCK>(img, smem);
  T12* frames = reinterpret_cast<T12*>(reinterpret_cast<char*>(smem) + img.bytes);
  f32x4* const lh = reinterpret_cast<f32x4*>(reinterpret_cast<char*>(smem) + img.bytes + sizeof(T12) * kMaxDofDev);
  const History H{lh + threadIdx.x, kMaxIter, BLOCK, nullptr};
  __shared__ int s_word;
  const float* q = qs.q[blockIdx.x];
  if (threadIdx.x < 64) {
    // check_boundaries(q) (robotconfigspace.cpp:795-802)
    const int j = threadIdx.x;
    const bool out_of = j < rb.ndof && (q[j] < rb.mins[j] || q[j] > rb.maxs[j]);
    const bool ob = __ballot(out_of) != 0ull;
    if (j == 0) s_word = ob ? kWordOutOfBounds : kWordFree;
    if (!ob) fk_frames(rb, q, frames);
  }
  __syncthreads();
  if (s_word != kWordOutOfBounds) {
    for (int pair = threadIdx.x; pair < img.M; pair += BLOCK) {
      const int4 pd = L.pairs[pair];
      const int crs = pd.z;
      if ((__hip_atomic_load(&s_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) >> 4) <= crs) continue;
      const int sP = pd.y & 255, sQ = pd.y >> 8;
      T12 tp, tq;
#pragma unroll
      for (int i = 0; i < 12; ++i) tp.m[i] = tq.m[i] = 0.0f;
      if (sP != 0) tp = frames[sP - 1];
      if (sQ != 0) tq = frames[sQ - 1];
      const int code = sva_pair_full(L, tp, tq, sP == 0, sQ == 0, pd.x & 0xffff, (int)((unsigned)pd.x >> 16),
                                     pd.w & 0xffff, (int)((unsigned)pd.w >> 16), H);
      if (code != 0) atomicMin(&s_word, ((crs + 1) << 4) | (code + 1));
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int w = s_word;
    out[blockIdx.x] = w == kWordFree ? 0 : (w & 15) - 1;
  }
}

// Kinematics of the configurations of many scenes in one launch; block b
// belongs to the task with the largest block0 <= b.
template <int NDOF>
__global__ void __launch_bounds__(kFkBlock) fk_points_multi_kernel(const FkTask* __restrict__ tasks, int ntasks) {
  int lo = 0, hi = ntasks - 1;
  const int b = blockIdx.x;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tasks[mid].block0 <= b) lo = mid;
    else hi = mid - 1;
  }
  const FkTask& T = tasks[lo];
  const int i = (b - T.block0) * kFkBlock + threadIdx.x;
  if (i >= T.n) return;
  const int nd = NDOF > 0 ? NDOF : T.rb.ndof;
  float qq[kMaxDofDev];
#pragma unroll
  for (int j = 0; j < (NDOF > 0 ? NDOF : kMaxDofDev); ++j)
    if (NDOF > 0 || j < nd) qq[j] = T.q[i + T.offset * j];
  int st = 0;
  for (int j = 0; j < nd; ++j)
    if (qq[j] < T.rb.mins[j] || qq[j] > T.rb.maxs[j]) { st = 1; break; }
  T.word[i] = st ? kWordOutOfBounds : kWordFree;
  fk_store<NDOF>(T.rb, qq, T.frames, i, T.fstride, [](int, const T12&) {});
}

// codes of every task from its result words (same block map).
__global__ void finalize_points_multi_kernel(const FkTask* __restrict__ tasks, int ntasks) {
  int lo = 0, hi = ntasks - 1;
  const int b = blockIdx.x;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tasks[mid].block0 <= b) lo = mid;
    else hi = mid - 1;
  }
  const FkTask& T = tasks[lo];
  const int i = (b - T.block0) * kFkBlock + threadIdx.x;
  if (i >= T.n) return;
  const int w = T.word[i];
  T.codes[i] = w == kWordFree ? 0 : (w & 15) - 1;
}

}  // namespace

// ----------------------------------------------------------------------------
// launchers
// ----------------------------------------------------------------------------

// Dynamic LDS of a separating-vector block without its history entries: the
// deferral rings and the scene image.
size_t sva_lds_bytes(const SceneImg& img, int block, int gscene) {
  return (gscene ? 0 : (size_t)img.bytes) + sva_ring_bytes(block);
}

int sva_max_lds_bytes() { return 160 * 1024; }

#define GPRM_FK_DISPATCH(KERNEL, GRID, BLOCK, LDS, ST, ...)                                   \
  switch (rb.ndof) {                                                                          \
    case 2: hipLaunchKernelGGL(KERNEL<2>, GRID, BLOCK, LDS, ST, __VA_ARGS__); break;         \
    case 3: hipLaunchKernelGGL(KERNEL<3>, GRID, BLOCK, LDS, ST, __VA_ARGS__); break;         \
    case 4: hipLaunchKernelGGL(KERNEL<4>, GRID, BLOCK, LDS, ST, __VA_ARGS__); break;         \
    case 5: hipLaunchKernelGGL(KERNEL<5>, GRID, BLOCK, LDS, ST, __VA_ARGS__); break;         \
    case 6: hipLaunchKernelGGL(KERNEL<6>, GRID, BLOCK, LDS, ST, __VA_ARGS__); break;         \
    case 7: hipLaunchKernelGGL(KERNEL<7>, GRID, BLOCK, LDS, ST, __VA_ARGS__); break;         \
    case 8: hipLaunchKernelGGL(KERNEL<8>, GRID, BLOCK, LDS, ST, __VA_ARGS__); break;         \
    default: hipLaunchKernelGGL(KERNEL<0>, GRID, BLOCK, LDS, ST, __VA_ARGS__); break;        \
  }

// Threads per kinematics block: kFkBlock when that still gives at least two
// blocks per CU, else 256 (65,536 configurations in 1024-thread blocks
// would occupy 64 of the 256 CUs).
static int fk_block(long long n) { return n >= 2LL * 256 * kFkBlock ? kFkBlock : 256; }

hipError_t launch_fk_points(const DevRobot& rb, const float* q, long long offset, int n, float* frames,
                            long long fstride, int* word, int check_bounds, unsigned* zero_counter,
                            hipStream_t st, const unsigned char* skip, int* group_done) {
  if (n <= 0) return hipSuccess;
  const int fb = fk_block(n);
  dim3 grid((n + fb - 1) / fb), block(fb);
  GPRM_FK_DISPATCH(fk_points_kernel, grid, block, 0, st, rb, q, offset, n, frames, fstride, word,
                   check_bounds, zero_counter, skip, group_done);
  return hipGetLastError();
}

hipError_t launch_frames_unpack(const DevRobot& rb, const float* frames, long long fstride, int n, float* out,
                               hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(frames_unpack_kernel, dim3((n + 255) / 256), dim3(256), 0, st, rb, frames, fstride, n, out);
  return hipGetLastError();
}

hipError_t launch_finalize_points(const int* word, int* codes, int n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(finalize_points_kernel, dim3((n + 255) / 256), dim3(256), 0, st, word, codes, n);
  return hipGetLastError();
}

hipError_t launch_edge_fk(const DevRobot& rb, EdgeArgs ea, const int* item_edge, const int* item_pos,
                          const int* nitems, int cap, float* frames, const SceneImg& img, unsigned long long* mask,
                          hipStream_t st) {
  if (cap <= 0) return hipSuccess;
  int fb = fk_block(cap);
  if (mask != nullptr && !cull_fits(img, fb)) fb = 256;
  if (mask != nullptr && !cull_fits(img, fb)) return hipErrorInvalidValue;
  const size_t lds = mask != nullptr ? cull_lds_bytes(img.nworld, img.nmov, fb) : 0;
  int blocks = (cap + fb - 1) / fb;
  if (blocks > 4096) blocks = 4096;
  dim3 grid(blocks), block(fb);
  GPRM_FK_DISPATCH(fk_edges_kernel, grid, block, lds, st, rb, ea, item_edge, item_pos, nitems, cap, frames,
                   (long long)cap, img, mask);
  return hipGetLastError();
}

template <int EDGE, int BLOCK, int WAVES, int GS>
static const void* sva_fn() {
  return reinterpret_cast<const void*>(&sva_kernel<EDGE, BLOCK, WAVES, GS>);
}

template <int GS>
static const void* sva_variant_gs(int edge_mode, int block, int waves) {
  if (block == 256 && waves == 5) return edge_mode ? sva_fn<1, 256, 5, GS>() : sva_fn<0, 256, 5, GS>();
  if (block == 256 && waves == 4) return edge_mode ? sva_fn<1, 256, 4, GS>() : sva_fn<0, 256, 4, GS>();
  if (block == 1024 && waves == 4) return edge_mode ? sva_fn<1, 1024, 4, GS>() : sva_fn<0, 1024, 4, GS>();
  return nullptr;
}

// The kernel variants a shape may name: (block, waves per SIMD), the scene
// in LDS or (gscene) in the global image.
static const void* sva_variant(int edge_mode, int block, int waves, int gscene) {
  return gscene ? sva_variant_gs<1>(edge_mode, block, waves) : sva_variant_gs<0>(edge_mode, block, waves);
}

template <int EDGE, int BLOCK, int WAVES>
static const void* sva_multi_fn() {
  return reinterpret_cast<const void*>(&sva_multi_kernel<EDGE, BLOCK, WAVES>);
}

static const void* sva_multi_variant(int edge_mode, int block, int waves) {
  if (block == 256 && waves == 5) return edge_mode ? sva_multi_fn<1, 256, 5>() : sva_multi_fn<0, 256, 5>();
  if (block == 256 && waves == 4) return edge_mode ? sva_multi_fn<1, 256, 4>() : sva_multi_fn<0, 256, 4>();
  if (block == 1024 && waves == 4) return edge_mode ? sva_multi_fn<1, 1024, 4>() : sva_multi_fn<0, 1024, 4>();
  return nullptr;
}

// LDS is handed out in granules; of a block's last one 64 bytes are left for
// the kernels' static variables.
constexpr size_t kLdsGranule = 1280, kLdsStatic = 64;

// The history entries per lane that fit into LDS beside `lds` other bytes of
// each block, with as many blocks per CU as a launch of sh.grid blocks needs
// at once: none of them waits for another's LDS.
static int history_entries(const SvaShape& sh, size_t lds) {
  if (sh.cus < 1 || sh.grid < 1) return 0;
  const size_t per_cu = (size_t)((sh.grid + sh.cus - 1) / sh.cus);
  const size_t room = (size_t)sva_max_lds_bytes() / kLdsGranule / per_cu * kLdsGranule;
  if (room < lds + kLdsStatic) return 0;
  return (int)std::min<size_t>(kMaxIter, (room - lds - kLdsStatic) / (sizeof(float4) * (size_t)sh.block));
}
static size_t history_lds(int entries, int block) { return sizeof(float4) * (size_t)entries * (size_t)block; }

// Resident blocks over all CUs of a kernel variant with lds dynamic bytes.
static hipError_t resident_grid(const void* const fns[2], int block, size_t lds, int device, int* grid, int* cus) {
  int blocks = 0;
  hipError_t e = hipDeviceGetAttribute(cus, hipDeviceAttributeMultiprocessorCount, device);
  if (e != hipSuccess) return e;
  // the occupancy query sees the dynamic LDS only once the attribute allows
  // it, and small launches add history entries up to all of a CU's
  const size_t most = std::max(lds, (size_t)sva_max_lds_bytes() - kLdsStatic);
  for (int em = 0; em < 2; ++em) {
    if (!fns[em]) return hipErrorInvalidValue;
    if ((e = hipFuncSetAttribute(fns[em], hipFuncAttributeMaxDynamicSharedMemorySize, (int)most)) != hipSuccess)
      return e;
  }
  e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, fns[1], block, lds);
  if (e != hipSuccess) return e;
  if (blocks < 1) return hipErrorInvalidConfiguration;
  *grid = *cus * blocks;
  return hipSuccess;
}

hipError_t sva_multi_shape_finish(size_t img_bytes, SvaShape* sh, int device) {
  const size_t lds = img_bytes + sva_ring_bytes(sh->block);
  if (lds > (size_t)sva_max_lds_bytes() - 16) return hipErrorInvalidValue;
  if (sh->ppu < 1 || sh->ppu > 256) return hipErrorInvalidValue;
  const void* fns[2] = {sva_multi_variant(0, sh->block, sh->waves), sva_multi_variant(1, sh->block, sh->waves)};
  return resident_grid(fns, sh->block, lds, device, &sh->grid, &sh->cus);
}

hipError_t sva_shape_finish(const SceneImg& img, SvaShape* sh, int device) {
  sh->gscene = sva_lds_bytes(img, sh->block) > (size_t)sva_max_lds_bytes() ? 1 : 0;
  const size_t lds = sva_lds_bytes(img, sh->block, sh->gscene);
  if (lds > (size_t)sva_max_lds_bytes()) return hipErrorInvalidValue;
  if (sh->ppu < 1 || sh->ppu > 256) return hipErrorInvalidValue;
  const void* fns[2] = {sva_variant(0, sh->block, sh->waves, sh->gscene),
                        sva_variant(1, sh->block, sh->waves, sh->gscene)};
  return resident_grid(fns, sh->block, lds, device, &sh->grid, &sh->cus);
}

SvaShape sva_default_shape(const SceneImg& img) {
  SvaShape sh;
  // 256-thread blocks at five waves per SIMD (five blocks per CU) when five
  // scene copies fit in LDS, at four when four fit, else one 1024-thread
  // block sharing a single copy; units of up to 128 pairs (measured fastest
  // on the edge-checking workload; launches shrink them when there are too
  // few items, see unit_pairs in the host runtime)
  if (5 * sva_lds_bytes(img, 256) <= (size_t)sva_max_lds_bytes()) {
    sh.block = 256;
    sh.waves = 5;
  } else if (4 * sva_lds_bytes(img, 256) <= (size_t)sva_max_lds_bytes()) {
    sh.block = 256;
    sh.waves = 4;
  } else if (sva_lds_bytes(img, 1024) <= (size_t)sva_max_lds_bytes()) {
    sh.block = 1024;
    sh.waves = 4;
  } else {
    // beyond LDS: the scene is read from the global image (sva_shape_finish
    // sets gscene), and LDS holds only the rings
    sh.block = 256;
    sh.waves = 5;
  }
  sh.ppu = 128;
  return sh;
}

hipError_t launch_sva(const SvaArgs& a, int edge_mode, const SvaShape& sh, hipStream_t st) {
  size_t lds = sva_lds_bytes(a.img, sh.block, sh.gscene);
  if (lds > (size_t)sva_max_lds_bytes() || a.hist == nullptr || sh.grid < 1) return hipErrorInvalidValue;
  const void* fn = sva_variant(edge_mode, sh.block, sh.waves, sh.gscene);
  if (!fn) return hipErrorInvalidValue;
  SvaArgs b = a;
  b.lds_hist = history_entries(sh, lds);
  lds += history_lds(b.lds_hist, sh.block);
  void* args[] = {&b};
  return hipLaunchKernel(fn, dim3(sh.grid), dim3(sh.block), args, lds, st);
}

// LDS of a small point-check block: the image, the frames and BLOCK lanes'
// iteration history.
static size_t point_small_lds(const SceneImg& img, int block) {
  return (size_t)img.bytes + sizeof(T12) * kMaxDofDev + sizeof(float4) * kMaxIter * (size_t)block;
}

hipError_t launch_support_factors(const SceneImg& img, char* blob, hipStream_t st) {
  if (img.N <= 0) return hipSuccess;
  hipLaunchKernelGGL(support_factor_kernel, dim3(img.N), dim3(kCertBlock), 0, st, img, blob);
  return hipGetLastError();
}

hipError_t point_small_prepare(const SceneImg& img) {
  for (int block : {256, 64}) {
    const size_t lds = point_small_lds(img, block);
    if (lds > (size_t)sva_max_lds_bytes()) continue;
    const void* fn = block == 256 ? reinterpret_cast<const void*>(&point_small_kernel<256>)
                                  : reinterpret_cast<const void*>(&point_small_kernel<64>);
    if (lds > 64 * 1024) return hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    return hipSuccess;
  }
  return hipErrorInvalidValue;
}

hipError_t launch_point_small(const SceneImg& img, const DevRobot& rb, const SmallPoints& qs, int* out,
                              hipStream_t st) {
  if (qs.n <= 0) return hipSuccess;
  if (qs.n > kSmallMax) return hipErrorInvalidValue;
  if (point_small_lds(img, 256) <= (size_t)sva_max_lds_bytes())
    hipLaunchKernelGGL(point_small_kernel<256>, dim3(qs.n), dim3(256), point_small_lds(img, 256), st, img, rb, qs, out);
  else if (point_small_lds(img, 64) <= (size_t)sva_max_lds_bytes())
    hipLaunchKernelGGL(point_small_kernel<64>, dim3(qs.n), dim3(64), point_small_lds(img, 64), st, img, rb, qs, out);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_sva_multi(const SceneTask* d_tasks, int ntasks, int edge_mode, const SvaShape& sh, size_t img_bytes,
                            unsigned long long* t_start, unsigned long long* tally, hipStream_t st) {
  if (ntasks <= 0) return hipSuccess;
  size_t lds = img_bytes + sva_ring_bytes(sh.block);
  if (lds > (size_t)sva_max_lds_bytes() - 16 || sh.grid < 1) return hipErrorInvalidValue;
  const void* fn = sva_multi_variant(edge_mode, sh.block, sh.waves);
  if (!fn) return hipErrorInvalidValue;
  int entries = history_entries(sh, lds);
  lds += history_lds(entries, sh.block);
  void* args[] = {const_cast<SceneTask**>(&d_tasks), &ntasks, &t_start, &tally, &entries};
  return hipLaunchKernel(fn, dim3(sh.grid), dim3(sh.block), args, lds, st);
}

hipError_t launch_fk_points_multi(const FkTask* d_tasks, int ntasks, int nblocks, int ndof, hipStream_t st) {
  if (ntasks <= 0 || nblocks <= 0) return hipSuccess;
  dim3 grid(nblocks), block(kFkBlock);
  switch (ndof) {
    case 2: hipLaunchKernelGGL(fk_points_multi_kernel<2>, grid, block, 0, st, d_tasks, ntasks); break;
    case 3: hipLaunchKernelGGL(fk_points_multi_kernel<3>, grid, block, 0, st, d_tasks, ntasks); break;
    case 4: hipLaunchKernelGGL(fk_points_multi_kernel<4>, grid, block, 0, st, d_tasks, ntasks); break;
    case 5: hipLaunchKernelGGL(fk_points_multi_kernel<5>, grid, block, 0, st, d_tasks, ntasks); break;
    case 6: hipLaunchKernelGGL(fk_points_multi_kernel<6>, grid, block, 0, st, d_tasks, ntasks); break;
    case 7: hipLaunchKernelGGL(fk_points_multi_kernel<7>, grid, block, 0, st, d_tasks, ntasks); break;
    default: hipLaunchKernelGGL(fk_points_multi_kernel<0>, grid, block, 0, st, d_tasks, ntasks); break;
  }
  return hipGetLastError();
}

hipError_t launch_finalize_points_multi(const FkTask* d_tasks, int ntasks, int nblocks, hipStream_t st) {
  if (ntasks <= 0 || nblocks <= 0) return hipSuccess;
  hipLaunchKernelGGL(finalize_points_multi_kernel, dim3(nblocks), dim3(kFkBlock), 0, st, d_tasks, ntasks);
  return hipGetLastError();
}

hipError_t launch_edge_prologue(const DevRobot& rb, float dq, EdgeArgs ea, int* testnum_out, int* max_testnum,
                                unsigned long long* total, unsigned* blocks, EdgePinned* host, hipStream_t st) {
  if (ea.nedges <= 0) return hipSuccess;
  dim3 grid((ea.nedges + kPrologueBlock - 1) / kPrologueBlock), block(kPrologueBlock);
  hipLaunchKernelGGL(edge_prologue_kernel, grid, block, 0, st, rb.ndof, dq, ea, testnum_out,
                     max_testnum, total, blocks, host);
  return hipGetLastError();
}

hipError_t launch_edge_compact(EdgeArgs ea, const EdgeLaunch& p, int* item_edge, int* item_pos, int* nitems,
                               int* nsamples, int* overflow, unsigned* zero_queues, hipStream_t st) {
  if (p.e1 <= p.e0) return hipSuccess;
  const int x = (p.e1 - p.e0 + kCompactBlock - 1) / kCompactBlock, ranks = p.r1 - p.r0;
  dim3 grid(x, edge_slices(ranks, x)), block(kCompactBlock);
  hipLaunchKernelGGL(edge_compact_kernel, grid, block, 0, st, ea, p, item_edge, item_pos, nitems, nsamples,
                     zero_queues, edge_slice(ranks, x), overflow);
  return hipGetLastError();
}

hipError_t launch_edge_prologue_multi(const EdgeTask* d_tasks, int ntasks, int nblocks, hipStream_t st) {
  if (ntasks <= 0 || nblocks <= 0) return hipSuccess;
  hipLaunchKernelGGL(edge_prologue_multi_kernel, dim3(nblocks), dim3(256), 0, st, d_tasks, ntasks);
  return hipGetLastError();
}

hipError_t launch_edge_compact_multi(const EdgeTask* d_tasks, int ntasks, int nblocks, hipStream_t st) {
  if (ntasks <= 0 || nblocks <= 0) return hipSuccess;
  hipLaunchKernelGGL(edge_compact_multi_kernel, dim3(nblocks), dim3(kCompactBlockMulti), 0, st, d_tasks, ntasks);
  return hipGetLastError();
}

hipError_t launch_edge_fk_multi(const EdgeTask* d_tasks, int ntasks, int nblocks, int ndof, size_t cull_lds,
                                hipStream_t st) {
  if (ntasks <= 0 || nblocks <= 0) return hipSuccess;
  dim3 grid(nblocks), block(kFkBlock);
  switch (ndof) {
    case 2: hipLaunchKernelGGL(fk_edges_multi_kernel<2>, grid, block, cull_lds, st, d_tasks, ntasks); break;
    case 3: hipLaunchKernelGGL(fk_edges_multi_kernel<3>, grid, block, cull_lds, st, d_tasks, ntasks); break;
    case 4: hipLaunchKernelGGL(fk_edges_multi_kernel<4>, grid, block, cull_lds, st, d_tasks, ntasks); break;
    case 5: hipLaunchKernelGGL(fk_edges_multi_kernel<5>, grid, block, cull_lds, st, d_tasks, ntasks); break;
    case 6: hipLaunchKernelGGL(fk_edges_multi_kernel<6>, grid, block, cull_lds, st, d_tasks, ntasks); break;
    case 7: hipLaunchKernelGGL(fk_edges_multi_kernel<7>, grid, block, cull_lds, st, d_tasks, ntasks); break;
    default: hipLaunchKernelGGL(fk_edges_multi_kernel<0>, grid, block, cull_lds, st, d_tasks, ntasks); break;
  }
  return hipGetLastError();
}

CellGrid make_cell_grid_dims(int dims, const float* mins, const float* maxs, float D);

CellGrid make_cell_grid(int ndof, const float* mins, const float* maxs, float D) {
  // as many gridded coordinates as kGridMaxCells allows (at most kGridDims)
  for (int dims = ndof < kGridDims ? ndof : kGridDims; dims >= 1; --dims) {
    CellGrid g = make_cell_grid_dims(dims, mins, maxs, D);
    if (g.ncells <= kGridMaxCells || dims == 1) return g;
  }
  return make_cell_grid_dims(1, mins, maxs, D);
}

CellGrid make_cell_grid_dims(int dims, const float* mins, const float* maxs, float D) {
  CellGrid g{};
  g.dims = dims;
  g.ncells = 1;
  for (int d = 0; d < kGridDims; ++d) {
    g.cells[d] = 1;
    g.lo[d] = 0.0f;
    g.inv[d] = 0.0f;
    if (d >= g.dims) continue;
    const float span = maxs[d] - mins[d];
    int c = (span > 0.0f && D > 0.0f) ? (int)std::floor(span / D) : 1;
    c = c < 1 ? 1 : (c > 64 ? 64 : c);
    g.cells[d] = c;
    g.lo[d] = mins[d];
    g.inv[d] = span > 0.0f ? (float)c / span : 0.0f;
    // a cell must stay at least D wide after rounding of inv
    while (g.cells[d] > 1 && (float)(1.0 / g.inv[d]) < D) {
      g.cells[d] -= 1;
      g.inv[d] = (float)g.cells[d] / span;
    }
    g.ncells *= g.cells[d];
  }
  return g;
}

hipError_t launch_grid_build(const CellGrid& g, int ndof, const float* nodes, int n, long long noff, int* cell_id,
                             int* counts, int* starts, int* cursor, float* sorted, int* sid, hipStream_t st) {
  hipError_t e = launch_fill_i32(counts, 0, g.ncells, st);
  if (e != hipSuccess || n <= 0) return e;
  const dim3 grid((n + 255) / 256), block(256);
  hipLaunchKernelGGL(grid_count_kernel, grid, block, 0, st, g, nodes, n, noff, cell_id, counts);
  hipLaunchKernelGGL(grid_scan_kernel, dim3(1), dim3(1024), 0, st, counts, starts, cursor, g.ncells);
  hipLaunchKernelGGL(grid_scatter_kernel, grid, block, 0, st, ndof, nodes, n, noff, cell_id, cursor, sorted, sid);
  return hipGetLastError();
}

hipError_t launch_near_grid(int ndof, const float* queries, int nq, long long qoff, const CellGrid& g,
                            const int* starts, const int* counts, const float* sorted, const int* sid, int n, float D2,
                            int* qcount, long long* qstart, long long* total, int* out_q, int* out_node,
                            float* out_d2, int cap, hipStream_t st) {
  if (nq > 0)
    hipLaunchKernelGGL(near_grid_kernel<0>, dim3(nq), dim3(256), 0, st, ndof, queries, nq, qoff, g, starts, counts,
                       sorted, sid, n, D2, qcount, qstart, out_q, out_node, out_d2, cap);
  hipLaunchKernelGGL(near_scan_kernel, dim3(1), dim3(1024), 0, st, qcount, nq, qstart, total);
  if (nq > 0)
    hipLaunchKernelGGL(near_grid_kernel<1>, dim3(nq), dim3(256), 0, st, ndof, queries, nq, qoff, g, starts, counts,
                       sorted, sid, n, D2, qcount, qstart, out_q, out_node, out_d2, cap);
  return hipGetLastError();
}

hipError_t launch_fill_i32(int* p, int v, long long n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  long long b = (n + 255) / 256;
  if (b > 4096) b = 4096;
  hipLaunchKernelGGL(fill_i32_kernel, dim3((unsigned)b), dim3(256), 0, st, p, v, n);
  return hipGetLastError();
}

hipError_t launch_fill_u32(unsigned int* p, unsigned int v, long long n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  long long b = (n + 255) / 256;
  if (b > 4096) b = 4096;
  hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)b), dim3(256), 0, st, p, v, n);
  return hipGetLastError();
}

}  // namespace gprm
