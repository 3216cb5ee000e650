// kd_adjoint.hip -- reverse sweep of the kD-tree step on gfx950.
//
// The step (simple_sim, Parallel/RustVersion/src/array_kd_tree.rs:623-664)
// with its tree topology frozen: the tree of step k and every body's
// accept/open decisions are those of the forward run, so within the step the
// accelerations are a smooth function of positions p and masses m:
//   a_i = sum_{j in P2P(i)} f(p_i - p_j, m_j) + sum_{n in M2P(i)} f(p_i - c_n, M_n),
//   f(d, m) = -m d / |d|^3,  M_n = sum m_j,  c_n = sum m_j p_j / M_n.
// Backward through v' = v + dt a(p), p' = p + dt v' (array_kd_tree.rs:649-662):
//   lv += dt lp;  u = dt lv;  lp += (da/dp)^T u;  lm += (da/dm)^T u.
// k_adj_walk replays the forward walk (FP64: the same decisions; mixed: but
// for nodes within an ulp or two of the opening threshold, whose |d|^2 is
// rounded after every operation here and fused there) and adds, per term,
//   d/dp_i (u_i . f) = -m (u_i / r^3 - 3 (d.u_i) d / r^5)  to body i,
// its negative to the partner body (P2P) or to the node's centre of mass
// (M2P), and -(u_i . d) / r^3 to the partner's mass or the node's mass.
// k_adj_nodes carries node terms to the members: dc/dp_j = m_j / M,
// dc/dm_j = (p_j - c) / M, dM/dm_j = 1.  All adjoint sums are FP64 (global
// FP64 atomics); the mixed path evaluates its terms in FP32 like its forward
// walk.  Adjoint arrays are in original body order.
//
// What bounds the walk is latency: at 100,000 bodies there are 1,563
// wavefronts of 64 bodies, each a chain of some 1,000 node and 750 leaf-body
// visits.  So a workgroup of S wavefronts walks 64 bodies, each taking every
// S-th subtree of depth log2(S) + 2 (the sums are atomic, so their order is
// free); leaf bodies come in batches of scalar loads; and the reactions of a
// batch, one column of 64 lanes per value, are summed in registers by
// exchanging halves: a stage adds two columns into one (the lanes of one half
// keep the first, of the other half the second), 16 columns take 15 such adds
// and 2 more, and one atomic instruction adds the batch to consecutive words (the
// reactions are kept in tree order).  At 100,000 ring bodies the mixed walk
// takes 0.63 ms against 1.57 with one wavefront, bodies one by one and the
// reactions through LDS (a row of 34 doubles a lane, 17 KB a wavefront); the
// atomics are 0.18 ms of it.  0.27 ms of the difference came with records and
// bodies through the scalar unit (uniform_load), the next record fetched while
// a node is worked on: FP64 needs 84 registers instead of 110, five wavefronts
// a SIMD instead of four.
#include <algorithm>

#include "kd_internal.hpp"

namespace kd {

__device__ __forceinline__ uint32_t uni_a(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)x);
}

// gd = d/dd (u . f(d, mq)), gm = d/dmq (u . f(d, mq)), FP64; d2 = |d|^2.
// One reciprocal stands for the quotients by r^3, r^2 and r^3 again; residuals
// and fused operations take away the roundings that brings in: over 2e6 random
// terms the error of gd is 2.11 (rms; at most 11.9) times 2^-53 of its length,
// gm's 0.78, and with five quotients and no fused operations 2.21 (11.9) and
// 0.82.  Gradients of 20 steps in ms with three quotients / plain products
// of the reciprocal (errors 2.50, 13.3 and 0.85) / this: 9.40 / 9.20 / 9.35 at 1,000
// ring bodies, 35.9 / 34.1 / 34.7 at 40,000, 53.8 / 51.0 / 51.4 at 100,000.
__device__ __forceinline__ void vjp64(double dx, double dy, double dz, double d2, double mq,
                                      double ux, double uy, double uz, double &gx, double &gy,
                                      double &gz, double &gm) {
#pragma clang fp contract(off)
  const double r = sqrt(d2), r3 = d2 * r, ri3 = 1.0 / r3, ri2 = r * ri3;
  const double du = __builtin_fma(dz, uz, __builtin_fma(dy, uy, dx * ux));
  // du / d2 and du / r3, each corrected by its residual
  double e = du * ri2, t = du * ri3;
  e = __builtin_fma(__builtin_fma(-d2, e, du), ri2, e);
  t = __builtin_fma(__builtin_fma(-r3, t, du), ri3, t);
  const bool far = ri3 == 0.0;  // r^3 overflows: no term
  const double k = far ? 0.0 : -3.0 * e, w = -mq * ri3;
  gx = w * __builtin_fma(k, dx, ux);
  gy = w * __builtin_fma(k, dy, uy);
  gz = w * __builtin_fma(k, dz, uz);
  gm = far ? 0.0 : -t;
}

// The same in FP32 with a hardware reciprocal square root (mixed path), from
// the differences and their d2.  The fused operations are written out, so that
// a term's rounding does not depend on the code around it.
__device__ __forceinline__ void vjp32(float dx, float dy, float dz, float d2, float mq, float ux,
                                      float uy, float uz, float &gx, float &gy, float &gz,
                                      float &gm) {
#pragma clang fp contract(off)
  const float ri = __builtin_amdgcn_rsqf(d2);
  const float ri2 = ri * ri;
  const float ri3 = ri2 * ri;
  const float du = __builtin_fmaf(dz, uz, __builtin_fmaf(dx, ux, dy * uy));
  const float k = 3.f * du * ri3 * ri2;
  gx = -mq * __builtin_fmaf(ux, ri3, -(k * dx));
  gy = -mq * __builtin_fmaf(uy, ri3, -(k * dy));
  gz = -mq * __builtin_fmaf(uz, ri3, -(k * dz));
  gm = -du * ri3;
}

struct AdjWalk {
  const NodeRec64 *rec64;  // one step's tree (heap order)
  const NodeRec32 *rec32;
  const double4 *pos64;    // tree order (x, y, z, m)
  const float4 *pos32;
  const uint32_t *oid;     // tree position -> original index
  const double *ux, *uy, *uz;  // seed, original order
  double *react;  // per tree position: d/dp (x, y, z) and d/dm of this step
  double *gnode;  // per heap slot: d/dc (x, y, z) and d/dM
  uint32_t n;
  uint32_t leaf;
  double theta2;
};

// a + b, where lane l of a column gives to lane l ^ 32 (SWAP 32) or l ^ 16
// (SWAP 16) and the lanes with that bit clear keep column a, the others b.
template <int SWAP>
__device__ __forceinline__ double fold_swap(double a, double b) {
  typedef uint32_t pair __attribute__((ext_vector_type(2)));
  const uint32_t al = (uint32_t)__double2loint(a), ah = (uint32_t)__double2hiint(a);
  const uint32_t bl = (uint32_t)__double2loint(b), bh = (uint32_t)__double2hiint(b);
  pair lo, hi;
  if (SWAP == 32) {
    lo = __builtin_amdgcn_permlane32_swap(al, bl, false, false);
    hi = __builtin_amdgcn_permlane32_swap(ah, bh, false, false);
  } else {
    lo = __builtin_amdgcn_permlane16_swap(al, bl, false, false);
    hi = __builtin_amdgcn_permlane16_swap(ah, bh, false, false);
  }
  return __hiloint2double((int)hi.x, (int)lo.x) + __hiloint2double((int)hi.y, (int)lo.y);
}
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
// The same within a row of 16, where CTRL takes lane l to one whose bit
// differs and `second` says whether the lane keeps column b.
template <int CTRL>
__device__ __forceinline__ double fold_row(double a, double b, bool second) {
  const double keep = second ? b : a, give = second ? a : b;
  return keep + dpp_f64<CTRL>(give);
}
constexpr int ROW_ROR8 = 0x128, ROW_HALF_MIRROR = 0x141, QUAD_2301 = 0x4E, QUAD_1032 = 0xB1;

// Sums of the wavefront's 4 columns v: lane 16 q + r holds column
// fold4_col(lane).
__device__ __forceinline__ double fold4(const double v[4]) {
  double s = fold_swap<16>(fold_swap<32>(v[0], v[1]), fold_swap<32>(v[2], v[3]));
  s += dpp_f64<ROW_ROR8>(s);
  s += dpp_f64<ROW_HALF_MIRROR>(s);
  s += dpp_f64<QUAD_2301>(s);
  s += dpp_f64<QUAD_1032>(s);
  return s;
}
__device__ __forceinline__ uint32_t fold4_col(uint32_t lane) {
  return (lane >> 5) | ((lane >> 3) & 2u);
}
// Sums of 16 columns: lane l holds column fold16_col(l).
__device__ __forceinline__ double fold16(const double v[16], uint32_t lane) {
  double a[8], b[4], c[2];
#pragma unroll
  for (int i = 0; i < 8; ++i) a[i] = fold_swap<32>(v[2 * i], v[2 * i + 1]);
#pragma unroll
  for (int i = 0; i < 4; ++i) b[i] = fold_swap<16>(a[2 * i], a[2 * i + 1]);
#pragma unroll
  for (int i = 0; i < 2; ++i)
    c[i] = fold_row<ROW_ROR8>(b[2 * i], b[2 * i + 1], (lane & 8u) != 0);
  double s = fold_row<ROW_HALF_MIRROR>(c[0], c[1], (lane & 4u) != 0);
  s += dpp_f64<QUAD_2301>(s);
  s += dpp_f64<QUAD_1032>(s);
  return s;
}
__device__ __forceinline__ uint32_t fold16_col(uint32_t lane) {
  return (lane >> 5) | ((lane >> 3) & 2u) | ((lane >> 1) & 4u) | ((lane << 1) & 8u);
}

// A node record or a body at a wave-uniform byte offset.  The address is given
// as constant memory, so that the scalar unit loads it: beside the walk's
// atomics the compiler takes a plain load for one that may change, and loads
// into vector registers, a lane each, what every lane reads alike.
template <class T>
__device__ __forceinline__ T uniform_load(const T *base, uint64_t off) {
  typedef uint32_t words __attribute__((ext_vector_type(sizeof(T) / 4), aligned(16)));
  typedef const words __attribute__((address_space(4))) *ptr;
  const words w = *(ptr)(reinterpret_cast<uintptr_t>(base) + off);
  T r;
  __builtin_memcpy(&r, &w, sizeof(T));
  return r;
}
template <class Rec>
__device__ __forceinline__ Rec adj_rec(const Rec *nodes_m1, uint32_t off) {
  return uniform_load(nodes_m1, uni_a(off));
}

template <bool MIXED>
struct AdjForm {
  using Rec = NodeRec64;
  using Body = double4;
  __device__ static const Rec *nodes(const AdjWalk &a) { return a.rec64 - 1; }
  __device__ static const Body *bodies(const AdjWalk &a) { return a.pos64; }
};
template <>
struct AdjForm<true> {
  using Rec = NodeRec32;
  using Body = float4;
  __device__ static const Rec *nodes(const AdjWalk &a) { return a.rec32 - 1; }
  __device__ static const Body *bodies(const AdjWalk &a) { return a.pos32; }
};

// Positions in the tree are byte offsets h RS of the records, and a lane's
// acceptance level is kept as in the forward walk (kd_traverse.hip).
template <bool MIXED, int S>
__global__ __launch_bounds__(64 * S) void k_adj_walk(AdjWalk a, int lzd) {
#pragma clang fp contract(off)
  using F = AdjForm<MIXED>;
  using Rec = typename F::Rec;
  using Body = typename F::Body;
  constexpr uint32_t RS = sizeof(Rec);
  constexpr int RSL = RS == 32 ? 5 : 6;
  constexpr int BATCH = 4;  // leaf bodies whose reactions are summed together
  const Rec *nodes = F::nodes(a);
  const Body *bodies = F::bodies(a);
  const uint32_t wbase = xcd_block() * 64u, lane = threadIdx.x & 63;
  const uint32_t w = uni_a(threadIdx.x >> 6);
  const uint32_t me = wbase + lane;
  const bool valid = me < a.n;
  const uint32_t ms = valid ? me : wbase;
  const Body p = bodies[ms];
  const uint32_t o = a.oid[ms];
  const double ux = valid ? a.ux[o] : 0.0, uy = valid ? a.uy[o] : 0.0,
               uz = valid ? a.uz[o] : 0.0;
  const float uxf = (float)ux, uyf = (float)uy, uzf = (float)uz;
  double sx = 0.0, sy = 0.0, sz = 0.0;
  int E = valid ? -RSL : 32 - RSL;
  const uint32_t col4 = fold4_col(lane), col16 = fold16_col(lane);

  // one term of a lane that takes it (use), 0 otherwise: the lane's own sum,
  // and the reaction v
  auto term = [&](auto dx, auto dy, auto dz, auto d2, auto m, bool use, double v[4]) {
    double gx, gy, gz, gm;
    if constexpr (MIXED) {
      float fx, fy, fz, fm;
      vjp32(dx, dy, dz, d2, m, uxf, uyf, uzf, fx, fy, fz, fm);
      gx = use ? fx : 0.f, gy = use ? fy : 0.f, gz = use ? fz : 0.f, gm = use ? fm : 0.f;
    } else {
      vjp64(dx, dy, dz, d2, m, ux, uy, uz, gx, gy, gz, gm);
      gx = use ? gx : 0.0, gy = use ? gy : 0.0, gz = use ? gz : 0.0, gm = use ? gm : 0.0;
    }
    sx += gx;
    sy += gy;
    sz += gz;
    v[0] = -gx, v[1] = -gy, v[2] = -gz, v[3] = gm;
  };
  // the next record is loaded as soon as its position is known
  auto inner = [&](Rec &r, uint32_t h, int lz, bool mine) {
    const uint64_t actm = __builtin_amdgcn_ballot_w64(lz >= E);
    const auto dx = p.x - r.cx, dy = p.y - r.cy, dz = p.z - r.cz;
    const auto d2 = dx * dx + dy * dy + dz * dz;
    bool ok;
    if constexpr (MIXED)
      // size^2 / theta^2 < d2.  (The forward walk fuses its d2, so a node that
      // lies that close to the threshold may be taken by one and opened by the
      // other: some of a step's 1e8 tests at 100,000 bodies, 4e-8 of a gradient
      // whose FP32 terms are 5e-4 off.)
      ok = r.size2 < d2;
    else
      ok = r.size2 < a.theta2 * d2;
    const uint64_t tm = actm & __builtin_amdgcn_ballot_w64(ok);
    const uint64_t om = actm & ~tm;
    const uint32_t hn = om ? 2 * h : r.skip;
    const auto m = scalar_copy(r.m);
    r = adj_rec(nodes, hn);
    if (mine && tm) {
      double v[4];
      term(dx, dy, dz, d2, m, __builtin_amdgcn_inverse_ballot_w64(tm), v);
      const double s = fold4(v);
      if ((lane & 15u) == 0) atomicAdd(a.gnode + 4 * (size_t)(h / RS - 1) + col4, s);
    }
    E = __builtin_amdgcn_inverse_ballot_w64(om) ? -RSL : max(E, lz);
    return hn;
  };
  auto leaf = [&](uint32_t start, uint32_t count, int lz) {
    const bool active = lz >= E;
    for (uint32_t b = 0; b < count; b += BATCH) {
      const uint32_t j0 = start + b, m = min((uint32_t)BATCH, count - b);
      struct Batch {
        Body q[BATCH];
      };
      // past the leaf: still inside the padded body arrays
      const Batch t = uniform_load(reinterpret_cast<const Batch *>(bodies),
                                   (uint64_t)j0 * sizeof(Body));
      const Body *q = t.q;
      double v[4 * BATCH];
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        if ((uint32_t)i < m) {  // wave-uniform
          const auto dx = p.x - q[i].x, dy = p.y - q[i].y, dz = p.z - q[i].z;
          auto d2 = dx * dx + dy * dy + dz * dz;
          if constexpr (MIXED) d2 = __builtin_fmaf(dz, dz, __builtin_fmaf(dx, dx, dy * dy));
          term(dx, dy, dz, d2, q[i].w, active && j0 + i != me, v + 4 * i);
        } else {
          v[4 * i] = v[4 * i + 1] = v[4 * i + 2] = v[4 * i + 3] = 0.0;
        }
      }
      const double s = fold16(v, lane);
      if ((lane & 3u) == 0 && col16 < 4 * m) atomicAdd(a.react + 4 * (size_t)j0 + col16, s);
    }
  };

  uint32_t h = RS, parts = 0;
  bool mine = w == 0;
  do {
    const int lz = __builtin_clz(h);
    if (lz == lzd) {
      mine = (parts++ & (S - 1u)) == w;
      uint32_t x = h / RS;
      x >>= __builtin_ctz(~x);
      const uint32_t next = x == 0 ? 0 : (x + 1) * RS;
      if (mine) {
        Rec r = adj_rec(nodes, h);
        do {
          const int l = __builtin_clz(h);
          if (r.count <= a.leaf) {
            const uint32_t start = scalar_copy(r.start), count = scalar_copy(r.count);
            h = r.skip;
            r = adj_rec(nodes, h);
            leaf(start, count, l);
          } else {
            h = inner(r, h, l, true);
          }
        } while (h != next);
      }
      h = next;
    } else {
      Rec r = adj_rec(nodes, h);
      h = inner(r, h, lz, mine);
    }
  } while (h != 0);
  if (valid) {
    atomicAdd(a.react + 4 * (size_t)me, sx);
    atomicAdd(a.react + 4 * (size_t)me + 1, sy);
    atomicAdd(a.react + 4 * (size_t)me + 2, sz);
  }
}

// The step's reactions to the bodies' adjoints, with the node terms: one
// thread per heap slot that is a leaf.  The sums over its ancestors of
// A = G/M and B = H - c.A give  lp_j += m_j A,  lm_j += p_j . A + B  for every
// member j.  (The ancestors' slots are known beforehand, so four are loaded at
// a time.)
__global__ __launch_bounds__(256) void k_adj_nodes(
    const uint32_t *__restrict__ seg_count, const NodeRec64 *__restrict__ rec64,
    const double4 *__restrict__ pos64, const uint32_t *__restrict__ oid,
    const double4 *__restrict__ gnode, const double4 *__restrict__ react, uint32_t slots,
    uint32_t leaf, double *lpx, double *lpy, double *lpz, double *lm) {
#pragma clang fp contract(off)
  const uint32_t h = blockIdx.x * blockDim.x + threadIdx.x;
  if (h >= slots) return;
  const uint32_t c = seg_count[h];
  if (c == 0 || c > leaf) return;
  if (h > 0 && seg_count[(h - 1) / 2] <= leaf) return;  // below a leaf: unused slot
  double ax = 0.0, ay = 0.0, az = 0.0, b = 0.0;
  for (uint32_t q = h; q > 0;) {
    double4 g[4];
    NodeRec64 r[4];
    bool use[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      use[i] = q > 0;
      q = q > 0 ? (q - 1) / 2 : 0;
      g[i] = gnode[q];
      r[i] = rec64[q];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (!use[i] || (g[i].x == 0.0 && g[i].y == 0.0 && g[i].z == 0.0 && g[i].w == 0.0)) continue;
      const double Ax = g[i].x / r[i].m, Ay = g[i].y / r[i].m, Az = g[i].z / r[i].m;
      ax += Ax;
      ay += Ay;
      az += Az;
      b += g[i].w - (r[i].cx * Ax + r[i].cy * Ay + r[i].cz * Az);
    }
  }
  const NodeRec64 lr = rec64[h];
  for (uint32_t t = lr.start; t < lr.start + lr.count; ++t) {
    const double4 p = pos64[t], v = react[t];
    const uint32_t o = oid[t];
    lpx[o] += p.w * ax + v.x;
    lpy[o] += p.w * ay + v.y;
    lpz[o] += p.w * az + v.z;
    lm[o] += p.x * ax + p.y * ay + p.z * az + b + v.w;
  }
}

// lv += dt lp;  u = dt lv  (original order); clears the step's reactions and
// node adjoints.
__global__ void k_adj_begin(double *lpx, double *lpy, double *lpz, double *lvx, double *lvy,
                            double *lvz, double *ux, double *uy, double *uz, uint32_t n, double dt,
                            double4 *react, double4 *gnode, uint32_t slots) {
#pragma clang fp contract(off)
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  const double4 zero = make_double4(0.0, 0.0, 0.0, 0.0);
  if (i < slots) gnode[i] = zero;
  if (i >= n) return;
  react[i] = zero;
  double a = lvx[i] + dt * lpx[i], b = lvy[i] + dt * lpy[i], c = lvz[i] + dt * lpz[i];
  lvx[i] = a;
  lvy[i] = b;
  lvz[i] = c;
  ux[i] = dt * a;
  uy[i] = dt * b;
  uz[i] = dt * c;
}

// The depth of the subtrees dealt to the wavefronts of a workgroup (0: one
// wavefront).  Backward of a step (with its recomputed forward, 506 us at
// 100,000 ring bodies, 350 at 10,000, 162 at 2,000) in us at depths 0, 3, 4, 5,
// 6: mixed 1272, 1250, 1166, 1224 (to 5) at 100,000, 2216, 2171, 2129, 2214 (to
// 5) at 300,000 and 783, 673, 550, 488, 470 at 10,000; FP64 466, 364, 290, 253,
// 247 at 2,000.
static int adj_depth(uint32_t n) { return n <= 16384 ? 6 : n <= 65536 ? 5 : n <= 400000 ? 4 : 0; }

template <bool MIXED>
static void launch_adj_walk(const AdjWalk &a, int levels, hipStream_t s) {
  const unsigned groups = (a.n + 63) / 64;
  int d = adj_depth(a.n);
  if (d > levels - 2) d = levels - 2;  // every node above the depth is internal
  if (d < 3) d = 0;
  const int lzd = 31 - (MIXED ? 5 : 6) - d;
  if (d == 0)
    k_adj_walk<MIXED, 1><<<groups, 64, 0, s>>>(a, lzd);
  else if (d == 3)
    k_adj_walk<MIXED, 2><<<groups, 128, 0, s>>>(a, lzd);
  else if (d == 4)
    k_adj_walk<MIXED, 4><<<groups, 256, 0, s>>>(a, lzd);
  else if (d == 5)
    k_adj_walk<MIXED, 8><<<groups, 512, 0, s>>>(a, lzd);
  else
    k_adj_walk<MIXED, 16><<<groups, 1024, 0, s>>>(a, lzd);
}

hipError_t launch_adj_step(const AdjStep &st, hipStream_t s) {
  const uint32_t n = st.n, work = std::max(n, st.slots);
  double4 *react = reinterpret_cast<double4 *>(st.react);
  double4 *gnode = reinterpret_cast<double4 *>(st.gnode);
  k_adj_begin<<<(work + 255) / 256, 256, 0, s>>>(st.lp[0], st.lp[1], st.lp[2], st.lv[0], st.lv[1],
                                                 st.lv[2], st.u[0], st.u[1], st.u[2], n, st.dt,
                                                 react, gnode, st.slots);
  const AdjWalk a{st.rec64, st.rec32, st.pos64, st.pos32, st.oid, st.u[0], st.u[1], st.u[2],
                  st.react, st.gnode, n, st.leaf, st.theta * st.theta};
  const int levels = make_shape(n, (int)st.leaf).levels;
  if (st.mixed)
    launch_adj_walk<true>(a, levels, s);
  else
    launch_adj_walk<false>(a, levels, s);
  k_adj_nodes<<<(st.slots + 255) / 256, 256, 0, s>>>(st.seg_count, st.rec64, st.pos64, st.oid,
                                                     gnode, react, st.slots, st.leaf, st.lp[0],
                                                     st.lp[1], st.lp[2], st.lm);
  return hipGetLastError();
}

}  // namespace kd
