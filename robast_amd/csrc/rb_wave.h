// rb_wave.h -- navigation of the lane kernels, a wavefront at a time
// (device).
//
// One lane owns one ray, as in rb_trace.h, and every lane of the wavefront
// goes through the same loop: locate the lanes that moved, apply the optics
// of the boundary they reached, search the next boundary of those that go
// on. No lane leaves the loop before its wavefront, so the lanes can work
// for each other: the daughters of a node are culled against the whole
// wavefront's bundle of rays, one daughter box per lane, instead of each
// lane walking the node's BVH, and the shape code runs once per distinct
// shape with the shape's data in scalar registers.
#pragma once

#include "rb_trace.h"

namespace rbd {

// ---------------------------------------------------------------- wavefront
#ifndef RB_HOST_EMULATION
constexpr int kWave = 64;
__device__ __forceinline__ int wave_lane() { return int(__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u))); }
__device__ __forceinline__ unsigned long long wave_ballot(bool b) { return __ballot(b); }
__device__ __forceinline__ int wave_get(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }
__device__ __forceinline__ float wave_get(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}
__device__ __forceinline__ int first_lane(unsigned long long m) { return __ffsll(m) - 1; }
// The largest of one non-negative float per lane, every lane taking part:
// compared as integers, which orders them, with NaN above everything.
template <int CTRL, int ROWS> __device__ __forceinline__ unsigned dpp_max(unsigned v) {
  return max(v, unsigned(__builtin_amdgcn_update_dpp(int(v), int(v), CTRL, ROWS, 0xf, false)));
}
__device__ __forceinline__ float wave_max(float x) {
  unsigned v = unsigned(__float_as_int(x));
  v = dpp_max<0x111, 0xf>(v);  // row_shr 1, 2, 4, 8
  v = dpp_max<0x112, 0xf>(v);
  v = dpp_max<0x114, 0xf>(v);
  v = dpp_max<0x118, 0xf>(v);
  v = dpp_max<0x142, 0xa>(v);  // row_bcast 15, 31
  v = dpp_max<0x143, 0xc>(v);
  return __int_as_float(__builtin_amdgcn_readlane(int(v), 63));
}
__device__ __forceinline__ float wave_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
#else
constexpr int kWave = 1;
inline int wave_lane() { return 0; }
inline unsigned long long wave_ballot(bool b) { return b ? 1ull : 0ull; }
inline int wave_get(int v, int) { return v; }
inline float wave_get(float v, int) { return v; }
inline int first_lane(unsigned long long) { return 0; }
inline float wave_max(float x) { return x; }
inline float wave_rcp(float x) { return 1.0f / x; }
#endif
__device__ __forceinline__ bool wave_any(bool b) { return wave_ballot(b) != 0ull; }

// ---------------------------------------------------------------- shapes, one nesting level
// The queries of rb_device.h's Csg for a primitive or a one-level composite,
// written as loops over the operands so that each primitive's code is there
// once: inlined into the wavefront loop, with no calls, the kernel's whole
// state stays in registers.
#ifndef RB_WPRIM_FN
#define RB_WPRIM_FN __noinline__
#endif
template <typename T, unsigned SH>
__device__ RB_WPRIM_FN T wave_prim_dist_out(int type, const double* p, V3<T> q, V3<T> d) {
  return prim_dist_out<T, SH>(uniform(type), (ParamPtr)uniform(p), q, d);
}
template <typename T, unsigned SH>
__device__ RB_WPRIM_FN T wave_prim_dist_in(int type, const double* p, V3<T> q, V3<T> d) {
  return prim_dist_in<T, SH>(uniform(type), (ParamPtr)uniform(p), q, d);
}
template <typename T, unsigned SH> __device__ RB_WPRIM_FN bool wave_prim_contains(int type, const double* p, V3<T> q) {
  return prim_contains<T, SH>(uniform(type), (ParamPtr)uniform(p), q);
}
template <typename T, unsigned SH>
__device__ RB_WPRIM_FN V3<T> wave_prim_normal(int type, const double* p, V3<T> q, V3<T> d) {
  return prim_normal<T, SH>(uniform(type), (ParamPtr)uniform(p), q, d);
}
template <typename T, unsigned SH>
__device__ __forceinline__ T prim_dist(int type, ParamPtr p, V3<T> q, V3<T> d, bool out) {
  return out ? wave_prim_dist_out<T, SH>(type, (const double*)p, q, d) : wave_prim_dist_in<T, SH>(type, (const double*)p, q, d);
}

template <typename T, unsigned SH> __device__ __forceinline__ bool flat_contains(const ShapeRef<>& R, V3<T> q) {
  const bool comp = R.type == RB_SHAPE_COMPOSITE;
  const int op = R.sh->op;
  bool a = false;
#pragma unroll 1
  for (int side = 0; side < (comp ? 2 : 1); side++) {
    // the right operand decides where the left one has not
    if (side == 1 && a == (op == RB_OP_UNION)) continue;
    V3<T> lq = q;
    int type = R.type;
    ParamPtr p = R.p;
    if (comp) {
      const ParamPtr m = R.placement(side);
      lq = m2l<T>((R.sh->turned >> side & 1) != 0, m, m + 9, q);
      const ShapePtr c = (ShapePtr)R.V.shapes + R.child(side);
      type = c->type;
      p = (ParamPtr)R.V.params + c->off;
    }
    const bool in = wave_prim_contains<T, SH>(type, (const double*)p, lq);
    a = side == 1 && op == RB_OP_SUBTRACTION ? !in : in;
  }
  return a;
}

// Distance to enter (out) or leave the shape; see Csg::dist_out / dist_in.
// A difference's right operand is crossed the other way round.
template <typename T, unsigned SH>
__device__ __forceinline__ Hit flat_dist(const ShapeRef<>& R, bool out, V3<T> q, V3<T> d, double lim) {
  const bool comp = R.type == RB_SHAPE_COMPOSITE;
  const int op = R.sh->op;
  // boundary to boundary: entering an intersection or a difference, leaving a union
  const bool walk = comp && (out ? op != RB_OP_UNION : op == RB_OP_UNION);
  const T push = bool_push<T>();
  T s = T(0);
  Hit last = {0.0, 0u, out ? 0u : 1u};
  for (int it = 0; it < 64; it++) {
    const V3<T> x = axpy(q, s, d);
    bool in[2] = {false, false};
    bool need[2] = {true, comp};
    if (walk) {
      const V3<T> xp = axpy(x, push, d);
#pragma unroll 1
      for (int side = 1; side >= 0; side--) {
        // a difference's left operand is tested outside its right one only
        if (side == 0 && op == RB_OP_SUBTRACTION && in[1]) continue;
        const ParamPtr m = R.placement(side);
        const ShapePtr c = (ShapePtr)R.V.shapes + R.child(side);
        const bool r = wave_prim_contains<T, SH>(c->type, R.V.params + c->off, m2l<T>((R.sh->turned >> side & 1) != 0, m, m + 9, xp));
        if (side) in[1] = r; else in[0] = r;
      }
      const bool there = op == RB_OP_INTERSECTION ? in[0] && in[1] : op == RB_OP_SUBTRACTION ? !in[1] && in[0] : !in[0] && !in[1];
      if (there) return {double(s), last.leaf, last.exiting};
      need[0] = op == RB_OP_INTERSECTION ? !in[0] : op == RB_OP_SUBTRACTION ? !in[1] : in[0];
      need[1] = op == RB_OP_INTERSECTION ? !in[1] : in[1];
    }
    T h0 = T(0), h1 = T(0);
#pragma unroll 1
    for (int side = 0; side < (comp ? 2 : 1); side++) {
      if (side ? !need[1] : !need[0]) continue;
      V3<T> lq = x, ld = d;
      int type = R.type;
      ParamPtr p = R.p;
      bool o = out;
      if (comp) {
        const ParamPtr m = R.placement(side);
        const bool turned = (R.sh->turned >> side & 1) != 0;
        lq = m2l<T>(turned, m, m + 9, x);
        ld = m2lv<T>(turned, m, d);
        const ShapePtr c = (ShapePtr)R.V.shapes + R.child(side);
        type = c->type;
        p = (ParamPtr)R.V.params + c->off;
        o = (op == RB_OP_SUBTRACTION && side == 1) != out;
      }
      const T h = prim_dist<T, SH>(type, p, lq, ld, o);
      if (side) h1 = h; else h0 = h;
      // an operand that is never entered is never in the intersection or difference
      if (walk && out && o && double(h) >= kBig) return {kBig, 0u, 0u};
    }
    if (!comp) return {double(h0), 0u, out ? 0u : 1u};
    const bool right = !walk ? h1 < h0
                       : op == RB_OP_SUBTRACTION ? need[1]
                                                 : !(need[0] && (!need[1] || h0 >= h1));
    const T h = right ? h1 : h0;
    const bool o = (op == RB_OP_SUBTRACTION && right) != out;
    const Hit hit = {double(h), leaf_push(0u, right ? 1 : 0), o ? 0u : 1u};
    if (!walk) return hit;
    last = hit;
    s += h < push ? push : h;
    if (out && double(s) >= lim) return {kBig, 0u, 0u};
  }
  if (out) return {kBig, 0u, 0u};
  return {double(s), last.leaf, last.exiting};
}

template <typename T, unsigned SH>
__device__ __forceinline__ V3<T> flat_normal(const ShapeRef<>& R, uint32_t leaf, V3<T> q, V3<T> d) {
  const bool comp = R.type == RB_SHAPE_COMPOSITE;
  const int mine = (leaf >> 24) > 0u ? int(leaf & 1u) : 0;
  V3<T> n = mk<T>(T(0), T(0), T(1));
#pragma unroll 1
  for (int side = 0; side < (comp ? 2 : 1); side++) {
    if (comp && side != mine) continue;
    V3<T> lq = q, ld = d;
    int type = R.type;
    ParamPtr p = R.p;
    const ParamPtr m = R.placement(side);
    if (comp) {
      lq = m2l<T>((R.sh->turned >> side & 1) != 0, m, m + 9, q);
      ld = m2lv<T>(m, d);
      const ShapePtr c = (ShapePtr)R.V.shapes + R.child(side);
      type = c->type;
      p = (ParamPtr)R.V.params + c->off;
    }
    n = wave_prim_normal<T, SH>(type, (const double*)p, lq, ld);
    if (comp) n = l2mv<T>(m, n);
  }
  return n;
}

// The lane's shape among the wavefront's, in turns.
template <typename T, typename SC>
__device__ __forceinline__ bool wave_contains(const SC& S, int shape, V3<T> q) {
  static_assert(SC::max_depth == 1, "the wavefront forms handle one nesting level");
  bool in = false;
  in_turns(shape, [&](int u) { in = flat_contains<T, SC::shape_set>(ShapeRef<>(shape_view(S), u), q); });
  return in;
}
template <typename T, typename SC>
__device__ __forceinline__ Hit wave_dist(const SC& S, int shape, V3<T> q, V3<T> d, bool out, double lim) {
  Hit h = {kBig, 0u, 0u};
  // the lanes that enter and those that leave a shape take turns too
  in_turns(2 * shape + (out ? 1 : 0), [&](int u) {
    h = flat_dist<T, SC::shape_set>(ShapeRef<>(shape_view(S), u >> 1), (u & 1) != 0, q, d, lim);
  });
  return h;
}
template <typename T, typename SC>
__device__ __forceinline__ V3<T> wave_normal(const SC& S, int shape, uint32_t leaf, V3<T> q, V3<T> d) {
  V3<T> n = mk<T>(T(0), T(0), T(1));
  in_turns(shape, [&](int u) { n = flat_normal<T, SC::shape_set>(ShapeRef<>(shape_view(S), u), leaf, q, d); });
  return n;
}

// ---------------------------------------------------------------- culling a node's daughters
// A bundle of rays about one of them: at distance t every ray of the bundle
// lies in [o - do + (d - dd) t, o + do + (d + dd) t] on each axis. All members
// are uniform.
struct Bundle {
  float lo[3], hi[3];        // o - do, o + do
  float slo[3], shi[3];      // d - dd, d + dd
  float rlo[3], rhi[3];      // their reciprocals
  bool finite;
};
// Called by the whole wavefront for its lanes `mine`, of which `lead` is one;
// points only without d.
__device__ __forceinline__ Bundle wave_bundle(bool mine, int lead, const float* o, const float* d) {
  Bundle B;
  B.finite = true;
  for (int k = 0; k < 3; k++) {
    // widened by the roundings of the differences and sums here
    const float o0 = wave_get(o[k], lead), dev = wave_max(mine ? fabsf(o[k] - o0) : 0.0f);
    B.finite = B.finite && dev < 1.0e30f && fabsf(o0) < 1.0e30f;
    const float wo = dev * 1.000001f + (fabsf(o0) * 1.0e-6f + 2.0e-3f);
    B.lo[k] = o0 - wo;
    B.hi[k] = o0 + wo;
    if (!d) continue;
    const float d0 = wave_get(d[k], lead), dd = wave_max(mine ? fabsf(d[k] - d0) : 0.0f);
    B.finite = B.finite && dd < 1.0e30f && fabsf(d0) < 1.0e30f;
    const float wd = dd * 1.000001f + 4.0e-7f;
    B.slo[k] = d0 - wd;
    B.shi[k] = d0 + wd;
    B.rlo[k] = wave_rcp(B.slo[k]);
    B.rhi[k] = wave_rcp(B.shi[k]);
  }
  return B;
}
// Whether some ray of the bundle may cross the box: on each axis the bundle
// must reach lo (its upper edge) and stay below hi (its lower edge) at a
// common distance. Never false for a box that a ray of the bundle passes by
// box_pass: the margins are twice that test's.
__device__ __forceinline__ bool bundle_pass(const Bundle& B, const DBvh& b) {
  float tn = 0.0f, tf = 3.0e38f;
  bool ok = true;
  for (int k = 0; k < 3; k++) {
    const float u = b.lo[k] - B.hi[k], v = B.lo[k] - b.hi[k];  // > 0: not there yet
    if (B.shi[k] > 0.0f) tn = fmaxf(tn, u * B.rhi[k]);
    else {
      ok = ok && u <= 0.0f;
      tf = fminf(tf, B.shi[k] < 0.0f ? u * B.rhi[k] : 3.0e38f);
    }
    if (B.slo[k] < 0.0f) tn = fmaxf(tn, -v * B.rlo[k]);
    else {
      ok = ok && v <= 0.0f;
      tf = fminf(tf, B.slo[k] > 0.0f ? -v * B.rlo[k] : 3.0e38f);
    }
  }
  return ok && tn <= tf * 1.0002f + 2e-3f;
}
// A point bundle: every point of the bundle lies in [lo, hi].
__device__ __forceinline__ bool bundle_near(const Bundle& B, const DBvh& b) {
  bool ok = true;
  for (int k = 0; k < 3; k++) ok = ok && b.lo[k] <= B.hi[k] && B.lo[k] <= b.hi[k];
  return ok;
}

// A node with more daughters than this, or a bundle that meets more than
// kBundleMax of them (an incoherent wavefront), has its BVH walked by each
// lane. A daughter box of the bundle costs the wavefront about 50
// instructions and a visited BVH entry as many; the walks of the 85-facet
// reflector visit 39 entries per search.
constexpr int kBundleLeaves = 256;
constexpr int kBundleMax = 24;
// A node with so few daughters has them all tested: the bundle costs about as
// much as six boxes.
constexpr int kBundleMin = 6;

// Leaf `i` of node n's daughters (BVH order), from the LDS copy when staged.
__device__ __forceinline__ DBvh leaf_box(const DScene& S, int i) {
#ifndef RB_HOST_EMULATION
  if (unsigned(i) < unsigned(S.leaf_stage_n)) {
    const float4* l = reinterpret_cast<const float4*>(&g_leaf_stage[i]);
    const float4 a = l[0], c = l[1];
    return {{a.x, a.y, a.z}, __float_as_int(a.w), {c.x, c.y, c.z}, __float_as_int(c.w)};
  }
#endif
  return S.leaves[i];
}
__device__ __forceinline__ DBvh wave_get(const DBvh& b, int lane) {
  DBvh u;
  for (int k = 0; k < 3; k++) {
    u.lo[k] = wave_get(b.lo[k], lane);
    u.hi[k] = wave_get(b.hi[k], lane);
  }
  u.escape = 0;
  u.prim = wave_get(b.prim, lane);
  return u;
}

// One lane's candidates: the kCand daughters with the smallest (box entry,
// node id), in that order, of those beyond (from_tn, from_node); `drop` the
// smallest entry of the others.
struct Picks {
  int n;
  float drop;
  float from_tn;
  int from_node;
};
__device__ __forceinline__ void pick(const Cand& cand, Picks& K, float tn, int node) {
  if (tn < K.from_tn || (tn == K.from_tn && node <= K.from_node)) return;
  int k = K.n;
  if (K.n == kCand) {
    const float last = cand.tn[(kCand - 1) * kCandStride];
    if (tn > last || (tn == last && node > cand.node[(kCand - 1) * kCandStride])) {
      K.drop = fminf(K.drop, tn);
      return;
    }
    K.drop = fminf(K.drop, last);
    k = kCand - 1;
  } else {
    K.n++;
  }
  while (k > 0 && (cand.tn[(k - 1) * kCandStride] > tn ||
                   (cand.tn[(k - 1) * kCandStride] == tn && cand.node[(k - 1) * kCandStride] > node))) {
    cand.tn[k * kCandStride] = cand.tn[(k - 1) * kCandStride];
    cand.node[k * kCandStride] = cand.node[(k - 1) * kCandStride];
    k--;
  }
  cand.tn[k * kCandStride] = tn;
  cand.node[k * kCandStride] = node;
}

// The candidates of every lane with `need`, in node `cur` (one of several
// daughters): the boxes of the node's daughters that the lane's ray crosses.
// Called by the whole wavefront.
__device__ __forceinline__ void wave_gather(const DScene& S, bool need, int cur, V3<double> p, V3<double> d,
                                            const Cand& cand, Picks& K) {
  const float o[3] = {float(p.x), float(p.y), float(p.z)}, v[3] = {float(d.x), float(d.y), float(d.z)};
  const float ix = 1.0f / v[0], iy = 1.0f / v[1], iz = 1.0f / v[2];
  K.n = 0;
  K.drop = 3.0e38f;
  bool walk = false;
  for (unsigned long long left = wave_ballot(need); left != 0ull;) {
    const int lead = first_lane(left);
    const int c = wave_get(cur, lead);
    const bool mine = need && cur == c;
    left &= ~wave_ballot(mine);
    const int first = node_ptr(S, c)->leaf0, nl = node_ptr(S, c)->n_children;
    bool apart = nl > kBundleLeaves;
    if (!apart) {
      Bundle B;
      B.finite = true;
      if (nl > kBundleMin) B = wave_bundle(mine, lead, o, v);
      apart = !B.finite;
      int met = 0;
      for (int base = 0; base < nl && !apart; base += kWave) {
        const int l = base + wave_lane();
        DBvh b{};
        bool pass = false;
        if (l < nl) {
          b = leaf_box(S, first + l);
          pass = nl <= kBundleMin || bundle_pass(B, b);
        }
        unsigned long long m = wave_ballot(pass);
#ifndef RB_HOST_EMULATION
        met += __popcll(m);
#endif
        if (met > kBundleMax) apart = true;
        for (; m != 0ull && !apart; m &= m - 1ull) {
          const DBvh u = wave_get(b, first_lane(m));
          float tn;
          if (mine && box_pass(u, o[0], o[1], o[2], ix, iy, iz, K.drop, tn)) pick(cand, K, tn, u.prim);
        }
      }
    }
    if (apart) walk = walk || mine;
  }
  if (walk) {
    K.n = 0;
    K.drop = 3.0e38f;
    int i = S.nodes[cur].bvh_root;
    const int end = S.bvh[i].escape;
    while (i < end) {
      const DBvh b = S.bvh[i];
      float tn;
      if (!box_pass(b, o[0], o[1], o[2], ix, iy, iz, K.drop, tn)) {
        i = b.escape;
        continue;
      }
      if (b.prim >= 0) pick(cand, K, tn, b.prim);
      i++;
    }
  }
}

// A node's point and ray in its frame: with scalar loads where all active
// lanes ask for one node.
template <typename SC> __device__ __forceinline__ bool at_node_contains(const SC& S, int n, V3<double> p) {
  V3<double> q;
  int u, shape;
  if (all_one(n, u)) {
    const NodePtr nd = node_ptr(S, u);
    shape = nd->shape;
    q = m2l<double>((nd->kind & kNodeTurned) != 0, nd->rot, nd->tr, p);
  } else {
    const DNode& nd = S.nodes[n];
    shape = nd.shape;
    q = m2l<double>(nd.rot, nd.tr, p);
  }
  return wave_contains<double>(S, shape, q);
}

// Where the point p of each lane with `req` lies: TGeoNavigator::SearchNode
// from node `n` (up until inside, unless `inside`, then down through the
// daughters; `skip` is not entered), -1 outside the top node. Lanes without
// `req` get n back. Called by the whole wavefront.
template <typename SC>
__device__ __forceinline__ int wave_locate(const SC& S, bool req, int n, int skip, bool inside, V3<double> p) {
  inside = inside || n == skip;
  while (wave_any(req && !inside)) {
    if (req && !inside) {
      if (at_node_contains(S, n, p)) {
        inside = true;
      } else {
        skip = n;
        n = node_ints(S, n).parent;
        if (n < 0) req = false;
      }
    }
  }
  const float o[3] = {float(p.x), float(p.y), float(p.z)};
  for (int guard = 0; guard < 64; guard++) {
    if (req) req = node_ints(S, n).n_children > 0;
    const unsigned long long all = wave_ballot(req);
    if (all == 0ull) break;
    int found = 0x7fffffff;
    bool walk = false;
    for (unsigned long long left = all; left != 0ull;) {
      const int lead = first_lane(left);
      const int c = wave_get(n, lead);
      const bool mine = req && n == c;
      left &= ~wave_ballot(mine);
      const int first = node_ptr(S, c)->leaf0, nl = node_ptr(S, c)->n_children;
      bool apart = nl > kBundleLeaves;
      if (!apart) {
        Bundle B;
        B.finite = true;
        if (nl > kBundleMin) B = wave_bundle(mine, lead, o, nullptr);
        apart = !B.finite;
        int met = 0;
        for (int base = 0; base < nl && !apart; base += kWave) {
          const int l = base + wave_lane();
          DBvh b{};
          bool pass = false;
          if (l < nl) {
            b = leaf_box(S, first + l);
            pass = nl <= kBundleMin || bundle_near(B, b);
          }
          unsigned long long m = wave_ballot(pass);
#ifndef RB_HOST_EMULATION
          met += __popcll(m);
#endif
          if (met > kBundleMax) apart = true;
          for (; m != 0ull && !apart; m &= m - 1ull) {
            const DBvh u = wave_get(b, first_lane(m));
            if (mine && u.prim != skip && u.prim < found && box_has(u, o[0], o[1], o[2]) &&
                at_node_contains(S, u.prim, p))
              found = u.prim;
          }
        }
      }
      if (apart) walk = walk || mine;
    }
    if (walk) {
      found = 0x7fffffff;
      int i = S.nodes[n].bvh_root;
      const int end = S.bvh[i].escape;
      while (i < end) {
        const DBvh b = S.bvh[i];
        if (!box_has(b, o[0], o[1], o[2])) {
          i = b.escape;
          continue;
        }
        if (b.prim >= 0 && b.prim != skip && b.prim < found && at_node_contains(S, b.prim, p)) found = b.prim;
        i++;
      }
    }
    if (req) {
      if (found == 0x7fffffff) {
        req = false;
      } else {
        n = found;
        skip = -1;
      }
    }
  }
  return n;
}

template <typename SC>
__device__ __forceinline__ Hit at_node_dist(const SC& S, int n, V3<double> p, V3<double> d, bool out, double lim) {
  V3<double> q, e;
  int u, shape;
  if (all_one(n, u)) {
    const NodePtr nd = node_ptr(S, u);
    const bool turned = (nd->kind & kNodeTurned) != 0;
    shape = nd->shape;
    q = m2l<double>(turned, nd->rot, nd->tr, p);
    e = m2lv<double>(turned, nd->rot, d);
  } else {
    const DNode& nd = S.nodes[n];
    shape = nd.shape;
    q = m2l<double>(nd.rot, nd.tr, p);
    e = m2lv<double>(nd.rot, d);
  }
  return wave_dist<double>(S, shape, q, e, out, lim);
}

// The nearest boundary of every lane with `go`: its own node's exit (or,
// outside, the top node's entry; crossed = -1), a daughter's entry (crossed =
// node id) or none (-2), as search_boundary_fp64 finds it. The candidates are
// tested in order of box entry, the lanes' k-th together, up to the first
// entry beyond the best crossing; should the dropped boxes hold a nearer
// crossing, the next kCand are picked. Called by the whole wavefront.
template <typename SC>
__device__ __forceinline__ void wave_search(const SC& S, bool go, int cur, V3<double> p, V3<double> d,
                                            const Cand& cand, double& best, int& crossed, Hit& hit) {
  best = kBig;
  crossed = -2;
  hit = {kBig, 0u, 0u};
  bool more = go && cur >= 0;
  if (more) more = node_ints(S, cur).n_children > 0;
  Picks K{0, 3.0e38f, -1.0f, -1};
  for (int k = -1;; k = 0) {
    wave_gather(S, more, cur, p, d, cand, K);
    for (;; k++) {
      const bool mine = k < 0 ? go : more && k < K.n && !(cand.tn[k * kCandStride] > float(best) * 1.0001f + 1e-2f);
      if (!wave_any(mine)) break;
      if (mine) {
        const int c = k < 0 ? (cur < 0 ? 0 : cur) : cand.node[k * kCandStride];
        const Hit h = at_node_dist(S, c, p, d, k >= 0 || cur < 0, k < 0 ? kBig : best + kTol);
        if (k >= 0) {
          rank_fp64(c, h, best, crossed, hit);
        } else if (h.s < best - kTol) {
          best = h.s;
          crossed = -1;
          hit = h;
        }
      }
    }
    more = more && K.drop <= float(best) * 1.0001f + 1e-2f;
    if (!wave_any(more)) break;
    if (more) {
      K.from_tn = cand.tn[(kCand - 1) * kCandStride];
      K.from_node = cand.node[(kCand - 1) * kCandStride];
    }
  }
}

// The whole trace of the wavefront's rays, those with `act`; see step_lane
// and next_boundary for the rules of one segment.
template <typename Rec, typename IO, typename SC>
__device__ __forceinline__ void wave_trace(const SC& S, const TraceParams& P, const IO& io, int64_t& i, bool act,
                                           Lane& L, Rec& rec) {
  volatile ColdState& C = *L.cold;
  const int me = L.slot;
  // where to locate a lane, and from which node
  bool req = act, inside = false, arrived = false, on_b = false;
  int n = 0, skip = -1, cur = -1, status = L.status;
  V3<double> p = L.p, d = L.d;
  C.ray[me] = i;
  C.push[me] = 0.0;
  C.t[me] = L.t;
  C.lambda[me] = L.lambda;
  C.npoints[me] = L.npoints;
  C.last_node[me] = L.last_node;
  C.draw[me] = 0;
  while (wave_any(act)) {
    n = wave_locate(S, req, n, skip, inside, axpy(p, C.push[me], d));
    if (req) cur = n;
    req = false;
    if (act && arrived) {
      // the optics of the boundary between the node left and the one located
      L.p = p;
      L.d = d;
      L.t = C.t[me];
      L.lambda = C.lambda[me];
      L.step = C.step[me];
      L.npoints = C.npoints[me];
      L.last_node = C.last_node[me];
      L.hit_node = C.hit_node[me];
      L.hit_leaf = C.hit_leaf[me];
      L.draw = C.draw[me];
      L.status = RB_RUN;
      L.on_b = on_b;
      const V3<double> x1 = mk<double>(C.x1[0][me], C.x1[1][me], C.x1[2][me]);
      const int64_t ray = C.ray[me];
      L.ray = P.id_base + uint64_t(ray);
      const bool reflected = interact(S, P, io, ray, L, x1, C.from[me], cur, rec);
      p = L.p;
      d = L.d;
      status = L.status;
      on_b = L.on_b;
      C.t[me] = L.t;
      C.npoints[me] = L.npoints;
      C.last_node[me] = L.last_node;
      C.draw[me] = L.draw;
      act = status == RB_RUN;
      if (reflected) {
        // locate the point stepped back to
        req = act;
        n = cur < 0 ? 0 : cur;
        skip = -1;
        inside = false;
        C.push[me] = 0.0;
      }
    }
    arrived = act && !req;
    if (!wave_any(arrived)) continue;
    const double extra = on_b ? kTol : 0.0;
    if (arrived) {
      C.x1[0][me] = p.x;
      C.x1[1][me] = p.y;
      C.x1[2][me] = p.z;
      C.from[me] = cur;
      p = axpy(p, extra, d);
    }
    double best;
    int crossed;
    Hit hit;
    wave_search(S, arrived, cur, p, d, L.cand, best, crossed, hit);
    if (arrived) {
      int hit_node = -1;
      double step = kBig;
      on_b = crossed != -2;
      if (cur >= 0 || crossed != -2) {  // (a ray outside may never meet the top node)
        // TGeoNavigator: do not stay on the exit surface; step by the tolerance
        const bool stay = cur >= 0 && crossed == -1 && best <= kTol;
        p = axpy(p, stay ? kTol : best, d);
        step = stay ? kTol : best + extra;
        if (crossed != -2) {
          hit_node = crossed >= 0 ? crossed : cur < 0 ? 0 : cur;
          // locate from the node entered, or from the mother of the one left
          const int parent = cur < 0 ? -1 : node_ints(S, cur).parent;
          n = crossed >= 0 ? crossed : cur < 0 ? 0 : stay ? cur : parent;
          skip = cur < 0 ? -1 : cur;
          inside = crossed >= 0 || cur < 0;
          if (n < 0) {
            cur = -1;
          } else {
            req = true;
            C.push[me] = locate_push(S, n, step);
          }
        }
      }
      C.step[me] = step;
      C.hit_node[me] = hit_node;
      C.hit_leaf[me] = crossed == -2 ? 0u : hit.leaf;
    }
  }
  L.p = p;
  L.d = d;
  L.status = status;
  L.t = C.t[me];
  L.lambda = C.lambda[me];
  L.npoints = C.npoints[me];
  L.last_node = C.last_node[me];
  i = C.ray[me];
}

}  // namespace rbd
