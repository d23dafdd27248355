// Tree-aware gated delta net (GDN) state update for tree verification on MI355X.
//
// Reference semantics (cf/ = src/chain_flow/): cf/kernels/tree_scan.py:23-73 -- every node n of a
// BFS-ordered draft tree (parent[n] < n, -1 = root) starts from its parent's state (roots from S0):
//     S = S_parent * exp(g);  delta = (v - S^T k) * beta;  S = S + k (x) delta;  o = S^T q
// with q, k l2-normalised (x / (|x| + 1e-6), or x / sqrt(|x|^2 + 1e-6) as in the Triton kernels of
// cf/vllm_tree/tree_ssm.py:60-62) and q scaled by Dk^-1/2.  State layout [H][Dk][Dv].
//
// Execution plan (path-parallel): one workgroup per (node, head, 64-column value slice), four
// waves of it each holding 32 of the Dk = 128 state rows (lane j: column j) in registers.  The
// workgroup replays the node's ancestor chain from the root, so every node's state and output come
// from the same sequential per-path recurrence (tree_scan.py:78-90) and no workgroup waits for
// another; each step's dot products are summed over the four waves through LDS.  k of each path
// step is normalised once and broadcast through LDS; q only for the node itself (the output).
// The recompute costs depth x 3 Dk FMA-class operations per column per node, below the state
// traffic (S0 read, node state written).
#include "cfh_kernels.h"
#include "cfh_host.h"

namespace {

constexpr int GDN_DK = 128;
constexpr int GDN_MAXN = 256;

struct GdnArgs {
  const uint16_t* q;     // [N][H][Dk] bf16
  const uint16_t* k;     // [N][H][Dk] bf16
  const uint16_t* v;     // [N][H][Dv] bf16
  const float* g;        // [N][H] log decay
  const float* beta;     // [N][H]
  const float* S0;       // [H][Dk][Dv]
  const int* parent;     // [N]
  float* out;            // [N][H][Dv]
  float* states;         // [N][H][Dk][Dv] or null
  int N, H, Dv, l2norm, l2mode;
  float scale;
};

__device__ __forceinline__ float bf16f(uint16_t b) { return __uint_as_float((unsigned)b << 16); }

// The ancestor chain comes from the parents staged in LDS by one coalesced load; each batch of up to
// GDN_LB path steps issues all its loads (k, v, gates) before any math, and the step scalars wait
// in LDS for the sequential replay.  The dot products over Dk run as four partial sums.
constexpr int GDN_LB = 8;

// Lane 0 walks n, parent(n), ..., root through the staged parents; *len = path length, returns
// nonzero if a parent does not precede its child (not BFS-ordered).
__device__ int gdn_path(const int* __restrict__ parent, int n, int* par, int* path, int* plen_s, int* bad_s) {
  for (int i = threadIdx.x; i <= n; i += blockDim.x) par[i] = parent[i];
  __syncthreads();
  if (threadIdx.x == 0) {
    int len = 0, bad = 0, cur = n;
    while (true) {
      path[len++] = cur;
      const int p = par[cur];
      if (p < 0) break;
      if (p >= cur) { bad = 1; break; }
      cur = p;
    }
    *plen_s = len;
    *bad_s = bad;
  }
  __syncthreads();
  return *bad_s;
}

// GDN_NW waves per (node, head, 64-column value slice): wave w holds state rows
// [GDN_HK w, GDN_HK (w + 1)) of the slice's columns, so the deepest nodes' replays (the critical
// path) spread over GDN_NW times the SIMDs.  Each step's dot product is the sum of the waves'
// partials, exchanged through LDS (one barrier a step, buffers alternating by step).
constexpr int GDN_NW = 4;                  // waves per (node, head, value slice)
constexpr int GDN_HK = GDN_DK / GDN_NW;    // state rows a wave holds

// kv partial = S^T k over the wave's rows after S *= e (k broadcast from LDS), four partial sums
__device__ __forceinline__ float gdn_decay_dot_h(float* S, const float* kk, float e) {
  float p0 = 0.f, p1 = 0.f, p2 = 0.f, p3 = 0.f;
#pragma unroll
  for (int i = 0; i < GDN_HK; i += 4) {
    const float4 k4 = *(const float4*)(kk + i);
    S[i] *= e; S[i + 1] *= e; S[i + 2] *= e; S[i + 3] *= e;
    p0 += S[i] * k4.x; p1 += S[i + 1] * k4.y; p2 += S[i + 2] * k4.z; p3 += S[i + 3] * k4.w;
  }
  return (p0 + p1) + (p2 + p3);
}

__device__ __forceinline__ float gdn_dot_h(const float* S, const float* qq) {
  float p0 = 0.f, p1 = 0.f, p2 = 0.f, p3 = 0.f;
#pragma unroll
  for (int i = 0; i < GDN_HK; i += 4) {
    const float4 q4 = *(const float4*)(qq + i);
    p0 += S[i] * q4.x; p1 += S[i + 1] * q4.y; p2 += S[i + 2] * q4.z; p3 += S[i + 3] * q4.w;
  }
  return (p0 + p1) + (p2 + p3);
}

__device__ __forceinline__ void gdn_rank1_h(float* S, const float* kk, float delta) {
#pragma unroll
  for (int i = 0; i < GDN_HK; i += 4) {
    const float4 k4 = *(const float4*)(kk + i);
    S[i] += k4.x * delta; S[i + 1] += k4.y * delta; S[i + 2] += k4.z * delta; S[i + 3] += k4.w * delta;
  }
}

__global__ void __launch_bounds__(64 * GDN_NW) k_gdn_tree(GdnArgs a) {
  __shared__ __align__(16) float qs[GDN_DK];
  __shared__ __align__(16) float ks[GDN_LB][GDN_DK];
  __shared__ float egs[GDN_LB], bts[GDN_LB], vjs[GDN_LB][64];
  __shared__ float red[2][GDN_NW][64];                       // [step parity][wave][lane]
  __shared__ int par[GDN_MAXN], path[GDN_MAXN];
  __shared__ int plen_s, bad_s;
  const int nvs = a.Dv / 64;
  int u = blockIdx.x;
  const int vs = u % nvs;
  u /= nvs;
  const int h = u % a.H;
  const int n = u / a.H;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int j = vs * 64 + lane;
  const int i0 = wave * GDN_HK;                              // this wave's state rows

  // the node's own q (for the output) and the initial state do not depend on the path: issued
  // before the parents, they share its memory round trip
  const size_t qn = ((size_t)n * a.H + h) * GDN_DK;
  float q0 = bf16f(a.q[qn + lane]), q1 = bf16f(a.q[qn + 64 + lane]);
  float S[GDN_HK];
  const float* s0 = a.S0 + ((size_t)h * GDN_DK + i0) * a.Dv + j;
#pragma unroll
  for (int i = 0; i < GDN_HK; ++i) S[i] = s0[(size_t)i * a.Dv];
  if (gdn_path(a.parent, n, par, path, &plen_s, &bad_s)) {   // not BFS-ordered: NaN outputs
    const float nan = __builtin_nanf("");
    if (wave == 0) a.out[((size_t)n * a.H + h) * a.Dv + j] = nan;
    if (a.states)
      for (int i = 0; i < GDN_HK; ++i)
        a.states[(((size_t)n * a.H + h) * GDN_DK + i0 + i) * a.Dv + j] = nan;
    return;
  }
  const int len = plen_s;
  int rb = 0;                                                // red buffer of the next exchange

  for (int t0 = len - 1; t0 >= 0; t0 -= GDN_LB) {
    const int nb = min(GDN_LB, t0 + 1);                      // steps t0, t0 - 1, ..., t0 - nb + 1
    if (wave == 0) {                                         // wave 0 stages the batch for both
      float k0[GDN_LB], k1[GDN_LB], vj[GDN_LB], gg[GDN_LB], bb[GDN_LB];
#pragma unroll
      for (int b = 0; b < GDN_LB; ++b) {
        const int m = path[t0 - min(b, nb - 1)];             // past nb: a repeat, never used
        const size_t qk = ((size_t)m * a.H + h) * GDN_DK;
        k0[b] = bf16f(a.k[qk + lane]);
        k1[b] = bf16f(a.k[qk + 64 + lane]);
        vj[b] = bf16f(a.v[((size_t)m * a.H + h) * a.Dv + j]);
        gg[b] = a.g[(size_t)m * a.H + h];
        bb[b] = a.beta[(size_t)m * a.H + h];
      }
#pragma unroll
      for (int b = 0; b < GDN_LB; ++b) {
        if (b < nb) {
          float ik = 1.0f;
          if (a.l2norm) {
            const float sk = wave_sum(k0[b] * k0[b] + k1[b] * k1[b]);
            ik = a.l2mode ? 1.0f / sqrtf(sk + 1e-6f) : 1.0f / (sqrtf(sk) + 1e-6f);
          }
          ks[b][lane] = k0[b] * ik;
          ks[b][lane + 64] = k1[b] * ik;
          vjs[b][lane] = vj[b];
          if (lane == 0) { egs[b] = expf(gg[b]); bts[b] = bb[b]; }
        }
      }
    }
    __syncthreads();
    for (int b = 0; b < nb; ++b) {
      red[rb][wave][lane] = gdn_decay_dot_h(S, ks[b] + i0, egs[b]);
      __syncthreads();
      float kv = 0.f;
#pragma unroll
      for (int w = 0; w < GDN_NW; ++w) kv += red[rb][w][lane];
      rb ^= 1;
      gdn_rank1_h(S, ks[b] + i0, (vjs[b][lane] - kv) * bts[b]);
    }
    __syncthreads();   // the batch's reads of ks / vjs are done before the next batch writes them
  }
  if (wave == 0) {
    if (a.l2norm) {
      const float sq = wave_sum(q0 * q0 + q1 * q1);
      const float iq = a.l2mode ? 1.0f / sqrtf(sq + 1e-6f) : 1.0f / (sqrtf(sq) + 1e-6f);
      q0 *= iq; q1 *= iq;
    }
    qs[lane] = q0 * a.scale;
    qs[lane + 64] = q1 * a.scale;
  }
  __syncthreads();
  red[rb][wave][lane] = gdn_dot_h(S, qs + i0);
  __syncthreads();
  if (wave == 0) {
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < GDN_NW; ++w) o += red[rb][w][lane];
    a.out[((size_t)n * a.H + h) * a.Dv + j] = o;
  }
  if (a.states) {
    float* st = a.states + (((size_t)n * a.H + h) * GDN_DK + i0) * a.Dv + j;
#pragma unroll
    for (int i = 0; i < GDN_HK; ++i) st[(size_t)i * a.Dv] = S[i];
  }
}

// ---------------------------------------------------------------------------- vLLM layout
// The serving form (cf/vllm_tree/tree_ssm.py:256-311, path-parallel; bit-identical by construction to
// the per-node slot form :34-77): q, k, v are rows of the post-conv `mixed_qkv` [N][2 H K + HV V]
// (q heads, k heads, then HV value heads; value head hv uses q/k head hv / (HV / H)); the gates come
// from the projections a, b [N][HV]:
//     g = -exp(A_log) * softplus(a + dt_bias)   (softplus(x) = x above 20)
//     beta = bf16(sigmoid(b))
// q, k are normalised as x / sqrt(|x|^2 + 1e-6) and q scaled by `scale`.  States live in slots of
// `ssm_state` [slots][HV][V][K] (value-major, bf16 or fp32).  Every node starts from the prefix slot
// and follows its root->node path; each ancestor's state is rounded to the storage type (exactly
// what storing and re-reading its slot does), the node's own state stays fp32 for its output and
// is stored to node_slots[n].  Output o [N][HV][V] bf16.
struct GdnVArgs {
  const uint16_t* qkv;   // [N][ld] bf16
  const uint16_t* ga;    // [N][HV] bf16
  const uint16_t* gb;    // [N][HV] bf16
  const float* A_log;    // [HV]
  const float* dt_bias;  // [HV]
  void* state;           // [slots][HV][V][K]
  const int* slots;      // [N]
  const int* parent;     // [N]
  uint16_t* out;         // [N][HV][V] bf16
  int* status;           // [1] or null: set to 1 when a node's slot is refused
  int N, H, HV, V, ld, prefix, nslots, l2norm, chains;
  float scale;
};

// round to nearest even, as torch's cast does: gfx950 converts in hardware (v_cvt_pk_bf16_f32, two
// values an instruction), inf unchanged, NaN stays NaN
__device__ __forceinline__ float round_bf16(float x) { return (float)(__bf16)x; }
__device__ __forceinline__ uint16_t to_bf16(float x) { return __builtin_bit_cast(uint16_t, (__bf16)x); }

// The nodes are cut into one chain per leaf (every node belongs to the chain of its lowest child).  A
// workgroup takes a (chain, value head, 64 value rows): it replays its leaf's path from the root once
// and writes the outputs and states of the chain's own nodes as it passes them.  Bound by the
// replay's arithmetic (about 200 vector instructions a step and wave, 80 more at an own node):
// a workgroup per node replayed every node's path for itself, 231 steps a head for a 41-node width-4
// tree of depth 11 against 74 with ten leaves, the longest path the same.
//   state   lane 16 g + p of wave w holds an 8-element share of K of rows 16 w + 4 g + (0..3):
//           bf16 elements 8 p .. 8 p + 7 (a row is 16 lanes' 16-byte loads), fp32 elements 4 p ..
//           4 p + 3 and 64 + 4 p ..  Loads and stores are whole rows in global memory (no pass through
//           LDS); a dot product is 8 products and a 16-lane DPP sum (no exchange between waves).
//   k, q    GDN_VB steps of the path staged in LDS in the lanes' element order, the waves taking steps
//           in turn.
//   chains  GDN_GRID workgroups in all, at least GDN_CHAINS a (head, rows), take the leaves in turn, last
//           (deepest) first.  A workgroup a node, most of which then end, took 28.3 us where this takes
//           18.7 (with the paired bf16 rounding below).  GDN_CHAINS alone left a bushy tree's leaves in
//           line where few heads fill a part of the chip: 4 value heads, 200 roots 34.2 us, so 14.8; a
//           random tree of 200 nodes 53 and 21; at 32 heads the two are one.
// 41 nodes of that tree, 32 value heads, K = V = 128, bf16 states (44 MB): 46.4 -> 18.7 us.
constexpr int GDN_VB = 16;   // path steps staged at once
constexpr int GDN_VW = 4;    // waves of 16 value rows
constexpr int GDN_CHAINS = 16;   // workgroups a (value head, 64 rows) that share the leaves, at least
constexpr int GDN_GRID = 1024;   // workgroups to fill the chip with where the heads are fewer

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));
// two values rounded by one instruction (rounded one by one, each takes one and two more to join them)
__device__ __forceinline__ unsigned pack_bf16(float lo, float hi) {
  const f32x2 v = {lo, hi};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, b16x2));
}

// Element order of k and q in LDS: the lanes' first float4s, then their second ones.
template <typename T>
__device__ __forceinline__ int kq_pos(int x) {
  return sizeof(T) == 2 ? ((x >> 2) & 1) * 64 + (x >> 3) * 4 + (x & 3) : x;
}

// One lane's share of a state row: 8 elements from global memory and back.
__device__ __forceinline__ void row_load(const uint16_t* row, int p, uint4 (&r)[1]) { r[0] = *(const uint4*)(row + 8 * p); }
__device__ __forceinline__ void row_load(const float* row, int p, uint4 (&r)[2]) {
  r[0] = *(const uint4*)(row + 4 * p);
  r[1] = *(const uint4*)(row + 64 + 4 * p);
}
__device__ __forceinline__ void row_store(uint16_t* row, int p, const uint4 (&r)[1]) { *(uint4*)(row + 8 * p) = r[0]; }
__device__ __forceinline__ void row_store(float* row, int p, const uint4 (&r)[2]) {
  *(uint4*)(row + 4 * p) = r[0];
  *(uint4*)(row + 64 + 4 * p) = r[1];
}
__device__ __forceinline__ void row_widen(const uint4 (&r)[1], float (&S)[8]) {
  const unsigned w[4] = {r[0].x, r[0].y, r[0].z, r[0].w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    S[2 * e] = __uint_as_float(w[e] << 16);
    S[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
  }
}
__device__ __forceinline__ void row_widen(const uint4 (&r)[2], float (&S)[8]) {
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    S[4 * q] = __uint_as_float(r[q].x); S[4 * q + 1] = __uint_as_float(r[q].y);
    S[4 * q + 2] = __uint_as_float(r[q].z); S[4 * q + 3] = __uint_as_float(r[q].w);
  }
}
__device__ __forceinline__ void row_pack(const float (&S)[8], uint4 (&r)[1]) {
  r[0] = make_uint4(pack_bf16(S[0], S[1]), pack_bf16(S[2], S[3]), pack_bf16(S[4], S[5]), pack_bf16(S[6], S[7]));
}
__device__ __forceinline__ void row_pack(const float (&S)[8], uint4 (&r)[2]) {
#pragma unroll
  for (int q = 0; q < 2; ++q)
    r[q] = make_uint4(__float_as_uint(S[4 * q]), __float_as_uint(S[4 * q + 1]), __float_as_uint(S[4 * q + 2]),
                      __float_as_uint(S[4 * q + 3]));
}

template <typename T>
__global__ void __launch_bounds__(64 * GDN_VW) k_gdn_tree_vllm(GdnVArgs a) {
  constexpr int NR = sizeof(T) / 2;                          // 16-byte vectors of a lane's row share
  __shared__ __align__(16) float ks[GDN_VB][GDN_DK], qs[GDN_VB][GDN_DK];
  __shared__ __align__(16) float vjs[GDN_VB][64];
  __shared__ float egs[GDN_VB], bts[GDN_VB];
  __shared__ __align__(16) int slot[GDN_MAXN];
  __shared__ int par[GDN_MAXN], first[GDN_MAXN], path[GDN_MAXN], refused[GDN_MAXN];
  __shared__ int leaf[GDN_MAXN], plen_s, pown_s, bad_s;
  __shared__ unsigned long long leaves_s[GDN_VW];
  static_assert(GDN_MAXN <= 64 * GDN_VW, "a thread a node");
  const int nvs = a.V / 64;
  int u = blockIdx.x;
  const int vs = u % nvs;
  u /= nvs;
  const int hv = u % a.HV;
  const int c0 = u / a.HV;                                   // leaves c0, c0 + chains, ... from the last
  const int h = hv / (a.HV / a.H);
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
  const int p = lane & 15, r0 = wave * 16 + (lane >> 4) * 4; // this lane's share of K; its first row

  // lowest child of every node (a parent that does not precede its node is no parent)
  const int mypar = t < a.N ? a.parent[t] : -1, myslot = t < a.N ? a.slots[t] : -1;
  par[t] = mypar;
  slot[t] = myslot;
  first[t] = a.N;
  lds_barrier();
  if (mypar >= 0 && mypar < t) atomicMin(&first[mypar], t);
  lds_barrier();
  const unsigned long long lb = __ballot(t < a.N && first[t] == a.N);
  if (lane == 0) leaves_s[wave] = lb;
  lds_barrier();
  int nleaf = 0, later = 0;                                  // leaves in all, and after node t
#pragma unroll
  for (int w = 0; w < GDN_VW; ++w) {
    const int c = __popcll(leaves_s[w]);
    nleaf += c;
    later += w > wave ? c : 0;
  }
  if (c0 >= nleaf) return;                                   // (the whole workgroup)
  if (lb >> lane & 1) leaf[later + __popcll(lb >> lane) - 1] = t;

  const size_t srow = (size_t)a.HV * a.V * GDN_DK;                 // elements per slot
  const size_t sblk = ((size_t)hv * a.V + vs * 64 + r0) * GDN_DK;  // the lane's first row in a slot
  T* const state = (T*)a.state;
  const size_t qoff = (size_t)h * GDN_DK, koff = (size_t)a.H * GDN_DK + qoff;
  const size_t voff = 2 * (size_t)a.H * GDN_DK + (size_t)hv * a.V + vs * 64;
  const float Aexp = expf(a.A_log[hv]), dtb = a.dt_bias[hv];
  // a node's slot must lie in ssm_state, differ from the prefix slot and from every other node's
  // (checked here rather than on the host, so that a caller never synchronises to validate them)
  if (t < a.N) {
    int same = 0;
    for (int m = 0; m < a.N; m += 4) {                       // (entries past N are -1)
      const int4 s4 = *(const int4*)(slot + m);
      same += (s4.x == myslot) + (s4.y == myslot) + (s4.z == myslot) + (s4.w == myslot);
    }
    refused[t] = same > 1 || myslot < 0 || myslot >= a.nslots || myslot == a.prefix;
  }
  lds_barrier();
  for (int l = c0; l < nleaf; l += a.chains) {
    // the prefix state is in flight while the path is walked
    uint4 raw[4][NR];
#pragma unroll
    for (int i = 0; i < 4; ++i) row_load(state + a.prefix * srow + sblk + i * GDN_DK, p, raw[i]);
    if (t == 0) {                                              // the leaf, its parent, ..., the root
      int len = 0, own = 0, bad = 0, cur = leaf[l];
      bool mine = true;
      while (true) {
        path[len++] = cur;
        if (mine) own = len;
        const int q = par[cur];
        if (q < 0) break;
        if (q >= cur) { bad = 1; break; }
        mine = mine && first[q] == cur;
        cur = q;
      }
      plen_s = len;
      pown_s = own;
      bad_s = bad;
    }
    lds_barrier();
    const int len = plen_s, own = pown_s;                      // path[0 .. own) are this workgroup's
    if (t < own && refused[path[t]] && a.status) a.status[0] = 1;
    if (bad_s) {                                               // not BFS-ordered: NaN outputs, no slot written
      for (int i = wave; i < own; i += GDN_VW) a.out[((size_t)path[i] * a.HV + hv) * a.V + vs * 64 + lane] = 0x7fc0;
      lds_barrier();
      continue;
    }
    float S[4][8];
#pragma unroll
    for (int i = 0; i < 4; ++i) row_widen(raw[i], S[i]);
    for (int t0 = len - 1; t0 >= 0; t0 -= GDN_VB) {
      const int nb = min(GDN_VB, t0 + 1);                      // steps t0, t0 - 1, ..., t0 - nb + 1
      constexpr int SB = GDN_VB / GDN_VW;                      // steps a wave stages: wave, wave + GDN_VW, ...
      float k0[SB], k1[SB], q0[SB], q1[SB], vj[SB];
#pragma unroll
      for (int c = 0; c < SB; ++c) {
        const uint16_t* row = a.qkv + (size_t)path[t0 - min(wave + c * GDN_VW, nb - 1)] * a.ld;   // past nb: a repeat
        k0[c] = bf16f(row[koff + lane]);
        k1[c] = bf16f(row[koff + 64 + lane]);
        q0[c] = bf16f(row[qoff + lane]);
        q1[c] = bf16f(row[qoff + 64 + lane]);
        vj[c] = bf16f(row[voff + lane]);
      }
      if (t < nb) {
        const size_t m = (size_t)path[t0 - t] * a.HV + hv;
        const float x = bf16f(a.ga[m]) + dtb;
        const float sp = x <= 20.0f ? logf(1.0f + expf(x)) : x;
        egs[t] = expf(-Aexp * sp);
        bts[t] = round_bf16(1.0f / (1.0f + expf(-bf16f(a.gb[m]))));
      }
#pragma unroll
      for (int c = 0; c < SB; ++c) {
        const int b = wave + c * GDN_VW;
        if (b >= nb) break;
        float ik = 1.0f, iq = 1.0f;
        if (a.l2norm) {
          ik = 1.0f / sqrtf(wave_sum(k0[c] * k0[c] + k1[c] * k1[c]) + 1e-6f);
          iq = 1.0f / sqrtf(wave_sum(q0[c] * q0[c] + q1[c] * q1[c]) + 1e-6f);
        }
        ks[b][kq_pos<T>(lane)] = k0[c] * ik;
        ks[b][kq_pos<T>(lane + 64)] = k1[c] * ik;
        qs[b][kq_pos<T>(lane)] = q0[c] * iq * a.scale;
        qs[b][kq_pos<T>(lane + 64)] = q1[c] * iq * a.scale;
        vjs[b][lane] = vj[c];
      }
      lds_barrier();
      for (int b = 0; b < nb; ++b) {
        const float e = egs[b], bt = bts[b];
        const float4 ka = *(const float4*)&ks[b][4 * p], kb = *(const float4*)&ks[b][64 + 4 * p];
        const float4 v4 = *(const float4*)&vjs[b][r0];
        const float kk[8] = {ka.x, ka.y, ka.z, ka.w, kb.x, kb.y, kb.z, kb.w};
        const float vv[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float d0 = 0.f, d1 = 0.f;
#pragma unroll
          for (int x = 0; x < 8; x += 2) {
            S[i][x] *= e; S[i][x + 1] *= e;
            d0 += S[i][x] * kk[x]; d1 += S[i][x + 1] * kk[x + 1];
          }
          const float delta = (vv[i] - row_sum(d0 + d1)) * bt;
#pragma unroll
          for (int x = 0; x < 8; ++x) S[i][x] += kk[x] * delta;
        }
        const int at = t0 - b;                                 // position on the path (0: the leaf)
        const int node = path[at];
        const bool no = refused[node];                         // NaN outputs, no slot written
        if (at < own) {
          const float4 qa = *(const float4*)&qs[b][4 * p], qb = *(const float4*)&qs[b][64 + 4 * p];
          const float qq[8] = {qa.x, qa.y, qa.z, qa.w, qb.x, qb.y, qb.z, qb.w};
          float o[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            float d0 = 0.f, d1 = 0.f;
#pragma unroll
            for (int x = 0; x < 8; x += 2) { d0 += S[i][x] * qq[x]; d1 += S[i][x + 1] * qq[x + 1]; }
            o[i] = row_sum(d0 + d1);
          }
          const float mine = p & 2 ? (p & 1 ? o[3] : o[2]) : (p & 1 ? o[1] : o[0]);
          if (p < 4) a.out[((size_t)node * a.HV + hv) * a.V + vs * 64 + r0 + p] = no ? 0x7fc0 : to_bf16(mine);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) row_pack(S[i], raw[i]);
        if (at < own && !no) {
          T* const dst = state + (size_t)slot[node] * srow + sblk;
#pragma unroll
          for (int i = 0; i < 4; ++i) row_store(dst + i * GDN_DK, p, raw[i]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) row_widen(raw[i], S[i]);   // what a child reads is the stored state
      }
      lds_barrier();   // the batch's reads of ks / qs / vjs are done before the next batch writes them
    }
  }
}

}  // namespace

extern "C" {

int cfh_gdn_tree(const void* q, const void* k, const void* v, const float* g, const float* beta, const float* S0,
                 const int32_t* parent, int N, int H, int Dk, int Dv, int use_l2norm, int l2mode, float* out,
                 float* states, void* stream) {
  if (!q || !k || !v || !g || !beta || !S0 || !parent || !out) return CFH_E_INVALID;
  if (N < 1 || N > GDN_MAXN || H < 1 || Dv < 64 || Dv % 64) return CFH_E_INVALID;
  if (Dk != GDN_DK) return CFH_E_UNSUPPORTED;
  GdnArgs a = {};
  a.q = (const uint16_t*)q; a.k = (const uint16_t*)k; a.v = (const uint16_t*)v; a.g = g; a.beta = beta;
  a.S0 = S0; a.parent = parent; a.out = out; a.states = states; a.N = N; a.H = H; a.Dv = Dv;
  a.l2norm = use_l2norm ? 1 : 0; a.l2mode = l2mode ? 1 : 0; a.scale = 1.0f / sqrtf((float)Dk);
  const long long blocks = (long long)N * H * (Dv / 64);
  hipLaunchKernelGGL(k_gdn_tree, dim3((unsigned)blocks), dim3(64 * GDN_NW), 0, (hipStream_t)stream, a);
  CFH_LAUNCH_CHECK();
  return CFH_OK;
}

int cfh_gdn_tree_vllm(const void* mixed_qkv, const void* a, const void* b, const float* A_log, const float* dt_bias,
                      void* ssm_state, int state_bf16, int nslots, const int32_t* node_slots, const int32_t* parent,
                      int prefix_slot, int N, int H, int HV, int K, int V, int use_l2norm, float scale,
                      void* out, int32_t* status, void* stream) {
  if (!mixed_qkv || !a || !b || !A_log || !dt_bias || !ssm_state || !node_slots || !parent || !out)
    return CFH_E_INVALID;
  if (N < 1 || N > GDN_MAXN || H < 1 || HV < H || HV % H || V < 64 || V % 64 || prefix_slot < 0 ||
      prefix_slot >= nslots)
    return CFH_E_INVALID;
  if (K != GDN_DK) return CFH_E_UNSUPPORTED;
  GdnVArgs g = {};
  g.qkv = (const uint16_t*)mixed_qkv; g.ga = (const uint16_t*)a; g.gb = (const uint16_t*)b;
  g.A_log = A_log; g.dt_bias = dt_bias; g.state = ssm_state; g.slots = node_slots; g.parent = parent;
  g.out = (uint16_t*)out; g.N = N; g.H = H; g.HV = HV; g.V = V; g.ld = 2 * H * K + HV * V;
  g.prefix = prefix_slot; g.nslots = nslots; g.status = status; g.l2norm = use_l2norm ? 1 : 0; g.scale = scale;
  g.chains = std::min(N, std::max(GDN_CHAINS, GDN_GRID / (HV * (V / 64))));
  const long long blocks = (long long)g.chains * HV * (V / 64);
  if (state_bf16)
    hipLaunchKernelGGL(k_gdn_tree_vllm<uint16_t>, dim3((unsigned)blocks), dim3(64 * GDN_VW), 0, (hipStream_t)stream, g);
  else
    hipLaunchKernelGGL(k_gdn_tree_vllm<float>, dim3((unsigned)blocks), dim3(64 * GDN_VW), 0, (hipStream_t)stream, g);
  CFH_LAUNCH_CHECK();
  return CFH_OK;
}

}  // extern "C"
