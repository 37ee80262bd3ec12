// Ancestor-only tree verification over a shared paged prefix for gfx950.
//
// Reference: tree_kernel / tree_verify (src/tree_attention.cu:14-71,
// 93-105).  The reference gives every (request, node, query head) one warp
// that walks the whole prefix token by token.  Here the query rows of one KV
// head -- nodes x GQA group, e.g. 7 x 4 = 28 -- fill the 32 columns of a
// v_mfma_f32_32x32x16_f16 tile, so each K/V token is read once per request
// and KV head and serves every candidate:
//
//   S^T[32 tok x 32 rows] = K[32 tok x D] . Q^T[D x 32 rows]   (D/16 MFMAs)
//   O^T[D x 32 rows]     += V^T[D x 32 tok] . P^T[32 tok x 32 rows]
//
// P enters the second product as an FP16 hi/lo pair (two MFMAs), so the
// only rounding left is the FP32 accumulation.  The S^T accumulator layout
// is, lane for lane, the B operand of the P.V product once the token order
// inside a 16-token step is permuted, so P never leaves registers; V^T is
// read from LDS with ds_read_b64_tr_b16.  The draft nodes form extra 32-token
// tiles whose scores are masked by the row's ancestor set, walked from the
// parent array (at most N steps, stopping at a parent outside [0, N)).
//
// Kernels:
//  - tree_split_kernel (16-byte aligned tensors, the common path): unit =
//    (request, KV head, row tile); each of a unit's `parts` workgroups takes
//    a range of 32-token tiles (draft tiles first, then prefix tiles), its
//    waves take the range's tiles round-robin with whole-row 16-byte loads
//    staged through per-wave LDS, and merge through LDS; with parts > 1
//    merge_split_kernel combines the FP32 partials.  A single pass over
//    more units than CUs may give one eight-wave workgroup two requests,
//    four waves each on the same tiles.  Workgroup ids put
//    (KV head, row tile) in the low bits, so requests that share prefix
//    pages run on the same XCD and reuse its L2.
//  - tree_wide_kernel: trees of several row tiles per (request, KV head): four
//    waves take four row tiles (or two, two waves each) and share K/V tiles
//    that are loaded straight into LDS, whole units or shares of them.
//  - tree_flat_kernel: small trees over batches that may be long and ragged:
//    every workgroup takes an equal range of the batch's tiles.
//  - tree_whole_kernel, behind a launch of shares or ranges: the host sees only
//    what a page table could hold, so those launches read the lengths and leave
//    a batch that is better off whole to this kernel, which verifies it in a
//    single pass; else it combines the partials of the units that were cut.
//  - tree_rows_kernel, tree_kernel: element-wise loads and stores, for tensors
//    that are not 16-byte aligned (and, tree_kernel, calls without the pool
//    size): a K/V tile shared by four row tiles, and one row tile each.
#include <type_traits>

#include "bc_device.h"
#include "bc_host.h"
#include "bc_slots.h"

namespace {

using namespace bcd;

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kTile = 32;       // tokens per MFMA tile (two pages)
// Halves per staged V row: D + 32 spaces the four token rows a 16-lane
// transpose read touches 16 banks apart.
template <int D>
constexpr int v_pitch() { return D + 32; }

struct TreeParams {
  const uint16_t* k;        // prefix K [P,16,Hkv,D]
  const uint16_t* v;        // prefix V
  const int32_t* pages;     // [B, max_pages]
  const int32_t* lengths;   // [B]
  const uint16_t* dq;       // draft Q [B,N,Hq,D]
  const uint16_t* dk;       // draft K [B,N,Hkv,D]
  const uint16_t* dv;       // draft V
  const int32_t* parent;    // [B,N]
  float* out;               // [B,N,Hq,D]
  float* part_acc;          // split-kernel partials (null: one part per unit)
  float* part_ml;
  int batch, nodes, hq, hkv, group, max_pages, phys_pages;
  int rows, row_tiles;      // rows = nodes * group per (request, KV head)
  float scale_log2;
  // tree_split_kernel: parts per unit and tiles per part; with parts > 1,
  // part_acc/part_ml hold P.parts slots per output row.  tree_wide_kernel:
  // workgroups that split the units (1: none are split), with a slot per
  // workgroup and row of its.  tree_flat_kernel: ranges.
  int parts, tiles_per_part;
  // The device's CUs, and the rounds over them of the same units whole
  // (tree_wide_kernel's shares and tree_flat_kernel).
  int cus, whole_rounds;
  // ceil(2^32 / d) for d = group and d = row_tiles (0: divide plainly), and
  // whether the launch is a (KV head x row tile, request group, part) grid.
  unsigned long long group_mul, rt_mul;
  int grid3d;
};

// Every kernel argument into scalar registers at the kernel's start, in one
// round of loads.  Otherwise the compiler loads each field where it is first
// used, and a field first used after a branch costs one more serial round
// trip before the kernel's first memory access.
__device__ __forceinline__ void pin_params(const TreeParams& P) {
  asm volatile("" ::"s"(P.k), "s"(P.v), "s"(P.pages), "s"(P.lengths), "s"(P.dq), "s"(P.dk),
               "s"(P.dv), "s"(P.parent), "s"(P.out), "s"(P.part_acc), "s"(P.part_ml),
               "s"(P.batch), "s"(P.nodes), "s"(P.hq), "s"(P.hkv), "s"(P.group),
               "s"(P.max_pages), "s"(P.phys_pages), "s"(P.rows), "s"(P.row_tiles),
               "s"(P.scale_log2), "s"(P.parts), "s"(P.tiles_per_part), "s"(P.group_mul),
               "s"(P.rt_mul), "s"(P.grid3d), "s"(P.cus), "s"(P.whole_rounds));
  __builtin_amdgcn_sched_barrier(0);  // nothing that uses them moves above
}

// n / d, as a multiply-high when the host passed mul = ceil(2^32 / d) (exact
// for n * d < 2^32, which the host checks), else a plain division.
__device__ __forceinline__ int div_by(int n, int d, unsigned long long mul) {
  return mul ? (int)(((unsigned long long)(unsigned)n * mul) >> 32) : n / d;
}

__device__ __forceinline__ f16x8 as_f16x8(const uint4 u) {
  return __builtin_bit_cast(f16x8, u);
}

typedef short i16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f16x4 lds_read_tr(const _Float16* p) {
  const i16x4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) i16x4*)(p));
  return __builtin_bit_cast(f16x4, r);
}

template <int D, bool VEC>
__global__ __launch_bounds__(kThreads, 2) void tree_kernel(TreeParams P) {
  pin_params(P);
  constexpr int KS = D / 16;  // MFMA k-steps over the head dimension
  constexpr int DT = D / 32;  // 32-row output tiles over the head dimension
  constexpr int VP = v_pitch<D>();

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5;   // lane half
  const int lr = lane & 31;  // tile column (query row) / token slot

  const int zdim = P.hkv * P.row_tiles;
  const int z = blockIdx.x % zdim;
  const int b = blockIdx.x / zdim;
  const int kvh = z / P.row_tiles;
  const int rt = z % P.row_tiles;

  // Page ids of this wave's first prefix tile, requested together with the
  // length (they do not depend on it) so the first K/V loads wait for one
  // memory round trip instead of two.
  int ida[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int pg = wave * (kTile / BC_PAGE_SIZE) + q;
    ida[q] = pg < P.max_pages ? P.pages[(size_t)b * P.max_pages + pg] : -1;
  }
  const int len = max(0, min(P.lengths[b], P.max_pages * BC_PAGE_SIZE));
  const int ntile_p = (len + kTile - 1) / kTile;
  const int ntile_d = (P.nodes + kTile - 1) / kTile;

  // This lane's query row (tile column lr).
  const int r = rt * 32 + lr;
  const bool rvalid = r < P.rows;
  const int node = rvalid ? r / P.group : 0;
  const int h = kvh * P.group + (rvalid ? r % P.group : 0);
  // Q^T B operand fragments, the same for every wave of the workgroup: wave
  // 0 stages them in LDS (lane-major per k-step), all waves read them back.
  __shared__ uint4 s_q[KS][64];
  __shared__ int s_parent[BC_MAX_TREE_NODES];
  __shared__ __attribute__((aligned(16))) char s_mem[kWaves * kTile * VP * 2];
  __shared__ float s_m[2][32], s_l[2][32];
  // The loads before the first barrier go out together and on one path, so
  // the waits before the LDS stores cover Q and the parents only: the parent
  // array (one entry per thread, the index clamped so every lane loads),
  // each wave's quarter of the Q^T fragments and, further down, the first
  // tile's K.  Rows past the tile's query rows read row (node 0, head h) and
  // store zeros.
  static_assert(BC_MAX_TREE_NODES <= kThreads, "one parent entry per thread");
  constexpr int QS = KS / kWaves;  // Q^T k-steps staged per wave
  static_assert(QS * kWaves == KS, "Q^T k-steps split evenly over the waves");
  const bool has_parent = (int)threadIdx.x < P.nodes;
  const int par = P.parent[(size_t)b * P.nodes + min((int)threadIdx.x, P.nodes - 1)];
  uint4 qf[QS];
  {
    const uint16_t* qp = P.dq + (((size_t)b * P.nodes + node) * P.hq + h) * D + 8 * g;
#pragma unroll
    for (int j = 0; j < QS; ++j) qf[j] = load8<VEC>(qp + 16 * (wave * QS + j));
  }

  _Float16* vs = reinterpret_cast<_Float16*>(s_mem) + wave * kTile * VP;
  // Transpose-read address of this lane: group G = lane/16, j = lane%16.
  const int trG = lane >> 4, trj = lane & 15;
  const _Float16* vtr = vs + (4 * (trG >> 1) + (trj >> 2)) * VP + 16 * (trG & 1) + 4 * (trj & 3);
  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[dt][j] = 0.f;
  float m = kNegInf, l = 0.f;

  const size_t tok_stride = (size_t)P.hkv * D;  // elements between slots
  const int ntile = ntile_p + ntile_d;
  const int nmine = ntile > wave ? (ntile - wave + kWaves - 1) / kWaves : 0;

  // Tile `idx` of this wave is tile wave + kWaves*idx of the workgroup.  The
  // loads of a tile are issued one tile ahead of its MFMAs; issues past the
  // wave's last tile repeat that tile (L2 hits), so every iteration has the
  // same loads in flight and the loop body never exits early.
  auto tile_of = [&](int idx) { return wave + kWaves * min(idx, max(nmine - 1, 0)); };
  // Physical ids of a prefix tile's two pages: uniform scalar loads, fetched
  // one tile before the K/V loads that use them.
  auto ids_of = [&](int idx, int (&ph)[2]) {
    const int it = tile_of(idx);
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int pg = it * (kTile / BC_PAGE_SIZE) + q;
      ph[q] = it < ntile_p && pg < P.max_pages ? P.pages[(size_t)b * P.max_pages + pg] : -1;
    }
  };
  // K is loaded one tile ahead; V is requested when its tile starts and is
  // consumed after the scores and softmax.
  auto issue = [&](int idx, const int (&ph)[2], uint4 (&kr)[KS], const uint16_t*& vp, bool& tv,
                   bool (&pok)[2]) {
    const int it = tile_of(idx);
    const uint16_t* kp;
    if (it < ntile_p) {
      const int tbase = it * kTile;
#pragma unroll
      for (int q = 0; q < 2; ++q) pok[q] = ph[q] >= 0 && ph[q] < P.phys_pages;
      const int t = tbase + lr;
      tv = t < len && pok[lr >> 4];
      const size_t phys = (size_t)(tv ? (lr >> 4 ? ph[1] : ph[0]) : 0);
      const size_t off =
          tv ? (phys * BC_PAGE_SIZE + t % BC_PAGE_SIZE) * tok_stride + (size_t)kvh * D : 0;
      // Rows that are not tokens read draft row 0 (always present): with the
      // pool size not given, page 0 of the pool may not exist.
      kp = tv ? P.k + off : P.dk;
      vp = tv ? P.v + off : P.dv;
    } else {
      pok[0] = pok[1] = true;
      const int dn = (it - ntile_p) * kTile + lr;
      tv = dn < P.nodes;
      const size_t off = tv ? (((size_t)b * P.nodes + dn) * P.hkv + kvh) * D : 0;
      kp = P.dk + off;
      vp = P.dv + off;
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) kr[s] = load8<VEC>(kp + 16 * s + 8 * g);
  };

  auto process = [&](int idx, const uint4 (&kr)[KS], const uint16_t* vp, bool tv,
                     const bool (&pok)[2]) {
    if (idx >= nmine) return;  // padding step
    uint4 vr[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) vr[s] = load8<VEC>(vp + 16 * s + 8 * g);
    const int it = wave + kWaves * idx;
    const bool is_draft = it >= ntile_p;
    const int tbase = (is_draft ? it - ntile_p : it) * kTile;
    // Valid token rows of the tile as a bit mask (bit i = token tbase + i):
    // prefix tiles stop at the length and drop pages outside the pool
    // (uniform over the wave); draft tiles take this row's ancestor-or-self
    // set.
    uint32_t okbits;
    if (!is_draft) {
      const int hi = min(max(len - tbase, 0), kTile);
      okbits = (hi >= kTile ? ~0u : (1u << hi) - 1u) &
               ((pok[0] ? 0x0000ffffu : 0u) | (pok[1] ? 0xffff0000u : 0u));
    } else {
      okbits = 0;
      int cur = node;
      for (int steps = 0; steps < P.nodes && cur >= 0 && cur < P.nodes; ++steps) {
        if (cur >= tbase && cur < tbase + kTile) okbits |= 1u << (cur - tbase);
        cur = s_parent[cur];
      }
    }
    // Rows past the prefix or the node count may hold any bits (NaN
    // included); their weight is zero, so their V row must be zero too.
    if (is_draft || okbits != ~0u) {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        vr[s].x = tv ? vr[s].x : 0u;
        vr[s].y = tv ? vr[s].y : 0u;
        vr[s].z = tv ? vr[s].z : 0u;
        vr[s].w = tv ? vr[s].w : 0u;
      }
    }

    // ---- S^T = K Q^T ----
    f32x16 sc;
#pragma unroll
    for (int j = 0; j < 16; ++j) sc[j] = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s)
      sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_f16x8(kr[s]),
                                                  as_f16x8(s_q[s][lane]), sc, 0, 0, 0);

    // ---- stage V row-major while the MFMAs drain ----
#pragma unroll
    for (int s = 0; s < KS; ++s)
      *reinterpret_cast<uint4*>(vs + lr * VP + 16 * s + 8 * g) = vr[s];

    // ---- mask and online softmax (column lr = query row) ----
    // sc[j] holds token row 8*(j/4) + 4*g + j%4.
    const uint32_t ob = okbits >> (4 * g);
    float sv[16];
    float tmax = kNegInf;
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const bool ok = (ob >> (8 * (j >> 2) + (j & 3))) & 1u;
      sv[j] = ok ? sc[j] * P.scale_log2 : kNegInf;
      tmax = __builtin_fmaxf(tmax, sv[j]);
    }
    tmax = __builtin_fmaxf(tmax, shfl_xor_f(tmax, 32));
    // The running max moves only when it would grow by more than
    // kRescaleSlack (log2 units): weights then stay below 2^kRescaleSlack and
    // most tiles skip rescaling the accumulators.
    const float mnew = __builtin_fmaxf(m, tmax);
    if (__builtin_amdgcn_ballot_w64(mnew > m + kRescaleSlack)) {
      const float alpha = fast_exp2(m - safe_max(mnew));
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[dt][j] *= alpha;
      m = mnew;
    }
    // P is split into FP16 hi + lo parts (two MFMAs each) so the P.V product
    // carries ~21 bits of P instead of FP16's 11.
    const float mb = safe_max(m);
    f16x8 pb[2], pl[2];
    float pr[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      pr[j] = fast_exp2(sv[j] - mb);
      l += pr[j];
    }
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      uint32_t wh[4], wl[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        split_hi_lo(pr[8 * hh + 2 * q], pr[8 * hh + 2 * q + 1], wh[q], wl[q]);
      pb[hh] = __builtin_bit_cast(f16x8, u32x4{wh[0], wh[1], wh[2], wh[3]});
      pl[hh] = __builtin_bit_cast(f16x8, u32x4{wl[0], wl[1], wl[2], wl[3]});
    }

    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // ---- O^T += V^T P^T; A operand tokens 16st + 8hf + 4g + k, dim lr ----
    // The MFMAs go round the DT accumulators, so consecutive ones are
    // independent: one accumulator's chain of four would wait out each
    // MFMA's latency in turn.
    f16x8 av[DT][2];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const f16x4 lo = lds_read_tr(vtr + (16 * st) * VP + 32 * dt);
        const f16x4 hi = lds_read_tr(vtr + (16 * st + 8) * VP + 32 * dt);
        av[dt][st] = f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[dt][st], pb[st], acc[dt], 0, 0, 0);
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[dt][st], pl[st], acc[dt], 0, 0, 0);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  uint4 ka[KS], kb[KS];
  const uint16_t* va = P.v;
  const uint16_t* vb = P.v;
  bool ta = false, tb = false;
  bool pa[2] = {true, true}, pbk[2] = {true, true};
  int idb[2];
  // The first tile's loads go out before Q and the parent array are stored
  // and published by the barrier.  A wave without tiles issues them too
  // (tile_of clamps, and every address stays inside its tensor) so that all
  // waves run the same code up to the barrier.
  issue(0, ida, ka, va, ta, pa);
#pragma unroll
  for (int j = 0; j < QS; ++j)
    s_q[wave * QS + j][lane] = rvalid ? qf[j] : make_uint4(0, 0, 0, 0);
  if (has_parent) s_parent[threadIdx.x] = par;
  ids_of(1, idb);
  __syncthreads();
  if (nmine > 0) {
    for (int idx = 0; idx < nmine; idx += 2) {
      issue(idx + 1, idb, kb, vb, tb, pbk);
      ids_of(idx + 2, ida);
      process(idx, ka, va, ta, pa);
      issue(idx + 2, ida, ka, va, ta, pa);
      ids_of(idx + 3, idb);
      process(idx + 1, kb, vb, tb, pbk);
    }
  }
  // Both lane halves share m; combine their partial sums.
  l += shfl_xor_f(l, 32);

  // ---- merge the four waves: 3,2 -> 1,0 then 1 -> 0 through LDS ----
  // Rows are padded to D + 4 floats so the 32 rows a float4 access touches
  // fall in different LDS banks.
  constexpr int XP = D + 4;
  static_assert(kWaves * kTile * VP * 2 >= 2 * 32 * XP * 4, "merge buffer fits");
  float* xacc = reinterpret_cast<float*>(s_mem);  // [2][32 rows][XP]
  auto put = [&](int slot) {
    float* dst = xacc + (size_t)slot * 32 * XP + (size_t)lr * XP;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) {
        float4 v4 = make_float4(acc[dt][4 * jq], acc[dt][4 * jq + 1],
                                acc[dt][4 * jq + 2], acc[dt][4 * jq + 3]);
        *reinterpret_cast<float4*>(dst + 32 * dt + 8 * jq + 4 * g) = v4;
      }
    if (g == 0) {
      s_m[slot][lr] = m;
      s_l[slot][lr] = l;
    }
  };
  auto take = [&](int slot) {
    const float* src = xacc + (size_t)slot * 32 * XP + (size_t)lr * XP;
    const float m2 = s_m[slot][lr], l2 = s_l[slot][lr];
    const float mm = __builtin_fmaxf(m, m2);
    const float a1 = fast_exp2(m - safe_max(mm)), a2 = fast_exp2(m2 - safe_max(mm));
    l = l * a1 + l2 * a2;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) {
        const float4 v4 = *reinterpret_cast<const float4*>(src + 32 * dt + 8 * jq + 4 * g);
        acc[dt][4 * jq] = acc[dt][4 * jq] * a1 + v4.x * a2;
        acc[dt][4 * jq + 1] = acc[dt][4 * jq + 1] * a1 + v4.y * a2;
        acc[dt][4 * jq + 2] = acc[dt][4 * jq + 2] * a1 + v4.z * a2;
        acc[dt][4 * jq + 3] = acc[dt][4 * jq + 3] * a1 + v4.w * a2;
      }
    m = mm;
  };
  __syncthreads();  // V^T staging area is reused below
  if (wave >= 2) put(wave - 2);
  __syncthreads();
  if (wave < 2) take(wave);
  __syncthreads();
  if (wave == 1) put(0);
  __syncthreads();
  if (wave != 0) return;
  take(0);
  if (!rvalid) return;

  // ---- write: lane holds O^T[32dt + 8jq + 4g + e][row r] ----
  float* dst = P.out + (((size_t)b * P.nodes + node) * P.hq + h) * D;
  const float inv = 1.f / l;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int jq = 0; jq < 4; ++jq)
      store4f<VEC>(dst + 32 * dt + 8 * jq + 4 * g, acc[dt][4 * jq] * inv,
                   acc[dt][4 * jq + 1] * inv, acc[dt][4 * jq + 2] * inv,
                   acc[dt][4 * jq + 3] * inv);
}

// ---- per-tile pieces of tree_split_kernel ----

// Valid tokens of a prefix tile: the first `valid` rows (clipped to
// [0, 32]), minus the 16-row halves whose page id lies outside the pool.
__device__ __forceinline__ uint32_t prefix_bits(int valid, int id0, int id1, int phys) {
  const int hi = min(max(valid, 0), kTile);
  return (hi >= kTile ? ~0u : (1u << hi) - 1u) &
         ((id0 >= 0 && id0 < phys ? 0x0000ffffu : 0u) |
          (id1 >= 0 && id1 < phys ? 0xffff0000u : 0u));
}

// parent[i] for i in [0, nodes) from the parent registers (lane i of
// register c holds parent[i + 64c]).
__device__ __forceinline__ int parent_at(const int (&parr)[4], int nodes, int i) {
  if (nodes <= 64) return __shfl(parr[0], i, 64);
  const int c0 = __shfl(parr[0], i & 63, 64), c1 = __shfl(parr[1], i & 63, 64);
  const int c2 = __shfl(parr[2], i & 63, 64), c3 = __shfl(parr[3], i & 63, 64);
  const int c = i >> 6;
  return c == 0 ? c0 : c == 1 ? c1 : c == 2 ? c2 : c3;
}

// Valid tokens of the draft tile starting at node tbase for the lane's
// query row: its node and that node's ancestors.  Lanes walk different
// chains, so the loop runs until every lane's walk has ended (a parent
// outside [0, nodes) ends it; at most `nodes` steps).
__device__ __forceinline__ uint32_t ancestor_bits(const int (&parr)[4], int nodes, int node,
                                                  int tbase) {
  uint32_t okbits = 0;
  int cur = node;
  for (int steps = 0; steps < nodes; ++steps) {
    const bool live = cur >= 0 && cur < nodes;
    if (!__builtin_amdgcn_ballot_w64(live)) break;
    if (live && cur >= tbase && cur < tbase + kTile) okbits |= 1u << (cur - tbase);
    const int nx = parent_at(parr, nodes, live ? cur : 0);
    cur = live ? nx : -1;
  }
  return okbits;
}

// One 32-token tile staged in LDS (K rows at a pitch of D + 8 halves, V
// rows at D + 16), in two steps.  tile_scores: S^T = K Q^T as one MFMA
// chain over the k-steps and the masked online-softmax update of (m, l,
// acc), leaving P as an FP16 hi/lo pair; tile_pv: O^T += V^T P^T.  kr is
// this lane's K row (token lr), vtr its transpose-read address in the V
// rows, qf this lane's Q^T B-operand fragments (k-step s at qf[QS s]: in
// LDS, QS = 64; in registers, QS = 1) and okbits the valid tokens of the
// lane's query row.
// FIRST: the wave's first tile; its running max starts at -inf and acc is
// not yet defined, so the rescale is skipped (tile_pv then starts acc from
// zero).
template <int D, int QS, bool FIRST>
__device__ __forceinline__ void tile_scores(const _Float16* kr, const uint4* qf,
                                            uint32_t okbits, float scale_log2, int g,
                                            f32x16 (&acc)[D / 32], float& m, float& l,
                                            f16x8 (&pb)[2], f16x8 (&pl)[2]) {
  constexpr int KS = D / 16;
  constexpr int DT = D / 32;
  f32x16 sc;
#pragma unroll
  for (int j = 0; j < 16; ++j) sc[j] = 0.f;
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const uint4 k0 = *reinterpret_cast<const uint4*>(kr + 16 * s + 8 * g);
    sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_f16x8(k0), as_f16x8(qf[QS * s]), sc, 0, 0, 0);
  }
  // sc[j] holds token row 8*(j/4) + 4*g + j%4.  Scores stay unscaled here;
  // the scale enters the running max once and the exp2 argument as an FMA.
  float sv[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) sv[j] = sc[j];
  if (__builtin_amdgcn_ballot_w64(okbits != ~0u)) {  // masked tokens in the tile
    const uint32_t ob = okbits >> (4 * g);
#pragma unroll
    for (int j = 0; j < 16; ++j)
      sv[j] = (ob >> (8 * (j >> 2) + (j & 3))) & 1u ? sv[j] : kNegInf;
  }
  float tmax = kNegInf;
#pragma unroll
  for (int j = 0; j < 16; ++j) tmax = __builtin_fmaxf(tmax, sv[j]);
  tmax = __builtin_fmaxf(tmax, shfl_xor_f(tmax, 32)) * scale_log2;
  if constexpr (FIRST) {
    m = tmax;  // l is still 0
  } else {
    const float mnew = __builtin_fmaxf(m, tmax);
    if (__builtin_amdgcn_ballot_w64(mnew > m + kRescaleSlack)) {
      const float alpha = fast_exp2(m - safe_max(mnew));
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[dt][j] *= alpha;
      m = mnew;
    }
  }
  // P splits into an FP16 hi part (p truncated to FP16, exact for p in
  // [2^-14, 2^8]) and lo = p - hi rounded to FP16, so P.V carries ~21 bits
  // of P.
  const float mb = safe_max(m);
  float pr[16];
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    pr[j] = fast_exp2(__builtin_fmaf(sv[j], scale_log2, -mb));
    l += pr[j];
  }
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    uint32_t wh[4], wl[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) split_hi_lo(pr[8 * h + 2 * q], pr[8 * h + 2 * q + 1], wh[q], wl[q]);
    pb[h] = __builtin_bit_cast(f16x8, u32x4{wh[0], wh[1], wh[2], wh[3]});
    pl[h] = __builtin_bit_cast(f16x8, u32x4{wl[0], wl[1], wl[2], wl[3]});
  }
}

// FIRST: acc starts from zero (the first MFMA of each accumulator takes a
// zero C operand).
template <int D, bool FIRST>
__device__ __forceinline__ void tile_pv(const _Float16* vtr, const f16x8 (&pb)[2],
                                        const f16x8 (&pl)[2], f32x16 (&acc)[D / 32]) {
  constexpr int DT = D / 32;
  constexpr int VP = D + 16;
  // ---- O^T += V^T P^T; A operand tokens 16st + 8hf + 4g + k, dim lr ----
  // The MFMAs go round the DT accumulators, so consecutive ones are
  // independent.
  f16x8 av[DT][2];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const f16x4 lo = lds_read_tr(vtr + (16 * st) * VP + 32 * dt);
      const f16x4 hi = lds_read_tr(vtr + (16 * st + 8) * VP + 32 * dt);
      av[dt][st] = f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    }
  const f32x16 zero = {};
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[dt][st], pb[st],
                                                       FIRST && st == 0 ? zero : acc[dt], 0, 0,
                                                       0);
#pragma unroll
  for (int st = 0; st < 2; ++st)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[dt][st], pl[st], acc[dt], 0, 0, 0);
}

// Wave-local LDS handoff: this wave's LDS writes are visible to its own
// later reads (and its reads done before its later writes).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Split tree verification.  Unit = (request, KV head, row tile); its work is
// one tile space: the draft tiles [0, ntd) followed by the prefix tiles (32
// tokens each, up to the request's length).  Workgroup `part` of a unit
// takes tiles [part*T, part*T + T), T = P.tiles_per_part, and its W waves
// take those tiles round-robin.  The row tile's Q^T fragments are fetched
// once per workgroup into LDS, where the score MFMAs read them.  A wave
// loads a tile's K and V as whole token rows (each 16-byte load instruction
// covers complete 128-byte lines: measured 2x the tile rate of loading K in
// the MFMA operand layout, where an instruction touches 32 rows), stages
// them in its own LDS area -- K rows at a pitch for conflict-free A-operand
// reads, V rows at a pitch for transpose reads -- and issues the next tile's
// loads as soon as the rows are staged, so they are in flight during the
// current tile's MFMAs.  Masks, softmax and the hi/lo P.V product are
// tree_kernel's.  The waves merge through LDS, each thread combining the
// waves' states for its share of a row; with one part per unit (no
// workspace) that share goes to the output, otherwise every part with tiles
// writes an FP32 partial per row, slot (row, part), and merge_split_kernel
// combines them.
// WHOLE: one part per unit on a flat grid (tree_whole_kernel), whatever the
// parameters say of parts.
template <int D, int W, int RQ, bool WHOLE>
__device__ __forceinline__ void tree_split_body(const TreeParams& P) {
  constexpr int KS = D / 16;      // MFMA k-steps; also load instructions per tile
  constexpr int DT = D / 32;      // 32-row output tiles over the head dimension
  constexpr int KP = D + 8;       // halves per staged K row
  constexpr int VP = D + 16;      // halves per staged V row
  constexpr int LPR = D / 8;      // lanes per token row in a whole-row load
  constexpr int RPI = 64 / LPR;   // token rows per load instruction
  static_assert(RPI * KS == kTile, "KS whole-row loads cover a tile");
  constexpr int STAGE = kTile * (KP + VP);  // halves per wave
  constexpr int LN = W / RQ;      // waves per request

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5;   // lane half
  const int lr = lane & 31;  // tile column (query row) / token slot

  // RQ requests per workgroup: wave w serves request RQ*group + w/LN and
  // takes every LN-th tile from w%LN, so the RQ requests walk the same
  // tiles at the same time (their shared pages then meet in the CU's L1).
  const int rq = wave / LN;
  const int ln = wave % LN;
  // Workgroup ids put (KV head, row tile) in the low bits, then the request
  // group, then the part (a 3-D grid, or the same order flattened).
  int z, b0, part;
  if (!WHOLE && P.grid3d) {
    z = blockIdx.x;
    b0 = blockIdx.y * RQ;
    part = blockIdx.z;
  } else {
    const int zdim = P.hkv * P.row_tiles;
    const int units = zdim * ((P.batch + RQ - 1) / RQ);
    const int unit = WHOLE ? blockIdx.x : blockIdx.x % units;
    part = WHOLE ? 0 : blockIdx.x / units;
    if (WHOLE && unit >= units) return;  // uniform: the grid has a workgroup per CU at least
    z = unit % zdim;
    b0 = (unit / zdim) * RQ;
  }
  const bool present = b0 + rq < P.batch;  // uniform per wave
  const int b = present ? b0 + rq : b0;    // absent waves read request b0, unused
  const int kvh = div_by(z, P.row_tiles, P.rt_mul);
  const int rt = z - kvh * P.row_tiles;
  const int T = WHOLE ? 1 << 30 : P.tiles_per_part;
  const int tbeg = part * T;

  // Page ids of this wave's tiles as vector loads (lane j: page j%2 of the
  // wave's tile j/2, 32 tiles per register, the next 32 fetched a chunk
  // ahead).  Scalar loads would share lgkmcnt with the LDS reads of every
  // tile, whose waits would then also wait for the prefetched ids.
  //
  // Every load of the start is unconditional, from an address inside the
  // request's table row (the page index clamped), and what the entry means
  // is decided where it is used: a load under a condition is a branch, and
  // after one the compiler's wait for the kernel arguments also waits for
  // every scalar load in flight, which made the first two ids and the length
  // three serial round trips ahead of the first Q and K/V loads.  The values
  // that depend on the length are formed after those loads are issued.
  const int ntd = (P.nodes + kTile - 1) / kTile;  // draft tiles come first
  const size_t prow = (size_t)b * P.max_pages;
  auto table_entry = [&](int pg) { return P.pages[prow + min(max(pg, 0), P.max_pages - 1)]; };
  // Raw entries of chunk `chunk` (ids_of keeps those that are ids).
  auto load_ids = [&](int chunk) {
    const int it = tbeg + ln + LN * (chunk * 32 + (lane >> 1));
    return table_entry((it - ntd) * (kTile / BC_PAGE_SIZE) + (lane & 1));
  };
  int idv = load_ids(0);
  int idv_next = load_ids(1);

  const int r = rt * 32 + lr;
  const bool rvalid = r < P.rows;
  const int rnode = div_by(r, P.group, P.group_mul);
  const int node = rvalid ? rnode : 0;
  const int h = kvh * P.group + (rvalid ? r - rnode * P.group : 0);

  // Q stays in LDS (see s_q below) except in the D = 64 two-request
  // workgroups.
  constexpr bool QL = !(D == 64 && RQ == 2);
  // Q^T fragments: with Q in LDS, the LN waves of a request load KS / LN of
  // them each into s_q, so the workgroup fetches each fragment once instead
  // of once per wave (every wave of a request reads the same rows).  Q and
  // the parents load without selects (a select right after a load would wait
  // for it there): lanes past the tile's query rows read row (node 0, head
  // h), whose scores land in columns that are never written out, and parent
  // entries past the node count repeat the last one and are never read
  // (walks visit nodes in [0, nodes) only).
  constexpr int QPW = QL ? (KS + LN - 1) / LN : KS;  // fragments loaded per wave
  uint4 qown[QPW];
  {
    const uint16_t* qp = P.dq + (((size_t)b * P.nodes + node) * P.hq + h) * D + 8 * g;
#pragma unroll
    for (int j = 0; j < QPW; ++j)
      qown[j] = ldg16(qp + 16 * (QL ? min(ln + LN * j, KS - 1) : j));
  }

  // A wave whose first tile is a draft tile (part 0's first waves: draft
  // tiles come first) needs neither a page id nor the length for it, which
  // the launch geometry alone tells; the other waves load tile 0's two
  // entries and the length as scalar loads, together, after the vector loads
  // above.  Only scalar loads sit under this condition: vector loads under a
  // condition would leave the compiler's wait counts after it assuming the
  // fewest either side issued.
  const bool early = tbeg + ln < ntd;  // uniform
  const int pg0 = (tbeg + ln - ntd) * (kTile / BC_PAGE_SIZE);
  int raw0 = -1, raw1 = -1, len_raw = 0;
  if (!early) {
    raw0 = table_entry(pg0);
    raw1 = table_entry(pg0 + 1);
    len_raw = P.lengths[b];
  }
  int cur[2] = {-1, -1};
  int len = 0, ntot = 0, nmine = 0;
  auto set_lengths = [&]() {
    len = max(0, min(len_raw, P.max_pages * BC_PAGE_SIZE));
    ntot = ntd + (len + kTile - 1) / kTile;
    const int tend = min(tbeg + T, ntot);
    nmine = present && tend > tbeg + ln ? (tend - tbeg - ln + LN - 1) / LN : 0;
  };

  __shared__ __attribute__((aligned(16))) _Float16 s_stage[W * STAGE];
  // Q^T B operand of each request's row tile: lane (g, lr) of k-step s
  // holds Q[row lr][16s + 8g .. +8] (rows past the tile's query rows: row
  // (node 0, head h), unused).  It stays in LDS for the whole kernel (read
  // back per tile, which keeps 32 registers free), except in the D = 64
  // two-request workgroups, where it would leave room for one workgroup per
  // CU instead of two: there every wave holds it in registers.  The parent
  // array in registers: lane i holds parent[i + 64c] (c < 4), so a wave
  // walks ancestor chains with lane shuffles.
  __shared__ uint4 s_q[QL ? RQ * KS * 64 : 1];
  uint4 qreg[QL ? 1 : KS];
  static_assert(BC_MAX_TREE_NODES <= 256, "four parent registers per lane");
  int parr[4];

  _Float16* const ks = s_stage + wave * STAGE;
  _Float16* const vs = ks + kTile * KP;
  const int trG = lane >> 4, trj = lane & 15;
  const _Float16* vtr = vs + (4 * (trG >> 1) + (trj >> 2)) * VP + 16 * (trG & 1) + 4 * (trj & 3);
  // Whole-row load geometry: load s of a lane covers token row
  // s*RPI + lane/LPR, dims 8*(lane%LPR) .. +8.
  const int lrow = lane / LPR, lcol = 8 * (lane % LPR);
  const size_t tok_stride = (size_t)P.hkv * D;

  f32x16 acc[DT];  // defined by the first tile, or zeroed for a wave without tiles
  float m = kNegInf, l = 0.f;

  uint4 kreg[KS], vreg[KS];
  uint32_t rowok = 0;  // bit s: this lane's row of load s is a valid token
  constexpr uint32_t kAllRows = (1u << KS) - 1;
  // Byte offset of this lane's 16 bytes in whole-row load j of a page (j <
  // KS/2 loads per page: token row j*RPI + lrow, dims lcol .. +8); a prefix
  // tile's loads are then a uniform page base plus these offsets.
  constexpr int LPP = KS / 2;
  unsigned loff[LPP];
#pragma unroll
  for (int j = 0; j < LPP; ++j)
    loff[j] = (unsigned)((((size_t)(j * RPI + lrow)) * tok_stride + lcol) * sizeof(uint16_t));
  const size_t page_elems = (size_t)BC_PAGE_SIZE * tok_stride;
  // Issue the loads of this wave's tile `idx` from page ids ph.  Pages
  // outside the pool read page 0 and rows past the length read their page's
  // rows (all in bounds); both are masked.
  // K and V are issued apart (K first), so a wave can wait for K alone;
  // draft_tag (std::true_type: a draft tile) picks the address form at
  // compile time.
  auto issue_half = [&](int idx, const int (&ph)[2], bool is_v, auto draft_tag) {
    const int it = tbeg + ln + LN * idx - ntd;  // prefix tile index when >= 0
    uint4 (&dst)[KS] = is_v ? vreg : kreg;
    if constexpr (!decltype(draft_tag)::value) {
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const bool okp = ph[q] >= 0 && ph[q] < P.phys_pages;
        const size_t base = (size_t)(okp ? ph[q] : 0) * page_elems + (size_t)kvh * D;
        const char* src = reinterpret_cast<const char*>((is_v ? P.v : P.k) + base);
#pragma unroll
        for (int j = 0; j < LPP; ++j) dst[q * LPP + j] = *reinterpret_cast<const uint4*>(src + loff[j]);
      }
    } else {
      // Rows past the node count read the last node's row (masked); the
      // clamp, unlike a select of addresses, keeps the loads branch-free.
      const uint16_t* src = is_v ? P.dv : P.dk;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int dn = min((it + ntd) * kTile + s * RPI + lrow, P.nodes - 1);
        dst[s] = ldg16(src + (((size_t)b * P.nodes + dn) * P.hkv + kvh) * D + lcol);
      }
    }
  };
  // Rows of the wave's tile `idx` that hold valid tokens (bit s: this
  // lane's row of load s).
  auto rows_of = [&](int idx, const int (&ph)[2]) {
    const int it = tbeg + ln + LN * idx - ntd;
    uint32_t ok = 0;
    if (it >= 0) {
      const int tb = it * kTile;
      const bool okp0 = ph[0] >= 0 && ph[0] < P.phys_pages;
      const bool okp1 = ph[1] >= 0 && ph[1] < P.phys_pages;
      if (okp0 && okp1 && tb + kTile <= len) return kAllRows;  // uniform: every row valid
#pragma unroll
      for (int s = 0; s < KS; ++s)
        ok |= (s < LPP ? okp0 : okp1) && tb + s * RPI + lrow < len ? 1u << s : 0u;
    } else {
#pragma unroll
      for (int s = 0; s < KS; ++s)
        ok |= (it + ntd) * kTile + s * RPI + lrow < P.nodes ? 1u << s : 0u;
    }
    return ok;
  };
  // One tile's loads: K (is_v false), V (true), or both.
  auto issue_part = [&](int idx, const int (&ph)[2], bool k, bool v) {
    if (tbeg + ln + LN * idx < ntd) {
      if (k) issue_half(idx, ph, false, std::true_type{});
      if (v) issue_half(idx, ph, true, std::true_type{});
    } else {
      if (k) issue_half(idx, ph, false, std::false_type{});
      if (v) issue_half(idx, ph, true, std::false_type{});
    }
    if (v) rowok = rows_of(idx, ph);
  };
  auto issue = [&](int idx, const int (&ph)[2]) { issue_part(idx, ph, true, true); };

  // first_tag: std::true_type for the wave's first tile (a separate copy
  // of the tile code), std::false_type for the rest.
  // Valid token rows of tile idx as a bit mask (bit i = token tbase + i):
  // prefix tiles clip at the length and drop pages outside the pool; draft
  // tiles take this row's ancestor-or-self set.
  auto okbits_of = [&](int idx, const int (&ph)[2], bool is_draft) {
    const int it = tbeg + ln + LN * idx;
    const int tbase = (is_draft ? it : it - ntd) * kTile;
    return is_draft ? ancestor_bits(parr, P.nodes, node, tbase)
                    : prefix_bits(len - tbase, ph[0], ph[1], P.phys_pages);
  };
  // staged: the tile's rows are in the staging area already (an early
  // wave's first tile, see below).
  auto process = [&](int idx, uint32_t okbits, const int (&next_ids)[2], auto first_tag,
                     bool staged = false) {
    // Stage K and V rows; rows that are not valid tokens may hold any bits
    // (NaN included): their weight is zero, so their V row must be zero.
    auto stage_v = [&]() {
#pragma unroll
      for (int s = 0; s < KS; ++s)
        *reinterpret_cast<uint4*>(vs + (s * RPI + lrow) * VP + lcol) = vreg[s];
      if (__builtin_amdgcn_ballot_w64(rowok != kAllRows)) {  // rows past the data: zero V
#pragma unroll
        for (int s = 0; s < KS; ++s)
          if (!((rowok >> s) & 1u))
            *reinterpret_cast<uint4*>(vs + (s * RPI + lrow) * VP + lcol) = make_uint4(0, 0, 0, 0);
      }
    };
    constexpr bool first = decltype(first_tag)::value;
    if (!staged) {
#pragma unroll
      for (int s = 0; s < KS; ++s)
        *reinterpret_cast<uint4*>(ks + (s * RPI + lrow) * KP + lcol) = kreg[s];
      // The first tile's scores start as soon as its K is staged (its V was
      // issued after K and Q); later tiles stage both, then issue the next
      // tile's loads, which are then in flight during this tile's MFMAs.
      if (!first) stage_v();
    }
    wave_lds_sync();
    if (!first && idx + 1 < nmine) issue(idx + 1, next_ids);
    // The first tile's K registers are free once K is staged: the next
    // tile's K loads go out now, its V loads once this tile's V is staged.
    if (first && idx + 1 < nmine) issue_part(idx + 1, next_ids, true, false);
    f16x8 pb[2], pl[2];
    if constexpr (QL)
      tile_scores<D, 64, first>(ks + lr * KP, s_q + (size_t)rq * KS * 64 + lane, okbits,
                                P.scale_log2, g, acc, m, l, pb, pl);
    else
      tile_scores<D, 1, first>(ks + lr * KP, qreg, okbits, P.scale_log2, g, acc, m, l, pb, pl);
    if constexpr (first) {
      stage_v();
      wave_lds_sync();
      if (idx + 1 < nmine) issue_part(idx + 1, next_ids, false, true);
    }
    tile_pv<D, first>(vtr, pb, pl, acc);
    // The staging area is rewritten by the next tile.
    wave_lds_sync();
  };

  // Ids of the wave's tile idx < nmine: entries past the page table read as
  // -1 (a draft tile's entries are never used).
  auto ids_of = [&](int idx, int (&ph)[2]) {
    if ((idx & 31) == 0 && idx > 0) {  // uniform: move to the next chunk of ids
      idv = idv_next;
      if (T > 32 * LN * ((idx >> 5) + 1)) idv_next = load_ids((idx >> 5) + 1);
    }
    const int pg = (tbeg + ln + LN * idx - ntd) * (kTile / BC_PAGE_SIZE);
    const int r0 = __builtin_amdgcn_readlane(idv, 2 * (idx & 31));
    const int r1 = __builtin_amdgcn_readlane(idv, 2 * (idx & 31) + 1);
    ph[0] = pg >= 0 && pg < P.max_pages ? r0 : -1;
    ph[1] = pg >= 0 && pg + 1 < P.max_pages ? r1 : -1;
  };
  auto load_parents = [&]() {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      parr[c] = P.parent[(size_t)b * P.nodes + min(lane + 64 * c, P.nodes - 1)];
  };
  // This wave's Q fragments into s_q.  Each path below writes them itself:
  // the compiler's wait for Q at a point both paths reach is the stricter of
  // the two, and it would make the later path wait for its whole first tile.
  auto publish_q = [&]() {
    if constexpr (QL) {
#pragma unroll
      for (int j = 0; j < QPW; ++j)
        if (ln + LN * j < KS) s_q[((size_t)rq * KS + ln + LN * j) * 64 + lane] = qown[j];
    }
  };
  // Tile 0's loads, one straight-line sequence for draft and prefix tiles
  // alike (each address selected per wave): K, the parents, then V, so a
  // prefix tile's scores wait for Q and K only.  A wave without tiles issues
  // them too (pages outside the pool read page 0, draft rows past the node
  // count the last node's row, all in bounds), so every wave runs the same
  // loads and barriers.  Only a prefix tile's addresses wait for the scalar
  // loads above; an early wave issues its draft tile's loads at once and
  // stages the tile before the Q barrier, and after the barrier its first
  // step issues the second tile's loads (in single passes over short
  // prefixes this is the wave with the extra tile: one request over 256
  // tokens has 9 tiles for 8 waves).
  auto issue_first = [&](bool is_v) {
    uint4 (&dst)[KS] = is_v ? vreg : kreg;
    const uint16_t* pbase = is_v ? P.v : P.k;
    const uint16_t* dbase = is_v ? P.dv : P.dk;
    const int dn0 = (tbeg + ln) * kTile + lrow;  // draft row of load 0 (early waves)
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const bool okp = cur[q] >= 0 && cur[q] < P.phys_pages;
      const char* pg = reinterpret_cast<const char*>(
          pbase + (size_t)(okp ? cur[q] : 0) * page_elems + (size_t)kvh * D);
#pragma unroll
      for (int j = 0; j < LPP; ++j) {
        const int s = q * LPP + j;
        const int dn = min(dn0 + s * RPI, P.nodes - 1);
        const uint16_t* da = dbase + (((size_t)b * P.nodes + dn) * P.hkv + kvh) * D + lcol;
        dst[s] = *(early ? reinterpret_cast<const uint4*>(da)
                         : reinterpret_cast<const uint4*>(pg + loff[j]));
      }
    }
  };
  __builtin_amdgcn_sched_barrier(0);  // Q's loads go out before the id wait
  if (!early) {
    cur[0] = pg0 >= 0 && pg0 < P.max_pages ? raw0 : -1;
    cur[1] = pg0 >= 0 && pg0 + 1 < P.max_pages ? raw1 : -1;
  }
  issue_first(false);
  load_parents();
  issue_first(true);
  publish_q();
  if (early) {
    // The draft tile's rows into the staging area (V rows that are not
    // tokens zeroed by a mask), then the length.  No vector load is issued
    // here: the waits after this block are then exactly the other path's
    // (issuing the second tile here made that path's first K wait also
    // cover most of its V).
    rowok = rows_of(0, cur);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const unsigned keep = 0u - ((rowok >> s) & 1u);
      *reinterpret_cast<uint4*>(ks + (s * RPI + lrow) * KP + lcol) = kreg[s];
      *reinterpret_cast<uint4*>(vs + (s * RPI + lrow) * VP + lcol) =
          make_uint4(vreg[s].x & keep, vreg[s].y & keep, vreg[s].z & keep, vreg[s].w & keep);
    }
    len_raw = P.lengths[b];
  }
  set_lengths();
  rowok = rows_of(0, cur);
  if constexpr (QL) {
    __syncthreads();  // every wave's Q fragments are in s_q
  } else {
#pragma unroll
    for (int j = 0; j < KS; ++j) qreg[j] = qown[j];
  }
  if (nmine > 0 && !early) {
    int nxt[2] = {-1, -1};
    if (1 < nmine) ids_of(1, nxt);
    process(0, okbits_of(0, cur, false), nxt, std::true_type{});
    cur[0] = nxt[0];
    cur[1] = nxt[1];
  } else {
    // No tile yet, or an early wave's staged first tile, which the loop
    // below takes with the later tiles' code from acc = 0, m = -inf, l = 0:
    // the rescale then multiplies zeros by 0, and the result is the
    // first-tile code's bit for bit.
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[dt][j] = 0.f;
  }
  // The loads run one tile ahead of the MFMAs: while tile idx is processed,
  // tile idx+1's rows are loading.
  for (int idx = early ? 0 : 1; idx < nmine; ++idx) {
    int nxt[2] = {-1, -1};
    if (idx + 1 < nmine) ids_of(idx + 1, nxt);
    process(idx, okbits_of(idx, cur, tbeg + ln + LN * idx < ntd), nxt, std::false_type{},
            early && idx == 0);
    cur[0] = nxt[0];
    cur[1] = nxt[1];
  }
  l += shfl_xor_f(l, 32);  // both lane halves share m

  // ---- merge each request's LN waves through LDS in one step ----
  // Every wave stores its state in its own staging area as soon as its
  // tiles are done: no other wave uses that area, so the stores need no
  // barrier and overlap the waves still computing.  After one barrier each
  // thread combines the LN states of its request's share of the tile (row
  // mrow, DPT dims) and writes it.
  constexpr int XP = D + 4;      // padded rows: a float4 access spreads over banks
  constexpr int XW = STAGE / 2;  // floats in a wave's staging area
  static_assert(32 * XP + 64 <= XW, "a wave's state fits its staging area");
  // Wave w's state: [32 rows][XP] accumulators, then (max, sum) per row.
  auto xw = [&](int w) { return reinterpret_cast<float*>(s_stage) + (size_t)w * XW; };
  {
    float* dst = xw(wave) + (size_t)lr * XP;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq)
        *reinterpret_cast<float4*>(dst + 32 * dt + 8 * jq + 4 * g) =
            make_float4(acc[dt][4 * jq], acc[dt][4 * jq + 1], acc[dt][4 * jq + 2],
                        acc[dt][4 * jq + 3]);
    if (g == 0) *reinterpret_cast<float2*>(xw(wave) + 32 * XP + 2 * lr) = make_float2(m, l);
  }
  __syncthreads();
  constexpr int TPR = 2 * LN;   // threads per row
  constexpr int DPT = D / TPR;  // dims per thread
  static_assert(DPT % 4 == 0, "float4 steps");
  const int t = threadIdx.x % (64 * LN);  // the request's waves hold its rows
  const int mrow = t / TPR;
  const int md0 = (t % TPR) * DPT;
  const int rr = rt * 32 + mrow;
  if (!present || rr >= P.rows) return;
  const int w0 = rq * LN;
  float mw[LN], mm = kNegInf;
#pragma unroll
  for (int w = 0; w < LN; ++w) {
    mw[w] = xw(w0 + w)[32 * XP + 2 * mrow];
    mm = __builtin_fmaxf(mm, mw[w]);
  }
  const float ms = safe_max(mm);  // all waves empty: every weight is 0
  float ll = 0.f, o[DPT];
#pragma unroll
  for (int j = 0; j < DPT; ++j) o[j] = 0.f;
#pragma unroll
  for (int w = 0; w < LN; ++w) {
    const float wt = fast_exp2(mw[w] - ms);  // 0 for a wave without tiles
    ll += wt * xw(w0 + w)[32 * XP + 2 * mrow + 1];
    const float* src = xw(w0 + w) + (size_t)mrow * XP + md0;
#pragma unroll
    for (int j = 0; j < DPT; j += 4) {
      const float4 v4 = *reinterpret_cast<const float4*>(src + j);
      o[j] += wt * v4.x;
      o[j + 1] += wt * v4.y;
      o[j + 2] += wt * v4.z;
      o[j + 3] += wt * v4.w;
    }
  }
  const int rrn = div_by(rr, P.group, P.group_mul);
  const size_t orow =
      ((size_t)b * P.nodes + rrn) * P.hq + kvh * P.group + (rr - rrn * P.group);
  if (WHOLE || P.parts == 1) {
    const float inv = 1.f / ll;  // every row sees its own node: ll > 0
    float* dst = P.out + orow * D + md0;
#pragma unroll
    for (int j = 0; j < DPT; j += 4)
      *reinterpret_cast<float4*>(dst + j) =
          make_float4(o[j] * inv, o[j + 1] * inv, o[j + 2] * inv, o[j + 3] * inv);
  } else if (tbeg < ntot) {
    const size_t slot = orow * P.parts + part;
    float* dst = P.part_acc + slot * D + md0;
#pragma unroll
    for (int j = 0; j < DPT; j += 4)
      *reinterpret_cast<float4*>(dst + j) = make_float4(o[j], o[j + 1], o[j + 2], o[j + 3]);
    if (md0 == 0) *reinterpret_cast<float2*>(P.part_ml + 2 * slot) = make_float2(mm, ll);
  }
}

template <int D, int W, int RQ>
__global__ __launch_bounds__(64 * W, 2) void tree_split_kernel(TreeParams P) {
  pin_params(P);
  tree_split_body<D, W, RQ, false>(P);
}

// Combines tree_split_kernel's partials: one wave per output row (b, node,
// h); the parts that held tiles, [0, nparts) with nparts from the request's
// length, wrote slots (row, part).  Lane p holds slot p's (max, sum); the
// weights are formed once and every lane accumulates its dims from the
// slots.  The (max, sum) loads and the first 8 * NB slots' accumulators go
// out together with the length, in one memory round (NB = ceil(parts / 8),
// at most 4); slots past nparts are masked afterwards (their contents are
// whatever the workspace held).  Rows of more than 8 * NB parts load the
// rest eight slots at a time.
template <int D, int NB>
__global__ __launch_bounds__(256) void merge_split_kernel(TreeParams P) {
  pin_params(P);
  constexpr int PER = D / 64;
  constexpr int NS = 8 * NB;  // slots loaded in the first round
  const int lane = threadIdx.x & 63;
  const size_t row = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);  // (b*N+node)*Hq+h
  if (row >= (size_t)P.batch * P.nodes * P.hq) return;
  const int b = row / ((size_t)P.nodes * P.hq);
  const int lraw = P.lengths[b];
  const size_t base = row * P.parts;  // P.parts <= 64
  auto load_slot = [&](int sidx, float (&v)[PER]) {
    const float* src = P.part_acc + (base + sidx) * D + lane;
#pragma unroll
    for (int j = 0; j < PER; ++j) v[j] = src[64 * j];
  };
  const float2 ml0 = *reinterpret_cast<const float2*>(P.part_ml + 2 * (base + min(lane, P.parts - 1)));
  float v[NS][PER];
#pragma unroll
  for (int u = 0; u < NS; ++u) load_slot(min(u, P.parts - 1), v[u]);
  // Nothing that waits for the length moves above the last slot load.
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < PER; ++j)
#pragma unroll
    for (int u = 0; u < NS; ++u) asm volatile("" ::"v"(v[u][j]));
  const int len = max(0, min(lraw, P.max_pages * BC_PAGE_SIZE));
  const int ntot = (len + kTile - 1) / kTile + (P.nodes + kTile - 1) / kTile;
  const int nparts = (ntot + P.tiles_per_part - 1) / P.tiles_per_part;  // >= 1
  const bool written = lane < nparts;
  const float mp = written ? ml0.x : kNegInf;
  const float lp = written ? ml0.y : 0.f;
  const float mm = wave_max(mp);
  const float w = fast_exp2(mp - mm);  // every row sees its own node: mm finite
  const float lsum = wave_sum(w * lp);
  auto weight = [&](int i) {
    return __builtin_bit_cast(float,
                              __builtin_amdgcn_readlane(__builtin_bit_cast(int, w), i));
  };
  float a[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) a[j] = 0.f;
#pragma unroll
  for (int u = 0; u < NS; ++u) {
    if (u < nparts) {  // uniform
      const float wi = weight(u);
#pragma unroll
      for (int j = 0; j < PER; ++j) a[j] += wi * v[u][j];
    }
  }
  for (int i0 = NS; i0 < nparts; i0 += 8) {
    float x[8][PER];
#pragma unroll
    for (int u = 0; u < 8; ++u) load_slot(min(i0 + u, nparts - 1), x[u]);
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if (i0 + u < nparts) {  // uniform
        const float wi = weight(i0 + u);
#pragma unroll
        for (int j = 0; j < PER; ++j) a[j] += wi * x[u][j];
      }
    }
  }
  const float inv = 1.f / lsum;
#pragma unroll
  for (int j = 0; j < PER; ++j) P.out[row * D + lane + 64 * j] = a[j] * inv;
}

template <int D>
void launch_merge_split(const TreeParams& P, dim3 grid, hipStream_t st) {
  if (P.parts <= 8) merge_split_kernel<D, 1><<<grid, 256, 0, st>>>(P);
  else if (P.parts <= 16) merge_split_kernel<D, 2><<<grid, 256, 0, st>>>(P);
  else if (P.parts <= 24) merge_split_kernel<D, 3><<<grid, 256, 0, st>>>(P);
  else merge_split_kernel<D, 4><<<grid, 256, 0, st>>>(P);
}

// ---- softmax pieces of tree_wide_kernel and tree_flat_kernel ----

// Scores of the lane's query row at the tokens outside ok to -inf: sc[j] holds
// token row 8*(j/4) + 4*g + j%4.
__device__ __forceinline__ void row_mask(f32x16& sc, uint32_t ok, int g) {
  const uint32_t ob = ok >> (4 * g);
#pragma unroll
  for (int j = 0; j < 16; ++j) sc[j] = (ob >> (8 * (j >> 2) + (j & 3))) & 1u ? sc[j] : kNegInf;
}

// Online softmax: moves the row's running max m (log2 units) for the raw
// scores of NT tiles and rescales l and acc.  The max moves only when it
// would grow by more than kRescaleSlack, so the two lane halves of a row
// compare their own maxima and exchange them only then.
template <int DT, int NT>
__device__ __forceinline__ void row_max(const f32x16 (&sc)[NT], float scale_log2, float& m,
                                         float& l, f32x16 (&acc)[DT]) {
  float tmax = kNegInf;
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) tmax = __builtin_fmaxf(tmax, sc[i][j]);
  tmax *= scale_log2;
  if (__builtin_amdgcn_ballot_w64(tmax > m + kRescaleSlack)) {
    const float mnew = __builtin_fmaxf(m, __builtin_fmaxf(tmax, shfl_xor_f(tmax, 32)));
    const float alpha = fast_exp2(m - safe_max(mnew));
    l *= alpha;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[dt][j] *= alpha;
    m = mnew;
  }
}

// Weights of the 16 tokens 16 half .. of a tile as an FP16 hi/lo pair (see
// split_hi_lo), added to l; mb is the exponent base.
__device__ __forceinline__ void row_weights(const f32x16& sc, int half, float scale_log2,
                                             float mb, float& l, f16x8& pb, f16x8& pl) {
  uint32_t wh[4], wl[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    const float p0 = fast_exp2(__builtin_fmaf(sc[8 * half + 2 * x], scale_log2, -mb));
    const float p1 = fast_exp2(__builtin_fmaf(sc[8 * half + 2 * x + 1], scale_log2, -mb));
    l += p0;
    l += p1;
    split_hi_lo(p0, p1, wh[x], wl[x]);
  }
  pb = __builtin_bit_cast(f16x8, u32x4{wh[0], wh[1], wh[2], wh[3]});
  pl = __builtin_bit_cast(f16x8, u32x4{wl[0], wl[1], wl[2], wl[3]});
}

// 16-byte chunk c of token row `row` sits at chunk c ^ swz<D>(row) of the
// row's place in LDS: rows need no padding (a load straight into LDS fills
// consecutive lanes' chunks), and both the K reads (16 rows, one chunk each)
// and the V transpose reads (four rows, four chunks each) touch every bank
// once.
template <int D>
__device__ __forceinline__ int swz(int row) {
  return D == 128 ? ((row & 3) << 2) | ((row >> 2) & 3) : (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}

// 16 bytes per lane straight into LDS, lane i's at dst + 16 i (dst
// wave-uniform).  No register waits for it: the caller waits with
// wait_loads() before the barrier that publishes the data.
__device__ __forceinline__ void load_to_lds(const void* src, unsigned dst) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(src), "s"(dst)
               : "memory");
}

__device__ __forceinline__ void load_to_lds(const void* base, unsigned off, unsigned dst) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(off), "s"(base), "s"(dst)
               : "memory");
}

__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Tiles of one (KV head, row tile) of a request of length len: its draft
// tiles, then its prefix tiles.
__device__ __forceinline__ int flat_tiles(const TreeParams& P, int len) {
  return (P.nodes + kTile - 1) / kTile + (len + kTile - 1) / kTile;
}

__device__ __forceinline__ int flat_len(const TreeParams& P, int b) {
  return max(0, min(P.lengths[b], P.max_pages * BC_PAGE_SIZE));
}

// A workgroup's share of a wide tree: steps [t0, tend) of unit (request b, z =
// (KV head, row group)), one of `parts` shares of the unit.
struct WidePart {
  int b, z, len, t0, tend, parts;
};

constexpr int kWideStep = 2 * kTile;     // tokens per step
constexpr int kWideRequests = 4 * 64;    // requests of a split launch, four per lane
constexpr int kWideParts = 63;           // most shares of a unit
constexpr int kWideLeast = 6;            // fewest steps per share of a long unit
constexpr float kWideSlack = 11.f;       // steps that a batch's partials cost

// Per request: the first of its shares in the launch's order, and how many.
// They stand after the partials' (max, sum) pairs.
template <int RT>
__device__ __forceinline__ int2* wide_records(const TreeParams& P) {
  return reinterpret_cast<int2*>(P.part_ml + (size_t)P.parts * RT * 32 * 2);
}

// Set by the split launch for tree_whole_kernel behind it: whether the shares
// were taken, and not left to that kernel as whole units.
template <int RT>
__device__ __forceinline__ int* wide_taken(const TreeParams& P) {
  return reinterpret_cast<int*>(wide_records<RT>(P) + P.batch);
}

// The tiles that one CU takes one after the other where a single pass runs
// whole units (tree_whole_kernel), as far as the lengths tell: `all` tiles of
// the requests together, `longest` of the longest.  Each round over the CUs
// ends with its longest unit at the latest, and no CU gets more than its equal
// part and a unit.
__device__ __forceinline__ float whole_chain(const TreeParams& P, int all, int longest) {
  return __builtin_fminf((float)P.whole_rounds * (float)longest,
                         (float)all * (float)(P.hkv * P.row_tiles) / (float)P.cus + (float)longest);
}

// Whether shares of the batch's units beat whole ones.  Shares take a CU's part
// of the row groups, and finding, leaving and merging them costs the time of 56
// tiles (15 us); 44 where the tiles, each read once per row tile by whole units,
// are more than the L2s hold.  With two units per CU (D = 64: more) shares win
// at any length.  Over 119 batches of 1 to 64 requests x 33 to 8192 tokens,
// under tables of up to 32768, the rule takes 0.1 % longer than the faster of
// both on average and 5 % at most.  Shares against whole units, us, 32/8 heads
// and D = 128 unless noted: 1 x 300 x 256 nodes 28 against 17, 16 x 64-512 x 16
// 20 against 17, 5 x 2102 x 33 (32/4, one shared prefix) 35 against 27, 16 x
// 2454 x 16 (24/8, D = 64, shared) 25 against 22, 16 x 64-512 x 33 (28/4, D =
// 64) 19 against 16; 2 x 1058-2117 x 9 19 against 24, 14 x 2319 x 32 54 against
// 90, 16 x 200-900 x 64 39 against 62, 16 x 300-3000 x 33 (28/4, D = 64) 31
// against 47.
template <int D>
__device__ __forceinline__ bool wide_pays(const TreeParams& P, int all, int longest, int zdim) {
  const float cus = (float)P.cus;
  const float units = (float)P.batch * (float)(P.hkv * P.row_tiles);
  const bool far = (float)all * (float)(kTile * 4 * D) * (float)P.hkv > 32e6f;
  return units >= 2.f * cus + (D == 64 ? 1.f : 0.f) ||
         whole_chain(P, all, longest) > (float)all * (float)zdim / cus + (far ? 44.f : 56.f);
}

// Workgroup blockIdx.x's share when P.parts workgroups split the units on
// P.cus CUs: the shortest share of at least kWideLeast steps with
// which the batch, however ragged, needs no more than P.parts workgroups,
// from the lengths themselves (parts == 0: none left).  A request's units
// take equal shares.
// Every wave finds it for itself, a lane holding four requests; counts of a
// share per lane add up by ballots of their six bits.
template <int D, int RT>
__device__ __forceinline__ WidePart wide_part(const TreeParams& P, int lane, int zdim) {
  constexpr int NW = kWideRequests / 64;
  int len[NW], steps[NW], sum = 0, most = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    len[w] = steps[w] = 0;
    if (64 * w < P.batch) {  // uniform
      len[w] = flat_len(P, min(64 * w + lane, P.batch - 1));
      steps[w] = 64 * w + lane < P.batch ? (flat_tiles(P, len[w]) + 1) / 2 : 0;
    }
    sum += steps[w];
    most = max(most, steps[w]);
  }
  // Uniform values in scalar registers keep the search scalar.
  const int all = __builtin_amdgcn_readfirstlane(wave_sum_i(sum));
  const int longest = __builtin_amdgcn_readfirstlane((int)wave_max((float)most));
  const bool taken = wide_pays<D>(P, 2 * all, 2 * longest, zdim);
  if (blockIdx.x == 0 && threadIdx.x == 0) *wide_taken<RT>(P) = taken;
  if (!taken) return WidePart{0, 0, 0, 0, 0, 0};
  const int cap = P.parts / zdim;  // shares of all requests, >= P.batch
  // About ceil(steps / per): 1 to kWideParts, no more than steps, and 1 for
  // per == longest.  Shares follow from the count, so that it need not be exact.
  auto shares = [&](int w, int per) {
    return max((int)((float)steps[w] * __builtin_amdgcn_rcpf((float)per) + 0.999f), min(steps[w], 1));
  };
  int per = max(max((all + cap - 1) / cap, (longest + kWideParts - 1) / kWideParts),
                kWideLeast);
  // An even batch (equal lengths, most CUs with a unit) runs whole units, one
  // per CU, unless they are long: two workgroups per CU hide a fifth of the
  // steps behind each other, and a batch's partials cost about kWideSlack
  // steps.  Whole against shares, 32/8 heads and D = 128 unless noted: 8 x 2048
  // x 128 nodes 69.6 against 71.2 us, 30 x 2048 x 32 72.9 against 76.7; 57 x
  // 3696 x 11 (28/4 heads) 129 against 114, 8 x 8000 x 128 217 against 206, 28
  // x 6000 x 48 (16/4, D = 64) 111 against 94, 16 x 4096 x 64 (D = 64) 83
  // against 79.
  if (1.2f * (float)longest <= (float)all * (float)zdim / (float)P.cus + kWideSlack)
    per = max(per, longest);
  for (int hi = max(per, longest); per < hi;) {
    const int mid = (per + hi) >> 1;
    int total = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w)
      if (64 * w < P.batch) {
        const int n = shares(w, mid);
#pragma unroll
        for (int bit = 0; bit < 6; ++bit)
          total += __builtin_popcountll(__builtin_amdgcn_ballot_w64((n >> bit) & 1)) << bit;
      }
    if (total <= cap) hi = mid;
    else per = mid + 1;
  }
  WidePart p{0, 0, 0, 0, 0, 0};
  const int idx = blockIdx.x / zdim;
  p.z = blockIdx.x - idx * zdim;
  int before = 0;  // shares of the requests of earlier windows
#pragma unroll
  for (int w = 0; w < NW; ++w)
    if (64 * w < P.batch) {
      const int n = shares(w, per);
      int pre = before, total = 0;
#pragma unroll
      for (int bit = 0; bit < 6; ++bit) {
        const unsigned long long set = __builtin_amdgcn_ballot_w64((n >> bit) & 1);
        pre += __builtin_amdgcn_mbcnt_hi((unsigned)(set >> 32),
                                         __builtin_amdgcn_mbcnt_lo((unsigned)set, 0)) << bit;
        total += __builtin_popcountll(set) << bit;
      }
      const unsigned long long hit = __builtin_amdgcn_ballot_w64(pre <= idx && idx < pre + n);
      if (hit) {  // uniform
        const int at = __builtin_ffsll((long long)hit) - 1;
        const int first = __builtin_amdgcn_readlane(pre, at);
        const int all_steps = __builtin_amdgcn_readlane(steps[w], at);
        p.b = 64 * w + at;
        p.len = __builtin_amdgcn_readlane(len[w], at);
        p.parts = __builtin_amdgcn_readlane(n, at);
        p.t0 = (idx - first) * all_steps / p.parts;
        p.tend = (idx - first + 1) * all_steps / p.parts;
        if (idx == first && p.z == 0 && threadIdx.x == 0)
          wide_records<RT>(P)[p.b] = make_int2(first, p.parts);
      }
      before += total;
    }
  return p;
}

// Wide trees: a workgroup takes RT row tiles of one (request, KV head) and
// all of its steps, or with SPLIT the share that wide_part gives it (a step
// is two 32-token tiles: draft tiles first, then prefix tiles).  Its four
// waves share the steps through LDS, 4 / RT waves on each row tile: with RT =
// 4 a wave takes both tiles of a step, with RT = 2 one.  Each step's K and V
// go straight into the other of two LDS buffers while the current one is
// computed, one barrier per step, and hold no registers, so the reads of a
// whole step's K can be in flight at once.  A whole unit's rows go to the
// output, a share leaves an FP32 partial of each row, in the workgroup's own
// slots, for merge_wide.
// Bound by the matrix units and their clock: 8 requests x 2048 tokens x 256
// nodes (32/8 heads, D = 128) take 112 us, 617 TFLOP/s (925 with the second
// MFMA that P's low part takes); the MFMAs alone fill half the cycles, and
// the clock falls from 2.4 to 1.8 GHz under them.  One 32-token tile per
// barrier, staged through registers, took 143 us.
template <int D, int RT, bool SPLIT>
__global__ __launch_bounds__(256, D == 64 ? 3 : 2) void tree_wide_kernel(TreeParams P) {
  constexpr int KS = D / 16;      // MFMA k-steps over the head dimension
  constexpr int DT = D / 32;      // 32-row output tiles over the head dimension
  constexpr int TPS = 2;          // tiles per step
  constexpr int TS = 4 / RT;      // waves per row tile
  constexpr int TPW = TPS / TS;   // tiles per wave and step
  static_assert(TPW >= 1, "RT is 2 or 4");
  constexpr int CPR = D / 8;      // 16-byte chunks per token row
  constexpr int CPT = kTile * CPR / 256;  // chunks per thread and tile, K and V each
  constexpr int HALF = kTile * D;   // halves of a tile's K (then as many of V)
  constexpr int TILE = 2 * HALF;
  constexpr int PPS = TPS * kTile / BC_PAGE_SIZE;  // pages per step
  constexpr int SPC = 64 / PPS;                    // steps per register of page ids

  pin_params(P);
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 5;   // lane half
  const int lr = lane & 31;  // tile column (query row) / token slot
  const int wrt = wave % RT, wts = wave / RT;  // this wave's row tile and tile of a step

  __shared__ __attribute__((aligned(256))) _Float16 s_kv[2][TPS * TILE];
  __shared__ uint4 s_anc[BC_MAX_TREE_NODES][2];  // ancestor-or-self set per node, 256 bits
  __shared__ int s_ptr[BC_MAX_TREE_NODES];

  // Workgroup ids put (KV head, row group) in the low bits, then the share,
  // then the request.
  const int rgroups = (P.row_tiles + RT - 1) / RT;
  const int zdim = P.hkv * rgroups;
  WidePart w{0, 0, 0, 0, 0, 1};
  if constexpr (SPLIT) {
    w = wide_part<D, RT>(P, lane, zdim);
    if (w.parts == 0) return;  // uniform
  } else {
    w.b = blockIdx.x / zdim;
    w.z = blockIdx.x - w.b * zdim;
  }
  const int b = w.b, t0 = w.t0;
  const int kvh = w.z / rgroups;
  int rg = w.z - kvh * rgroups;
  // Whole units: the later row groups of a tree see more of its draft tiles
  // (below), so every other round of workgroups over the CUs takes them in the
  // opposite order.
  if (!SPLIT && ((b * P.hkv + kvh) * rgroups / P.cus) & 1) rg = rgroups - 1 - rg;

  // First round of loads: the page ids (lane i of a register: entry i of the
  // 64 table entries from step t on, from inside the request's table row),
  // the row's Q^T fragments (rows past the tree read row (node 0, head 0),
  // whose columns are never written out), the parents and the length.
  int ntd = (P.nodes + kTile - 1) / kTile;
  auto load_ids = [&](int t) {
    const int pg = t * PPS - ntd * (kTile / BC_PAGE_SIZE) + lane;
    return P.pages[(size_t)b * P.max_pages + min(max(pg, 0), P.max_pages - 1)];
  };
  int ids = load_ids(t0), ids_next = load_ids(t0 + SPC);
  const int r = (rg * RT + wrt) * 32 + lr;
  const int rnode = div_by(r, P.group, P.group_mul);
  const int node = r < P.rows ? rnode : 0;
  const int h = kvh * P.group + (r < P.rows ? r - rnode * P.group : 0);
  uint4 qB[KS];
  {
    const uint16_t* qp = P.dq + (((size_t)b * P.nodes + node) * P.hq + h) * D + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) qB[s] = ldg16(qp + 16 * s);
  }
  const int me = min(tid, P.nodes - 1);
  int up = P.parent[(size_t)b * P.nodes + me];
  const int len = SPLIT ? w.len : flat_len(P, b);
  int tend = SPLIT ? w.tend : (flat_tiles(P, len) + TPS - 1) / TPS;

  // Loads: chunk c of a tile is token row (tid + 256c) / CPR, 16 bytes at
  // 8 * (tid % CPR); a wave's chunk lies in one page.
  const int lrow = tid / CPR, lcol = 8 * (tid % CPR ^ swz<D>(lrow));
  const size_t tok_stride = (size_t)P.hkv * D;
  const unsigned loff = (unsigned)(((lrow % BC_PAGE_SIZE) * tok_stride + lcol) * sizeof(uint16_t));
  const unsigned page_bytes = (unsigned)(BC_PAGE_SIZE * tok_stride * sizeof(uint16_t));
  const char* const kb = reinterpret_cast<const char*>(P.k + (size_t)kvh * D);
  const char* const vb = reinterpret_cast<const char*>(P.v + (size_t)kvh * D);
  // LDS byte address of this wave's first chunk of tile 0's K in buffer 0.
  const unsigned lds0 = __builtin_amdgcn_readfirstlane(
      (unsigned)(uintptr_t)(__attribute__((address_space(3))) _Float16*)s_kv + wave * 1024);
  auto lds_of = [&](int buf, int i, int c) {
    return lds0 + (unsigned)(buf * TPS * TILE * 2 + i * TILE * 2 + c * 4096);
  };
  // Chunk x of a prefix step from page ids inside the pool, K and V.
  constexpr int NX = TPS * CPT;
  auto issue_chunk = [&](int x, const int (&ph)[PPS], int buf) {
    const int i = x / CPT, c = x % CPT;
    const unsigned id = CPT == 2 ? ph[2 * i + c] : wave < 2 ? ph[2 * i] : ph[2 * i + 1];
    const unsigned long long off = (unsigned long long)id * page_bytes;
    load_to_lds(kb + off, loff, lds_of(buf, i, c));
    load_to_lds(vb + off, loff, lds_of(buf, i, c) + HALF * 2);
  };
  // Any step.  Pages outside the pool read page 0, rows past the length
  // their page's rows and draft rows past the node count the last node's: all
  // in bounds, all masked (a draft tile's page ids are unused).
  auto issue = [&](int t, const int (&ph)[PPS], int buf) {
    int in[PPS];
#pragma unroll
    for (int q = 0; q < PPS; ++q) in[q] = (unsigned)ph[q] < (unsigned)P.phys_pages ? ph[q] : 0;
#pragma unroll
    for (int x = 0; x < NX; ++x) {
      const int i = x / CPT, c = x % CPT, it = t * TPS + i;
      if (it >= ntd) {
        issue_chunk(x, in, buf);
      } else {
        const int dn = min(it * kTile + lrow + 256 / CPR * c, P.nodes - 1);
        const size_t off = (((size_t)b * P.nodes + dn) * P.hkv + kvh) * D + lcol;
        load_to_lds(P.dk + off, lds_of(buf, i, c));
        load_to_lds(P.dv + off, lds_of(buf, i, c) + HALF * 2);
      }
    }
  };
  // Whether every token of the step is a valid prefix token; else the valid
  // ones per tile (of draft tiles: of the node count) in rows.
  auto whole_step = [&](int t, const int (&ph)[PPS], uint32_t (&rows)[TPS]) {
    bool ok = t * TPS >= ntd && ((t + 1) * TPS - ntd) * kTile <= len;
#pragma unroll
    for (int q = 0; q < PPS; ++q) ok = ok && (unsigned)ph[q] < (unsigned)P.phys_pages;
    if (ok) return true;
#pragma unroll
    for (int i = 0; i < TPS; ++i) {
      const int it = t * TPS + i;
      rows[i] = __builtin_amdgcn_readfirstlane(
          it < ntd ? prefix_bits(P.nodes - it * kTile, 0, 0, 1)
                   : prefix_bits(len - (it - ntd) * kTile, ph[2 * i], ph[2 * i + 1], P.phys_pages));
    }
    return false;
  };
  // V rows that are not valid tokens may hold any bits (NaN included): their
  // weight is zero, so the rows must be zero.  Each lane clears the chunks
  // that its own loads, already waited for, have filled.
  auto clear = [&](const uint32_t (&rows)[TPS], _Float16* buf) {
#pragma unroll
    for (int i = 0; i < TPS; ++i)
#pragma unroll
      for (int c = 0; c < CPT; ++c)
        if (!((rows[i] >> (lrow + 256 / CPR * c)) & 1u))
          *reinterpret_cast<uint4*>(buf + i * TILE + HALF + (tid + 256 * c) * 8) =
              make_uint4(0, 0, 0, 0);
  };
  auto take_ids = [&](int v, int step, int (&ph)[PPS]) {
#pragma unroll
    for (int q = 0; q < PPS; ++q) ph[q] = __builtin_amdgcn_readlane(v, step * PPS + q);
  };

  int ph[PPS];
  uint32_t rows[TPS] = {~0u, ~0u};
  take_ids(ids, 0, ph);
  issue(t0, ph, 0);
  bool whole = whole_step(t0, ph, rows);

  // Ancestor sets, while the first step loads.  Pointer doubling: after round
  // k thread i holds the nodes within 2^k steps of node i and the node 2^k
  // steps up, so a chain of any depth (or a cycle) takes at most eight
  // rounds; a serial walk pays one LDS round trip per step of the chain, in
  // every draft tile (2 requests x 333 tokens x a 256-node chain: 88.6 us).
  if (t0 * TPS < ntd && P.nodes <= 64) {
    // One node per lane of the first wave: no LDS and no barrier a round (64 x
    // 8-64 tokens x 33 nodes, 32/8 heads, D = 128: 29.0 -> 26.1 us; 64 x 16-128
    // x 64, D = 64: 24.8 -> 21.8).  The barrier below publishes the sets.
    if (wave == 0) {
      uint32_t set0 = lane < 32 ? 1u << lane : 0u, set1 = lane < 32 ? 0u : 1u << (lane - 32);
      if (lane >= P.nodes || up < 0 || up >= P.nodes) up = -1;
      for (int round = 0; round < 6 && __builtin_amdgcn_ballot_w64(up >= 0); ++round) {
        const int from = max(up, 0);
        const uint32_t a0 = __shfl(set0, from, 64), a1 = __shfl(set1, from, 64);
        const int next = __shfl(up, from, 64);
        if (up >= 0) {
          set0 |= a0;
          set1 |= a1;
          up = next;
        }
      }
      s_anc[lane][0] = make_uint4(set0, set1, 0, 0);
    }
  } else if (t0 * TPS < ntd) {  // uniform: the share holds draft tiles
    uint32_t set[8];
#pragma unroll
    for (int w = 0; w < 8; ++w) set[w] = (me >> 5) == w ? 1u << (me & 31) : 0u;
    if (up < 0 || up >= P.nodes) up = -1;
    for (int round = 0;; ++round) {
      s_anc[tid][0] = make_uint4(set[0], set[1], set[2], set[3]);
      s_anc[tid][1] = make_uint4(set[4], set[5], set[6], set[7]);
      s_ptr[tid] = up;
      if (!__syncthreads_or(up >= 0) || round == 8) break;  // uniform
      if (up >= 0) {
        const uint4 s0 = s_anc[up][0], s1 = s_anc[up][1];
        set[0] |= s0.x;
        set[1] |= s0.y;
        set[2] |= s0.z;
        set[3] |= s0.w;
        set[4] |= s1.x;
        set[5] |= s1.y;
        set[6] |= s1.z;
        set[7] |= s1.w;
        up = s_ptr[up];
      }
      __syncthreads();
    }
    // A whole unit ends its draft tiles with the last one that holds an
    // ancestor of its rows (parents stand before their children, so that is
    // half of them on average); the two that the first step has loaded stay.
    // The prefix tiles move up, and their page ids with them.  28 requests x
    // 14-113 tokens x 221 nodes (32/8 heads, D = 128) 88 -> 71 us, 8 x 2048 x
    // 256 nodes 120 -> 116.
    if (!SPLIT && ntd > TPS) {
      const int r0 = rg * RT * 32, r1 = min(r0 + RT * 32, P.rows) - 1;
      const int n1 = div_by(r1, P.group, P.group_mul);
      int last = 0;
      for (int n0 = div_by(r0, P.group, P.group_mul); n0 <= n1; n0 += 64) {
        const int n = min(n0 + lane, n1);
        const uint4 s0 = s_anc[n][0], s1 = s_anc[n][1];
        const int mine = s1.w ? 7 : s1.z ? 6 : s1.y ? 5 : s1.x ? 4 : s0.w ? 3 : s0.z ? 2 : 0;
        last = max(last, mine);
      }
      int used = TPS;
#pragma unroll
      for (int i = TPS; i < 8; ++i) used = __builtin_amdgcn_ballot_w64(last >= i) ? i + 1 : used;
      const int off = ntd - used;
      ntd = used;
      tend = (flat_tiles(P, len) - off + TPS - 1) / TPS;
      const int from = lane + off * (kTile / BC_PAGE_SIZE);
      const int lo = __shfl(ids, from & 63, 64), hi = __shfl(ids_next, from & 63, 64);
      ids = from < 64 ? lo : hi;
      ids_next = load_ids(SPC);
    }
  }

  // Read offsets in a staged tile (halves): K chunk 2s + g of row lr, and the
  // V transpose reads' [token 4 * (trG / 2) + trj / 4 (+ 8 hf)][dim
  // 16 * (trG % 2) + 4 * (trj % 4) (+ 32 dt)].
  const int trG = lane >> 4, trj = lane & 15;
  int koff[KS], voff[2][DT];
#pragma unroll
  for (int s = 0; s < KS; ++s) koff[s] = lr * D + ((2 * s + g) ^ swz<D>(lr)) * 8;
#pragma unroll
  for (int hf = 0; hf < 2; ++hf)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const int row = 4 * (trG >> 1) + (trj >> 2) + 8 * hf;
      const int dim = 32 * dt + 16 * (trG & 1) + 4 * (trj & 3);
      voff[hf][dt] = HALF + row * D + ((dim >> 3) ^ swz<D>(row)) * 8 + (dim & 7);
    }
  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[dt][j] = 0.f;
  float m = kNegInf, l = 0.f;
  constexpr int NG = 2 * TPW;  // 16-token groups per wave and step
  static_assert(KS / 2 >= NX, "a step's loads fit between its score MFMAs");
  // The wait for Q belongs here: left to its first use, inside the step
  // loop, the compiler's wait there also covers the loads each step has just
  // issued.
#pragma unroll
  for (int s = 0; s < KS; ++s)
    asm volatile("" : "+v"(qB[s].x), "+v"(qB[s].y), "+v"(qB[s].z), "+v"(qB[s].w));
  wait_loads();
  if (!whole) clear(rows, s_kv[0]);
  __syncthreads();

  int k = 0;
  for (int t = t0; t < tend; ++t) {
    // The next step's page ids; a step of other than valid prefix tokens
    // only is issued here, the others between the score MFMAs below: issued
    // together, the four waves' loads queue for the CU's 64 bytes per clock
    // and hold up the math behind them.
    bool whole_n = true, next = false;
    uint32_t rows_n[TPS] = {~0u, ~0u};
    if (t + 1 < tend) {
      const int i = (t + 1 - t0) % SPC;
      if (i == 0) {
        ids = ids_next;
        ids_next = load_ids(t + 1 + SPC);
      }
      take_ids(ids, i, ph);
      whole_n = next = whole_step(t + 1, ph, rows_n);
      if (!next) issue(t + 1, ph, k ^ 1);
    }
    const _Float16* base = s_kv[k] + (TS == 1 ? 0 : wts * TILE);
    f16x8 kf[TPW][KS], av[2][DT];
    f32x16 sc[TPW];
    auto read_v = [&](int grp) {
      const _Float16* v0 = base + grp / 2 * TILE + grp % 2 * 16 * D;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        const f16x4 lo = lds_read_tr(v0 + voff[0][dt]);
        const f16x4 hi = lds_read_tr(v0 + voff[1][dt]);
        av[grp % 2][dt] = f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
    };
    // ---- S^T = K Q^T ----
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int i = 0; i < TPW; ++i)
        kf[i][s] = as_f16x8(*reinterpret_cast<const uint4*>(base + i * TILE + koff[s]));
#pragma unroll
    for (int i = 0; i < TPW; ++i)
#pragma unroll
      for (int j = 0; j < 16; ++j) sc[i][j] = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
#pragma unroll
      for (int i = 0; i < TPW; ++i)
        sc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[i][s], as_f16x8(qB[s]), sc[i], 0, 0, 0);
      if (s % 2 == 1 && s / 2 < NX) {
        if (next) issue_chunk(s / 2, ph, k ^ 1);  // uniform
      }
    }
    // ---- mask and online softmax (column lr = query row) ----
    if (!whole) {
#pragma unroll
      for (int i = 0; i < TPW; ++i) {
        const int it = t * TPS + (TS == 1 ? i : wts);
        const uint32_t ok = it < ntd ? reinterpret_cast<const uint32_t*>(s_anc[node])[it]
                                     : TS == 1 ? rows[i] : wts ? rows[1] : rows[0];
        row_mask(sc[i], ok, g);
      }
    }
    row_max<DT, TPW>(sc, P.scale_log2, m, l, acc);
    // ---- O^T += V^T P^T, the next group's weights between the MFMAs ----
    const float mb = safe_max(m);
    f16x8 pb[2], pl[2];
    auto weights = [&](int grp) {
      row_weights(sc[grp / 2], grp % 2, P.scale_log2, mb, l, pb[grp % 2], pl[grp % 2]);
    };
    read_v(0);
    weights(0);
#pragma unroll
    for (int grp = 0; grp < NG; ++grp) {
      if (grp + 1 < NG) {
        read_v(grp + 1);
        weights(grp + 1);
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        acc[dt] =
            __builtin_amdgcn_mfma_f32_32x32x16_f16(av[grp % 2][dt], pb[grp % 2], acc[dt], 0, 0, 0);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        acc[dt] =
            __builtin_amdgcn_mfma_f32_32x32x16_f16(av[grp % 2][dt], pl[grp % 2], acc[dt], 0, 0, 0);
    }
    wait_loads();
    if (!whole_n) clear(rows_n, s_kv[k ^ 1]);
    __syncthreads();
    k ^= 1;
    whole = whole_n;
#pragma unroll
    for (int i = 0; i < TPS; ++i) rows[i] = rows_n[i];
  }

  // ---- the rows' output, or this part's partial of them ----
  l += shfl_xor_f(l, 32);  // both lane halves share m
  if constexpr (TS > 1) {
    // The waves of a row tile merge through LDS (every staged tile has been
    // read).  Four-float chunk c of row lr sits at c ^ (lr % (D / 4)), so an
    // access of 32 rows spreads over the banks; (max, sum) go to s_ptr.
    static_assert(RT * 32 * D * 4 <= TPS * TILE * 2, "the states fit one buffer");
    static_assert(RT * 64 <= BC_MAX_TREE_NODES, "(max, sum) pairs fit s_ptr");
    float* mine = reinterpret_cast<float*>(s_kv[0]) + wrt * 32 * D + lr * D;
    float2* mine_ml = reinterpret_cast<float2*>(s_ptr) + wrt * 32 + lr;
    auto at = [&](int d) { return mine + (((d >> 2) ^ (lr % (D / 4))) << 2); };
    if (wts == 1) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int jq = 0; jq < 4; ++jq)
          *reinterpret_cast<float4*>(at(32 * dt + 8 * jq + 4 * g)) =
              make_float4(acc[dt][4 * jq], acc[dt][4 * jq + 1], acc[dt][4 * jq + 2],
                          acc[dt][4 * jq + 3]);
      if (g == 0) *mine_ml = make_float2(m, l);
    }
    __syncthreads();
    if (wts == 1) return;
    const float2 ml = *mine_ml;
    const float mm = __builtin_fmaxf(m, ml.x);
    const float a1 = fast_exp2(m - safe_max(mm)), a2 = fast_exp2(ml.x - safe_max(mm));
    l = l * a1 + ml.y * a2;
    m = mm;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq) {
        const float4 v4 = *reinterpret_cast<const float4*>(at(32 * dt + 8 * jq + 4 * g));
        acc[dt][4 * jq] = acc[dt][4 * jq] * a1 + v4.x * a2;
        acc[dt][4 * jq + 1] = acc[dt][4 * jq + 1] * a1 + v4.y * a2;
        acc[dt][4 * jq + 2] = acc[dt][4 * jq + 2] * a1 + v4.z * a2;
        acc[dt][4 * jq + 3] = acc[dt][4 * jq + 3] * a1 + v4.w * a2;
      }
  }
  float inv = 1.f;
  float* to = P.out;
  size_t idx = ((size_t)b * P.nodes + node) * P.hq + h;  // this lane's row of `to`
  if (w.parts == 1) {
    inv = 1.f / l;  // every row sees its own node: l > 0
  } else {
    to = P.part_acc;
    idx = (size_t)blockIdx.x * (RT * 32) + wrt * 32 + lr;
    if (g == 0 && r < P.rows) *reinterpret_cast<float2*>(P.part_ml + 2 * idx) = make_float2(m, l);
  }
  if constexpr (TS > 1) {
    if (r >= P.rows) return;
    float* dst = to + idx * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int jq = 0; jq < 4; ++jq)
        *reinterpret_cast<float4*>(dst + 32 * dt + 8 * jq + 4 * g) =
            make_float4(acc[dt][4 * jq] * inv, acc[dt][4 * jq + 1] * inv,
                        acc[dt][4 * jq + 2] * inv, acc[dt][4 * jq + 3] * inv);
    return;
  }
  // Rows leave through LDS, each wave's in its own part of the staged tiles
  // (all read by now), so that a store covers whole rows; stored from the
  // accumulators, as where only half of the waves have rows to write (64 x
  // 1024 tokens x 9 nodes: 48.8 us, 49.2 through LDS), it writes 32 bytes of
  // each of 32 rows.  41 x 48-97 tokens x 137 nodes (28/4 heads, D = 128) 60.9
  // -> 57.3 us, 31 x 30-61 x 100 (32/8, D = 64) 25.0 -> 23.8, partials of 8 x
  // 4096 x 64 (32/8, D = 128) 70.3 -> 67.0.
  static_assert(RT * 32 * D * 4 <= sizeof(s_kv), "the rows fit the staged tiles");
  float* const mine = reinterpret_cast<float*>(s_kv[0]) + wrt * 32 * D;
  constexpr int C4 = D / 4;  // four-float chunks per row, chunk c of row i at c ^ (i % C4)
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int jq = 0; jq < 4; ++jq)
      *reinterpret_cast<float4*>(mine + lr * D + (((8 * dt + 2 * jq + g) ^ (lr % C4)) << 2)) =
          make_float4(acc[dt][4 * jq] * inv, acc[dt][4 * jq + 1] * inv,
                      acc[dt][4 * jq + 2] * inv, acc[dt][4 * jq + 3] * inv);
  wave_lds_sync();
  const int nrow = P.rows - (rg * RT + wrt) * 32;  // valid rows, from the first one on
  constexpr int RPS = 64 / C4;                     // rows per store
#pragma unroll
  for (int i = 0; i < 32; i += RPS) {
    const int row = i + lane / C4, c = lane % C4;
    const float4 v = *reinterpret_cast<const float4*>(mine + row * D + ((c ^ (row % C4)) << 2));
    const size_t at = __shfl((unsigned long long)idx, row, 64);
    if (row < nrow) *reinterpret_cast<float4*>(to + at * D + 4 * c) = v;
  }
}

// Combines the partials of the units that a split launch of tree_wide_kernel
// cut: wave `worker` of `workers` takes every workers-th group of CH rows of a
// unit, D / 4 lanes on a row, so that the count of shares is the wave's own and
// the rows' loads of a round, U shares of each, are in flight together.
template <int RT, int CH>
__device__ __forceinline__ int2 merge_wide_record(const TreeParams& P, int item) {
  const int zdim = P.hkv * ((P.row_tiles + RT - 1) / RT);
  constexpr int chunks = RT * 32 / CH;
  return wide_records<RT>(P)[min(item / chunks / zdim, P.batch - 1)];
}

template <int D, int RT, int CH, int U>
__device__ __forceinline__ void merge_wide(const TreeParams& P, int worker, int workers,
                                           int2 rec_next) {
  constexpr int C4 = D / 4;      // lanes per row, four dims each
  constexpr int RPW = 64 / C4;   // rows side by side in a wave
  constexpr int R = CH / RPW;
  constexpr int chunks = RT * 32 / CH;
  const int lane = threadIdx.x & 63;
  const int sub = lane / C4, c = 4 * (lane % C4);
  const int rgroups = (P.row_tiles + RT - 1) / RT, zdim = P.hkv * rgroups;
  const int items = P.batch * zdim * chunks;
  const size_t next = (size_t)zdim * (RT * 32);  // from a share's slot to the next one's
  for (int item = worker; item < items; item += workers) {
    const int2 rec = rec_next;
    rec_next = merge_wide_record<RT, CH>(P, item + workers);
    const int unit = item / chunks, ch = item % chunks;
    const int b = unit / zdim, z = unit - b * zdim;
    const int kvh = z / rgroups, rg = z - kvh * rgroups;
    const int r0 = rg * (RT * 32) + ch * CH;
    const int parts = __builtin_amdgcn_readfirstlane(rec.y);
    if (r0 >= P.rows || parts < 2) continue;  // no rows, or written by its only share
    const size_t slot0 =
        ((size_t)__builtin_amdgcn_readfirstlane(rec.x) * zdim + z) * (RT * 32) + ch * CH + sub;
    float m[R], l[R];
    float4 a[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      m[i] = kNegInf;
      l[i] = 0.f;
      a[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    for (int p0 = 0; p0 < parts; p0 += U) {
      float2 ml[U][R];
      float4 v[U][R];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const size_t at = slot0 + min(p0 + u, parts - 1) * next;
#pragma unroll
        for (int i = 0; i < R; ++i) {
          ml[u][i] = *reinterpret_cast<const float2*>(P.part_ml + 2 * (at + i * RPW));
          v[u][i] = *reinterpret_cast<const float4*>(P.part_acc + (at + i * RPW) * D + c);
        }
      }
#pragma unroll
      for (int i = 0; i < R; ++i) {
        float mn = m[i];
#pragma unroll
        for (int u = 0; u < U; ++u) mn = __builtin_fmaxf(mn, ml[u][i].x);  // the last one again
        const float ms = safe_max(mn);
        const float keep = fast_exp2(m[i] - ms);
        l[i] *= keep;
        a[i].x *= keep;
        a[i].y *= keep;
        a[i].z *= keep;
        a[i].w *= keep;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float w = p0 + u < parts ? fast_exp2(ml[u][i].x - ms) : 0.f;
          l[i] += w * ml[u][i].y;
          a[i].x += w * v[u][i].x;
          a[i].y += w * v[u][i].y;
          a[i].z += w * v[u][i].z;
          a[i].w += w * v[u][i].w;
        }
        m[i] = mn;
      }
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int r = r0 + sub + i * RPW;
      if (r < P.rows) {
        const int node = div_by(r, P.group, P.group_mul);
        const float inv = 1.f / l[i];  // every row sees its own node
        *reinterpret_cast<float4*>(
            P.out + (((size_t)b * P.nodes + node) * P.hq + kvh * P.group + (r - node * P.group)) * D +
            c) = make_float4(a[i].x * inv, a[i].y * inv, a[i].z * inv, a[i].w * inv);
      }
    }
  }
}

// ---- flat ranges: equal shares of a ragged batch's tiles ----

__device__ __forceinline__ int wave_incl_scan_i(int x, int lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  return x;
}

// Lengths of 64 consecutive requests, lane i holding request base + i's, so
// that stepping into the next request reads a register; a step out of the
// window loads the one it needs.
struct FlatLens {
  int base, len;
  __device__ __forceinline__ int at(const TreeParams& P, int lane, int b) {
    if (b < base || b - base >= 64) {
      base = b & ~63;
      len = flat_len(P, min(base + lane, P.batch - 1));
    }
    return __builtin_amdgcn_readlane(len, __builtin_amdgcn_readfirstlane(b - base));
  }
};

// Position in a range's tiles: tile t of segment `ord`, the part of unit
// (z, b) that the range covers, which ends before tile tend; `rest` tiles of
// the range follow the segment.
struct FlatPos {
  int ord, z, b, len, t, tend, rest;
};

// What merge_flat_range needs of each range, after the partials' (max, sum)
// pairs (two slots of 32 rows per range): the unit it begins in and how many
// tiles into it (an empty range: unit -1, tile 0).
__device__ __forceinline__ int2* flat_records(const TreeParams& P) {
  return reinterpret_cast<int2*>(P.part_ml + (size_t)P.parts * 2 * 32 * 2);
}

// As wide_taken.
__device__ __forceinline__ int* flat_taken(const TreeParams& P) {
  return reinterpret_cast<int*>(flat_records(P) + P.parts);
}

// Whether equal ranges beat whole units: where the longest chain of a single
// pass exceeds an equal part by the time that ranges cost, 48 tiles.  Over 118
// batches as at wide_pays 0.3 % longer than the faster of both on average, 11 %
// at most.  Ranges against whole units, us, 7 nodes, 32/8 heads and D = 128
// unless noted: 64 x 16-200 29 against 16, 64 x 32-1024 46 against 42, 64 x 2048
// (one shared prefix) 54 against 49, 32 x 64-2048 45 against 41; 64 x 128-4096
// 115 against 134 (D = 64: 67 against 77), 16 x 128-4096 47 against 60, 4 x
// 500-8000 x 8 nodes 30 against 74.
__device__ __forceinline__ bool flat_pays(const TreeParams& P, int all, int longest, int zdim) {
  return whole_chain(P, all, longest) > (float)all * (float)zdim / (float)P.cus + 48.f;
}

// Range rid's first position (ord -1: the range is empty), of P.parts equal
// ranges.  Units are ordered z (KV head, row tile) outermost, then request:
// a range of one KV head's tiles finds requests that share pages next to
// each other.
__device__ __forceinline__ FlatPos flat_first(const TreeParams& P, int lane, int rid, int zdim,
                                              FlatLens& lens) {
  const int len0 = flat_len(P, min(lane, P.batch - 1));
  int sum = lane < P.batch ? flat_tiles(P, len0) : 0, most = sum;
  for (int base = 64; base < P.batch; base += 64) {
    const int i = base + lane;
    const int n = i < P.batch ? flat_tiles(P, flat_len(P, min(i, P.batch - 1))) : 0;
    sum += n;
    most = max(most, n);
  }
  // Sums in scalar registers keep the whole walk scalar.
  const int all = __builtin_amdgcn_readfirstlane(wave_sum_i(sum));
  const int longest = __builtin_amdgcn_readfirstlane((int)wave_max((float)most));
  const bool taken = flat_pays(P, all, longest, zdim);
  if (blockIdx.x == 0 && threadIdx.x == 0) *flat_taken(P) = taken;
  const int total = all * zdim;
  const int per = (total + P.parts - 1) / P.parts;
  const int f0 = rid * per;
  const int count = taken ? min(total - f0, per) : 0;
  FlatPos p{-1, 0, 0, 0, 0, 0, 0};
  lens = FlatLens{0, len0};
  if (count <= 0) return p;
  p.ord = 0;
  p.z = f0 / all;
  int rem = f0 - p.z * all;
  for (int base = 0;; base += 64) {
    if (base > 0) lens = FlatLens{base, flat_len(P, min(base + lane, P.batch - 1))};
    const int n = base + lane < P.batch ? flat_tiles(P, lens.len) : 0;
    const int inc = wave_incl_scan_i(n, lane);
    const int tot = __builtin_amdgcn_readlane(inc, 63);
    if (rem < tot) {
      const unsigned long long hit = __builtin_amdgcn_ballot_w64(inc > rem);
      const int first = __builtin_ffsll((long long)hit) - 1;
      p.b = base + first;
      p.t = rem - __builtin_amdgcn_readlane(inc - n, first);
      p.len = __builtin_amdgcn_readlane(lens.len, first);
      break;
    }
    rem -= tot;
  }
  p.tend = min(flat_tiles(P, p.len), p.t + count);
  p.rest = count - (p.tend - p.t);
  return p;
}

// The segment after p's (p.rest > 0): the next request, or the first one of
// the next z.
__device__ __forceinline__ void flat_next(const TreeParams& P, int lane, FlatLens& lens,
                                          FlatPos& p) {
  ++p.ord;
  if (++p.b == P.batch) {
    p.b = 0;
    ++p.z;
  }
  p.len = lens.at(P, lane, p.b);
  p.t = 0;
  p.tend = min(flat_tiles(P, p.len), p.rest);
  p.rest -= p.tend;
}

// Workgroup ids go round the eight XCDs: each XCD takes a contiguous eighth
// of the ranges, so neighbouring ranges share an L2.
__device__ __forceinline__ int flat_range_id(const TreeParams& P) {
  const int n = P.parts, i = blockIdx.x;
  return n % 8 == 0 ? i % 8 * (n / 8) + i / 8 : i;
}

__device__ __forceinline__ void flat_record(const TreeParams& P, int rid, const FlatPos& p) {
  if (threadIdx.x == 0)
    flat_records(P)[rid] = p.ord < 0 ? make_int2(-1, 0) : make_int2(p.z * P.batch + p.b, p.t);
}

// Tree verification of a ragged batch in equal shares.  The batch's tiles
// (per unit, a (KV head, row tile) of a request: its draft tiles, then its
// prefix tiles) form one sequence, and workgroup r takes the r-th of
// P.parts equal ranges of it, crossing unit boundaries as it goes: however
// ragged the prefixes are, every workgroup streams the same number of
// tiles.  Within a unit's segment the W waves take tiles round-robin, each
// with its own staging area and no barrier; at the segment's end they merge
// through LDS.  A unit that lies inside one range is written directly; the
// others leave one FP32 partial per range (slot 2r for the range's first
// segment, 2r + 1 for its last), which merge_flat_range combines.
// Bound by HBM: a wave requests its next tile, also across a segment's end,
// before it computes the current one, with non-temporal loads (plain ones: 13
// us more at the shape below), ahead of the waves that compute.  64 requests x
// 128-4096 tokens x 7 nodes (520 MB) take 126 us with a workgroup per two
// requests, 100-105 us so (two boxes), 5 TB/s for the call.  Tile loads without
// the math, reach 6.9 TB/s over prefixes of equal length; a ragged batch's
// boundaries (partials, LDS merges, their kernel) cost 11 us, and four-wave
// workgroups over 512 ranges would leave twice the partials (105 us).
template <int D, int W>
__global__ __launch_bounds__(64 * W, 2) void tree_flat_kernel(TreeParams P) {
  constexpr int KS = D / 16;      // MFMA k-steps; also load instructions per tile
  constexpr int DT = D / 32;      // 32-row output tiles over the head dimension
  constexpr int KP = D + 8;       // halves per staged K row
  constexpr int VP = D + 16;      // halves per staged V row
  constexpr int LPR = D / 8;      // lanes per token row in a whole-row load
  constexpr int RPI = 64 / LPR;   // token rows per load instruction
  constexpr int LPP = KS / 2;     // load instructions per page
  constexpr int STAGE = kTile * (KP + VP);  // halves per wave
  constexpr int QPW = KS / W > 0 ? KS / W : 1;  // Q fragments loaded per wave

  pin_params(P);
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5;   // lane half
  const int lr = lane & 31;  // tile column (query row) / token slot

  __shared__ __attribute__((aligned(16))) _Float16 s_stage[W * STAGE];
  __shared__ uint4 s_q[KS * 64];            // Q^T fragments, lane-major per k-step
  __shared__ int s_parent[BC_MAX_TREE_NODES];

  const int rid = flat_range_id(P);
  const int zdim = P.hkv * P.row_tiles;
  const int ntd = (P.nodes + kTile - 1) / kTile;
  FlatLens lens{0, 0};
  FlatPos seg = flat_first(P, lane, rid, zdim, lens);
  flat_record(P, rid, seg);
  if (seg.ord < 0) return;  // uniform over the workgroup

  // Page ids of a wave's tiles, every W-th from tile t of request b: lane i
  // of a register holds page i % 2 of the i / 2-th of them, loaded from
  // inside the request's table row.
  constexpr int TPC = 32;  // tiles per register
  auto load_ids = [&](int b, int t) {
    const int pg = (t + W * (lane >> 1) - ntd) * (kTile / BC_PAGE_SIZE) + (lane & 1);
    return P.pages[(size_t)b * P.max_pages + min(max(pg, 0), P.max_pages - 1)];
  };

  _Float16* const ks = s_stage + wave * STAGE;
  _Float16* const vs = ks + kTile * KP;
  const int trG = lane >> 4, trj = lane & 15;
  const _Float16* vtr = vs + (4 * (trG >> 1) + (trj >> 2)) * VP + 16 * (trG & 1) + 4 * (trj & 3);
  // Whole-row load geometry: load s of a lane covers token row
  // s*RPI + lane/LPR, dims 8*(lane%LPR) .. +8.
  const int lrow = lane / LPR, lcol = 8 * (lane % LPR);
  const size_t tok_stride = (size_t)P.hkv * D;
  unsigned loff[LPP];
#pragma unroll
  for (int j = 0; j < LPP; ++j)
    loff[j] = (unsigned)((((size_t)(j * RPI + lrow)) * tok_stride + lcol) * sizeof(uint16_t));
  const unsigned page_bytes = (unsigned)(BC_PAGE_SIZE * tok_stride * sizeof(uint16_t));

  uint4 kreg[KS], vreg[KS];
  // Tile t of unit (kvh, b) from page ids id0 and id1 (a draft tile's are
  // unused).  Pages outside the pool read page 0, rows past the length their
  // page's rows and draft rows past the node count the last node's: all in
  // bounds, all masked.
  auto issue = [&](int kvh, int b, int t, int id0, int id1) {
    if (t >= ntd) {
      const char* kb = reinterpret_cast<const char*>(P.k + (size_t)kvh * D);
      const char* vb = reinterpret_cast<const char*>(P.v + (size_t)kvh * D);
      unsigned long long off[2];
      off[0] = (unsigned long long)((unsigned)id0 < (unsigned)P.phys_pages ? id0 : 0) * page_bytes;
      off[1] = (unsigned long long)((unsigned)id1 < (unsigned)P.phys_pages ? id1 : 0) * page_bytes;
#pragma unroll
      for (int s = 0; s < KS; ++s)
        kreg[s] = ldg16_stream(reinterpret_cast<const uint16_t*>(kb + off[s / LPP] + loff[s % LPP]));
#pragma unroll
      for (int s = 0; s < KS; ++s)
        vreg[s] = ldg16_stream(reinterpret_cast<const uint16_t*>(vb + off[s / LPP] + loff[s % LPP]));
    } else {
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const int dn = min(t * kTile + s * RPI + lrow, P.nodes - 1);
        const size_t off = (((size_t)b * P.nodes + dn) * P.hkv + kvh) * D + lcol;
        kreg[s] = ldg16(P.dk + off);
        vreg[s] = ldg16(P.dv + off);
      }
    }
  };
  // Valid tokens of a tile (draft tiles: of the node count).
  auto rows_of = [&](int len, int t, int id0, int id1) {
    if (t >= ntd && (t + 1 - ntd) * kTile <= len && (unsigned)id0 < (unsigned)P.phys_pages &&
        (unsigned)id1 < (unsigned)P.phys_pages)
      return ~0u;
    return (uint32_t)__builtin_amdgcn_readfirstlane(
        t < ntd ? prefix_bits(P.nodes - t * kTile, 0, 0, 1)
                : prefix_bits(len - (t - ntd) * kTile, id0, id1, P.phys_pages));
  };

  // ---- a segment's Q^T fragments and parents: registers, then LDS ----
  uint4 qown[QPW];
  int par_own = 0;
  auto load_q = [&](int z, int b) {
    const int kvh = div_by(z, P.row_tiles, P.rt_mul);
    const int r = (z - kvh * P.row_tiles) * 32 + lr;
    const int rnode = div_by(r, P.group, P.group_mul);
    // Lanes past the tile's query rows read row (node 0, head 0), whose
    // columns are never written out.
    const int node = r < P.rows ? rnode : 0;
    const int h = kvh * P.group + (r < P.rows ? r - rnode * P.group : 0);
    const uint16_t* qp = P.dq + (((size_t)b * P.nodes + node) * P.hq + h) * D + 8 * g;
#pragma unroll
    for (int j = 0; j < QPW; ++j) qown[j] = ldg16(qp + 16 * min(wave + W * j, KS - 1));
    par_own = P.parent[(size_t)b * P.nodes + min((int)threadIdx.x, P.nodes - 1)];
  };
  auto publish_q = [&]() {
#pragma unroll
    for (int j = 0; j < QPW; ++j)
      if (wave + W * j < KS) s_q[(wave + W * j) * 64 + lane] = qown[j];
    if ((int)threadIdx.x < P.nodes) s_parent[threadIdx.x] = par_own;
  };
  static_assert(BC_MAX_TREE_NODES <= 64 * W, "one parent entry per thread");

  // Entering a segment: ids holds the page ids of this wave's first TPC
  // tiles, ids_next the following ones and ids_seg the next segment's first.
  int ids = load_ids(seg.b, seg.t + wave);
  load_q(seg.z, seg.b);
  FlatPos nseg = seg;
  if (seg.rest > 0) flat_next(P, lane, lens, nseg);
  int ids_next = load_ids(seg.b, seg.t + wave + W * TPC);
  int ids_seg = load_ids(nseg.b, wave);
  uint32_t rows = 0;     // valid tokens of the tile in the registers
  bool loaded = false;   // whether it is the segment's first
  publish_q();
  __syncthreads();

  f32x16 acc[DT];
  for (;;) {
    const int t0 = seg.t;
    float m = kNegInf, l = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int j = 0; j < 16; ++j) acc[dt][j] = 0.f;
    const int kvh = div_by(seg.z, P.row_tiles, P.rt_mul);
    const int kvh_n = div_by(nseg.z, P.row_tiles, P.rt_mul);
    const int rt = seg.z - kvh * P.row_tiles;
    const int r = rt * 32 + lr;
    const int node = r < P.rows ? div_by(r, P.group, P.group_mul) : 0;
    // A round loads the wave's next tile -- of this segment, or the next
    // one's first -- between staging its current one and the math on it.  A
    // segment whose first tile is not in the registers yet begins with a
    // round that only loads it.
    for (int t = loaded ? t0 + wave : t0 + wave - W, i = loaded ? 0 : -1; t < seg.tend; t += W) {
      const bool math = i >= 0;
      const uint32_t now = rows;
      // A wave about to load goes ahead of one that computes.
      __builtin_amdgcn_s_setprio(2);
      if (math) {
        // Stage the tile; V rows that are not valid tokens may hold any bits
        // (NaN included): their weight is zero, so the rows must be zero.
#pragma unroll
        for (int s = 0; s < KS; ++s) {
          *reinterpret_cast<uint4*>(ks + (s * RPI + lrow) * KP + lcol) = kreg[s];
          *reinterpret_cast<uint4*>(vs + (s * RPI + lrow) * VP + lcol) = vreg[s];
        }
        if (now != ~0u) {  // uniform
#pragma unroll
          for (int s = 0; s < KS; ++s)
            if (!((now >> (s * RPI + lrow)) & 1u))
              *reinterpret_cast<uint4*>(vs + (s * RPI + lrow) * VP + lcol) =
                  make_uint4(0, 0, 0, 0);
        }
      }
      wave_lds_sync();
      const bool here = t + W < seg.tend;
      loaded = !here && seg.rest > 0 && wave < nseg.tend;
      if (here && ++i == TPC) {
        i = 0;
        ids = ids_next;
        ids_next = load_ids(seg.b, t + W + W * TPC);
      }
      if (here || loaded) {
        const int v = here ? ids : ids_seg, at = here ? 2 * i : 0, tn = here ? t + W : wave;
        const int id0 = __builtin_amdgcn_readlane(v, at);
        const int id1 = __builtin_amdgcn_readlane(v, at + 1);
        issue(here ? kvh : kvh_n, here ? seg.b : nseg.b, tn, id0, id1);
        rows = rows_of(here ? seg.len : nseg.len, tn, id0, id1);
      }
      __builtin_amdgcn_s_setprio(0);
      if (!math) continue;
      // ---- S^T = K Q^T ----
      f32x16 sc[1];
#pragma unroll
      for (int j = 0; j < 16; ++j) sc[0][j] = 0.f;
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const uint4 k0 = *reinterpret_cast<const uint4*>(ks + lr * KP + 16 * s + 8 * g);
        sc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_f16x8(k0), as_f16x8(s_q[s * 64 + lane]),
                                                       sc[0], 0, 0, 0);
      }
      if (now != ~0u || t < ntd) {
        uint32_t ok = now;
        if (t < ntd) {  // the row's ancestor-or-self set
          const int tbase = t * kTile;
          ok = 0;
          int cur = node;
          for (int steps = 0; steps < P.nodes && cur >= 0 && cur < P.nodes; ++steps) {
            if (cur >= tbase && cur < tbase + kTile) ok |= 1u << (cur - tbase);
            cur = s_parent[cur];
          }
        }
        row_mask(sc[0], ok, g);
      }
      row_max<DT, 1>(sc, P.scale_log2, m, l, acc);
      const float mb = safe_max(m);
      f16x8 pb[2], pl[2];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) row_weights(sc[0], hh, P.scale_log2, mb, l, pb[hh], pl[hh]);
      tile_pv<D, false>(vtr, pb, pl, acc);
      wave_lds_sync();
    }

    // ---- segment end: merge the W waves through LDS, write, move on ----
    const bool more = seg.rest > 0;
    if (more) load_q(nseg.z, nseg.b);
    l += shfl_xor_f(l, 32);  // both lane halves share m
    constexpr int XP = D + 4;
    constexpr int XW = STAGE / 2;  // floats in a wave's staging area
    static_assert(32 * XP + 64 <= XW, "a wave's state fits its staging area");
    auto xw = [&](int w) { return reinterpret_cast<float*>(s_stage) + (size_t)w * XW; };
    {
      float* dst = xw(wave) + (size_t)lr * XP;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int jq = 0; jq < 4; ++jq)
          *reinterpret_cast<float4*>(dst + 32 * dt + 8 * jq + 4 * g) =
              make_float4(acc[dt][4 * jq], acc[dt][4 * jq + 1], acc[dt][4 * jq + 2],
                          acc[dt][4 * jq + 3]);
      if (g == 0) *reinterpret_cast<float2*>(xw(wave) + 32 * XP + 2 * lr) = make_float2(m, l);
    }
    __syncthreads();
    constexpr int TPR = 2 * W;    // threads per row
    constexpr int DPT = D / TPR;  // dims per thread
    static_assert(DPT % 4 == 0, "float4 steps");
    const int mrow = threadIdx.x / TPR;
    const int md0 = (threadIdx.x % TPR) * DPT;
    const int rr = rt * 32 + mrow;
    float mw[W], mm = kNegInf;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      mw[w] = xw(w)[32 * XP + 2 * mrow];
      mm = __builtin_fmaxf(mm, mw[w]);
    }
    const float ms = safe_max(mm);
    float ll = 0.f, o[DPT];
#pragma unroll
    for (int j = 0; j < DPT; ++j) o[j] = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const float wt = fast_exp2(mw[w] - ms);  // 0 for a wave without tiles
      ll += wt * xw(w)[32 * XP + 2 * mrow + 1];
      const float* src = xw(w) + (size_t)mrow * XP + md0;
#pragma unroll
      for (int j = 0; j < DPT; j += 4) {
        const float4 v4 = *reinterpret_cast<const float4*>(src + j);
        o[j] += wt * v4.x;
        o[j + 1] += wt * v4.y;
        o[j + 2] += wt * v4.z;
        o[j + 3] += wt * v4.w;
      }
    }
    if (rr < P.rows) {
      if (t0 == 0 && seg.tend == flat_tiles(P, seg.len)) {  // the whole unit
        const int rrn = div_by(rr, P.group, P.group_mul);
        const size_t orow = ((size_t)seg.b * P.nodes + rrn) * P.hq + kvh * P.group +
                            (rr - rrn * P.group);
        const float inv = 1.f / ll;  // every row sees its own node: ll > 0
        float* dst = P.out + orow * D + md0;
#pragma unroll
        for (int j = 0; j < DPT; j += 4)
          *reinterpret_cast<float4*>(dst + j) =
              make_float4(o[j] * inv, o[j + 1] * inv, o[j + 2] * inv, o[j + 3] * inv);
      } else {
        const size_t slot = ((size_t)2 * rid + (seg.ord > 0)) * 32 + mrow;
        float* dst = P.part_acc + slot * D + md0;
#pragma unroll
        for (int j = 0; j < DPT; j += 4)
          *reinterpret_cast<float4*>(dst + j) = make_float4(o[j], o[j + 1], o[j + 2], o[j + 3]);
        if (md0 == 0) *reinterpret_cast<float2*>(P.part_ml + 2 * slot) = make_float2(mm, ll);
      }
    }
    if (!more) return;
    publish_q();
    seg = nseg;
    ids = ids_seg;
    if (seg.rest > 0) flat_next(P, lane, lens, nseg);
    ids_next = load_ids(seg.b, wave + W * TPC);
    ids_seg = load_ids(nseg.b, wave);
    __syncthreads();
  }
}

// Combines tree_flat_kernel's partials at range boundary r, 256 threads on it.
// The unit that range r starts inside is merged at the first boundary that cuts it, over
// range r - 1 and the ranges from r on that start inside it too; every other
// unit lies inside one range and was written by the attention kernel.  Range
// r - 1 holds the unit as its first segment (slot 2(r - 1)) or, when the
// unit begins inside it, its last (slot 2(r - 1) + 1); the others as their
// first.
template <int D>
__device__ __forceinline__ void merge_flat_range(const TreeParams& P, int r) {
  constexpr int NF = D / 32;  // float4s per thread: 8 threads per row
  constexpr int U = 4;        // parts loaded together
  const int lane = threadIdx.x & 63;
  const int2* rec = flat_records(P);
  const int2 m1 = rec[r], m0 = rec[r - 1];
  const int mv = rec[min(r + 1 + lane, P.parts - 1)].x;
  const int unit = m1.x;
  if (m1.y == 0) return;                       // r starts on a unit's first tile
  if (m0.x == unit && m0.y > 0) return;        // an earlier boundary cuts the unit too
  // The ranges after r that start inside the unit follow r: count them.
  int nparts = 2;
  for (int base = r + 1;; base += 64) {
    const int rr = base + lane;
    const int x = base == r + 1 ? mv : rec[min(rr, P.parts - 1)].x;
    const unsigned long long hit = __builtin_amdgcn_ballot_w64(rr < P.parts && x == unit);
    const int n = ~hit ? __builtin_ffsll((long long)~hit) - 1 : 64;
    nparts += n;
    if (n < 64 || base + 64 >= P.parts) break;
  }
  const int row = threadIdx.x % 256 >> 3, d0 = 4 * (threadIdx.x & 7);
  const int z = unit / P.batch, b = unit - z * P.batch;
  const int kvh = div_by(z, P.row_tiles, P.rt_mul);
  const int rr = (z - kvh * P.row_tiles) * 32 + row;
  if (rr >= P.rows) return;
  const int first = 2 * (r - 1) + (m0.x != unit);
  auto slot_of = [&](int p) { return p == 0 ? first : 2 * (r - 1 + p); };
  float mm = kNegInf, lsum = 0.f;
  float4 a[NF];
#pragma unroll
  for (int j = 0; j < NF; ++j) a[j] = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int p0 = 0; p0 < nparts; p0 += U) {
    float2 ml[U];
    float4 v[U][NF];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const size_t at = (size_t)slot_of(min(p0 + u, nparts - 1)) * 32 + row;
      ml[u] = *reinterpret_cast<const float2*>(P.part_ml + 2 * at);
#pragma unroll
      for (int j = 0; j < NF; ++j)
        v[u][j] = *reinterpret_cast<const float4*>(P.part_acc + at * D + 32 * j + d0);
    }
    float mn = mm;
#pragma unroll
    for (int u = 0; u < U; ++u)
      mn = __builtin_fmaxf(mn, p0 + u < nparts ? ml[u].x : kNegInf);
    const float ms = safe_max(mn);
    const float a1 = fast_exp2(mm - ms);
    lsum *= a1;
#pragma unroll
    for (int j = 0; j < NF; ++j) {
      a[j].x *= a1;
      a[j].y *= a1;
      a[j].z *= a1;
      a[j].w *= a1;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float w = p0 + u < nparts ? fast_exp2(ml[u].x - ms) : 0.f;
      lsum += w * ml[u].y;
#pragma unroll
      for (int j = 0; j < NF; ++j) {
        a[j].x += w * v[u][j].x;
        a[j].y += w * v[u][j].y;
        a[j].z += w * v[u][j].z;
        a[j].w += w * v[u][j].w;
      }
    }
    mm = mn;
  }
  const float inv = 1.f / lsum;  // every row sees its own node
  const int rrn = div_by(rr, P.group, P.group_mul);
  float* dst = P.out +
               (((size_t)b * P.nodes + rrn) * P.hq + kvh * P.group + (rr - rrn * P.group)) * D + d0;
#pragma unroll
  for (int j = 0; j < NF; ++j)
    *reinterpret_cast<float4*>(dst + 32 * j) =
        make_float4(a[j].x * inv, a[j].y * inv, a[j].z * inv, a[j].w * inv);
}

// Behind a launch that cut a batch's units by its lengths, or found that whole
// units serve it better (RT: row tiles a workgroup of tree_wide_kernel, 0:
// tree_flat_kernel): combines the partials, or verifies the whole units as
// tree_split_kernel does in a single pass.  One launch for both, as an empty one
// costs 1.5 us; its grid has a workgroup per CU at least.
template <int D, int RQ, int RT>
__global__ __launch_bounds__(512, 2) void tree_whole_kernel(TreeParams P) {
  pin_params(P);
  if constexpr (RT > 0) {
    // Eight rows a wave, or four where the units are few and so in many shares
    // each (22 x 1934 x 9 nodes, 16/2 heads, D = 128: 31.8 -> 29.0 us).  The
    // first record is loaded with the word that says whether there are any.
    const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 8 + (threadIdx.x >> 6));
    const int waves = P.cus * 8;  // of a workgroup per CU
    const bool few = P.batch * P.hkv * ((P.row_tiles + RT - 1) / RT) * (RT * 8) <= waves;
    const int taken = *wide_taken<RT>(P);
    int2 rec = few ? merge_wide_record<RT, 4>(P, wave) : merge_wide_record<RT, 8>(P, wave);
    asm volatile("" : "+v"(rec.x), "+v"(rec.y));
    if (!taken) tree_split_body<D, 8, RQ, true>(P);
    else if (wave >= waves) return;
    else if (few) merge_wide<D, RT, 4, 8>(P, wave, waves, rec);
    else merge_wide<D, RT, 8, 4>(P, wave, waves, rec);
  } else if (!*flat_taken(P)) {
    tree_split_body<D, 8, RQ, true>(P);
  } else {
    const int r = 1 + blockIdx.x * 2 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    if (r < P.parts) merge_flat_range<D>(P, r);  // a workgroup per CU and so per range
  }
}

// Row-sharing variant, for tensors that are not 16-byte aligned, of trees of
// four or more row tiles per (request, KV head), where tree_kernel would read
// the prefix once per row tile: the four
// waves take four row tiles and walk the same 32-token tiles, which the
// workgroup loads once (two 16-byte chunks of K and of V per thread) into a
// double-buffered LDS tile, one barrier per tile.  Each wave reads K back in
// the A-operand layout and V through transpose reads, and owns its rows to
// the end: no merge between waves.  Masks, softmax and the P.V product are
// those of tree_kernel.
template <int D>
__global__ __launch_bounds__(kThreads, 2) void tree_rows_kernel(TreeParams P) {
  // No pin_params here: this kernel's loop runs tens to hundreds of us, and
  // holding every argument in registers from the start measured 0.4-2%
  // slower on it (8 x 2048 x 256 nodes: 161.9 -> 164.0 us; 32 x 512 x 64:
  // 48.3 -> 49.3 us) against about 0.5 us saved at the start.
  constexpr int KS = D / 16;
  constexpr int DT = D / 32;
  constexpr int VP = v_pitch<D>();
  constexpr int KP = D + 8;            // halves per staged K row
  constexpr int CPR = D / 8;           // 16-byte chunks per token row
  constexpr int CPT = kTile * CPR / kThreads;  // chunks per thread, K and V each
  static_assert(CPT * kThreads == kTile * CPR, "tile chunks split evenly");
  constexpr int BUF = kTile * (KP + VP);       // halves per staged tile

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 5;
  const int lr = lane & 31;

  const int rgroups = (P.row_tiles + kWaves - 1) / kWaves;
  const int zdim = P.hkv * rgroups;
  const int z = blockIdx.x % zdim;
  const int b = blockIdx.x / zdim;
  const int kvh = z / rgroups;
  const int rt = (z % rgroups) * kWaves + wave;  // row tile; idle when >= row_tiles

  const int len = max(0, min(P.lengths[b], P.max_pages * BC_PAGE_SIZE));
  const int ntile_p = (len + kTile - 1) / kTile;
  const int ntile = ntile_p + (P.nodes + kTile - 1) / kTile;

  const int r = rt * 32 + lr;
  const bool rvalid = rt < P.row_tiles && r < P.rows;
  const int node = rvalid ? r / P.group : 0;
  const int h = kvh * P.group + (rvalid ? r % P.group : 0);

  __shared__ int s_parent[BC_MAX_TREE_NODES];
  __shared__ __attribute__((aligned(16))) _Float16 s_kv[2 * BUF];
  __shared__ bool s_pok[2][2];

  // Q^T B operand of this wave's row tile; parent entries (one per thread).
  uint4 qB[KS];
  {
    const uint16_t* qp = P.dq + (((size_t)b * P.nodes + node) * P.hq + h) * D + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) qB[s] = rvalid ? load8<false>(qp + 16 * s) : make_uint4(0, 0, 0, 0);
  }
  static_assert(BC_MAX_TREE_NODES <= kThreads, "one parent entry per thread");
  const bool has_parent = (int)threadIdx.x < P.nodes;
  const int par = P.parent[(size_t)b * P.nodes + min((int)threadIdx.x, P.nodes - 1)];

  const size_t tok_stride = (size_t)P.hkv * D;
  // Tile i's chunk c of this thread: token row c / CPR, dims 8 * (c % CPR).
  // Every address stays inside its tensor: rows of invalid pages read page
  // 0, draft rows past the node count read the last node; their V is staged
  // as zeros and their scores are masked.
  uint4 kreg[2][CPT], vreg[2][CPT];
  bool vok[2][CPT];
  int ph[2][2] = {{-1, -1}, {-1, -1}};
  auto page_ids = [&](int i, int (&pg)[2]) {
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int pi = i * (kTile / BC_PAGE_SIZE) + q;
      pg[q] = i < ntile_p && pi < P.max_pages ? P.pages[(size_t)b * P.max_pages + pi] : -1;
    }
  };
  auto load_tile = [&](int i, int set) {
    const int (&pg)[2] = ph[set];
    const bool is_draft = i >= ntile_p;
    const int tbase = (is_draft ? i - ntile_p : i) * kTile;
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      const int chunk = (int)threadIdx.x + kThreads * c;
      const int row = chunk / CPR, col = 8 * (chunk % CPR);
      size_t off;
      bool ok;
      if (!is_draft) {
        const int pgq = pg[row / BC_PAGE_SIZE];
        const bool pok = pgq >= 0 && pgq < P.phys_pages;
        const int t = tbase + row;
        ok = pok && t < len;
        off = (pok ? ((size_t)pgq * BC_PAGE_SIZE + row % BC_PAGE_SIZE) * tok_stride : 0) +
              (size_t)kvh * D + col;
        kreg[set][c] = load8<false>(P.k + off);
        vreg[set][c] = load8<false>(P.v + off);
      } else {
        const int dn = tbase + row;
        ok = dn < P.nodes;
        off = (((size_t)b * P.nodes + min(dn, P.nodes - 1)) * P.hkv + kvh) * D + col;
        kreg[set][c] = load8<false>(P.dk + off);
        vreg[set][c] = load8<false>(P.dv + off);
      }
      vok[set][c] = ok;
    }
  };
  auto store_tile = [&](int i, int set) {
    const int buf = i & 1;
    const int (&pg)[2] = ph[set];
    _Float16* sk = s_kv + buf * BUF;
    _Float16* sv = sk + kTile * KP;
#pragma unroll
    for (int c = 0; c < CPT; ++c) {
      const int chunk = (int)threadIdx.x + kThreads * c;
      const int row = chunk / CPR, col = 8 * (chunk % CPR);
      *reinterpret_cast<uint4*>(sk + row * KP + col) = kreg[set][c];
      *reinterpret_cast<uint4*>(sv + row * VP + col) =
          vok[set][c] ? vreg[set][c] : make_uint4(0, 0, 0, 0);
    }
    if (threadIdx.x < 2) {
      const int pgq = pg[threadIdx.x];
      s_pok[buf][threadIdx.x] = i >= ntile_p || (pgq >= 0 && pgq < P.phys_pages);
    }
  };

  f32x16 acc[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int j = 0; j < 16; ++j) acc[dt][j] = 0.f;
  float m = kNegInf, l = 0.f;
  // Transpose-read address of this lane in a staged V tile.
  const int trG = lane >> 4, trj = lane & 15;
  const int vtr_off = (4 * (trG >> 1) + (trj >> 2)) * VP + 16 * (trG & 1) + 4 * (trj & 3);

  auto compute = [&](int i, int buf) {
    const _Float16* sk = s_kv + buf * BUF;
    const _Float16* sv = sk + kTile * KP;
    const bool is_draft = i >= ntile_p;
    const int tbase = (is_draft ? i - ntile_p : i) * kTile;
    uint32_t okbits;
    if (!is_draft) {
      const int hi = min(max(len - tbase, 0), kTile);
      okbits = (hi >= kTile ? ~0u : (1u << hi) - 1u) &
               ((s_pok[buf][0] ? 0x0000ffffu : 0u) | (s_pok[buf][1] ? 0xffff0000u : 0u));
    } else {
      okbits = 0;
      int cur = node;
      for (int steps = 0; steps < P.nodes && cur >= 0 && cur < P.nodes; ++steps) {
        if (cur >= tbase && cur < tbase + kTile) okbits |= 1u << (cur - tbase);
        cur = s_parent[cur];
      }
    }
    // ---- S^T = K Q^T, K from the staged tile in the A-operand layout ----
    f32x16 sc;
#pragma unroll
    for (int j = 0; j < 16; ++j) sc[j] = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint4 ka = *reinterpret_cast<const uint4*>(sk + lr * KP + 16 * s + 8 * g);
      sc = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_f16x8(ka), as_f16x8(qB[s]), sc, 0, 0, 0);
    }
    // ---- mask and online softmax (column lr = query row) ----
    // Scores stay unscaled: the scale enters the running max once and the
    // exp2 argument as an FMA; fully valid tiles skip the mask.
    float svv[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) svv[j] = sc[j];
    if (__builtin_amdgcn_ballot_w64(okbits != ~0u)) {
      const uint32_t ob = okbits >> (4 * g);
#pragma unroll
      for (int j = 0; j < 16; ++j)
        svv[j] = (ob >> (8 * (j >> 2) + (j & 3))) & 1u ? svv[j] : kNegInf;
    }
    float tmax = kNegInf;
#pragma unroll
    for (int j = 0; j < 16; ++j) tmax = __builtin_fmaxf(tmax, svv[j]);
    tmax = __builtin_fmaxf(tmax, shfl_xor_f(tmax, 32)) * P.scale_log2;
    const float mnew = __builtin_fmaxf(m, tmax);
    if (__builtin_amdgcn_ballot_w64(mnew > m + kRescaleSlack)) {
      const float alpha = fast_exp2(m - safe_max(mnew));
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int j = 0; j < 16; ++j) acc[dt][j] *= alpha;
      m = mnew;
    }
    const float mb = safe_max(m);
    f16x8 pb[2], pl[2];
    float pr[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      pr[j] = fast_exp2(__builtin_fmaf(svv[j], P.scale_log2, -mb));
      l += pr[j];
    }
#pragma unroll
    for (int hh = 0; hh < 2; ++hh) {
      uint32_t wh[4], wl[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        split_hi_lo(pr[8 * hh + 2 * q], pr[8 * hh + 2 * q + 1], wh[q], wl[q]);
      pb[hh] = __builtin_bit_cast(f16x8, u32x4{wh[0], wh[1], wh[2], wh[3]});
      pl[hh] = __builtin_bit_cast(f16x8, u32x4{wl[0], wl[1], wl[2], wl[3]});
    }
    // ---- O^T += V^T P^T from the staged tile ----
    const _Float16* vtr = sv + vtr_off;
    f16x8 av[DT][2];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const f16x4 lo = lds_read_tr(vtr + (16 * st) * VP + 32 * dt);
        const f16x4 hi = lds_read_tr(vtr + (16 * st + 8) * VP + 32 * dt);
        av[dt][st] = f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[dt][st], pb[st], acc[dt], 0, 0, 0);
#pragma unroll
    for (int st = 0; st < 2; ++st)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av[dt][st], pl[st], acc[dt], 0, 0, 0);
  };

  // Loads run two tiles ahead in two register sets (set = tile & 1); LDS
  // holds two staged tiles (buffer = tile & 1).  Tiles 0 and 1 are loaded
  // and tile 0 staged before the first barrier, together with the parent
  // array.  Step i loads tile i + 2, computes tile i and stages tile i + 1,
  // then the barrier publishes tile i + 1 and frees tile i's buffer.
  if (ntile > 0) {
    page_ids(0, ph[0]);
    load_tile(0, 0);
  }
  if (ntile > 1) {
    page_ids(1, ph[1]);
    load_tile(1, 1);
  }
  if (ntile > 0) store_tile(0, 0);
  if (has_parent) s_parent[threadIdx.x] = par;
  __syncthreads();
  auto step = [&](int i, int set) {  // set = i & 1, a compile-time constant
    if (i >= ntile) return;
    if (i + 2 < ntile) {
      page_ids(i + 2, ph[set]);
      load_tile(i + 2, set);
    }
    if (rt < P.row_tiles) compute(i, set);
    if (i + 1 < ntile) store_tile(i + 1, set ^ 1);
    __syncthreads();
  };
  for (int i = 0; i < ntile; i += 2) {
    step(i, 0);
    step(i + 1, 1);
  }
  if (!rvalid) return;
  l += shfl_xor_f(l, 32);

  // ---- write: lane holds O^T[32dt + 8jq + 4g + e][row r] ----
  float* dst = P.out + (((size_t)b * P.nodes + node) * P.hq + h) * D;
  const float inv = 1.f / l;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int jq = 0; jq < 4; ++jq)
      store4f<false>(dst + 32 * dt + 8 * jq + 4 * g, acc[dt][4 * jq] * inv,
                   acc[dt][4 * jq + 1] * inv, acc[dt][4 * jq + 2] * inv,
                   acc[dt][4 * jq + 3] * inv);
}

// The reference's rules (src/tree_attention.cu:94-99): physical_pages is not
// among them, and a value below 1 means the pool size is not given.
bool tree_shape_ok(const bc_shape& s, int nodes) {
  return s.batch >= 1 && s.query_heads >= 1 && s.kv_heads >= 1 &&
         s.query_heads % s.kv_heads == 0 && (s.dim == 64 || s.dim == 128) &&
         s.max_pages >= 1 && nodes >= 1 && nodes <= BC_MAX_TREE_NODES;
}

bool tree_args_ok(const bc_shape& s, const bc_tree_inputs& in, int nodes) {
  return tree_shape_ok(s, nodes) && in.prefix.k && in.prefix.v && in.prefix.pages &&
         in.prefix.lengths && in.draft_q && in.draft_k && in.draft_v && in.parent && in.output;
}

// With the pool size given, ids outside [0, physical_pages) are masked and
// every padding load may read page 0.  Without it (physical_pages < 1, as an
// empty pool gives), the page-table entries inside a length are trusted as in
// the reference, and only tree_kernel runs: it reads pages for tokens inside
// the length only and points every other row at the draft tensors.
bool pool_known(const bc_shape& s) { return s.physical_pages >= 1; }

bool aligned16(const void* p) {
  return (reinterpret_cast<uintptr_t>(p) & 15) == 0;
}

TreeParams make_params(const bc_shape& s, const bc_tree_inputs& in, int nodes) {
  TreeParams P{};
  P.k = in.prefix.k;
  P.v = in.prefix.v;
  P.pages = in.prefix.pages;
  P.lengths = in.prefix.lengths;
  P.dq = in.draft_q;
  P.dk = in.draft_k;
  P.dv = in.draft_v;
  P.parent = in.parent;
  P.out = in.output;
  P.batch = s.batch;
  P.nodes = nodes;
  P.hq = s.query_heads;
  P.hkv = s.kv_heads;
  P.group = s.query_heads / s.kv_heads;
  P.max_pages = s.max_pages;
  // physical_pages is not part of the reference tree contract
  // (bindings/torch_ops.cpp:54 passes prefix_k.size(0)); below 1 the ids
  // are not range-checked (tree_kernel only, see pool_known).
  P.phys_pages = pool_known(s) ? s.physical_pages : 0x7fffffff;
  P.cus = bch::device_cus();
  P.rows = nodes * P.group;
  P.row_tiles = (P.rows + 31) / 32;
  P.scale_log2 = (float)(1.4426950408889634 / __builtin_sqrt((double)s.dim));
  // Multiply-high division needs n * d < 2^32 for every n it divides: row
  // indices stay below 32 * row_tiles, (KV head, row tile) indices below
  // hkv * row_tiles.
  const unsigned long long lim = 1ull << 32;
  if ((unsigned long long)P.row_tiles * 32 * P.group < lim)
    P.group_mul = (lim + P.group - 1) / P.group;
  if ((unsigned long long)P.hkv * P.row_tiles * P.row_tiles < lim)
    P.rt_mul = (lim + P.row_tiles - 1) / P.row_tiles;
  return P;
}

// Tensors that are not 16-byte aligned, and calls without the pool size:
// element-wise loads and stores.  tree_rows_kernel (one K/V tile shared by
// four row tiles) pays once its row groups fill the CUs.
hipError_t launch_tree(const TreeParams& P, int dim, bool known_pool, hipStream_t st) {
  const size_t groups = (size_t)P.batch * P.hkv * ((P.row_tiles + kWaves - 1) / kWaves);
  if (known_pool && P.row_tiles >= kWaves && groups >= (size_t)bch::device_cus()) {
    if (dim == 64) tree_rows_kernel<64><<<dim3((unsigned)groups), kThreads, 0, st>>>(P);
    else tree_rows_kernel<128><<<dim3((unsigned)groups), kThreads, 0, st>>>(P);
  } else {
    const dim3 grid((unsigned)((size_t)P.batch * P.hkv * P.row_tiles));
    if (dim == 64) tree_kernel<64, false><<<grid, kThreads, 0, st>>>(P);
    else tree_kernel<128, false><<<grid, kThreads, 0, st>>>(P);
  }
  return hipGetLastError();
}

bool tree_ptrs_aligned(const bc_tree_inputs& in) {
  return aligned16(in.prefix.k) && aligned16(in.prefix.v) &&
         aligned16(in.draft_q) && aligned16(in.draft_k) &&
         aligned16(in.draft_v) && aligned16(in.output);
}

// ---- aligned tensors: plan, workspace and launch ----

struct SplitPlan {
  int parts;  // workgroups per (request group, KV head, row tile), <= 64
  int tiles;  // 32-token tiles per workgroup and request (draft then prefix tiles)
  int waves;  // waves per workgroup: 4 or 8
  int rq = 1;  // requests per workgroup (waves / rq per request)
  int wide = 0;  // row tiles per workgroup of tree_wide_kernel (0: tree_split_kernel)
};

// Units (request, KV head, group of `rt` row tiles) of a launch.
long long row_groups(const bc_shape& s, int row_tiles, int rt) {
  return (long long)s.batch * s.kv_heads * ((row_tiles + rt - 1) / rt);
}

// tree_wide_kernel reads a K/V tile once for four row tiles (or two), where
// tree_split_kernel reads it per row tile, so it takes the trees of several
// row tiles whose groups fill the CUs (same box, 32/8 heads and D = 128 unless
// noted, tree_split_kernel or the kernel it replaced first):
//  - tables of 60 tiles and more, at most one group per CU, and room for at
//    least 17 steps per CU in all (D = 64, whose steps are half as long: 24), or
//    from 5 (D = 64: 12) where tables and pool have room for more than 32 MB,
//    which the eight L2s do not hold: two workgroups per CU split the groups by
//    the batch's lengths, four row tiles each (two, if there are no more), if
//    the lengths fill what the table has room for (wide_pays), else
//    tree_whole_kernel runs a single pass of whole units.  Below these lines no
//    lengths make the shares pay, and the second launch (2 us) is saved.  At
//    lengths that fill the table: 8 x 128-4096 tokens x 128 nodes 185 against
//    105 us, 14 x 2319 x 32 88 against 47, 9 x 450-3600 x 32 (32/4) 73 against
//    41, 32 x 256-2048 x 16 58 against 42, 16 x 300-3000 x 33 (28/4, D = 64) 45
//    against 31, 8 x 2048 x 128 108 against 80; near the lines 22 x 1934 x 9
//    (16/2) 29.5 against 29.3, 6 x 1079-2158 x 12 (24/8) 21.5 against 19.9.
//    Short lengths under a table of 4096: 8 x 100-300 x 33 15.7 against 17.8 (21
//    in shares), 16 x 64-512 x 16 14.6 against 17.1 (20.6);
//  - else four row tiles a workgroup from 7/8 CUs of groups on: 8 requests x
//    2048 tokens x 256 nodes 143 against 116 us, 16 x 1000 x 64 nodes 57
//    against 40, 64 x 30-500 x 64 nodes 73 against 64;
//  - else two a workgroup from two groups per CU on: 64 x 1024 x 9 nodes 50
//    against 35 us; and from one group per CU on where the prefixes are not
//    short (30 tiles): 16/16 heads, D = 64: 16 x 1000 x 33 nodes 25 against
//    20 us, while 28/4 heads, D = 64, 64 x 30-500 x 9 nodes would take 13.2
//    against 11.2.
// Without scratch memory (`scratch` false) there is no split.
SplitPlan wide_plan(const bc_shape& s, int row_tiles, int max_tiles, int cus, bool scratch) {
  SplitPlan p{0, 0, 4};
  if (row_tiles < 2) return p;
  const int rt = row_tiles > 2 ? 4 : 2;
  const long long g = row_groups(s, row_tiles, rt);
  const long long page = 2LL * BC_PAGE_SIZE * s.kv_heads * s.dim * sizeof(uint16_t);
  // The prefixes' bytes, as far as the shape tells, against eight L2s of 4 MB.
  const bool far =
      std::min((long long)s.batch * s.max_pages, (long long)s.physical_pages) * page > 32000000;
  const long long least = s.dim == 64 ? (far ? 24LL : 48LL) : (far ? 10LL : 34LL);
  if (scratch && max_tiles >= 60 && s.batch <= kWideRequests && g <= cus &&
      g * max_tiles >= least * cus) {
    p.parts = 2 * cus;
    p.wide = rt;
    return p;
  }
  p.parts = 1;
  p.wide = 4;
  if (rt == 4 && 8 * g >= 7LL * cus) return p;
  const long long u = row_groups(s, row_tiles, 2);
  p.wide = 2;
  if (u >= 2LL * cus || (max_tiles >= 30 && u >= cus)) return p;
  p.wide = 0;
  return p;
}

// A single pass of more (request, KV head, row tile) units than CUs runs
// its eight-wave workgroups (one per CU) in rounds.  Two requests per
// workgroup, four waves each on the same tiles, halve the workgroups and
// double each wave's tiles, so they pay where they at least halve the
// rounds; requests that share pages then also share them in the CU's L1.
// Measured against one request per workgroup (32 / 8 heads, D = 128, 7
// nodes, shared prefix): 33 x 2048 tokens 48.9 -> 45.3 us, 40 x 1024 31.6
// -> 28.2, 64 x 1024 32.4 -> 30.1, 128 x 512 46.3 -> 39.2; 96 x 512 (three
// rounds against two) 35.5 -> 37.9 and 32 x 2048 (one round) 27.9 -> 45.7,
// so neither of those pairs.
SplitPlan pair_requests(int batch, long long units, SplitPlan p, int cus) {
  if (p.parts != 1 || p.waves != 8 || batch < 2) return p;
  const long long per_request = units / batch;  // KV heads x row tiles
  const long long rounds1 = (units + cus - 1) / cus;
  const long long rounds2 = ((batch + 1) / 2 * per_request + cus - 1) / cus;
  if (2 * rounds2 <= rounds1) p.rq = 2;
  return p;
}

// Sets the rounds of a single pass and returns its requests per workgroup.
int whole_requests(TreeParams& P) {
  const long long units = (long long)P.batch * P.hkv * P.row_tiles;
  const int rq = pair_requests(P.batch, units, SplitPlan{1, 0, 8}, P.cus).rq;
  const long long wgs = (long long)((P.batch + rq - 1) / rq) * P.hkv * P.row_tiles;
  P.whole_rounds = rq * (int)((wgs + P.cus - 1) / P.cus);
  return rq;
}

// Parts per unit and tiles per part for `cus` compute units, sized from the
// page table's capacity (lengths stay on the device).  A CU holds one
// eight-wave or two four-wave workgroups (LDS), so both shapes offer eight
// wave slots per CU: eight-wave workgroups take about cus/units parts, four-
// wave ones about 2*cus/units.  The plan with more waves that have a tile
// wins (12 requests x 2048 tokens, 96 units: four waves x 5 parts 20.2 us
// against eight waves x 2 parts 20.8 and four waves x 2 parts 24.5); at about
// equal counts, the one spread over more CUs (one request x 2048 tokens:
// four waves x 17 parts, 10.4 against 11.8 us), else eight waves, which
// merge more tiles in LDS (8 and 16 requests), or run single-pass (24 and 32
// requests: one part, 28.6 against 31.7 us with two); see pair_requests for
// single passes of more units than CUs.
SplitPlan split_plan(const bc_shape& s, int nodes, int cus) {
  const int group = s.query_heads / s.kv_heads;
  const int row_tiles = (nodes * group + 31) / 32;
  const long long units = (long long)s.batch * s.kv_heads * row_tiles;
  const int max_tiles =
      (s.max_pages * BC_PAGE_SIZE + kTile - 1) / kTile + (nodes + kTile - 1) / kTile;
  auto plan_for = [&](int waves, long long want) {
    if (want > 64) want = 64;
    SplitPlan p{1, max_tiles, waves};
    if (want < 2) return p;
    int tiles = (int)((max_tiles + want - 1) / want);
    if (tiles < waves) tiles = waves;
    const int parts = (max_tiles + tiles - 1) / tiles;
    return parts < 2 ? p : SplitPlan{parts, tiles, waves};
  };
  const long long u = units > 0 ? units : 1;
  const SplitPlan wide = wide_plan(s, row_tiles, max_tiles, cus, true);
  if (wide.wide) return wide;
  // A single pass whose eight waves take two tiles or fewer each beats a
  // split, which adds the merge launch (one request over 256 tokens: 8.2
  // against 9.6 us, over 384: 8.4 against 9.3 us; 2 x 256: 8.5 against
  // 9.6 us; 16 x 256: 10.3 against 13.2 us).  Up to five tiles per wave it
  // still wins once its units fill (tiles per wave - 1) eighths of the CUs
  // (12 x 512 tokens: 9.5 against 12.1 us; 16 x 512: 9.4 against 12.1 us;
  // 12 x 768: 11.2 against 13.7 us; 8 x 1024 with 16 nodes: 13.3 against
  // 15.0 us); below that the split wins (one request over 512 tokens: 9.1
  // against 9.7 us).
  const int rounds = (max_tiles + 7) / 8;  // tiles per wave in a single pass
  if (max_tiles <= 2 * 8 || (rounds <= 5 && 8 * u >= (long long)cus * (rounds - 1)))
    return pair_requests(s.batch, u, SplitPlan{1, max_tiles, 8}, cus);
  const SplitPlan eight = plan_for(8, cus / u);
  const SplitPlan four = plan_for(4, 2LL * cus / u);
  // Waves with at least one tile, and CUs with a workgroup.
  auto busy = [&](const SplitPlan& p) {
    return u * std::min<long long>((long long)p.parts * p.waves, max_tiles);
  };
  auto spread = [&](const SplitPlan& p) { return std::min<long long>(u * p.parts, cus); };
  const long long b8 = busy(eight), b4 = busy(four);
  if (10 * b4 > 11 * b8) return four;
  if (eight.parts > 1 && 10 * b4 >= 9 * b8 && spread(four) > spread(eight)) return four;
  return pair_requests(s.batch, u, eight, cus);
}

// Workspace of a split plan: P.parts (acc; max, sum) slots per output row.
size_t split_workspace(const bc_shape& s, int nodes, const SplitPlan& plan, size_t* acc_bytes) {
  if (plan.parts < 2) return 0;
  const size_t slots = plan.wide ? (size_t)plan.parts * plan.wide * 32
                                 : (size_t)s.batch * nodes * s.query_heads * plan.parts;
  *acc_bytes = (slots * s.dim * sizeof(float) + 255) & ~(size_t)255;
  return *acc_bytes + slots * 2 * sizeof(float) + (plan.wide ? s.batch * sizeof(int2) + sizeof(int) : 0);
}

template <int D>
void launch_split_kernel(const TreeParams& P, const SplitPlan& plan, dim3 grid,
                         hipStream_t st) {
  if (plan.waves == 4)
    tree_split_kernel<D, 4, 1><<<grid, 256, 0, st>>>(P);
  else if (plan.rq == 2)
    tree_split_kernel<D, 8, 2><<<grid, 512, 0, st>>>(P);
  else
    tree_split_kernel<D, 8, 1><<<grid, 512, 0, st>>>(P);
}

// tree_whole_kernel, `rq` requests a workgroup where it runs whole units.
template <int D, int RT>
void launch_whole_kernel(const TreeParams& P, int rq, hipStream_t st) {
  const size_t units = (size_t)((P.batch + rq - 1) / rq) * P.hkv * P.row_tiles;
  const dim3 grid((unsigned)std::max<size_t>(units, P.cus));
  if (rq == 2) tree_whole_kernel<D, 2, RT><<<grid, 512, 0, st>>>(P);
  else tree_whole_kernel<D, 1, RT><<<grid, 512, 0, st>>>(P);
}

template <int D, int RT>
void launch_wide_kernel(TreeParams& P, hipStream_t st) {
  const size_t groups = (size_t)P.batch * P.hkv * ((P.row_tiles + RT - 1) / RT);
  if (P.parts == 1) {
    tree_wide_kernel<D, RT, false><<<dim3((unsigned)groups), 256, 0, st>>>(P);
    return;
  }
  const int rq = whole_requests(P);
  tree_wide_kernel<D, RT, true><<<dim3((unsigned)P.parts), 256, 0, st>>>(P);
  launch_whole_kernel<D, RT>(P, rq, st);
}

template <int D>
hipError_t launch_wide(TreeParams& P, int row_tiles, hipStream_t st) {
  if (row_tiles == 2) launch_wide_kernel<D, 2>(P, st);
  else launch_wide_kernel<D, 4>(P, st);
  return hipGetLastError();
}

hipError_t launch_split(TreeParams& P, int dim, const SplitPlan& plan, void* workspace,
                        size_t acc_bytes, hipStream_t st) {
  P.parts = plan.parts;
  P.tiles_per_part = plan.tiles;
  if (plan.parts > 1) {
    P.part_acc = static_cast<float*>(workspace);
    P.part_ml = reinterpret_cast<float*>(static_cast<char*>(workspace) + acc_bytes);
  }
  if (plan.wide)
    return dim == 64 ? launch_wide<64>(P, plan.wide, st) : launch_wide<128>(P, plan.wide, st);
  const size_t groups = ((size_t)P.batch + plan.rq - 1) / plan.rq;
  P.grid3d = groups <= 65535;
  const dim3 grid = P.grid3d
      ? dim3((unsigned)(P.hkv * P.row_tiles), (unsigned)groups, (unsigned)plan.parts)
      : dim3((unsigned)((size_t)plan.parts * groups * P.hkv * P.row_tiles));
  if (dim == 64) launch_split_kernel<64>(P, plan, grid, st);
  else launch_split_kernel<128>(P, plan, grid, st);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess || plan.parts < 2) return err;
  const size_t rows = (size_t)P.batch * P.nodes * P.hq;
  const dim3 mgrid((unsigned)((rows + 3) / 4));
  if (dim == 64) launch_merge_split<64>(P, mgrid, st);
  else launch_merge_split<128>(P, mgrid, st);
  return hipGetLastError();
}

// ---- tree_flat_kernel: ranges, workspace and launch ----

// Ranges of tree_flat_kernel (0: not taken): one eight-wave workgroup per CU
// for batches that may be long enough to stream their prefixes from HBM, by
// what the shape has room for: small trees (one row tile), page tables of at
// least 2048 tokens that could hold 400 MB, and a pool of at least 128 MB (a
// smaller one stays in the 256 MB cache, where equal shares gain nothing).  The
// kernel reads the lengths (flat_pays), and tree_whole_kernel takes what is
// better off whole.  7 nodes, 32/8 heads, D = 128 unless noted,
// tree_split_kernel first: 64 x 128-4096 tokens 130 against 115 us, 20 x
// 256-8192 99 against 84, 64 x 128-4096 at D = 64 73 against 67; under a table
// of 32768 tokens 16 x 128-4096 62 against 47, 4 x 500-8000 x 8 nodes 51
// against 30.  Left whole, the second launch and the lengths ahead of the first
// load cost 2 to 3 us: 64 x 32-1024 39 against 42, 64 x 2048 (one shared prefix)
// 46 against 49, 64 x 16-200 13 against 16 (in ranges 46, 54 and 29).  Below
// the lines ranges lose at any length: 64 x 32-1024 32 against 44, 16 x 128-4096
// 28 against 33.
int flat_ranges(const bc_shape& s, int nodes, int cus) {
  const int group = s.query_heads / s.kv_heads;
  const long long page = 2LL * BC_PAGE_SIZE * s.kv_heads * s.dim * sizeof(uint16_t);
  const long long table = (long long)s.batch * s.max_pages;  // pages
  if ((long long)nodes * group > 32 || s.max_pages * BC_PAGE_SIZE < 2048 ||
      table * page < 400000000LL || s.physical_pages * page < 128000000LL)
    return 0;
  if (table * s.kv_heads >= 1LL << 30) return 0;  // tile indices stay in an int
  return cus;
}

size_t flat_workspace(const bc_shape& s, int ranges, size_t* acc_bytes) {
  const size_t slots = (size_t)2 * ranges * 32;
  *acc_bytes = slots * s.dim * sizeof(float);
  return *acc_bytes + slots * 2 * sizeof(float) + (size_t)ranges * sizeof(int2) + sizeof(int);
}

template <int D>
void launch_flat_kernel(TreeParams& P, hipStream_t st) {
  const int rq = whole_requests(P);
  tree_flat_kernel<D, 8><<<dim3(P.parts), 512, 0, st>>>(P);
  launch_whole_kernel<D, 0>(P, rq, st);
}

hipError_t launch_flat(TreeParams& P, int dim, int ranges, void* workspace, size_t acc_bytes,
                       hipStream_t st) {
  P.parts = ranges;
  P.part_acc = static_cast<float*>(workspace);
  P.part_ml = reinterpret_cast<float*>(static_cast<char*>(workspace) + acc_bytes);
  if (dim == 64) launch_flat_kernel<64>(P, st);
  else launch_flat_kernel<128>(P, st);
  return hipGetLastError();
}

// One call, with the caller's workspace where it serves, else a slot of the
// library's scratch pool, else (under graph capture, or for a plan larger
// than a slot) without one.
int tree_call(bc_shape s, bc_tree_inputs in, int nodes, void* workspace, size_t workspace_bytes,
              bc_stream_t stream) {
  if (!tree_args_ok(s, in, nodes)) return BC_ERROR_INVALID_VALUE;
  TreeParams P = make_params(s, in, nodes);
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (!tree_ptrs_aligned(in) || !pool_known(s)) return launch_tree(P, s.dim, pool_known(s), st);
  const int cus = bch::device_cus();
  const bool ws_ok = workspace && aligned16(workspace);
  size_t acc = 0;
  if (const int flat = flat_ranges(s, nodes, cus)) {
    const size_t need = flat_workspace(s, flat, &acc);
    if (ws_ok && workspace_bytes >= need)
      return launch_flat(P, s.dim, flat, workspace, acc, st);
    const bch::ScratchLease lease(st, need);
    if (lease.get()) return launch_flat(P, s.dim, flat, lease.get(), acc, st);
  }
  SplitPlan plan = split_plan(s, nodes, cus);
  size_t need = split_workspace(s, nodes, plan, &acc);
  if (need == 0) return launch_split(P, s.dim, plan, nullptr, 0, st);
  if (ws_ok && workspace_bytes >= need) return launch_split(P, s.dim, plan, workspace, acc, st);
  // Four row tiles a workgroup at D = 128 with two workgroups per CU need more
  // than a slot holds; with one per CU they fit.
  if (plan.wide == 4 && need > bch::kSlotBytes) {
    plan.parts = cus;
    need = split_workspace(s, nodes, plan, &acc);
  }
  const bch::ScratchLease lease(st, need);
  if (lease.get()) return launch_split(P, s.dim, plan, lease.get(), acc, st);
  // One part per unit, by the rules for whole units: few wide ones would leave
  // most CUs idle.
  const int max_tiles =
      (s.max_pages * BC_PAGE_SIZE + kTile - 1) / kTile + (nodes + kTile - 1) / kTile;
  SplitPlan one = wide_plan(s, P.row_tiles, max_tiles, cus, false);
  if (!one.wide)
    one = pair_requests(P.batch, (long long)P.batch * P.hkv * P.row_tiles,
                        SplitPlan{1, max_tiles, 8}, cus);
  return launch_split(P, s.dim, one, nullptr, 0, st);
}

}  // namespace

extern "C" int bc_tree_verify(bc_shape s, bc_tree_inputs in, int nodes,
                              bc_stream_t stream) {
  return tree_call(s, in, nodes, nullptr, 0, stream);
}

// Calls without the pool size, and plans of one part, need no workspace.
extern "C" size_t bc_tree_verify_workspace_size(bc_shape s, int nodes) {
  if (!tree_shape_ok(s, nodes) || !pool_known(s)) return 0;
  const int cus = bch::device_cus();
  size_t a = 0;
  if (const int flat = flat_ranges(s, nodes, cus)) return flat_workspace(s, flat, &a);
  return split_workspace(s, nodes, split_plan(s, nodes, cus), &a);
}

extern "C" int bc_tree_verify_ws(bc_shape s, bc_tree_inputs in, int nodes,
                                 void* workspace, size_t workspace_bytes,
                                 bc_stream_t stream) {
  return tree_call(s, in, nodes, workspace, workspace_bytes, stream);
}
