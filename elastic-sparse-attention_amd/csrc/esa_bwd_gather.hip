// Gather backward (gfx950): dQ, dK and dV for any index source (explicit
// index lists, the elastic pattern at positions, float32 / bfloat16 /
// float16, any head_dim that is a multiple of 4 up to 256).
//
// Replaces the backward branch of the reference's Triton kernel
// (elastic_sparse_attention.py:168-233) as ElasticSparseAttentionFunction
// .backward launches it (:299-339), without its float atomics:
//
//   bwd_rows_kernel   one wave per (batch, head, query row): delta = dO . O,
//                     then per entry j (lane j): s = q . k_j * scale,
//                     p = exp(s - lse) (valid entries), dp = dO . v_j,
//                     dS = p (m_j dp - delta) with m_j the dropout factor,
//                     dQ = scale * sum_j dS_j k_j; each entry's dV
//                     coefficient m_j p and dK coefficient scale * dS go to
//                     the workspace (0 for an entry that is masked or whose
//                     key lies outside [0, kv_len): the Triton kernel's
//                     atomics skip those, :209-213, :226-228).  A row
//                     with a non-finite delta and an entry it does not
//                     attend gets a NaN dQ, as the Triton kernel's
//                     (0 - delta) * 0 term for that entry gives it.
//   radix sort        of (key, entry id), the key of an entry being kv_head *
//                     kv_len + key for a valid in-range entry, else a sentinel
//                     past every key: a stable LSD radix sort, 8 bits per
//                     pass (per-tile digit histograms, an exclusive scan of
//                     them, then a scatter ranked by wave ballots), so each
//                     key's entries end up contiguous, in entry order.
//   bwd_segments      the start of each (kv head, key) in the sorted order.
//   bwd_kv_kernel     one wave per (batch, kv head, key): dK = sum of
//                     coefficient * q row and dV = sum of coefficient * dO
//                     row over the key's entries, in entry order.
//
// The row and key-major passes have a cooperative-row form each
// (rows_coop_kernel, kv_coop_kernel, below), taken for 16-byte aligned rows;
// the per-lane forms above serve the rest.
//
// Every gradient element is summed by one wave (a long key segment by one wave
// per window, the windows in order) in a fixed order, so two runs agree bit
// for bit.  The index lists do not depend on the batch, so
// the sort serves every batch element.
#include <type_traits>

#include "esa_gather.hpp"

namespace esa {

namespace {

template <Elem E, bool PATTERN>
__global__ __launch_bounds__(256) void bwd_rows_kernel(GatherBwdArgs A) {
  using T = typename ElemT<E>::T;
  __shared__ float qs_all[4][256];
  __shared__ float dos_all[4][256];
  __shared__ float ds_all[4][64];
  __shared__ int ks_all[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = blockIdx.x * 4 + wave;
  const int h = blockIdx.y, b = blockIdx.z;
  if (r >= A.q_len) return;  // whole wave leaves; no block-level barrier below
  const int kvh = h / A.groups;
  const int D = A.D;
  float* qs = qs_all[wave];
  float* dos = dos_all[wave];
  float* dsl = ds_all[wave];
  int* ksl = ks_all[wave];

  const T* qrow = (const T*)A.q + (int64_t)b * A.qsb + (int64_t)h * A.qsh + (int64_t)r * A.qss;
  const T* orow = (const T*)A.o + (int64_t)b * A.osb + (int64_t)h * A.osh + (int64_t)r * A.oss;
  const T* dorow =
      (const T*)A.dout + (int64_t)b * A.dosb + (int64_t)h * A.dosh + (int64_t)r * A.doss;
  float dl = 0.f;
  for (int d = lane; d < D; d += 64) {
    qs[d] = ElemT<E>::load(qrow + d);
    const float g = ElemT<E>::load(dorow + d);
    dos[d] = g;
    dl += g * ElemT<E>::load(orow + d);
  }
  const float delta = wave_sum(dl);  // dO . O (the output the forward stored)
  wave_sync_lds();

  const T* kbase = (const T*)A.k + (int64_t)b * A.ksb + (int64_t)kvh * A.ksh;
  const T* vbase = (const T*)A.v + (int64_t)b * A.vsb + (int64_t)kvh * A.vsh;
  RowEntries row;
  row.init<PATTERN>(A.src, h, r);
  const float lse = A.lse[(int64_t)b * A.lsb + (int64_t)h * A.lsh + r];
  const int w = A.src.w;
  const int64_t e0 = ((int64_t)h * A.q_len + r) * w;  // entry id of (h, r, 0)
  float* cp = A.cp + (int64_t)b * A.E;
  float* cs = A.cs + (int64_t)b * A.E;

  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  bool dead = false;
  for (int c0 = 0; c0 < w; c0 += 64) {
    const int j = c0 + lane;
    bool valid = false;
    int64_t key = 0;
    if (j < w) row.entry<PATTERN>(A.src, h, r, j, valid, key);
    const bool in_range = key >= 0 && key < A.kv_len;
    const bool live = valid && in_range && !row.bad_pos;
    dead |= j < w && !live;
    float dsc = 0.f, pc = 0.f;
    if (live) {
      const float s = row_dot<E>(qs, kbase + key * A.kss, D) * A.sm_scale;
      const float dp = row_dot<E>(dos, vbase + key * A.vss, D);
      const float p = expf(s - lse);
      const float keep = drop_factor(A.drop, b, h, r, j, A.H, A.q_len, w);
      pc = keep * p;
      dsc = p * (keep * dp - delta) * A.sm_scale;
    }
    if (j < w) {
      cp[e0 + j] = pc;
      cs[e0 + j] = dsc;
    }
    dsl[lane] = dsc;
    ksl[lane] = live ? (int)key : -1;
    wave_sync_lds();
    const int nj = min(64, w - c0);
    for (int jj = 0; jj < nj; ++jj) {
      const float g = dsl[jj];
      const int kj = ksl[jj];
      if (kj >= 0) {
        const T* kr = kbase + (int64_t)kj * A.kss;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int d = lane + 64 * e;
          if (d < D) acc[e] += g * ElemT<E>::load(kr + d);
        }
      }
    }
    wave_sync_lds();
  }
  T* dqrow = (T*)A.dq + (int64_t)b * A.dqsb + (int64_t)h * A.dqsh + (int64_t)r * A.dqss;
  // an entry the row does not attend (masked, or a key outside [0, kv_len))
  // adds dS * 0 in the Triton kernel with dS = p (0 - delta) scale (:202-221):
  // NaN throughout when delta is not finite
  const bool all_nan = row.bad_pos || (__builtin_amdgcn_ballot_w64(dead) != 0 && !__builtin_isfinite(delta));
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int d = lane + 64 * e;
    if (d < D) ElemT<E>::store(dqrow + d, all_nan ? __builtin_nanf("") : acc[e]);
  }
}

// seg[g] = the first sorted position whose key is >= g, g = 0 .. Hkv * kv_len
__global__ __launch_bounds__(256) void bwd_segments(GatherBwdArgs A) {
  const int64_t n_keys = (int64_t)A.Hkv * A.kv_len;
  for (int64_t g = (int64_t)blockIdx.x * 256 + threadIdx.x; g <= n_keys;
       g += (int64_t)gridDim.x * 256) {
    int64_t lo = 0, hi = A.E;
    while (lo < hi) {
      const int64_t mid = (lo + hi) >> 1;
      if ((int64_t)A.keys_out[mid] < g)
        lo = mid + 1;
      else
        hi = mid;
    }
    A.seg[g] = (int32_t)lo;
  }
}

// dK and dV of one (batch, kv head, key): its entries in sorted (entry id)
// order, four at a time (their q / dO rows loaded together), lanes over D.
template <Elem E>
__global__ __launch_bounds__(256) void bwd_kv_kernel(GatherBwdArgs A) {
  using T = typename ElemT<E>::T;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int key = blockIdx.x * 4 + wave;
  const int kvh = blockIdx.y, b = blockIdx.z;
  if (key >= A.kv_len) return;
  const int D = A.D;
  const int w = A.src.w;
  const int64_t g = (int64_t)kvh * A.kv_len + key;
  const int i0 = A.seg[g], i1 = A.seg[g + 1];
  const float* cp = A.cp + (int64_t)b * A.E;
  const float* cs = A.cs + (int64_t)b * A.E;
  float dk[4] = {0.f, 0.f, 0.f, 0.f}, dv[4] = {0.f, 0.f, 0.f, 0.f};
  constexpr int U = 4;
  for (int i = i0; i < i1; i += U) {
    float qv[U][4], gv[U][4], c_s[U], c_p[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = i + u < i1;
      const uint32_t e = in ? A.vals_out[i + u] : A.vals_out[i0];
      const int64_t hr = e / (uint32_t)w;
      const int r = (int)(hr % A.q_len), h = (int)(hr / A.q_len);
      c_s[u] = in ? cs[e] : 0.f;
      c_p[u] = in ? cp[e] : 0.f;
      const T* qrow = (const T*)A.q + (int64_t)b * A.qsb + (int64_t)h * A.qsh + (int64_t)r * A.qss;
      const T* dorow =
          (const T*)A.dout + (int64_t)b * A.dosb + (int64_t)h * A.dosh + (int64_t)r * A.doss;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int d = lane + 64 * q;
        // (a padding slot's row counts 0, not 0 times that row)
        qv[u][q] = in && d < D ? ElemT<E>::load(qrow + d) : 0.f;
        gv[u][q] = in && d < D ? ElemT<E>::load(dorow + d) : 0.f;
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        dk[q] += c_s[u] * qv[u][q];
        dv[q] += c_p[u] * gv[u][q];
      }
    }
  }
  T* dkrow = (T*)A.dk + (int64_t)b * A.dksb + (int64_t)kvh * A.dksh + (int64_t)key * A.dkss;
  T* dvrow = (T*)A.dv + (int64_t)b * A.dvsb + (int64_t)kvh * A.dvsh + (int64_t)key * A.dvss;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int d = lane + 64 * q;
    if (d < D) {
      ElemT<E>::store(dkrow + d, dk[q]);
      ElemT<E>::store(dvrow + d, dv[q]);
    }
  }
}

// ---------------------------------------------------------------------------
// Cooperative-row forms of the two passes (rows_coop_kernel, kv_coop_kernel):
// LPK lanes read each row, 16 bytes a lane, so a load instruction covers KPI =
// 64 / LPK whole rows (bwd_rows_kernel walks a K row per lane, 64 cache lines
// an instruction, and reads K twice).  Taken when coop_applies: 16-byte
// aligned rows and spans that 32-bit buffer offsets reach.  Loads go through
// buffer resources: a masked entry, a slot past a key's entries or a lane past
// head_dim gets an offset past num_records and reads zeros without a fetch, so
// a row that is not listed never meets the sums (no 0 * Inf).  Kernel times,
// per-lane forms against these: bf16 B=2 H=8 L=4096 D=128 (2.1 GB of rows in
// each pass) row pass 520 -> 130 us, key pass 787 -> 149 us (14 TB/s);
// float32 B=2 H=8 L=4096 D=64 467 -> 91 and 564 -> 106 us; bf16 D=96 H=16/4
// L=5001 496 -> 130 and 1036 -> 226 us.

// One wave per (batch, head, query row): dQ and the row's (lse, delta).  The
// list is walked in chunks of NMAX load instructions of K and as many of V
// (bwd_in_flight), all of a chunk's in flight before its first score; K stays
// in registers for dQ, and each lane forms one entry's dS.  Bound by the L2 row
// gathers (2 w rows a query row).
template <Elem E, int LPK, bool PATTERN>
__global__ __launch_bounds__(256, 2) void rows_coop_kernel(GatherBwdArgs A) {
  using T = typename ElemT<E>::T;
  constexpr int EPL = ElemT<E>::kPerChunk;
  constexpr int KPI = 64 / LPK;
  constexpr int NMAX = bwd_in_flight<LPK>();
  constexpr int SK = NMAX * KPI < 64 ? NMAX * KPI : 64;  // entries per chunk
  constexpr int NI = SK / KPI;
  __shared__ float s_all[4][64];
  __shared__ float dp_all[4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // XCD x (blockIdx % 8) takes a contiguous range of rows, so it reads few
  // heads' K and V at a time
  const int blk = (int)(blockIdx.x & 7) * A.rows_per_xcd + (int)(blockIdx.x >> 3);
  const int hr = blk * 4 + wave;
  const int b = blockIdx.y;
  if (hr >= A.H * A.q_len) return;  // whole wave leaves; no block-level barrier below
  const int h = hr / A.q_len, r = hr % A.q_len;
  const int kvh = h / A.groups;
  const int gk = lane / LPK, ln = lane % LPK;
  const bool act = ln * EPL < A.D;
  const uint32_t lofs = act ? 16u * (uint32_t)ln : kLaneNone;
  float* sl = s_all[wave];
  float* dpl = dp_all[wave];

  u32x4 q16 = {0u, 0u, 0u, 0u}, g16 = q16, o16 = q16;
  if (act) {
    q16 = *(const u32x4*)((const T*)A.q + (int64_t)b * A.qsb + (int64_t)h * A.qsh +
                          (int64_t)r * A.qss + EPL * ln);
    g16 = *(const u32x4*)((const T*)A.dout + (int64_t)b * A.dosb + (int64_t)h * A.dosh +
                          (int64_t)r * A.doss + EPL * ln);
    o16 = *(const u32x4*)((const T*)A.o + (int64_t)b * A.osb + (int64_t)h * A.osh +
                          (int64_t)r * A.oss + EPL * ln);
  }
  RowEntries row;
  row.init<PATTERN>(A.src, h, r);
  const float lse = A.lse[(int64_t)b * A.lsb + (int64_t)h * A.lsh + r];
  const float delta = group_sum<LPK>(dot16<E>(g16, o16));

  const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const T*)A.k + (int64_t)b * A.ksb + (int64_t)kvh * A.ksh), (short)0, A.k_span,
      0x00020000);
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
      (void*)((const T*)A.v + (int64_t)b * A.vsb + (int64_t)kvh * A.vsh), (short)0, A.v_span,
      0x00020000);
  const int w = A.src.w;
  const uint32_t kst = (uint32_t)A.kss * sizeof(T), vst = (uint32_t)A.vss * sizeof(T);

  float acc[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) acc[e] = 0.f;
  bool dead = false;
  for (int c0 = 0; c0 < w; c0 += SK) {
    const int j = c0 + lane;
    bool valid = false;
    int64_t key = 0;
    if (lane < SK && j < w) row.entry<PATTERN>(A.src, h, r, j, valid, key);
    const bool live = valid && key >= 0 && key < A.kv_len && !row.bad_pos;
    dead |= lane < SK && j < w && !live;
    const uint32_t ko = live ? (uint32_t)key * kst : kOffNone;
    const uint32_t vo = live ? (uint32_t)key * vst : kOffNone;
    u32x4 kd[NI], vd[NI];
#pragma unroll
    for (int t = 0; t < NI; ++t) {
      kd[t] = load16(rk, from_lane(ko, KPI * t + gk) + lofs);
      vd[t] = load16(rv, from_lane(vo, KPI * t + gk) + lofs);
    }
#pragma unroll
    for (int t = 0; t < NI; ++t) {
      const float s = group_sum<LPK>(dot16<E>(q16, kd[t]));
      const float dp = group_sum<LPK>(dot16<E>(g16, vd[t]));
      if (ln == 0) {
        sl[KPI * t + gk] = s;
        dpl[KPI * t + gk] = dp;
      }
    }
    wave_sync_lds();
    float dsc = 0.f;
    if (live) {
      const float p = expf(sl[lane] * A.sm_scale - lse);
      const float keep = drop_factor(A.drop, b, h, r, j, A.H, A.q_len, w);
      dsc = p * (keep * dpl[lane] - delta) * A.sm_scale;
    }
    wave_sync_lds();
    if (lane < SK) sl[lane] = dsc;
    wave_sync_lds();
#pragma unroll
    for (int t = 0; t < NI; ++t) {
      const float g = sl[KPI * t + gk];
#pragma unroll
      for (int e = 0; e < EPL; ++e) acc[e] += g * ElemT<E>::chunk(kd[t], e);
    }
    wave_sync_lds();
  }
#pragma unroll
  for (int e = 0; e < EPL; ++e) acc[e] = slot_sum<LPK>(acc[e]);
  // (as bwd_rows_kernel: NaN for an entry not attended when delta is not finite)
  const bool all_nan = row.bad_pos || (__builtin_amdgcn_ballot_w64(dead) != 0 &&
                                       !__builtin_isfinite(delta));
  if (all_nan) {
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc[e] = __builtin_nanf("");
  }
  if (gk == 0 && act)
    *(u32x4*)((T*)A.dq + (int64_t)b * A.dqsb + (int64_t)h * A.dqsh + (int64_t)r * A.dqss +
              EPL * ln) = ElemT<E>::pack_chunk(acc);
  if (lane == 0) A.ld2[(int64_t)b * A.H * A.q_len + hr] = make_float2(lse, delta);
}

// dK and dV of one (batch, kv head, key) over sorted positions [i0, i1) of
// its entries, in entry order: each entry's p and dS are formed again from
// its q and dO rows and the row's (lse, delta), so no coefficient per entry
// passes through memory.  A lane decodes one of 64 entries (row offsets, lse,
// delta); U loads of KPI rows each of q and dO are in flight per step; the
// exponential of the step's U * KPI entries is formed once, lane ln of a row
// taking entry ln % U, and handed to the row's lanes by quad broadcasts.
template <Elem E, int LPK>
struct KvAcc {
  static constexpr int EPL = ElemT<E>::kPerChunk;
  static constexpr int KPI = 64 / LPK;
  static constexpr int U = 4;
  float dk[EPL], dv[EPL];

  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int e = 0; e < EPL; ++e) dk[e] = dv[e] = 0.f;
  }

  __device__ __forceinline__ void run(const GatherBwdArgs& A, int b, const u32x4& k16,
                                      const u32x4& v16, int i0, int i1, int lane) {
    using T = typename ElemT<E>::T;
    const int gk = lane / LPK, ln = lane % LPK;
    const uint32_t lofs = ln * EPL < A.D ? 16u * (uint32_t)ln : kLaneNone;
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((const T*)A.q + (int64_t)b * A.qsb), (short)0, A.q_span, 0x00020000);
    const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((const T*)A.dout + (int64_t)b * A.dosb), (short)0, A.do_span, 0x00020000);
    const float2* ld2 = A.ld2 + (int64_t)b * A.H * A.q_len;
    const int w = A.src.w;
    for (int ib = i0; ib < i1; ib += 64) {
      uint32_t qo = kOffNone, go = kOffNone;
      float lse = 0.f, delta = 0.f, keep = 1.f;
      if (ib + lane < i1) {
        const uint32_t e = A.vals_out[ib + lane];
        const uint32_t hr = fast_div(e, A.div_w);
        const uint32_t h = fast_div(hr, A.div_q);
        const uint32_t r = hr - h * (uint32_t)A.q_len;
        qo = (h * (uint32_t)A.qsh + r * (uint32_t)A.qss) * (uint32_t)sizeof(T);
        go = (h * (uint32_t)A.dosh + r * (uint32_t)A.doss) * (uint32_t)sizeof(T);
        const float2 x = ld2[hr];
        lse = x.x;
        delta = x.y;
        if (A.drop.p > 0.f)
          keep = drop_factor(A.drop, b, (int)h, (int)r, (int)(e - hr * (uint32_t)w), A.H, A.q_len,
                             w);
      }
      const int n = min(i1 - ib, 64);
      for (int t0 = 0; t0 < n; t0 += U * KPI) {
        u32x4 qd[U], gd[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int src = t0 + u * KPI + gk;
          qd[u] = load16(rq, from_lane(qo, src) + lofs);
          gd[u] = load16(rg, from_lane(go, src) + lofs);
        }
        // this lane's entry of the step's four: u = ln % 4
        const int mine = t0 + (ln & 3) * KPI + gk;
        const float lse_m = from_lane(lse, mine), delta_m = from_lane(delta, mine);
        float keep_m = 1.f;
        if (A.drop.p > 0.f) keep_m = from_lane(keep, mine);
        float s = 0.f, dp = 0.f;
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float su = group_sum<LPK>(dot16<E>(k16, qd[u]));
          const float du = group_sum<LPK>(dot16<E>(v16, gd[u]));
          s = (ln & 3) == u ? su : s;
          dp = (ln & 3) == u ? du : dp;
        }
        // (a slot past the entries: zero rows with coefficient 0, also where
        // the key's own row is not finite)
        const bool in = mine < n;
        const float p = expf(s * A.sm_scale - lse_m);
        const float pc = in ? keep_m * p : 0.f;
        const float dsc = in ? p * (keep_m * dp - delta_m) * A.sm_scale : 0.f;
        auto quad = [](float x, auto uc) {
          return __int_as_float(
              __builtin_amdgcn_mov_dpp(__float_as_int(x), 0x55 * decltype(uc)::value, 0xf, 0xf, true));
        };
        auto add = [&](auto uc) {
          constexpr int u = decltype(uc)::value;
          const float cs = quad(dsc, uc), cp = quad(pc, uc);
#pragma unroll
          for (int e = 0; e < EPL; ++e) {
            dk[e] += cs * ElemT<E>::chunk(qd[u], e);
            dv[e] += cp * ElemT<E>::chunk(gd[u], e);
          }
        };
        add(std::integral_constant<int, 0>{});
        add(std::integral_constant<int, 1>{});
        add(std::integral_constant<int, 2>{});
        add(std::integral_constant<int, 3>{});
      }
    }
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      dk[e] = slot_sum<LPK>(dk[e]);
      dv[e] = slot_sum<LPK>(dv[e]);
    }
  }
};

// this lane's 16 bytes of K and V row `key`
template <Elem E>
__device__ __forceinline__ void kv_chunks(const GatherBwdArgs& A, int b, int kvh, int key, int ln,
                                          u32x4& k16, u32x4& v16) {
  using T = typename ElemT<E>::T;
  constexpr int EPL = ElemT<E>::kPerChunk;
  k16 = v16 = u32x4{0u, 0u, 0u, 0u};
  if (ln * EPL < A.D) {
    k16 = *(const u32x4*)((const T*)A.k + (int64_t)b * A.ksb + (int64_t)kvh * A.ksh +
                          (int64_t)key * A.kss + EPL * ln);
    v16 = *(const u32x4*)((const T*)A.v + (int64_t)b * A.vsb + (int64_t)kvh * A.vsh +
                          (int64_t)key * A.vss + EPL * ln);
  }
}

// A key with more than 2 * part entries is summed in parts, the windows
// [p part, (p + 1) part) of the sorted order cut to its segment, one wave per
// window (kv_parts_kernel), and kv_coop_kernel adds the parts in window
// order: at the last layers every row lists the first keys, and one wave over
// such a key's q_len entries would outlast the rest of the grid.  A window
// meets at most two such segments (each longer than two windows): the one
// holding its first position (slot 2 p) and one starting inside it (2 p + 1).
template <Elem E, int LPK>
__global__ __launch_bounds__(256) void kv_parts_kernel(GatherBwdArgs A) {
  constexpr int EPL = ElemT<E>::kPerChunk;
  const int lane = threadIdx.x & 63;
  const int p = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int b = blockIdx.y;
  if (p >= A.n_windows) return;
  const int w0 = p * A.part, w1 = (int)min((int64_t)w0 + A.part, A.E);
  const int sentinel = A.Hkv * A.kv_len;
  const int g0 = (int)A.keys_out[w0], g1 = (int)A.keys_out[w1 - 1];
  const int ln = lane % LPK;
  for (int which = 0; which < 2; ++which) {
    const int g = which ? g1 : g0;
    if (g >= sentinel || (which && g1 == g0)) continue;
    const int i0 = A.seg[g], i1 = A.seg[g + 1];
    if (i1 - i0 <= 2 * A.part) continue;
    u32x4 k16, v16;
    kv_chunks<E>(A, b, g / A.kv_len, g % A.kv_len, ln, k16, v16);
    KvAcc<E, LPK> acc;
    acc.clear();
    acc.run(A, b, k16, v16, max(i0, w0), min(i1, w1), lane);
    float* dst = A.partial + (((int64_t)b * A.n_windows + p) * 2 + which) * 2 * A.D;
    if (lane < LPK && ln * EPL < A.D) {
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        dst[EPL * ln + e] = acc.dk[e];
        dst[A.D + EPL * ln + e] = acc.dv[e];
      }
    }
  }
}

template <Elem E, int LPK>
__global__ __launch_bounds__(256) void kv_coop_kernel(GatherBwdArgs A) {
  using T = typename ElemT<E>::T;
  constexpr int EPL = ElemT<E>::kPerChunk;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // XCD x takes a contiguous range of keys
  const int blk = (int)(blockIdx.x & 7) * A.keys_per_xcd + (int)(blockIdx.x >> 3);
  const int64_t gw = (int64_t)blk * 4 + wave;
  const int b = blockIdx.y;
  if (gw >= (int64_t)A.Hkv * A.kv_len) return;
  const int g = (int)gw;
  const int kvh = g / A.kv_len, key = g % A.kv_len;
  const int ln = lane % LPK;
  const int i0 = A.seg[g], i1 = A.seg[g + 1];
  KvAcc<E, LPK> acc;
  acc.clear();
  if (i1 - i0 <= 2 * A.part) {
    u32x4 k16, v16;
    kv_chunks<E>(A, b, kvh, key, ln, k16, v16);
    acc.run(A, b, k16, v16, i0, i1, lane);
  } else if (ln * EPL < A.D) {
    for (int p = i0 / A.part; p <= (i1 - 1) / A.part; ++p) {
      const float* src =
          A.partial + (((int64_t)b * A.n_windows + p) * 2 + (i0 > p * A.part)) * 2 * A.D;
#pragma unroll
      for (int e = 0; e < EPL; ++e) {
        acc.dk[e] += src[EPL * ln + e];
        acc.dv[e] += src[A.D + EPL * ln + e];
      }
    }
  }
  if (lane < LPK && ln * EPL < A.D) {
    *(u32x4*)((T*)A.dk + (int64_t)b * A.dksb + (int64_t)kvh * A.dksh + (int64_t)key * A.dkss +
              EPL * ln) = ElemT<E>::pack_chunk(acc.dk);
    *(u32x4*)((T*)A.dv + (int64_t)b * A.dvsb + (int64_t)kvh * A.dvsh + (int64_t)key * A.dvss +
              EPL * ln) = ElemT<E>::pack_chunk(acc.dv);
  }
}

unsigned grid_for(int64_t n) {
  const int64_t blocks = (n + 255) / 256;
  return (unsigned)(blocks < 65536 ? (blocks > 0 ? blocks : 1) : 65536);
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort of (uint32 key, uint32 entry id) pairs, 8 bits a pass.
// A tile is 4096 pairs: wave w of a 256-thread block owns tile positions
// [1024 w, 1024 (w + 1)), item i and lane l holding position 1024 w + 64 i + l,
// so (wave, item, lane) order is the input order.  Three launches a pass:
// digit counts per tile (the first pass forms the keys there), their scan (a
// block per digit) and the scatter.  2.1M pairs with 16-bit keys, the launches
// of both passes: 125 -> 60 us against one-pair-at-a-time stores and separate
// key and chunked-scan launches (first scatter 52 -> 16 us); 5.1M: 230 -> 105.
constexpr int kSortTile = 4096;

// Sort keys of every entry (batch-independent): kv_head * kv_len + key of a
// valid entry with a key in [0, kv_len), else the sentinel Hkv * kv_len; and
// hist[d * nb + blk] = entries of tile blk whose lowest digit is d
template <bool PATTERN>
__global__ __launch_bounds__(256) void sort_keys_hist(GatherBwdArgs A, int nb) {
  __shared__ int cnt[256];
  cnt[threadIdx.x] = 0;
  __syncthreads();
  const uint32_t sentinel = (uint32_t)A.Hkv * (uint32_t)A.kv_len;
  const int64_t t0 = (int64_t)blockIdx.x * kSortTile;
  for (int i = threadIdx.x; i < kSortTile && t0 + i < A.E; i += 256) {
    const uint32_t e = (uint32_t)(t0 + i);
    const uint32_t hr = fast_div(e, A.div_w);
    const int j = (int)(e - hr * (uint32_t)A.src.w);
    const int h = (int)fast_div(hr, A.div_q), r = (int)(hr - (uint32_t)h * (uint32_t)A.q_len);
    RowEntries row;
    row.init<PATTERN>(A.src, h, r);
    bool valid = false;
    int64_t key = 0;
    row.entry<PATTERN>(A.src, h, r, j, valid, key);
    const bool live = valid && key >= 0 && key < A.kv_len && !row.bad_pos;
    const uint32_t k =
        live ? (uint32_t)(h / A.groups) * (uint32_t)A.kv_len + (uint32_t)key : sentinel;
    A.keys_in[e] = k;
    atomicAdd(&cnt[k & 255u], 1);
  }
  __syncthreads();
  A.hist[(int64_t)threadIdx.x * nb + blockIdx.x] = cnt[threadIdx.x];
}

// hist[d * nb + blk] = pairs of tile blk whose digit is d
__global__ __launch_bounds__(256) void radix_hist(const uint32_t* __restrict__ keys, int64_t n,
                                                  int shift, int nb, int32_t* __restrict__ hist) {
  __shared__ int cnt[256];
  const int blk = blockIdx.x;
  cnt[threadIdx.x] = 0;
  __syncthreads();
  const int64_t t0 = (int64_t)blk * kSortTile;
  for (int i = threadIdx.x; i < kSortTile; i += 256) {
    const int64_t x = t0 + i;
    if (x < n) atomicAdd(&cnt[(keys[x] >> shift) & 255u], 1);
  }
  __syncthreads();
  hist[(int64_t)threadIdx.x * nb + blk] = cnt[threadIdx.x];
}

// exclusive scan of 256 per-thread values over the block (Hillis-Steele in
// LDS); returns the thread's exclusive prefix and the block total in *total
__device__ __forceinline__ int block_exclusive_scan(int v, int* buf, int* total) {
  const int t = threadIdx.x;
  buf[t] = v;
  __syncthreads();
  for (int off = 1; off < 256; off <<= 1) {
    const int add = t >= off ? buf[t - off] : 0;
    __syncthreads();
    buf[t] += add;
    __syncthreads();
  }
  *total = buf[255];
  const int incl = buf[t];
  __syncthreads();
  return incl - v;
}

// offs[d * nb + blk] = pairs of digit d in tiles before blk (one block a digit)
__global__ __launch_bounds__(256) void radix_scan(const int32_t* __restrict__ hist, int nb,
                                                  int32_t* __restrict__ offs) {
  __shared__ int buf[256];
  const int64_t row = (int64_t)blockIdx.x * nb;
  int carry = 0;
  for (int base = 0; base < nb; base += 256) {
    const int i = base + threadIdx.x;
    const int v = i < nb ? hist[row + i] : 0;
    int total = 0;
    const int ex = block_exclusive_scan(v, buf, &total);
    if (i < nb) offs[row + i] = carry + ex;
    carry += total;
  }
}

// Scatter of one pass: a pair goes to (pairs of smaller digits) + offs[d * nb
// + blk] + (pairs of digit d in earlier waves of the tile) + (pairs of digit d
// before it in its wave).  Ranks within a wave come from eight ballots per
// item (the lanes sharing the pair's digit) and per-wave running digit counts
// in LDS.  The tile is put in order in LDS first, so the stores go out in runs
// of equal digits instead of one pair at a time.  FIRST: entry ids are the
// input positions.
template <bool FIRST>
__global__ __launch_bounds__(256) void radix_scatter(const uint32_t* __restrict__ kin,
                                                     const uint32_t* __restrict__ vin, int64_t n,
                                                     int shift, int nb,
                                                     const int32_t* __restrict__ hist,
                                                     const int32_t* __restrict__ offs,
                                                     uint32_t* __restrict__ kout,
                                                     uint32_t* __restrict__ vout) {
  __shared__ int cnt[4][256];
  __shared__ int buf[256];
  __shared__ int base_g[256];  // global position of the digit's first pair, minus its local one
  __shared__ uint32_t lk[kSortTile], lv[kSortTile];
  constexpr int ITEMS = kSortTile / 256;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int blk = blockIdx.x;
  for (int i = threadIdx.x; i < 4 * 256; i += 256) (&cnt[0][0])[i] = 0;
  __syncthreads();
  const uint64_t below = lane ? (~0ull >> (64 - lane)) : 0ull;
  const int64_t t0 = (int64_t)blk * kSortTile;
  const int64_t p0 = t0 + (int64_t)wave * (64 * ITEMS);
  uint32_t key[ITEMS], val[ITEMS];
  int rank[ITEMS];
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const int64_t x = p0 + (int64_t)it * 64 + lane;
    const bool ok = x < n;
    key[it] = ok ? kin[x] : 0u;
    val[it] = FIRST ? (uint32_t)x : ok ? vin[x] : 0u;
  }
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const bool ok = p0 + (int64_t)it * 64 + lane < n;
    const uint32_t d = (key[it] >> shift) & 255u;
    uint64_t peers = __builtin_amdgcn_ballot_w64(ok);
#pragma unroll
    for (int bit = 0; bit < 8; ++bit) {
      const uint64_t bal = __builtin_amdgcn_ballot_w64(((d >> bit) & 1u) != 0u);
      peers &= ((d >> bit) & 1u) ? bal : ~bal;
    }
    const int base = cnt[wave][d];
    rank[it] = base + __builtin_popcountll(peers & below);
    wave_sync_lds();
    // the lowest lane of each digit group advances that digit's count
    if (ok && (peers & below) == 0ull) cnt[wave][d] = base + __builtin_popcountll(peers);
    wave_sync_lds();
  }
  __syncthreads();
  // thread d: its digit's pairs in the tile and in the whole input, both
  // scanned over the digits; cnt[w][d] becomes the local position of the
  // digit's first pair of wave w
  {
    const int d = threadIdx.x;
    int c[4];
#pragma unroll
    for (int w2 = 0; w2 < 4; ++w2) c[w2] = cnt[w2][d];
    const int64_t row = (int64_t)d * nb;
    const int all = offs[row + nb - 1] + hist[row + nb - 1];
    int total = 0;
    int at = block_exclusive_scan(c[0] + c[1] + c[2] + c[3], buf, &total);
    const int first = block_exclusive_scan(all, buf, &total);
    base_g[d] = first + offs[row + blk] - at;
#pragma unroll
    for (int w2 = 0; w2 < 4; ++w2) {
      cnt[w2][d] = at;
      at += c[w2];
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    if (p0 + (int64_t)it * 64 + lane >= n) continue;
    const int at = cnt[wave][(key[it] >> shift) & 255u] + rank[it];
    lk[at] = key[it];
    lv[at] = val[it];
  }
  __syncthreads();
  const int here = (int)(n - t0 < kSortTile ? n - t0 : kSortTile);
  for (int i = threadIdx.x; i < here; i += 256) {
    const uint32_t k = lk[i];
    const int dst = base_g[(k >> shift) & 255u] + i;
    kout[dst] = k;
    vout[dst] = lv[i];
  }
}

// Sorts the entries by key over the low key_bits bits; returns, through *keys
// / *vals, the buffers holding the result (the pair buffers alternate by pass).
hipError_t radix_sort(const GatherBwdArgs& A, bool pattern, const uint32_t** keys,
                      const uint32_t** vals, hipStream_t stream) {
  const int64_t n = A.E;
  const int nb = (int)((n + kSortTile - 1) / kSortTile);
  uint32_t* ka = A.keys_in;
  uint32_t* va = A.vals_in;
  uint32_t* kb = A.keys_out;
  uint32_t* vb = A.vals_out;
  for (int shift = 0; shift < A.key_bits; shift += 8) {
    if (shift > 0)
      radix_hist<<<nb, 256, 0, stream>>>(ka, n, shift, nb, A.hist);
    else if (pattern)
      sort_keys_hist<true><<<nb, 256, 0, stream>>>(A, nb);
    else
      sort_keys_hist<false><<<nb, 256, 0, stream>>>(A, nb);
    radix_scan<<<256, 256, 0, stream>>>(A.hist, nb, A.offs);
    if (shift > 0)
      radix_scatter<false><<<nb, 256, 0, stream>>>(ka, va, n, shift, nb, A.hist, A.offs, kb, vb);
    else
      radix_scatter<true><<<nb, 256, 0, stream>>>(ka, va, n, shift, nb, A.hist, A.offs, kb, vb);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    uint32_t* t = ka; ka = kb; kb = t;
    t = va; va = vb; vb = t;
  }
  *keys = ka;
  *vals = va;
  return hipSuccess;
}

// Whether the cooperative-row kernels take the call: 16-byte aligned rows of
// every tensor, and K / V heads and q / dO batch elements within 32-bit buffer
// offsets.  Fills what they need in a.
bool coop_applies(GatherBwdArgs& a, int es) {
  const int64_t epl = 16 / es;
  if (a.D % epl != 0) return false;
  const void* ptrs[] = {a.q, a.k, a.v, a.o, a.dout, a.dq, a.dk, a.dv};
  for (const void* p : ptrs)
    if (((uintptr_t)p & 15) != 0) return false;
  const int64_t st[] = {a.qsb,  a.qsh,  a.qss,  a.ksb,  a.ksh,  a.kss,  a.vsb,  a.vsh,
                        a.vss,  a.osb,  a.osh,  a.oss,  a.dosb, a.dosh, a.doss, a.dqsb,
                        a.dqsh, a.dqss, a.dksb, a.dksh, a.dkss, a.dvsb, a.dvsh, a.dvss};
  for (int64_t x : st)
    if (x % epl != 0) return false;
  auto span = [&](int64_t n0, int64_t s0, int64_t n1, int64_t s1) {
    return row_span(n0, s0, n1, s1, a.D, es);
  };
  const int64_t ks = span(a.kv_len, a.kss, 1, 0), vs = span(a.kv_len, a.vss, 1, 0);
  const int64_t qs = span(a.H, a.qsh, a.q_len, a.qss), gs = span(a.H, a.dosh, a.q_len, a.doss);
  if (ks >= kMaxSpan || vs >= kMaxSpan || qs >= kMaxSpan || gs >= kMaxSpan) return false;
  a.k_span = (int)ks;
  a.v_span = (int)vs;
  a.q_span = (int)qs;
  a.do_span = (int)gs;
  const int64_t rows = (int64_t)a.H * a.q_len;
  // (64 work-items a row and a key, 2^32 a grid dimension)
  constexpr int64_t kMost = (int64_t(1) << 26) - 64;
  if (rows > kMost || (int64_t)a.Hkv * a.kv_len > kMost) return false;
  // the per-entry coefficients' 2 B E floats hold the rows' (lse, delta) and
  // the partial sums of long segments, in windows of at least 512 entries
  a.ld2 = (float2*)a.cp;
  const int64_t head = 2 * a.B * rows, left = 2 * a.B * a.E - head;
  a.partial = a.cp + head;
  const int64_t per_window = 4 * (int64_t)a.D * a.B;  // floats
  const int64_t most = left / per_window;             // windows that fit
  int64_t part = most > 0 ? (a.E + most - 1) / most : a.E;
  part = (part < 512 ? 512 : part) + 63;
  part -= part % 64;
  a.part = (int)(part < (int64_t(1) << 30) ? part : (int64_t(1) << 30));
  // (segments of more than 2 part entries: none when the grid has no room)
  a.n_windows = a.E > 2 * (int64_t)a.part ? (int)((a.E + a.part - 1) / a.part) : 0;
  a.rows_per_xcd = (int)(((rows + 3) / 4 + 7) / 8);
  a.keys_per_xcd = (int)((((int64_t)a.Hkv * a.kv_len + 3) / 4 + 7) / 8);
  return true;
}

template <Elem E, int LPK>
void launch_rows_coop(const GatherBwdArgs& a, bool pattern, hipStream_t stream) {
  const dim3 grid(8u * (unsigned)a.rows_per_xcd, (unsigned)a.B);
  if (pattern)
    rows_coop_kernel<E, LPK, true><<<grid, 256, 0, stream>>>(a);
  else
    rows_coop_kernel<E, LPK, false><<<grid, 256, 0, stream>>>(a);
}

template <Elem E, int LPK>
void launch_kv_coop(const GatherBwdArgs& a, hipStream_t stream) {
  if (a.n_windows > 0)
    kv_parts_kernel<E, LPK>
        <<<dim3((unsigned)((a.n_windows + 3) / 4), (unsigned)a.B), 256, 0, stream>>>(a);
  kv_coop_kernel<E, LPK>
      <<<dim3(8u * (unsigned)a.keys_per_xcd, (unsigned)a.B), 256, 0, stream>>>(a);
}

// lanes per row: 8, 16, 32 or 64 of 16 bytes (lanes past head_dim idle)
#define ESA_LANES(E, fn, ...)                             \
  do {                                                    \
    const int lanes_ = a.D / ElemT<E>::kPerChunk;         \
    if (lanes_ <= 8)                                      \
      fn<E, 8>(__VA_ARGS__);                              \
    else if (lanes_ <= 16)                                \
      fn<E, 16>(__VA_ARGS__);                             \
    else if (lanes_ <= 32)                                \
      fn<E, 32>(__VA_ARGS__);                             \
    else if constexpr (ElemT<E>::kPerChunk == 4)          \
      fn<E, 64>(__VA_ARGS__);                             \
  } while (0)

template <Elem E>
hipError_t launch_elem(const GatherBwdArgs& a0, bool pattern, hipStream_t stream) {
  GatherBwdArgs a = a0;
  a.div_w = make_fast_div((uint32_t)a.src.w);
  a.div_q = make_fast_div((uint32_t)(a.q_len > 0 ? a.q_len : 1));
  const bool coop = coop_applies(a, ElemT<E>::kBytes);
  GatherBwdArgs s = a;
  hipError_t e = hipSuccess;
  if (a.E > 0) {
    const dim3 rows_grid((unsigned)((a.q_len + 3) / 4), (unsigned)a.H, (unsigned)a.B);
    if (coop)
      ESA_LANES(E, launch_rows_coop, a, pattern, stream);
    else if (pattern)
      bwd_rows_kernel<E, true><<<rows_grid, 256, 0, stream>>>(a);
    else
      bwd_rows_kernel<E, false><<<rows_grid, 256, 0, stream>>>(a);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    const uint32_t* sk = nullptr;
    const uint32_t* sv = nullptr;
    e = radix_sort(a, pattern, &sk, &sv, stream);
    if (e != hipSuccess) return e;
    s.keys_out = const_cast<uint32_t*>(sk);
    s.vals_out = const_cast<uint32_t*>(sv);
  }
  // with no entries every segment is empty and dK = dV = 0
  bwd_segments<<<grid_for((int64_t)a.Hkv * a.kv_len + 1), 256, 0, stream>>>(s);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (coop) {
    ESA_LANES(E, launch_kv_coop, s, stream);
    return hipGetLastError();
  }
  const dim3 kv_grid((unsigned)((a.kv_len + 3) / 4), (unsigned)a.Hkv, (unsigned)a.B);
  bwd_kv_kernel<E><<<kv_grid, 256, 0, stream>>>(s);
  return hipGetLastError();
}

}  // namespace

int64_t gather_bwd_hist_ints(int64_t n) { return 256 * ((n + kSortTile - 1) / kSortTile); }

hipError_t launch_gather_bwd(const GatherBwdArgs& a, bool pattern, hipStream_t stream) {
  if (a.B <= 0 || a.H <= 0 || a.kv_len <= 0) return hipSuccess;
  switch ((Elem)a.elem) {
    case Elem::f32: return launch_elem<Elem::f32>(a, pattern, stream);
    case Elem::bf16: return launch_elem<Elem::bf16>(a, pattern, stream);
    default: return launch_elem<Elem::f16>(a, pattern, stream);
  }
}

}  // namespace esa
