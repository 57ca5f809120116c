// Per-row index sources shared by the gather forward, the naive-path weights
// and the gather backward: a query row's w entries either regenerated from
// the elastic pattern (bit-exact with elastic_sparse_attention.py:470-535,
// masked entries 0 and clamped to [0, kv_len - 1] as _triton_forward does,
// :602-615) or read from explicit index / mask arrays (the operator
// ElasticSparseAttentionFunction, :241-297).
#pragma once
#include "esa_elem.hpp"
#include "esa_internal.hpp"

namespace esa {

struct RowEntries {
  HeadWeights hw;
  RowParams rp;
  int pos;       // the row's query position
  bool bad_pos;  // a position outside [-kv_len, kv_len): the row reads NaN

  template <bool PATTERN>
  __device__ __forceinline__ void init(const IndexSource& S, int h, int r) {
    pos = r;
    bad_pos = false;
    hw = HeadWeights{};
    rp = RowParams{};
    if (PATTERN) {
      if (S.positions) {
        // negative positions count from the end, as torch indexing does
        const int64_t p0 = S.positions[r];
        const int64_t p64 = p0 < 0 ? p0 + S.kv_len : p0;
        bad_pos = p64 < 0 || p64 >= S.kv_len;
        pos = bad_pos ? 0 : (int)p64;
      }
      hw = head_weights(S.pc, h);
      rp = row_params(S.pc, pos);
    }
  }

  // Entry j < w of the row: its key and whether it is valid.  A pattern key
  // is always in [0, kv_len); an explicit one may lie outside (the Triton
  // kernel then scores it 0 against zero K/V, :131-134).
  template <bool PATTERN>
  __device__ __forceinline__ void entry(const IndexSource& S, int h, int r, int j, bool& valid,
                                        int64_t& key) const {
    if (PATTERN) {
      const int idx = interp_index(oversized(rp, j), oversized(rp, j + 1), hw);
      valid = idx <= pos;
      int kk = valid ? idx : 0;
      kk = kk < 0 ? 0 : (kk > S.kv_len - 1 ? S.kv_len - 1 : kk);
      key = kk;
    } else {
      key = load_int_any(S.indices, S.index_bytes, (int64_t)h * S.ish + (int64_t)r * S.iss + j);
      valid = load_int_any(S.mask, S.mask_bytes, (int64_t)h * S.msh + (int64_t)r * S.mss + j) != 0;
    }
  }
};

// Dropout multiplier of entry j of row (b, h, r): 1 without dropout, else 0
// or 1 / (1 - p_drop) by the counter-based keep decision.
__device__ __forceinline__ float drop_factor(const DropoutArgs& dr, int b, int h, int r, int j,
                                             int H, int q_len, int w) {
  if (!(dr.p > 0.f)) return 1.f;
  const uint64_t idx = (((uint64_t)b * H + h) * (uint64_t)q_len + r) * (uint64_t)w + j;
  return dropout_keep(dr.seed, idx, dr.p) ? dr.scale : 0.f;
}

// Sum over aligned groups of N lanes (N = 8, 16, 32, 64), in every lane of
// the group: DPP within 16-lane rows (quad swaps and a half-row mirror for
// N = 8, row rotations by 8, 4, 2, 1 for 16), cross-row steps by lane swaps.
template <int N>
__device__ __forceinline__ float group_sum(float v) {
  auto dpp = [](float x, int ctrl) -> float {
    switch (ctrl) {  // the control word must be a constant
      case 0xB1: return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xf, 0xf, false));
      case 0x4E: return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xf, 0xf, false));
      case 0x141: return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x141, 0xf, 0xf, false));
      case 0x128: return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x128, 0xf, 0xf, false));
      case 0x124: return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x124, 0xf, 0xf, false));
      case 0x122: return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x122, 0xf, 0xf, false));
      default: return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x121, 0xf, 0xf, false));
    }
  };
  if (N == 8) {
    v += dpp(v, 0xB1);   // quad_perm [1, 0, 3, 2]
    v += dpp(v, 0x4E);   // quad_perm [2, 3, 0, 1]
    v += dpp(v, 0x141);  // row_half_mirror: the other quad of the 8
    return v;
  }
  v += dpp(v, 0x128);  // row_ror 8
  v += dpp(v, 0x124);  // row_ror 4
  v += dpp(v, 0x122);  // row_ror 2
  v += dpp(v, 0x121);  // row_ror 1
  if (N >= 32) {
    const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                    false);
    v = __uint_as_float(x[0]) + __uint_as_float(x[1]);
  }
  if (N >= 64) {
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                    false);
    v = __uint_as_float(x[0]) + __uint_as_float(x[1]);
  }
  return v;
}

// Orders LDS writes of a wave before its later reads (the wave's lanes run
// in lock step; the fences keep the compiler from reordering).
__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Row loads through buffer resources, LPK lanes a row: a masked entry, a slot
// past a list's end or a lane past head_dim gets an offset past num_records
// and reads zeros without a fetch.
constexpr uint32_t kOffNone = 0x80000000u;   // an entry's row offset: none
constexpr uint32_t kLaneNone = 0x7FFFF000u;  // a lane's offset within a row: past head_dim
// spans stay below both offsets
constexpr int64_t kMaxSpan = (int64_t(1) << 31) - 8192;

// Bytes from the first to past the last of n0 x n1 rows of D elements (es
// bytes each) at strides s0, s1, kMaxSpan at least when 32-bit offsets do not
// reach them (each factor is bounded before it is multiplied)
inline int64_t row_span(int64_t n0, int64_t s0, int64_t n1, int64_t s1, int D, int es) {
  if (n0 <= 0 || n1 <= 0) return 0;
  if (s0 < 0 || s1 < 0 || (n0 > 1 && s0 >= kMaxSpan) || (n1 > 1 && s1 >= kMaxSpan))
    return kMaxSpan;
  return ((n0 - 1) * s0 + (n1 - 1) * s1 + D) * es;
}

__device__ __forceinline__ u32x4 load16(__amdgpu_buffer_rsrc_t rs, uint32_t off) {
  return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, 0));
}

// v of lane `src` (0 .. 63)
__device__ __forceinline__ uint32_t from_lane(uint32_t v, int src) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute(4 * src, (int)v);
}
__device__ __forceinline__ float from_lane(float v, int src) {
  return __uint_as_float(from_lane(__float_as_uint(v), src));
}

// Row loads of K (and as many of V) a wave keeps in flight where the grid
// fills the chip: fewer than a row's list needs, so that more waves share a
// SIMD (180-210 VGPRs with 16 in flight, 100-140 with 8, 80 with 4) and one
// wave's sums overlap another's loads.  B=2 H=8 L=4096, 16 / 8 / 4 / 2 in flight,
// forward (H/Hkv = 4): float32 D=64 148 / 102 / 98 / 132 us, D=128 250 / 170 /
// 181 / 241, bf16 D=64 73 / 74 / 70 / 83, D=128 158 / 112 / 117 / 138, D=256
// 296 / 195 / 213 / 267; whole backward: float32 D=64 404 / 356 / 346 / 357,
// D=256 1116 / 1070 / 1092 / 1154, bf16 D=128 465 / 404 / 395 / 406.
template <Elem E, int LPK>
constexpr int fwd_in_flight() {
  return LPK <= (E == Elem::f32 ? 16 : 8) ? 4 : 8;
}
template <int LPK>
constexpr int bwd_in_flight() {
  return LPK <= 32 ? 4 : 8;
}

// Dot product of two 16-byte chunks.  bfloat16 pairs go through v_dot2_f32_bf16
// (exact products, float32 sums; over 128-element dots of normal values its
// error against float64 is 7.0e-8, a float32 fma chain's 7.3e-8; Inf, NaN and
// subnormals as in the chain): 4 instructions instead of 8 conversions and 8
// fmas (backward row pass bf16 D=128 155 -> 130 us, forward 133 -> 125).
template <Elem E>
__device__ __forceinline__ float dot16(const u32x4& a, const u32x4& b) {
  float acc = 0.f;
  if constexpr (E == Elem::bf16) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      // (copies: a bit cast of a vector's element itself reads element 0)
      const uint32_t x = a[e], y = b[e];
      acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, x),
                                            __builtin_bit_cast(bf16x2, y), acc, false);
    }
  } else {
#pragma unroll
    for (int e = 0; e < ElemT<E>::kPerChunk; ++e)
      acc += ElemT<E>::chunk(a, e) * ElemT<E>::chunk(b, e);
  }
  return acc;
}

// sum over the lanes l, l + LPK, l + 2 LPK, ... (a row slot each)
template <int LPK>
__device__ __forceinline__ float slot_sum(float v) {
#pragma unroll
  for (int off = LPK; off < 64; off <<= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// One query row (b, h, r) of the per-row gather forward, by one wave (the
// body of gather_rows_kernel, esa_fwd_gather.hip, which describes it): LPK
// lanes read a row of at most LPK 16-byte pieces; NMAX: load instructions of K
// (and of V) in flight; BUF: K and V by buffer loads (their spans allow it);
// sc: 64 floats of LDS private to the wave.
template <Elem E, int LPK, int NMAX, bool BUF, bool PATTERN>
__device__ __forceinline__ void gather_one_row(const GatherArgs& A, int b, int h, int r,
                                               float* sc, int lane) {
  using T = typename ElemT<E>::T;
  constexpr int EPL = ElemT<E>::kPerChunk;  // elements per lane per load
  constexpr int KPI = 64 / LPK;             // rows per load instruction
  constexpr int SK = NMAX * KPI < 64 ? NMAX * KPI : 64;  // keys per chunk
  constexpr int NI = SK / KPI;              // load instructions per chunk
  static_assert(LPK <= 64 && 64 % LPK == 0, "row split");
  const int kvh = h / A.groups;
  const int gk = lane / LPK;  // row of an instruction this lane loads
  const int ln = lane % LPK;  // its 16-byte piece: elements EPL ln .. + EPL
  const bool act = EPL * ln < A.D;

  u32x4 q16 = {0u, 0u, 0u, 0u};
  if (act)
    q16 = *(const u32x4*)((const T*)A.q + (int64_t)b * A.qsb + (int64_t)h * A.qsh +
                          (int64_t)r * A.qss + EPL * ln);
  const T* kbase = (const T*)A.k + (int64_t)b * A.ksb + (int64_t)kvh * A.ksh;
  const T* vbase = (const T*)A.v + (int64_t)b * A.vsb + (int64_t)kvh * A.vsh;
  const __amdgpu_buffer_rsrc_t rk =
      __builtin_amdgcn_make_buffer_rsrc((void*)kbase, (short)0, A.k_span, 0x00020000);
  const __amdgpu_buffer_rsrc_t rv =
      __builtin_amdgcn_make_buffer_rsrc((void*)vbase, (short)0, A.v_span, 0x00020000);
  const uint32_t lofs = act ? 16u * (uint32_t)ln : kLaneNone;
  const uint32_t kst = (uint32_t)A.kss * sizeof(T), vst = (uint32_t)A.vss * sizeof(T);
  RowEntries row;
  row.init<PATTERN>(A.src, h, r);

  float m = -INFINITY, l = 0.f;
  float acc[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) acc[e] = 0.f;
  const int w = A.src.w;
  for (int c0 = 0; c0 < w; c0 += SK) {
    // slot `lane` of the chunk: entry c0 + lane
    const int j = c0 + lane;
    bool valid = false;
    int64_t key = 0;
    if (lane < SK && j < w) row.entry<PATTERN>(A.src, h, r, j, valid, key);
    const bool in_range = key >= 0 && key < A.kv_len;
    const bool live = valid && in_range;
    u32x4 kd[NI], vd[NI];
    if constexpr (BUF) {
      const uint32_t ko = live ? (uint32_t)key * kst : kOffNone;
      const uint32_t vo = live ? (uint32_t)key * vst : kOffNone;
#pragma unroll
      for (int t = 0; t < NI; ++t) {
        kd[t] = load16(rk, from_lane(ko, KPI * t + gk) + lofs);
        vd[t] = load16(rv, from_lane(vo, KPI * t + gk) + lofs);
      }
    } else {
      const uint32_t kaddr = live ? (uint32_t)key : kOffNone;
#pragma unroll
      for (int t = 0; t < NI; ++t) {
        const uint32_t kk = from_lane(kaddr, KPI * t + gk);
        kd[t] = vd[t] = u32x4{0u, 0u, 0u, 0u};
        if (act && kk != kOffNone) {
          kd[t] = *(const u32x4*)(kbase + (int64_t)kk * A.kss + EPL * ln);
          vd[t] = *(const u32x4*)(vbase + (int64_t)kk * A.vss + EPL * ln);
        }
      }
    }
#pragma unroll
    for (int t = 0; t < NI; ++t) {
      const float part = group_sum<LPK>(dot16<E>(q16, kd[t]));
      if (ln == 0) sc[KPI * t + gk] = part;
    }
    wave_sync_lds();
    float s = -INFINITY;
    if (lane < SK && valid) s = in_range ? sc[lane] * A.sm_scale : 0.f;
    const float cmax = wave_max(s);
    const float m_new = fmaxf(m, cmax);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float p = valid ? expf(s - m_use) : 0.f;
    const float alpha = expf(m - m_use);
    l = l * alpha + wave_sum(p);
#pragma unroll
    for (int e = 0; e < EPL; ++e) acc[e] *= alpha;
    m = m_new;
    wave_sync_lds();
    // PV weight of the slot (dropout keep factor applied)
    if (lane < SK) {
      const float keep = j < w ? drop_factor(A.drop, b, h, r, j, A.H, A.q_len, w) : 0.f;
      sc[lane] = live ? p * keep : 0.f;
    }
    wave_sync_lds();
#pragma unroll
    for (int t = 0; t < NI; ++t) {
      const float pt = sc[KPI * t + gk];
#pragma unroll
      for (int e = 0; e < EPL; ++e) acc[e] += pt * ElemT<E>::chunk(vd[t], e);
    }
    wave_sync_lds();
  }
  // the KPI row groups' partial sums: lanes ln, ln + LPK, ...
#pragma unroll
  for (int e = 0; e < EPL; ++e) acc[e] = slot_sum<LPK>(acc[e]);

  const float inv = row.bad_pos ? __builtin_nanf("") : (l > 0.f ? 1.f / l : 0.f);
  if (gk == 0 && act) {
    T* orow = (T*)A.o + (int64_t)b * A.osb + (int64_t)h * A.osh + (int64_t)r * A.oss + EPL * ln;
    float x[EPL];
#pragma unroll
    for (int e = 0; e < EPL; ++e) x[e] = acc[e] * inv;
    *(u32x4*)orow = ElemT<E>::pack_chunk(x);
  }
  if (A.lse && lane == 0)
    A.lse[(int64_t)b * A.lsb + (int64_t)h * A.lsh + r] =
        row.bad_pos ? __builtin_nanf("") : (l > 0.f ? m + logf(l) : -INFINITY);
}

// dot(q, k_row) over D (D % 4 == 0); q in LDS as float
template <Elem E>
__device__ __forceinline__ float row_dot(const float* __restrict__ qs,
                                         const typename ElemT<E>::T* __restrict__ kr, int D) {
  float acc = 0.f;
  if constexpr (E == Elem::f32) {
    for (int d = 0; d < D; d += 4) {
      const f32x4 kv = *(const f32x4*)(kr + d);
      acc += qs[d] * kv[0];
      acc += qs[d + 1] * kv[1];
      acc += qs[d + 2] * kv[2];
      acc += qs[d + 3] * kv[3];
    }
  } else {
    for (int d = 0; d < D; d += 4) {
      const u32x2 kv = *(const u32x2*)(kr + d);
      const u32x4 raw = {kv[0], kv[1], 0u, 0u};
      acc += qs[d] * ElemT<E>::chunk(raw, 0);
      acc += qs[d + 1] * ElemT<E>::chunk(raw, 1);
      acc += qs[d + 2] * ElemT<E>::chunk(raw, 2);
      acc += qs[d + 3] * ElemT<E>::chunk(raw, 3);
    }
  }
  return acc;
}

// One query row (b, h, r) of the per-row gather forward for any head_dim (a
// multiple of 4, up to 256), by one wave (the body of gather_fwd_kernel,
// esa_fwd_gather.hip, which describes it; also the band forward's path for
// rows whose positions are not consecutive): scratch is 384 floats of LDS
// private to the wave (q, the chunk's probabilities and keys).
template <Elem E, bool PATTERN>
__device__ __forceinline__ void gather_one_row_any(const GatherArgs& A, int b, int h, int r,
                                                   float* scratch, int lane) {
  using T = typename ElemT<E>::T;
  const int kvh = h / A.groups;
  const int D = A.D;
  float* qs = scratch;                // D <= 256 floats
  float* ps = scratch + 256;          // 64
  int* ks = (int*)(scratch + 320);    // 64

  const T* qrow = (const T*)A.q + (int64_t)b * A.qsb + (int64_t)h * A.qsh + (int64_t)r * A.qss;
  for (int d = lane; d < D; d += 64) qs[d] = ElemT<E>::load(qrow + d);
  wave_sync_lds();

  const T* kbase = (const T*)A.k + (int64_t)b * A.ksb + (int64_t)kvh * A.ksh;
  const T* vbase = (const T*)A.v + (int64_t)b * A.vsb + (int64_t)kvh * A.vsh;
  RowEntries row;
  row.init<PATTERN>(A.src, h, r);

  float m = -INFINITY, l = 0.f;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  const int w = A.src.w;
  for (int c0 = 0; c0 < w; c0 += 64) {
    const int j = c0 + lane;
    bool valid = false;
    int64_t key = 0;
    if (j < w) row.entry<PATTERN>(A.src, h, r, j, valid, key);
    const bool in_range = key >= 0 && key < A.kv_len;
    float s = -INFINITY;
    if (valid) s = in_range ? row_dot<E>(qs, kbase + key * A.kss, D) * A.sm_scale : 0.f;
    const float cmax = wave_max(s);
    const float m_new = fmaxf(m, cmax);
    const float m_use = m_new == -INFINITY ? 0.f : m_new;
    const float p = valid ? expf(s - m_use) : 0.f;
    const float alpha = expf(m - m_use);
    l = l * alpha + wave_sum(p);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] *= alpha;
    m = m_new;
    const float keep = j < w ? drop_factor(A.drop, b, h, r, j, A.H, A.q_len, w) : 0.f;
    ps[lane] = p * keep;
    ks[lane] = (valid && in_range) ? (int)key : -1;
    wave_sync_lds();
    const int nj = min(64, w - c0);
    for (int jj = 0; jj < nj; ++jj) {
      const float pj = ps[jj];
      const int kj = ks[jj];
      if (kj >= 0 && pj != 0.f) {
        const T* vr = vbase + (int64_t)kj * A.vss;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int d = lane + 64 * e;
          if (d < D) acc[e] += pj * ElemT<E>::load(vr + d);
        }
      }
    }
    wave_sync_lds();
  }

  const float inv = row.bad_pos ? __builtin_nanf("") : (l > 0.f ? 1.f / l : 0.f);
  T* orow = (T*)A.o + (int64_t)b * A.osb + (int64_t)h * A.osh + (int64_t)r * A.oss;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int d = lane + 64 * e;
    if (d < D) ElemT<E>::store(orow + d, acc[e] * inv);
  }
  if (A.lse && lane == 0)
    A.lse[(int64_t)b * A.lsb + (int64_t)h * A.lsh + r] =
        row.bad_pos ? __builtin_nanf("") : (l > 0.f ? m + logf(l) : -INFINITY);
}

}  // namespace esa
