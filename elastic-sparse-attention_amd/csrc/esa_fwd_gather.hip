// Per-row gather forward (gfx950): one wave per (batch, head, query row).
//
// Two index sources share the kernels (esa_gather.hpp):
//   explicit  indices / mask arrays, the operator
//             ElasticSparseAttentionFunction.forward (elastic_sparse_attention.py:241-297)
//             with the Triton kernel's semantics (:117-166): a valid entry
//             whose index is outside [0, kv_len) scores 0 against zero K/V;
//             duplicates count once per entry.
//   pattern   each row's w indices regenerated on the device for query
//             position positions[r] (or r), masked entries set to 0 and
//             clamped to [0, kv_len - 1] as _triton_forward does (:602-615).
//
// q, k, v and o are float32, bfloat16 or float16; everything is computed in
// float32 with accurate expf (float32 inputs meet a 1e-4 bound), and o is
// stored in the inputs' type.  With dropout (the naive path in training
// mode, :674) each probability is multiplied by its entry's keep factor in
// PV; the normaliser and lse stay those of the undropped probabilities, as
// torch.dropout after the softmax leaves them.
//
// gather_fwd_kernel: lanes split the row's entries 64 at a time for QK (each
// lane one key, a full dot product over D in float32), then split D for PV
// (each lane up to four d columns, one 64-key chunk at a time with p and the
// key broadcast through LDS).  gather_rows_kernel (16-byte
// aligned rows) reads each K and V row with a lane per 16 bytes.
// gather_weights_kernel writes the naive path's attention weights from the
// forward's lse.
#include <algorithm>

#include "esa_gather.hpp"

namespace esa {

namespace {

template <Elem E, bool PATTERN>
__global__ __launch_bounds__(256) void gather_fwd_kernel(GatherArgs A) {
  __shared__ float scratch_all[4][384];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = blockIdx.x * 4 + wave;
  const int h = blockIdx.y, b = blockIdx.z;
  if (r >= A.q_len) return;  // whole wave leaves; no block-level barrier below
  gather_one_row_any<E, PATTERN>(A, b, h, r, scratch_all[wave], lane);
}

// ---------------------------------------------------------------------------
// Cooperative-row variant for 16-byte aligned rows (head dims of whole 16-byte
// pieces): one wave per (batch, head, query row) as above, waves numbered over
// (batch, head, row) with the row fastest (a one-row decode step fills every
// wave of a block; a block per row would leave three of its four waves idle),
// but each K and V row is read by LPK lanes (8, 16, 32 or 64: the smallest
// that hold a row, lanes past head_dim idle), 16 bytes each, so one load
// instruction covers KPI = 64 / LPK rows in whole cache lines, and a chunk's
// K and V rows (SK keys, NI = SK / KPI <= NMAX instructions each) are all in
// flight before the first score is formed.  Scores: each lane's 16-byte dot
// product, summed over the row's LPK lanes.  PV: each lane accumulates p * V
// over its 16 bytes of the rows it loaded; the KPI row groups are summed at
// the end.  Same online softmax, index semantics and float32 accuracy as
// gather_fwd_kernel (accurate expf; only the order of float32 additions
// differs).  Loads are buffer loads with 32-bit offsets (BUF; a masked entry
// reads zeros without a fetch) unless a head's K or V spans 2 GiB.
// Where an L2 holds the keys that a head's rows list (xcd_ranges), XCD x takes
// a contiguous range of the waves, so it reads the K and V of a few heads:
// explicit lists bf16 B=2 H=8 L=4096 D=128 200 -> 185 us, float32 D=64 158 ->
// 151 us, the decode steps unchanged.
template <Elem E, int LPK, int NMAX, bool BUF, bool PATTERN>
__global__ __launch_bounds__(256, 2) void gather_rows_kernel(GatherArgs A) {
  __shared__ float sc_all[4][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  // (in ranges, XCD x = blockIdx % 8 taking a contiguous one, or in turn)
  const int wv = (int)(blockIdx.x & 7) * A.xcd_step + (int)(blockIdx.x >> 3) * A.block_step + wave;
  if (wv >= A.waves) return;  // whole wave leaves; no block-level barrier below
  const int bh = wv / A.q_len, r = wv % A.q_len;
  const int b = bh / A.H, h = bh % A.H;
  gather_one_row<E, LPK, NMAX, BUF, PATTERN>(A, b, h, r, sc_all[wave], lane);
}

// ---------------------------------------------------------------------------
// The naive path's attention weights (elastic_sparse_attention.py:669-674):
// weights[b, h, r, j] = softmax over the row's valid entries, times the
// entry's dropout factor, 0 for a masked entry, in q's type.  One wave per
// (batch, head, row), lane j one entry, from the forward's lse (natural
// log): p_j = exp(s_j - lse).
template <Elem E, bool PATTERN>
__global__ __launch_bounds__(256) void gather_weights_kernel(GatherArgs A) {
  using T = typename ElemT<E>::T;
  __shared__ float qs_all[4][256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = blockIdx.x * 4 + wave;
  const int h = blockIdx.y, b = blockIdx.z;
  if (r >= A.q_len) return;
  const int kvh = h / A.groups;
  const int D = A.D;
  float* qs = qs_all[wave];
  const T* qrow = (const T*)A.q + (int64_t)b * A.qsb + (int64_t)h * A.qsh + (int64_t)r * A.qss;
  for (int d = lane; d < D; d += 64) qs[d] = ElemT<E>::load(qrow + d);
  wave_sync_lds();
  const T* kbase = (const T*)A.k + (int64_t)b * A.ksb + (int64_t)kvh * A.ksh;
  RowEntries row;
  row.init<PATTERN>(A.src, h, r);
  const float lse = A.lse[(int64_t)b * A.lsb + (int64_t)h * A.lsh + r];
  T* wrow = (T*)A.weights + (int64_t)b * A.wsb + (int64_t)h * A.wsh + (int64_t)r * A.wss;
  const int w = A.src.w;
  for (int c0 = 0; c0 < w; c0 += 64) {
    const int j = c0 + lane;
    if (j >= w) break;
    bool valid = false;
    int64_t key = 0;
    row.entry<PATTERN>(A.src, h, r, j, valid, key);
    const bool in_range = key >= 0 && key < A.kv_len;
    float p = 0.f;
    if (valid) {
      const float s = in_range ? row_dot<E>(qs, kbase + key * A.kss, D) * A.sm_scale : 0.f;
      p = expf(s - lse) * drop_factor(A.drop, b, h, r, j, A.H, A.q_len, w);
    }
    if (row.bad_pos) p = __builtin_nanf("");
    ElemT<E>::store(wrow + j, p);
  }
}

// The cooperative kernel needs every Q, K, V and O row 16-byte aligned (bases,
// strides and head_dim).
bool rows_aligned16(const GatherArgs& a, int es) {
  const int64_t epl = 16 / es;
  if (a.D % epl != 0) return false;
  const void* ptrs[] = {a.q, a.k, a.v, a.o};
  for (const void* p : ptrs)
    if (((uintptr_t)p & 15) != 0) return false;
  const int64_t st[] = {a.qsb, a.qsh, a.qss, a.ksb, a.ksh, a.kss,
                        a.vsb, a.vsh, a.vss, a.osb, a.osh, a.oss};
  for (int64_t x : st)
    if (x % epl != 0) return false;
  return true;
}

// Whether each XCD takes a contiguous range of the waves, or all of them take
// every head's rows in turn: by the bytes of K and V that a head's rows list,
// its window over the keys (interpolation weight x kv_len; half of kv_len for
// explicit lists) or, for few rows, w keys a row.  Ranges against turns, inputs
// changing from call to call, float32 and bf16, D 64 .. 256, L 2048 .. 65536: up
// to 5 MB ranges 1-30% faster (float32 H=8 L=4096 D=128 layer 4 of 8 169 against
// 183 us; 64 rows of H=32/8 L=32768 11.8 against 18.9); beyond, where a head's
// keys overflow an XCD's L2, turns 3-64% faster (presumably because eight
// XCDs then miss the same keys at about the same time; H=8/2 L=32768 D=128 layer
// 4 1216 -> 992 us, H=2/1 L=65536 712 -> 658); at weight 1 past 32 MB, with
// hardly a key shared, ranges 3-13% faster again.
bool xcd_ranges(const GatherArgs& a, int es, bool pattern) {
  const double weight = pattern ? (double)a.src.pc.a : 0.5;
  const double window = std::max(weight * a.kv_len, (double)a.src.w);
  const double keys = std::min(window, (double)a.q_len * a.src.w);
  const double bytes = 2.0 * keys * a.D * es;
  return bytes <= 5e6 || (pattern && a.src.pc.a == 1.0f && bytes > 32e6);
}

template <Elem E, int LPK, int NMAX, bool BUF>
void launch_rows(const GatherArgs& a, unsigned blocks, bool pattern, hipStream_t stream) {
  if (pattern)
    gather_rows_kernel<E, LPK, NMAX, BUF, true><<<blocks, 256, 0, stream>>>(a);
  else
    gather_rows_kernel<E, LPK, NMAX, BUF, false><<<blocks, 256, 0, stream>>>(a);
}

// A grid of at most one wave per SIMD (1024) is bound by one wave's latency:
// there 16 row loads of K and of V are in flight (one row of 32 heads: 7.2
// against 7.6 us); larger ones take fwd_in_flight (4096 rows 24.5 -> 23.2 us).
template <Elem E, int LPK>
void launch_rows_lanes(const GatherArgs& a, unsigned blocks, bool buf, bool pattern,
                       hipStream_t stream) {
  constexpr int NF = fwd_in_flight<E, LPK>();
  if (!buf)
    launch_rows<E, LPK, NF, false>(a, blocks, pattern, stream);
  else if (a.waves <= 1024)
    launch_rows<E, LPK, 16, true>(a, blocks, pattern, stream);
  else
    launch_rows<E, LPK, NF, true>(a, blocks, pattern, stream);
}

template <Elem E>
void launch_gather_elem(const GatherArgs& a, bool pattern, hipStream_t stream) {
  // the cooperative kernel's one-dimensional grid: four waves per block,
  // within the 2^32 work-items of a dispatch
  const int64_t waves = (int64_t)a.B * a.H * a.q_len;
  const int64_t per_xcd = (waves + 31) / 32;  // blocks
  if (rows_aligned16(a, ElemT<E>::kBytes) && per_xcd * 8 * 256 <= (int64_t)UINT32_MAX) {
    GatherArgs c = a;
    c.waves = (int)waves;  // (< 2^26: the test above)
    const bool ranges = xcd_ranges(a, ElemT<E>::kBytes, pattern);
    c.xcd_step = ranges ? (int)per_xcd * 4 : 4;
    c.block_step = ranges ? 4 : 32;
    const int64_t ks = row_span(a.kv_len, a.kss, 1, 0, a.D, ElemT<E>::kBytes);
    const int64_t vs = row_span(a.kv_len, a.vss, 1, 0, a.D, ElemT<E>::kBytes);
    const bool buf = ks < kMaxSpan && vs < kMaxSpan;
    c.k_span = (int)ks;
    c.v_span = (int)vs;
    const unsigned blocks = (unsigned)(8 * per_xcd);
    // lanes per row: 8, 16, 32 or 64 of 16 bytes (lanes past head_dim idle)
    const int lanes = a.D / ElemT<E>::kPerChunk;
    if (lanes <= 8)
      launch_rows_lanes<E, 8>(c, blocks, buf, pattern, stream);
    else if (lanes <= 16)
      launch_rows_lanes<E, 16>(c, blocks, buf, pattern, stream);
    else if (lanes <= 32)
      launch_rows_lanes<E, 32>(c, blocks, buf, pattern, stream);
    else if constexpr (ElemT<E>::kPerChunk == 4)
      launch_rows_lanes<E, 64>(c, blocks, buf, pattern, stream);
    return;
  }
  const dim3 grid((unsigned)((a.q_len + 3) / 4), (unsigned)a.H, (unsigned)a.B);
  if (pattern)
    gather_fwd_kernel<E, true><<<grid, 256, 0, stream>>>(a);
  else
    gather_fwd_kernel<E, false><<<grid, 256, 0, stream>>>(a);
}

template <Elem E>
void launch_weights_elem(const GatherArgs& a, bool pattern, hipStream_t stream) {
  dim3 grid((unsigned)((a.q_len + 3) / 4), (unsigned)a.H, (unsigned)a.B);
  if (pattern)
    gather_weights_kernel<E, true><<<grid, 256, 0, stream>>>(a);
  else
    gather_weights_kernel<E, false><<<grid, 256, 0, stream>>>(a);
}

}  // namespace

hipError_t launch_gather_fwd(const GatherArgs& a, bool pattern, hipStream_t stream) {
  if (a.q_len <= 0 || a.B <= 0 || a.H <= 0) return hipSuccess;
  switch ((Elem)a.elem) {
    case Elem::f32: launch_gather_elem<Elem::f32>(a, pattern, stream); break;
    case Elem::bf16: launch_gather_elem<Elem::bf16>(a, pattern, stream); break;
    default: launch_gather_elem<Elem::f16>(a, pattern, stream); break;
  }
  return hipGetLastError();
}

hipError_t launch_gather_weights(const GatherArgs& a, bool pattern, hipStream_t stream) {
  if (a.q_len <= 0 || a.B <= 0 || a.H <= 0) return hipSuccess;
  switch ((Elem)a.elem) {
    case Elem::f32: launch_weights_elem<Elem::f32>(a, pattern, stream); break;
    case Elem::bf16: launch_weights_elem<Elem::bf16>(a, pattern, stream); break;
    default: launch_weights_elem<Elem::f16>(a, pattern, stream); break;
  }
  return hipGetLastError();
}

}  // namespace esa
