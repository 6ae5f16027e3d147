// Paged decode in pieces that more than one kernel is built from: a block pair's loads and arithmetic, and the flat split of a step
// with the merge behind it as functions of the workgroup's number and its LDS -- the kernels of hipattn_paged_attention_*
// (paged_decode.hip) and that of a whole step's attention (step_attn.hip).  Device code; included by those two.
#pragma once

#include "common.h"
#include "device_types.h"

namespace hipattn {

constexpr int kBlockSize = 16;  // tokens per KV block handled by this kernel

struct DecodeParams {
  const void *q;
  int64_t q_stride;  // elements between sequences
  const void *kc;
  const void *vc;
  int64_t k_block_stride, k_head_stride, v_block_stride, v_head_stride;
  int64_t num_blocks;
  const int32_t *block_tables;
  int64_t max_blocks;  // row stride of block_tables
  int table_cols;      // columns of block_tables
  const int32_t *context_lens;
  const float *alibi;  // [Hq] or null
  float scale_log2;
  int Hq, Hkv, G;   // G = Hq / Hkv
  int col_groups;   // ceil(G / 16)
  int part_blocks;  // KV blocks per partition (even)
  int num_parts;
  int num_seqs;
  int waves;  // wavefronts per partition, 8 or the kernel's usual 4
  // split-K partials
  float *ws_acc;  // [S, Hq, P, HD]  (internal format)
  float *ws_m;    // [S, Hq, P]
  float *ws_l;    // [S, Hq, P]
  void *tmp_out;  // [S, Hq, P, HD] in T (reference v2 format)
  void *out;      // [S, Hq, HD]
  int64_t out_stride;
  int max_ctx;  // context lengths are clamped to this (the caller's max_context_len, at most what a table row holds)
  // flat split (paged_decode_flat_kernel)
  int *flat_prefix;  // [S + 1] block pairs before each sequence, written by workgroup 0
  int flat_waves;    // wavefronts of the main launch
  int flat_cols;   // query-head columns kept per partial slot: min(G, 16)
};

// What hipattn_paged_attention_v1 checks of its arguments and makes of them; false: nothing to do.
struct DecodeCall {
  const hipattn_tensor *query, *key_cache, *value_cache;
  int num_kv_heads;
  float scale;
  const hipattn_tensor *block_tables, *context_lens;
  int block_size, max_context_len;
  const hipattn_tensor *alibi;
  const char *op;
};
bool decode_params(const DecodeCall &c, hipattn_tensor *out, DecodeParams &p);
// Bytes of the library's scratch memory that hipattn_paged_attention_v1 takes for a call that decode_params has accepted.
size_t decode_scratch_bytes(const DecodeCall &c);

// Scratch memory of the flat split over `workgroups` workgroups: the prefix table of the block pairs, and behind it the partial results.
struct FlatScratch {
  int cols;  // query-head columns kept per partial result
  size_t prefix_bytes, slots, bytes;
};
FlatScratch flat_scratch(int64_t S, int G, int head_size, int workgroups);
void flat_scratch_set(DecodeParams &p, const FlatScratch &f, int workgroups, int head_size, char *ws);
// Block pairs of all sequences and kv heads at most, and whether the flat split can count them.
int64_t flat_units(int64_t S, int heads, int max_context_len);
bool flat_split_counts(int64_t S, int heads, int max_context_len);
// Whether a launch of decode rows alone would be one.
bool use_flat_split(int64_t S, int heads, int max_context_len);
// Compute units of the current device (asked of the runtime once).
int compute_units();

namespace {

template <typename T>
struct Mfma16;
template <>
struct Mfma16<half_t> {
  __device__ static __forceinline__ f32x4_t run(half8_t a, half8_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma16<bf16_t> {
  __device__ static __forceinline__ f32x4_t run(bf16x8_t a, bf16x8_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};

// A load of cache bytes.  Every byte of K and V is read once per launch and never again: the loads carry the
// non-temporal hint, so the lines are not kept in L2 and the memory-side cache at the expense of each other.
// Measured on MI355X, 64 sequences of 512..4096 tokens, 8 kv heads x 128: 120.8 -> 107.2 us per step.
template <typename V>
__device__ __forceinline__ V stream_load(const V *p) {
  return __builtin_nontemporal_load(p);
}

// The cache bytes of one block pair of one kv head, as MFMA operands.
template <int HD>
struct PairRegs {
  u32x4_t kra[(HD + 31) / 32], krb[(HD + 31) / 32];
  u32x2_t vra[HD / 16], vrb[HD / 16];
};

// Issues the loads of the block pair (pa, pb) of one kv head.
template <typename T, int HD>
__device__ __forceinline__ void pair_load(const DecodeParams &p, const T *kbase, const T *vbase, int64_t pa, int64_t pb,
                                          PairRegs<HD> &r) {
  constexpr int NCH = HD / 8;
  constexpr int NSTEP = (HD + 31) / 32;
  constexpr int NDT = HD / 16;
  const int lane = threadIdx.x & 63;
  const int kg = lane >> 4;
  const int col = lane & 15;
  const int64_t last_block = p.num_blocks - 1;
  pa = pa < 0 ? 0 : (pa > last_block ? last_block : pa);
  pb = pb < 0 ? 0 : (pb > last_block ? last_block : pb);
  const T *ka = kbase + pa * p.k_block_stride;
  const T *kb = kbase + pb * p.k_block_stride;
  const T *va = vbase + pa * p.v_block_stride;
  const T *vb = vbase + pb * p.v_block_stride;
  // K: step s of a block is the contiguous 1 KiB run of chunks 4s..4s+3.
#pragma unroll
  for (int s = 0; s < NSTEP; s++) {
    const int ch = 4 * s + kg;
    r.kra[s] = u32x4_t{0u, 0u, 0u, 0u};
    r.krb[s] = u32x4_t{0u, 0u, 0u, 0u};
    if (NCH % 4 == 0 || ch < NCH) {
      r.kra[s] = stream_load(reinterpret_cast<const u32x4_t *>(ka + (ch * kBlockSize + col) * 8));
      r.krb[s] = stream_load(reinterpret_cast<const u32x4_t *>(kb + (ch * kBlockSize + col) * 8));
    }
  }
  // V: tile dt of a block is the contiguous 512 B run of rows 16dt..16dt+15;
  // lane (kg, row) takes tokens 4kg..4kg+3 of its row.
#pragma unroll
  for (int dt = 0; dt < NDT; dt++) {
    r.vra[dt] = stream_load(reinterpret_cast<const u32x2_t *>(va + (dt * 16 + col) * kBlockSize + kg * 4));
    r.vrb[dt] = stream_load(reinterpret_cast<const u32x2_t *>(vb + (dt * 16 + col) * kBlockSize + kg * 4));
  }
}

// The same 32 tokens from caches with 8- or 32-token blocks, into the same registers: the kernels think in
// runs of 16 tokens ("blocks" below: what one MFMA tile of scores covers), and a pair of them is one
// 32-token block of the cache (id i0; its two halves) or four 8-token blocks (ids i0..i3; a lane's token
// says which one it reads).  Ids are clamped like those of pair_load: a pair's trailing ids may lie past
// the context, where the table holds anything; the tokens read through them are masked by the caller.
template <typename T, int HD, int BS>
__device__ __forceinline__ void pair_load_bs(const DecodeParams &p, const T *kbase, const T *vbase, int64_t i0, int64_t i1,
                                             int64_t i2, int64_t i3, PairRegs<HD> &r) {
  static_assert(BS == 8 || BS == 16 || BS == 32, "block sizes of the reference's support matrix");
  if constexpr (BS == 16) {
    pair_load<T, HD>(p, kbase, vbase, i0, i1, r);
  } else {
    constexpr int NCH = HD / 8;
    constexpr int NSTEP = (HD + 31) / 32;
    constexpr int NDT = HD / 16;
    const int lane = threadIdx.x & 63;
    const int kg = lane >> 4;
    const int col = lane & 15;
    const int64_t last_block = p.num_blocks - 1;
    auto clamp = [&](int64_t b) { return b < 0 ? (int64_t)0 : (b > last_block ? last_block : b); };
    const T *ka, *kb, *va, *vb;  // this lane's row of K (token col) and run of V (tokens 4kg..4kg+3) in each half
    if constexpr (BS == 32) {
      const int64_t b = clamp(i0);
      ka = kbase + b * p.k_block_stride + col * 8;
      kb = ka + 16 * 8;
      va = vbase + b * p.v_block_stride + kg * 4;
      vb = va + 16;
    } else {
      const int64_t ba = clamp(i0), bb = clamp(i1), bc = clamp(i2), bd = clamp(i3);
      ka = kbase + (col < 8 ? ba : bb) * p.k_block_stride + (col & 7) * 8;
      kb = kbase + (col < 8 ? bc : bd) * p.k_block_stride + (col & 7) * 8;
      va = vbase + (kg < 2 ? ba : bb) * p.v_block_stride + (kg & 1) * 4;
      vb = vbase + (kg < 2 ? bc : bd) * p.v_block_stride + (kg & 1) * 4;
    }
    // A load instruction reaches 4 KiB either side of its address register.  With 32-token blocks the steps of
    // a block lie 2 KiB apart and its tiles 1 KiB, so the lane addresses point 4 KiB into the block and the
    // steps and tiles are reached by constants on both sides: one address register per operand, as with
    // 16-token blocks (where everything lies within 4 KiB of the block's start).
    constexpr int BIAS = BS == 32 ? 2048 : 0;  // elements
    const T *kal = ka + kg * BS * 8 + BIAS, *kbl = kb + kg * BS * 8 + BIAS;
    const T *val = va + col * BS + BIAS, *vbl = vb + col * BS + BIAS;
#pragma unroll
    for (int s = 0; s < NSTEP; s++) {
      const int ch = 4 * s + kg;
      r.kra[s] = u32x4_t{0u, 0u, 0u, 0u};
      r.krb[s] = u32x4_t{0u, 0u, 0u, 0u};
      if (NCH % 4 == 0 || ch < NCH) {
        r.kra[s] = stream_load(reinterpret_cast<const u32x4_t *>(kal + (4 * s * BS * 8 - BIAS)));
        r.krb[s] = stream_load(reinterpret_cast<const u32x4_t *>(kbl + (4 * s * BS * 8 - BIAS)));
      }
    }
#pragma unroll
    for (int dt = 0; dt < NDT; dt++) {
      r.vra[dt] = stream_load(reinterpret_cast<const u32x2_t *>(val + (dt * 16 * BS - BIAS)));
      r.vrb[dt] = stream_load(reinterpret_cast<const u32x2_t *>(vbl + (dt * 16 * BS - BIAS)));
    }
  }
}

// Folds a loaded block pair -- blocks `blk` and `blk + 1` of the context, the
// second absent when !has_b -- into the running softmax state (m_run, l_run,
// acc).  qreg: lane (kg, col) holds q[head col][32*step + 8*kg .. +8].
template <typename T, int HD>
__device__ __forceinline__ void pair_compute(const DecodeParams &p, PairRegs<HD> &r, int blk, bool has_b, int ctx,
                                             float slope, const typename Vec8<T>::type (&qreg)[(HD + 31) / 32],
                                             float &m_run, float &l_run, f32x4_t (&acc)[HD / 16]) {
  typedef typename Vec8<T>::type vec8;
  constexpr int NSTEP = (HD + 31) / 32;
  constexpr int NDT = HD / 16;
  const int lane = threadIdx.x & 63;
  const int kg = lane >> 4;
  u32x4_t(&kra)[NSTEP] = r.kra;
  u32x4_t(&krb)[NSTEP] = r.krb;
  u32x2_t(&vra)[NDT] = r.vra;
  u32x2_t(&vrb)[NDT] = r.vrb;

  // S^T = K . Q^T : rows = tokens of the block, columns = query heads.
  f32x4_t sa = {0.f, 0.f, 0.f, 0.f}, sb = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < NSTEP; s++) {
    sa = Mfma16<T>::run(bit_cast<vec8>(kra[s]), qreg[s], sa);
    sb = Mfma16<T>::run(bit_cast<vec8>(krb[s]), qreg[s], sb);
  }

  // Lane (kg, col) now holds tokens 4kg..4kg+3 of both blocks for head col.
  const int tok_a = blk * kBlockSize + kg * 4;
  const int tok_b = has_b ? tok_a + kBlockSize : 0x3fffffff;
  float x[8];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    x[i] = sa[i] * p.scale_log2 + slope * (float)(tok_a + i - ctx + 1);
    x[4 + i] = sb[i] * p.scale_log2 + slope * (float)(tok_b + i - ctx + 1);
    if (tok_a + i >= ctx) x[i] = -INFINITY;
    if (tok_b + i >= ctx) x[4 + i] = -INFINITY;
  }
  float mx = fmaxf(fmaxf(fmaxf(x[0], x[1]), fmaxf(x[2], x[3])), fmaxf(fmaxf(x[4], x[5]), fmaxf(x[6], x[7])));
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  const float m_new = fmaxf(m_run, mx);
  const float m_safe = m_new == -INFINITY ? 0.f : m_new;
  const float alpha = fast_exp2(m_run - m_safe);
  float psum = 0.f;
  vec8 pv;
#pragma unroll
  for (int i = 0; i < 8; i++) {
    const float e = fast_exp2(x[i] - m_safe);
    psum += e;
    pv[i] = from_float<T>(e);
  }
  l_run = l_run * alpha + psum;
  m_run = m_new;
  if (__any(alpha != 1.0f)) {
#pragma unroll
    for (int dt = 0; dt < NDT; dt++) acc[dt] *= alpha;
  }

  // Tokens past the context hold whatever the cache held before; a zero
  // probability does not neutralise a NaN, so clear those V entries.
  if ((blk + 2) * kBlockSize > ctx || !has_b) {  // wave-uniform: only the context's last pair
#pragma unroll
    for (int dt = 0; dt < NDT; dt++) {
      uint16_t *ea = reinterpret_cast<uint16_t *>(&vra[dt]);
      uint16_t *eb = reinterpret_cast<uint16_t *>(&vrb[dt]);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if (tok_a + i >= ctx) ea[i] = 0;
        if (tok_b + i >= ctx) eb[i] = 0;
      }
    }
  }

  // O^T += V^T . P^T : contraction slot 8kg+j is token 4kg+j of block A
  // (j < 4) or token 4kg+j-4 of block B.
#pragma unroll
  for (int dt = 0; dt < NDT; dt++) {
    u32x4_t a = {vra[dt][0], vra[dt][1], vrb[dt][0], vrb[dt][1]};
    acc[dt] = Mfma16<T>::run(bit_cast<vec8>(a), pv, acc[dt]);
  }
}

// ---------------------------------------------------------------------------
// Flat split.  The launch above hands out (sequence, kv head, partition) items
// of unequal length, and every workgroup pays a chain of dependent loads
// (context length -> table -> cache) before its first byte streams.  Here the
// whole step is one list of units -- a unit is one block pair of one
// (sequence, kv head) segment, ordered sequence-major with the pair fastest --
// and the list is cut into equal contiguous ranges, one per wavefront of a
// launch sized to what the chip holds at once.  Every wavefront therefore
// streams the same number of bytes, starts once, and the launch drains
// together.  A range may begin inside a segment and end inside a later one, so
// a wavefront emits at most two partial results (slot 2w: the piece that
// begins where its range begins; slot 2w+1: a later piece cut by the range's
// end); segments that lie inside one range are normalised and written to
// `out` directly.  The reduce kernel recomputes which wavefronts cover a
// segment from the same arithmetic.
// ---------------------------------------------------------------------------
constexpr int kFlatMaxSeqs = 1024;

__device__ __forceinline__ int ctx_pairs(int ctx) {
  return ctx > 0 ? (ctx + 2 * kBlockSize - 1) / (2 * kBlockSize) : 0;
}

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// `units` cut into `waves` contiguous ranges whose lengths differ by at most
// one (the first `rem` ranges hold `base + 1` units).
struct FlatSplit {
  int base, rem;
  __device__ FlatSplit(int units, int waves) : base(units / waves), rem(units % waves) {}
  __device__ int start(int w) const { return w * base + min(w, rem); }
  __device__ int wave_of(int u) const {
    const int split = rem * (base + 1);
    return u < split ? u / (base + 1) : rem + (u - split) / base;
  }
};

template <int HD>
struct FlatLds {
  int ctx[kFlatMaxSeqs];
  int excl[kFlatMaxSeqs + 1];  // block pairs before sequence s; [S] = all
  int wsum[4];
  f32x4_t park[4][HD / 16][64];  // a wavefront's partial result waiting to be written (see below)
  float park_ml[4][2][64];
};

template <typename T, int HD, int BS>
__device__ __forceinline__ void decode_flat(const DecodeParams &p, const int wg, FlatLds<HD> &lds) {
  typedef typename Vec8<T>::type vec8;
  constexpr int NCH = HD / 8;
  constexpr int NSTEP = (HD + 31) / 32;
  constexpr int NDT = HD / 16;
  auto &s_ctx = lds.ctx;
  auto &s_excl = lds.excl;
  auto &s_wsum = lds.wsum;
  auto &s_park = lds.park;
  auto &s_park_ml = lds.park_ml;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int kg = lane >> 4;
  const int col = lane & 15;
  const int S = p.num_seqs;
  bool parked = false;

  // Exclusive prefix of the pair counts, thread t owning sequences 4t..4t+3.
  {
    int c[4], n[4], tsum = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int s = 4 * tid + j;
      c[j] = s < S ? min(p.context_lens[s], p.max_ctx) : 0;
      n[j] = ctx_pairs(c[j]);
      tsum += n[j];
    }
    int inc = tsum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(inc, o, 64);
      if (lane >= o) inc += t;
    }
    if (lane == 63) s_wsum[wave] = inc;
    __syncthreads();
    int run = inc - tsum;
    for (int k = 0; k < wave; k++) run += s_wsum[k];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int s = 4 * tid + j;
      if (s < S) {
        s_ctx[s] = c[j];
        s_excl[s] = run;
      }
      run += n[j];
    }
    if (tid == 0) s_excl[S] = s_wsum[0] + s_wsum[1] + s_wsum[2] + s_wsum[3];
    __syncthreads();
  }
  if (wg == 0) {
    for (int s = tid; s <= S; s += 256) p.flat_prefix[s] = s_excl[s];
  }

  const int hk = p.Hkv * p.col_groups;
  const int total_units = hk * uniform(s_excl[S]);  // the host bounds this below 2^31
  const FlatSplit split(total_units, p.flat_waves);
  const int w = wg * 4 + wave;
  const int u_first = split.start(w);
  const int u_end = split.start(w + 1);
  if (u_first >= u_end) return;

  // The sequence holding unit u_first: the first s with hk * pairs_before(s + 1) > u_first.
  int seq = 0;
  for (int s0 = 0; s0 < S; s0 += 64) {
    const int s = s0 + lane;
    const bool past = s < S && hk * s_excl[s + 1] > u_first;
    const unsigned long long b = __ballot(past);
    if (b) {
      seq = s0 + __ffsll(b) - 1;
      break;
    }
  }

  T *out = static_cast<T *>(p.out);
  int u = u_first;
  while (u < u_end) {
    const int before = uniform(s_excl[seq]);
    const int pairs = uniform(s_excl[seq + 1]) - before;
    if (pairs == 0) {  // u < total_units, so a longer sequence follows
      seq++;
      continue;
    }
    const int ctx = uniform(s_ctx[seq]);
    const int nblk = (ctx + kBlockSize - 1) / kBlockSize;
    const int r = u - hk * before;
    const int h = r / pairs;
    const int pr0 = r - h * pairs;
    const int n = min(pairs - pr0, u_end - u);
    const int kvh = h / p.col_groups;
    const int cg = h - kvh * p.col_groups;
    const int g_idx = cg * 16 + col;
    const bool col_ok = g_idx < p.G;
    const int qh = kvh * p.G + g_idx;

    vec8 qreg[NSTEP];
    {
      const T *qp = static_cast<const T *>(p.q) + seq * p.q_stride + (int64_t)qh * HD;
#pragma unroll
      for (int s = 0; s < NSTEP; s++) {
        const int ch = 4 * s + kg;
        u32x4_t raw = {0u, 0u, 0u, 0u};
        if (col_ok && ch < NCH) raw = *reinterpret_cast<const u32x4_t *>(qp + ch * 8);
        qreg[s] = bit_cast<vec8>(raw);
      }
    }
    const float slope = (p.alibi != nullptr && col_ok) ? p.alibi[qh] * kLog2e : 0.f;
    const T *kbase = static_cast<const T *>(p.kc) + (int64_t)kvh * p.k_head_stride;
    const T *vbase = static_cast<const T *>(p.vc) + (int64_t)kvh * p.v_head_stride;

    float m_run = -INFINITY, l_run = 0.f;
    f32x4_t acc[NDT];
#pragma unroll
    for (int dt = 0; dt < NDT; dt++) acc[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // The table entries of up to 32 pairs sit one per lane.
    for (int sp = 0; sp < n; sp += 32) {
      const int nsub = min(32, n - sp);
      const int b_first = 2 * (pr0 + sp);             // in runs of 16 tokens
      const int t_first = b_first * kBlockSize / BS;  // the table column of the first of them
      int tbl = 0;
      if (lane < 64 * kBlockSize / BS && t_first + lane < p.table_cols)
        tbl = p.block_tables[seq * p.max_blocks + t_first + lane];
      int tbl_hi = 0;  // 8-token blocks: 32 pairs span 128 columns
      if (BS == 8 && t_first + 64 + lane < p.table_cols) tbl_hi = p.block_tables[seq * p.max_blocks + t_first + 64 + lane];
      // Two register sets (heads up to 128 elements): the next pair's loads are
      // in flight while the current pair is folded in.
      auto issue = [&](int it, PairRegs<HD> &r) {
        if constexpr (BS == 16) {
          const bool has_b = b_first + 2 * it + 1 < nblk;
          const int64_t pa = __builtin_amdgcn_readlane(tbl, 2 * it);
          const int64_t pb = __builtin_amdgcn_readlane(tbl, has_b ? 2 * it + 1 : 2 * it);
          pair_load<T, HD>(p, kbase, vbase, pa, pb, r);
        } else if constexpr (BS == 32) {
          pair_load_bs<T, HD, BS>(p, kbase, vbase, __builtin_amdgcn_readlane(tbl, it), 0, 0, 0, r);
        } else {
          const int c = (4 * it) & 63;
          const int src = it < 16 ? tbl : tbl_hi;
          pair_load_bs<T, HD, BS>(p, kbase, vbase, __builtin_amdgcn_readlane(src, c), __builtin_amdgcn_readlane(src, c + 1),
                                  __builtin_amdgcn_readlane(src, c + 2), __builtin_amdgcn_readlane(src, c + 3), r);
        }
      };
      auto fold = [&](int it, PairRegs<HD> &r) {
        const int blk = b_first + 2 * it;
        pair_compute<T, HD>(p, r, blk, blk + 1 < nblk, ctx, slope, qreg, m_run, l_run, acc);
      };
      // The pairs of a batch are visited in bit-reversed order (of 32: 0, 16, 8, 24, 4, ...), not in the order of
      // the table; in a batch of fewer than 32 the largest power of two of them is, the rest follow in table order.
      // A sequence whose blocks lie in the pool in the order of their tokens -- what an allocator hands a fresh
      // prompt -- would otherwise be streamed with one constant stride by every wavefront at once, which the memory
      // system serves 5 % slower than scattered blocks (717 against 682 us on 128 x U[1k,16k] tokens; with this
      // order 670 us for either).  Which pair comes next is scalar arithmetic on the position in the batch -- the
      // same at every block size and in every launch, so results are too.
      const int pk = 31 - __builtin_clz((unsigned)nsub);  // the largest power of two within the batch
      auto pair_at = [&](int pos) -> int {
        return pos < (1 << pk) ? (int)((__builtin_bitreverse32((unsigned)pos) >> 1) >> (31 - pk)) : pos;
      };
      if (HD <= 128) {
        PairRegs<HD> ra, rb;
        issue(pair_at(0), ra);
        // the loop on a 256-byte boundary: 1 % on the whole step against where it happened to fall
        asm volatile(".p2align 8");
        for (int pos = 0; pos < nsub; pos += 2) {
          if (pos + 1 < nsub) issue(pair_at(pos + 1), rb);
          fold(pair_at(pos), ra);
          if (pos + 1 < nsub) {
            if (pos + 2 < nsub) issue(pair_at(pos + 2), ra);
            fold(pair_at(pos + 1), rb);
          }
        }
      } else {  // two register sets of 256-element heads do not fit
        for (int pos = 0; pos < nsub; pos++) {
          PairRegs<HD> ra;
          issue(pair_at(pos), ra);
          fold(pair_at(pos), ra);
        }
      }
    }

    float l_tot = l_run + __shfl_xor(l_run, 16, 64);
    l_tot += __shfl_xor(l_tot, 32, 64);
    if (col_ok) {
      if (pr0 == 0 && n == pairs) {
        const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
        T *op = out + seq * p.out_stride + (int64_t)qh * HD + kg * 4;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++) {
          T rr[4];
#pragma unroll
          for (int i = 0; i < 4; i++) rr[i] = from_float<T>(acc[dt][i] * inv);
          *reinterpret_cast<u32x2_t *>(op + dt * 16) = *reinterpret_cast<u32x2_t *>(rr);
        }
      } else if (u == u_first && u + n < u_end) {
          // The piece at the head of the range, with more of the range to stream after it: parked in LDS and
          // written out after the loop.  A store issued here would sit in the same in-order counter as the
          // loads that follow, and the first wait for those loads would also wait for the store to be
          // acknowledged (measured: 6.6 us of a 126 us step).
#pragma unroll
          for (int dt = 0; dt < NDT; dt++) s_park[wave][dt][lane] = acc[dt];
          s_park_ml[wave][0][lane] = m_run;
          s_park_ml[wave][1][lane] = l_tot;
          parked = true;
        } else {
          const int64_t pidx = (int64_t)(2 * w + (u != u_first ? 1 : 0)) * p.flat_cols + col;
          float *ap = p.ws_acc + pidx * HD + kg * 4;
#pragma unroll
          for (int dt = 0; dt < NDT; dt++) *reinterpret_cast<f32x4_t *>(ap + dt * 16) = acc[dt];
          if (kg == 0) {
            p.ws_m[pidx] = m_run;
            p.ws_l[pidx] = l_tot;
          }
        }
    }
    u += n;
    if (pr0 + n == pairs && h == hk - 1) seq++;
  }
  if (parked) {  // only lanes that hold a query head parked anything (slot 2w: the piece began the range)
    const int64_t pidx = (int64_t)(2 * w) * p.flat_cols + col;
    float *ap = p.ws_acc + pidx * HD + kg * 4;
#pragma unroll
    for (int dt = 0; dt < NDT; dt++) *reinterpret_cast<f32x4_t *>(ap + dt * 16) = s_park[wave][dt][lane];
    if (kg == 0) {
      p.ws_m[pidx] = s_park_ml[wave][0][lane];
      p.ws_l[pidx] = s_park_ml[wave][1][lane];
    }
  }
}

// Merge for the flat split, a workgroup of up to 128 threads per (query head, sequence).  The wavefronts that cover the
// segment of (sequence, kv head) follow from the unit arithmetic of the main
// kernel; a segment covered by one wavefront was already written.
template <typename T, int HD>
__device__ __forceinline__ void decode_flat_merge(const DecodeParams &p, const int qh, const int seq) {
  const int lane = threadIdx.x & 63;
  const int before = p.flat_prefix[seq];
  const int pairs = p.flat_prefix[seq + 1] - before;
  T *op = static_cast<T *>(p.out) + seq * p.out_stride + (int64_t)qh * HD;
  if (pairs == 0) {  // empty context: nobody else writes the row
    for (int d = threadIdx.x; d < HD; d += blockDim.x) op[d] = from_float<T>(0.f);
    return;
  }
  const int hk = p.Hkv * p.col_groups;
  const int total_units = hk * p.flat_prefix[p.num_seqs];
  const FlatSplit split(total_units, p.flat_waves);
  const int kvh = qh / p.G;
  const int g_idx = qh - kvh * p.G;
  const int h = kvh * p.col_groups + g_idx / 16;
  const int col = g_idx % 16;
  const int u0 = hk * before + h * pairs;
  const int w0 = split.wave_of(u0);
  const int w1 = split.wave_of(u0 + pairs - 1);
  if (w0 == w1) return;
  const int np = w1 - w0 + 1;
  const int first_odd = u0 > split.start(w0) ? 1 : 0;
  // slot of piece i: wavefront w0 + i; only the first piece can start inside its wavefront's range
  auto slot = [&](int i) -> int64_t { return (int64_t)(2 * (w0 + i) + (i == 0 ? first_odd : 0)) * p.flat_cols + col; };
  if (np <= 64) {
    // Lane i owns piece i's (max, sum); the first pieces' accumulator values are
    // requested before anything depends on them, so the kernel is two memory
    // round trips deep (prefix, then everything else).
    constexpr int NPRE = 8;
    const int d0 = threadIdx.x;
    float pre[NPRE];
#pragma unroll
    for (int i = 0; i < NPRE; i++) pre[i] = (i < np && d0 < HD) ? p.ws_acc[slot(i) * HD + d0] : 0.f;
    const float mi = lane < np ? p.ws_m[slot(lane)] : -INFINITY;
    const float li = lane < np ? p.ws_l[slot(lane)] : 0.f;
    float mmax = mi;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mmax = fmaxf(mmax, __shfl_xor(mmax, o, 64));
    const float wi = lane < np ? fast_exp2(mi - mmax) : 0.f;
    float denom = li * wi;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) denom += __shfl_xor(denom, o, 64);
    const float inv = denom > 0.f ? 1.0f / denom : 0.f;
    __shared__ float s_w[64];  // every wavefront computed the same weights; the first one publishes them
    if (threadIdx.x < 64) s_w[lane] = wi;
    __syncthreads();
    for (int d = d0; d < HD; d += blockDim.x) {
      float o = 0.f;
      if (d == d0) {
#pragma unroll
        for (int i = 0; i < NPRE; i++) o += pre[i] * s_w[i];
      } else {
        for (int i = 0; i < NPRE && i < np; i++) o += p.ws_acc[slot(i) * HD + d] * s_w[i];
      }
      for (int i = NPRE; i < np; i++) o += p.ws_acc[slot(i) * HD + d] * s_w[i];
      op[d] = from_float<T>(o * inv);
    }
    return;
  }
  float mmax = -INFINITY;
  for (int i = lane; i < np; i += 64) mmax = fmaxf(mmax, p.ws_m[slot(i)]);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mmax = fmaxf(mmax, __shfl_xor(mmax, o, 64));
  float denom = 0.f;
  for (int i = lane; i < np; i += 64) denom += p.ws_l[slot(i)] * fast_exp2(p.ws_m[slot(i)] - mmax);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) denom += __shfl_xor(denom, o, 64);
  const float inv = denom > 0.f ? 1.0f / denom : 0.f;
  for (int d = threadIdx.x; d < HD; d += blockDim.x) {
    float o = 0.f;
#pragma unroll 4
    for (int i = 0; i < np; i++) o += p.ws_acc[slot(i) * HD + d] * fast_exp2(p.ws_m[slot(i)] - mmax);
    op[d] = from_float<T>(o * inv);
  }
}

}  // namespace
}  // namespace hipattn
