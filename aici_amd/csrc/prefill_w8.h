// The prefill kernel of eight wavefronts, and its form with four, as a function of the workgroup's number and its LDS: the kernel of the
// varlen entry points (prefill_varlen.hip) and that of a whole step's attention (step_attn.hip) are built around it.  Device
// code; included by those two.
#pragma once

#include "prefill_common.h"

// The global -> LDS copies below set M0 inside inline asm and say so in their clobber lists, so that the
// compiler never assumes a value of its own survives them.  M0 is a register the compiler reserves, and
// naming a reserved register there draws a warning per use; the declaration is wanted all the same.
#pragma clang diagnostic ignored "-Winline-asm"

namespace hipattn {

namespace {

constexpr int BN = 64;  // keys per LDS tile

// ---------------------------------------------------------------------------
// Kernel of eight wavefronts for head sizes up to 128 (its form with four: NW below).  512 threads own 256 query rows (32 per wavefront) and run
// two wavefronts per SIMD within 256 registers each: every accumulator lives in a vector register the vector
// ALU can touch directly.  Three forms (MODE below) differ in how the 64-key tiles reach LDS and in the loop:
//   rows of k / v and block images of the paged cache: global -> LDS copies (no staging registers) into five
//     stages; the two wavefronts of a SIMD alternate between blocks of MFMAs and blocks of softmax, half a
//     period apart, one barrier per period.  K lies in LDS as block images [16-byte run][16 tokens], V as rows
//     (read with ds_read_b64_tr_b16) or, from the cache, as the [d][16 tokens] images that ds_read_b128 takes;
//   staged (paged cache, head sizes below 32 or on request): tiles through registers into three padded stages
//     (TileW8 below: K rows and V^T rows), one software-pipelined loop per wavefront.
// NW = 4: workgroups of four wavefronts, three to a compute unit (two at head sizes above 96, by their registers), so that every SIMD has
// a wavefront of each.  The alternation of the two pipes is left to chance; what it gains is that a workgroup's set-up and wind-down (block
// ids, Q, the first tile; the output) pass while the others work.  Same tiles, same order of the same operations: a row has the same bits
// in either form, so the form may follow the sizes of the whole batch (four_wavefronts_pay).  Tiles of 32 keys, which let three
// workgroups on a compute unit at head size 128 too (64 x 30..300 tokens 67 -> 60 us, 32 / 8 heads), give other last bits: not kept.  Three
// with tiles of 64 (one place for the values, a second barrier, 168 registers) keep part of Q in scratch memory: 67 -> 86 us.
// ---------------------------------------------------------------------------
// Where the eight-wavefront kernel takes its K/V tiles from.
enum { W8_ROWS = 0, W8_PAGED = 1, W8_PAGED_DMA = 2, W8_PAGED_DMA_PART = 3 };

// STEP: what else a launch holds.  Nothing, or (step_attn.hip) workgroups of paged decode in front or behind, and a row block's keys dealt out to up
// to n_parts workgroups: piece i takes tiles [i part_tiles, (i + 1) part_tiles), the last one the rest, and where a row block has more
// than one they leave sums, maximum and accumulators for the launch behind to merge.
struct PrefillAlone {
  typedef PrefillParams Params;
  static constexpr bool value = false;
};

// Wavefronts per SIMD and places for tiles in LDS of the forms with eight and four wavefronts.
constexpr int w8_wavefronts(int hdp, int nw) { return nw == 4 && hdp <= 96 ? 3 : 2; }
constexpr int w8_stages(int hdp, int nw) { return nw == 8 ? 5 : hdp <= 64 ? 3 : 2; }

// LDS geometry of the staged form.
template <int HDP>
struct TileW8 {
  static constexpr int KSTR = HDP + 8;   // K rows: key-major, +16 B
  static constexpr int VTSTR = BN + 8;   // V^T rows: head-element-major, 64 keys + 16 B
  static constexpr int K_ELEMS = BN * KSTR;
  static constexpr int V_ELEMS = HDP * VTSTR;
  static constexpr int STAGE_ELEMS = K_ELEMS + V_ELEMS;
  static constexpr size_t LDS_BYTES = 3 * (size_t)STAGE_ELEMS * 2;
};

template <typename T, int HDP, int MODE, typename STEP, int NW>
__global__ __launch_bounds__(NW * 64, STEP::value ? 2 : w8_wavefronts(HDP, NW)) void prefill_varlen_w8_kernel(typename STEP::Params p) {
  typedef typename Vec8<T>::type vec8;
  typedef TileW8<HDP> TL;
  constexpr bool PAGED = MODE != W8_ROWS;
  constexpr bool ROWS = MODE == W8_ROWS;
  constexpr bool DMA = MODE == W8_PAGED_DMA || MODE == W8_PAGED_DMA_PART;
  // W8_ROWS: K tiles are copied global -> LDS into the layout of the cache's block images (16-byte runs of a
  // row of k are the images' units, so a lane address per run is all it takes); V tiles are copied as the
  // rows they are and the second product reads its operands from them with the transposing LDS read.  Both
  // forms run the alternating MFMA / softmax blocks.
  constexpr bool KIMG = DMA || ROWS;      // K tiles lie in LDS as block images
  constexpr bool PINGPONG = DMA || ROWS;
  static_assert(NW == 8 || (NW == 4 && PINGPONG), "eight wavefronts, or four without staged tiles");
  // W8_PAGED_DMA_PART: head sizes below HDP (Phi-2's 80 in the 96-wide instance).  An image then fills only the
  // first d / HDP of its place in LDS; the rest is cleared once, so the contraction steps and output rows past d
  // work on zeros.
  constexpr bool DMA_PART = MODE == W8_PAGED_DMA_PART;
  // W8_PAGED_DMA keeps a tile as the four block images of the cache, unpadded.
  // Block images and rows: five stages (all of the 160 KB at head size 128) and one barrier per tile, with four wavefronts three or two
  // (48 KB, 64 at head sizes above 96); staged: three.  No tile is padded; where reads would collide, runs change places within their
  // row (see v_rows_dma).
  constexpr int NST = PINGPONG ? w8_stages(HDP, NW) : 3;
  constexpr int K_ELEMS = KIMG ? BN * HDP : TL::K_ELEMS;
  constexpr int STAGE_ELEMS = PINGPONG ? 2 * BN * HDP : K_ELEMS + TL::V_ELEMS;
  constexpr int KSTEPS = HDP / 16;
  constexpr int NDT = HDP / 32;
  constexpr int CPR = HDP / 8;                // 16-byte chunks per K row
  constexpr int K_CHUNKS = BN * CPR;          // per tile
  constexpr int NLOADK = (K_CHUNKS + 511) / 512;

  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  T *smem = reinterpret_cast<T *>(smem_raw);

  if constexpr (STEP::value) {
    const unsigned wg = blockIdx.x - (unsigned)p.decode_at;
    if (wg < (unsigned)p.decode_wgs) {
      STEP::decode(p, (int)wg, smem_raw);
      return;
    }
    // Ahead of the decode wavefronts on the same SIMD, which wait for memory whoever goes first (24 decode rows beside 718 new tokens, 32 / 8
    // heads x 128: 60 -> 51 us; 40 rows 84 -> 74).
    __builtin_amdgcn_s_setprio(3);
  }
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int g = lane >> 5;
  const int c = lane & 31;
  // The workgroup's eight wavefronts cover 2^hl query heads that share a kv head (and so the K/V tiles in
  // LDS) times 8 >> hl groups of 32 query rows.  With several heads per workgroup all wavefronts sit at
  // about the same rows, reach the diagonal of the causal mask together and skip the same tiles.
  const int hl = p.wg_heads_log2;
  const int BM = (NW * 32) >> hl;

  // Workgroups in launch order: query head fastest (the heads of a kv group land on one XCD and share its
  // L2), then the row blocks of a sequence, last rows -- the longest stretch of keys under the causal mask --
  // first, then the sequence: a sequence's row blocks run at the same time and find its keys in L2 (against
  // sequence-fastest order: -1.5 % on 8 x 4096 self-attention, -2.8 % on 512-row chunks over 8192 cached keys).
  int id = blockIdx.x, part = 0;
  if constexpr (STEP::value) id -= id >= p.decode_at ? p.decode_wgs : 0;
  const int n_slots = p.Hq >> hl;
  const int slot = id % n_slots;
  id /= n_slots;
  if constexpr (STEP::value) {
    part = id % p.n_parts;
    id /= p.n_parts;
  }
  const int b = id / p.n_qblocks;
  const int qb = p.n_qblocks - 1 - id % p.n_qblocks;
  const int head0 = ((slot % p.Hkv) * (p.G >> hl) + slot / p.Hkv) << hl;  // first query head of the workgroup
  const int h = head0 + (wave & ((1 << hl) - 1));
  const int kvh = head0 / p.G;

  const int q_begin = p.cu_q[b];
  const int Lq = p.cu_q[b + 1] - q_begin;
  const int k_begin = PAGED ? 0 : p.cu_k[b];
  int Lk = PAGED ? p.context_lens[b] : p.cu_k[b + 1] - k_begin;
  if (!PAGED && p.seqused_k) Lk = min(Lk, p.seqused_k[b]);
  const int wg_row0 = qb * BM;
  if (wg_row0 >= Lq) return;
  int off = Lk - Lq;
  const int wg_last_row = min(wg_row0 + BM, Lq) - 1;
  int kmax = p.causal ? min(Lk, wg_last_row + off + 1) : Lk;
  if (kmax < 0) kmax = 0;
  int n_tiles = (kmax + BN - 1) / BN;
  int first_tile = 0;
  bool whole = true;  // this workgroup sees all keys of its rows
  if constexpr (STEP::value) {
    whole = p.n_parts == 1 || n_tiles <= p.part_tiles;
    first_tile = part * p.part_tiles;
    if (part > 0 && first_tile >= n_tiles) return;
    n_tiles -= first_tile;
    if (part < p.n_parts - 1) n_tiles = min(n_tiles, p.part_tiles);  // (the last piece: whatever lies beyond the caller's bound, too)
    Lk -= first_tile * BN;  // keys are counted from the piece's first one on
    off -= first_tile * BN;
  }
  // Wavefronts w and w + 4 share a SIMD.  Under the causal mask a wavefront's work grows with its rows'
  // position in the block, so with one head per workgroup the two of a SIMD take row groups (w, 7 - w):
  // every SIMD gets the same sum.
  const int row_group = hl == 0 ? (wave < 4 ? wave : 11 - wave) : wave >> hl;  // (four wavefronts: one per SIMD)
  const int wave_row0 = wg_row0 + row_group * 32;
  const int wave_last_row = wave_row0 + 31;

  const T *qp = static_cast<const T *>(p.q) + (int64_t)q_begin * p.q_row + (int64_t)h * p.q_head;
  const T *kp = static_cast<const T *>(p.k) + (PAGED ? (int64_t)kvh * p.kc_head : (int64_t)k_begin * p.k_row + (int64_t)kvh * p.k_head);
  const T *vp = static_cast<const T *>(p.v) + (PAGED ? (int64_t)kvh * p.vc_head : (int64_t)k_begin * p.v_row + (int64_t)kvh * p.v_head);
  const int d_chunks = p.d / 8;

  // Q operands: lane (g, c) holds q[row c][16 ks + 8 g .. + 8] for every contraction step ks.  Read in
  // that shape an instruction touches 32 bytes of 32 rows; instead the rows are read whole (16 lanes x
  // 16 bytes per row, 4 rows per instruction) and turned through a private piece of LDS buffers 1 and 2,
  // which no tile reaches before the first barrier.  With four wavefronts, whose stages leave less room, only head sizes above 96 do so,
  // half of the columns at a time through the place of the values of tile 1, without padding (runs change places instead).  us, operand
  // shape / turned: 32 / 8 heads of 128, 64 x 30..300 tokens 70 / 67, 32 x 1024 395 / 373, 1 x 8000 522 / 496; at 80, where a half row is not
  // whole lines, turned 66 -> 78, at 64 +-1 %.
  constexpr int QSTR = HDP + 8;  // row pitch of the turned Q tile, elements
  // The alternating-block forms turn Q through stages 2.., so that tiles 0 and 1 can be on their way meanwhile.
  constexpr int Q_STAGE0 = PINGPONG && NST > 2 ? 2 : 1;
  constexpr bool Q_VIA_LDS = NW == 4 ? HDP == 128 : (size_t)NW * 32 * QSTR <= (size_t)(NST - Q_STAGE0) * STAGE_ELEMS;
  constexpr int Q_PARTS = NW == 4 && Q_VIA_LDS ? 2 : 1;
  constexpr int CPRQ = HDP / 8 / Q_PARTS;          // 16-byte runs of a row in a part
  constexpr int NQL1 = (32 * CPRQ + 63) / 64;      // loads per part
  constexpr int NQL = Q_PARTS * NQL1;
  vec8 qreg[KSTEPS];
  u32x4_t qraw[Q_VIA_LDS ? NQL : 1];
  // The loads of Q (the workgroup's longest wait: nothing else has touched these rows) ...
  auto q_issue = [&]() {
    if constexpr (Q_VIA_LDS) {
#pragma unroll
      for (int it = 0; it < NQL; it++) {
        const int idx = min(it % NQL1 * 64 + lane, 32 * CPRQ - 1);
        const int r = idx / CPRQ, ch = idx % CPRQ + it / NQL1 * CPRQ;
        const int row = min(wave_row0 + r, Lq - 1);
        qraw[it] = u32x4_t{0u, 0u, 0u, 0u};
        // (Q is read once and the output written once: with the non-temporal hint they do not displace the
        // K / V tiles that the other row blocks of the sequence are about to fetch from L2 -- 8 x 4096 tokens
        // 1.066 -> 1.051 ms from rows, 1.040 -> 1.019 ms from the paged cache; 16 x 1024 tokens 193 -> 188 us.  Not
        // with four wavefronts: 64 x 30..300 tokens 67 -> 73 us, 128 x 256 188 -> 178)
        if (ch < d_chunks) {
          const u32x4_t *run = reinterpret_cast<const u32x4_t *>(qp + (int64_t)row * p.q_row + ch * 8);
          qraw[it] = NW == 4 ? *run : __builtin_nontemporal_load(run);
        }
      }
    } else {
      const int row = min(wave_row0 + c, Lq - 1);
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ks++) {
        u32x4_t raw = {0u, 0u, 0u, 0u};
        const int ch = 2 * ks + g;
        if (ch < d_chunks) raw = *reinterpret_cast<const u32x4_t *>(qp + (int64_t)row * p.q_row + ch * 8);
        qreg[ks] = bit_cast<vec8>(raw);
      }
    }
  };
  // ... and their way through LDS into the operand registers.
  auto q_finish = [&]() {
    if constexpr (NW == 4 && Q_VIA_LDS) {
      T *qst = smem + Q_STAGE0 * STAGE_ELEMS + K_ELEMS + wave * (32 * CPRQ * 8);
#pragma unroll
      for (int part = 0; part < Q_PARTS; part++) {
#pragma unroll
        for (int it = 0; it < NQL1; it++) {
          const int idx = it * 64 + lane, r = idx / CPRQ, ch = idx % CPRQ;
          *reinterpret_cast<u32x4_t *>(qst + (r * CPRQ + (ch ^ (r & 7))) * 8) = qraw[part * NQL1 + it];
        }
#pragma unroll
        for (int ks = 0; ks < KSTEPS / Q_PARTS; ks++)
          qreg[part * (KSTEPS / Q_PARTS) + ks] = *reinterpret_cast<const vec8 *>(qst + (c * CPRQ + ((2 * ks + g) ^ (c & 7))) * 8);
      }
    } else if constexpr (Q_VIA_LDS) {
      T *qst = smem + Q_STAGE0 * STAGE_ELEMS + wave * (32 * QSTR);
#pragma unroll
      for (int it = 0; it < NQL; it++) {
        const int idx = it * 64 + lane;
        if ((32 * CPRQ) % 64 == 0 || idx < 32 * CPRQ)
          *reinterpret_cast<u32x4_t *>(qst + (idx / CPRQ) * QSTR + (idx % CPRQ) * 8) = qraw[it];
      }
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ks++)
        qreg[ks] = *reinterpret_cast<const vec8 *>(qst + c * QSTR + (2 * ks + g) * 8);
    } else {
      // (a use the compiler sees: its wait for these loads belongs here, not in front of every tile's first product)
#pragma unroll
      for (int ks = 0; ks < KSTEPS; ks++) asm volatile("" : "+v"(qreg[ks]));
    }
  };
  auto load_q = [&]() {
    q_issue();
    q_finish();
  };
  f32x16_t acc[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; dt++)
#pragma unroll
    for (int i = 0; i < 16; i++) acc[dt][i] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  // ---- tile staging ---------------------------------------------------------
  u32x4_t kst[NLOADK];
  // PAGED: blocks of the cache instead of rows of k / v.  A tile is 4 blocks; threads follow the cache's
  // own order so that consecutive lanes read consecutive 16-byte runs: K unit u = (block, chunk c8,
  // token) is the run [c8][token] of its block and lands in LDS row 16*block + token; V unit u = (block,
  // head element, half) is 8 tokens of the cache's [d][token] row -- already transposed.
  constexpr int K_PER_BLOCK = CPR * 16;            // 16-byte K runs per block
  constexpr int V_PER_BLOCK = HDP * 2;             // 16-byte V runs per block
  constexpr int NLOADVP = (4 * V_PER_BLOCK + 511) / 512;
  u32x4_t vstp[PAGED ? NLOADVP : 1];
  int staged_k0 = 0;  // first key of the tile held in the staging registers
  const int32_t *table_row = PAGED ? p.block_tables + (int64_t)b * p.table_stride : nullptr;
  if constexpr (STEP::value) table_row += first_tile * (BN / 16);
  // The block ids of 64 table columns (16 tiles) sit one per lane (columns past the context repeat its
  // last one), and a tile's four ids are lane reads into scalar registers: no tile waits for a table
  // read.  The next group is asked for one tile before it is needed and the ids are clamped to the cache
  // where they are used, so that nothing waits for the read where it is issued.
  int tbl_cur = 0, tbl_nxt = 0;
  auto load_ids = [&](int group) -> int {
    const int last_col = min((Lk - 1) >> 4, p.table_cols - first_tile * (BN / 16) - 1);
    return table_row[max(min(group * 64 + lane, last_col), 0)];
  };
  auto block_id = [&](int idx) -> int64_t {
    const int blk = __builtin_amdgcn_readlane(tbl_cur, idx);
    return blk < 0 ? 0 : (blk >= p.num_blocks ? p.num_blocks - 1 : (int64_t)blk);
  };
  // After a tile's ids are read: the last but one tile of a group asks for the next group's ids, the last
  // one switches to them.
  auto next_ids = [&](int tile) {
    if ((tile & 15) == 14) tbl_nxt = load_ids((tile >> 4) + 1);
    if ((tile & 15) == 15) tbl_cur = tbl_nxt;
  };
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  auto load_tile_paged = [&](int tile) {
    const int k0 = tile * BN;
    staged_k0 = k0;
    const int slot = tile & 15;
    // A wavefront's 64 runs lie in one block (a block has 2 HDP runs of K and of V), so the block's
    // address is scalar and the lane adds its run.  Blocks past the context re-read the last one
    // (their keys are masked, their V runs cleared before they reach LDS).
#pragma unroll
    for (int i = 0; i < NLOADK; i++) {
      const int ub = min(wave_u * 64 + 512 * i, K_CHUNKS - 64);
      const int r = ub / K_PER_BLOCK, rem = ub % K_PER_BLOCK + lane;
      const int c8 = min(rem / 16, d_chunks - 1), tok = rem % 16;
      const int64_t bs = block_id(slot * 4 + r);
      const char *base = reinterpret_cast<const char *>(kp + bs * p.kc_block);
      kst[i] = *reinterpret_cast<const u32x4_t *>(base + (uint32_t)((c8 * 16 + tok) * 8 * (int)sizeof(T)));
    }
#pragma unroll
    for (int i = 0; i < NLOADVP; i++) {
      const int ub = min(wave_u * 64 + 512 * i, 4 * V_PER_BLOCK - 64);
      const int r = ub / V_PER_BLOCK, rem = ub % V_PER_BLOCK + lane;
      const int drow = min(rem / 2, p.d - 1), half = rem % 2;
      const int64_t bs = block_id(slot * 4 + r);
      const char *base = reinterpret_cast<const char *>(vp + bs * p.vc_block);
      vstp[i] = *reinterpret_cast<const u32x4_t *>(base + (uint32_t)((drow * 16 + half * 8) * (int)sizeof(T)));
    }
    next_ids(tile);
  };
  // W8_PAGED_DMA (d == HDP): the tile's blocks go from the cache into LDS as they are, 1 KiB per
  // instruction (lane l's 16 bytes land at M0 + 16 l), no staging registers and no LDS writes.  A block of
  // one kv head is HDP * 32 contiguous bytes of K and as many of V.  Wavefront w copies one such image per
  // tile: K (w even) or V (w odd) of block w / 2, as HDP / 32 pieces.  K pieces keep the cache's order; in
  // a V piece (32 rows x 16 tokens) lane l fetches tokens 8 (l / 32) .. + 8 of row l % 32.  What sits one
  // per lane here is the byte offset of the block in this wavefront's cache, so that a tile costs two lane
  // reads and an add.
  constexpr int BLK_ELEMS = HDP * 16;
  constexpr int NDMA = HDP / 32;  // instructions per wavefront and tile
  const unsigned lds0 = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)smem_raw;
  constexpr int IMG = 8 / NW;  // images per wavefront: one, or K and V of block w
  auto dma_v = [&](int im) { return IMG == 1 ? wave_u & 1 : im; };
  const int dma_r = IMG == 1 ? wave_u >> 1 : wave_u;
  unsigned dma_lane[IMG];
  const char *dma_base[IMG];
  int64_t dma_blk_bytes[IMG];
  // The last piece of an image that is shorter than HDP: K lanes past the image's last 16-byte run and V
  // lanes whose row lies past d fetch nothing (what lies there belongs to the next head or block).
  const int dma_tail = p.d - 32 * (NDMA - 1);  // head elements in the last piece, 32 when d == HDP
  bool dma_last_ok[IMG];
  int64_t tbl_off[IMG];
#pragma unroll
  for (int im = 0; im < IMG; im++) {
    dma_lane[im] = dma_v(im) ? c * 32 + g * 16 : lane * 16;
    dma_base[im] = reinterpret_cast<const char *>(dma_v(im) ? vp : kp);
    dma_blk_bytes[im] = (dma_v(im) ? p.vc_block : p.kc_block) * (int64_t)sizeof(T);
    dma_last_ok[im] = !DMA_PART || (dma_v(im) ? c < dma_tail : lane < 2 * dma_tail);
    tbl_off[im] = 0;
  }
  auto id_to_offset = [&](int blk, int im) -> int64_t {
    const int64_t bid = blk < 0 ? 0 : (blk >= p.num_blocks ? p.num_blocks - 1 : (int64_t)blk);
    return bid * dma_blk_bytes[im];
  };
  auto dma_piece = [&](int tile, int i, int im) {
    const int idx = (tile & 15) * 4 + dma_r;
    const unsigned lo = __builtin_amdgcn_readlane((int)(uint32_t)tbl_off[im], idx);
    const unsigned hi = __builtin_amdgcn_readlane((int)(uint32_t)(tbl_off[im] >> 32), idx);
    // (an "s" operand is not made a scalar for the asm when the compiler holds the value in vector registers)
    const uint64_t src_v = reinterpret_cast<uint64_t>(dma_base[im]) + (((uint64_t)hi << 32) | lo);
    const char *src = reinterpret_cast<const char *>(
        ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(src_v >> 32)) << 32) |
        (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)src_v));
    // the instruction's offset field moves both ends of the copy: the address in memory and the one in LDS
    const unsigned dst = (unsigned)__builtin_amdgcn_readfirstlane(
        (int)(lds0 + (unsigned)(((tile % NST) * STAGE_ELEMS + dma_v(im) * K_ELEMS + dma_r * BLK_ELEMS) * (int)sizeof(T))));
#define HA_DMA_PIECE(OFF)                                                                          \
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:" #OFF \
               :                                                                                   \
               : "s"(dst), "v"(dma_lane[im]), "s"(src)                                                 \
               : "memory", "m0")
    if (!DMA_PART || i < NDMA - 1 || dma_last_ok[im]) {
      switch (i) {
        case 0: HA_DMA_PIECE(0); break;
        case 1: HA_DMA_PIECE(1024); break;
        case 2: HA_DMA_PIECE(2048); break;
        default: HA_DMA_PIECE(3072); break;
      }
    }
#undef HA_DMA_PIECE
    if (NST == 2 && i == NDMA - 1) {
      // (K's image is one tile ahead of V's: the ids that are asked for with the one are still there when the other turns to them)
      if (im == 0 && (tile & 15) == 14) tbl_nxt = load_ids((tile >> 4) + 1);
      if ((tile & 15) == 15) tbl_off[im] = id_to_offset(tbl_nxt, im);
    } else if (NST > 2 && i == NDMA - 1 && im == IMG - 1) {
      if ((tile & 15) == 14) tbl_nxt = load_ids((tile >> 4) + 1);
      if ((tile & 15) == 15) {
#pragma unroll
        for (int m = 0; m < IMG; m++) tbl_off[m] = id_to_offset(tbl_nxt, m);
      }
    }
  };
  auto dma_image = [&](int tile, int im) {
#pragma unroll
    for (int i = 0; i < NDMA; i++) dma_piece(tile, i, im);
  };
  auto dma_tile = [&](int tile) {
#pragma unroll
    for (int im = 0; im < IMG; im++) dma_image(tile, im);
  };
  // W8_PAGED_DMA_PART: clears what the images leave untouched in stages first..last: per block the K runs of
  // head elements d..HDP and, in the last V piece, the rows d..HDP of both 8-token halves.
  auto clear_image_tails = [&](int first, int last) {
    if constexpr (DMA_PART) {
      const int R = HDP - p.d;       // a multiple of 8 below 32
      const int per_stage = 16 * R;  // 16-byte runs: 4 blocks x (2 R of K + 2 R of V)
      for (int st = first; st <= last; st++)
        for (int idx = tid; idx < per_stage; idx += NW * 64) {
          const int r = idx / (4 * R), rem = idx % (4 * R);
          int e;
          if (rem < 2 * R) {
            e = r * BLK_ELEMS + (2 * p.d + rem) * 8;
          } else {
            const int v = rem - 2 * R;
            e = K_ELEMS + r * BLK_ELEMS + (NDMA - 1) * 512 + ((v / R) * 32 + (32 - R) + v % R) * 8;
          }
          *reinterpret_cast<u32x4_t *>(smem + st * STAGE_ELEMS + e) = u32x4_t{0u, 0u, 0u, 0u};
        }
    }
  };
  // Waits until this wavefront's pieces of `tile` have landed (`newer`: the pieces of the tile after it
  // were issued later and may still fly), then clears the V tokens past the context in them: stale
  // cache contents may be NaN, which a zero probability would not neutralise.
  auto dma_wait = [&](int tile, bool newer) {
    if (newer)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NDMA * IMG) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (dma_v(IMG - 1) && tile * BN + BN > Lk) {
      T *vs = smem + (tile % NST) * STAGE_ELEMS + K_ELEMS + dma_r * BLK_ELEMS;
      const int alive = Lk - (tile * BN + dma_r * 16 + g * 8);  // tokens of this lane's runs inside the context
      if (alive < 8) {
#pragma unroll
        for (int i = 0; i < NDMA; i++) {
          u32x4_t *run = reinterpret_cast<u32x4_t *>(vs + i * 512 + lane * 8);
          u32x4_t o = *run;
#pragma unroll
          for (int w = 0; w < 4; w++) {
            const int a2 = alive - 2 * w;
            o[w] &= a2 <= 0 ? 0u : (a2 == 1 ? 0xffffu : 0xffffffffu);
          }
          *run = o;
        }
      }
    }
  };
  // W8_ROWS, K: the tile goes global -> LDS in 1 KiB pieces, 4 x HDP / 32 of them, dealt round the
  // wavefronts.  Piece q is runs [4 pi .. 4 pi + 4) x 16 tokens of block r = q / (HDP / 32), pi = q %
  // (HDP / 32), of the image layout [run][token][8 elements]: lane l fetches run 4 pi + l / 16 of token
  // l % 16.  On a full tile the lane's offset is the same for every piece (the piece's own part is added to
  // the scalar base); only the last piece of a block clamps runs past d, and the last tile keys past Lk.
  constexpr int KPB = HDP / 32;   // pieces per block
  constexpr int KNP = 4 * KPB;    // pieces per tile
  const int kd_tok = lane & 15, kd_run = lane >> 4;
  const uint32_t kd_off = (uint32_t)(((int64_t)kd_tok * p.k_row + kd_run * 8) * (int64_t)sizeof(T));
  const uint32_t kd_off_last =
      (uint32_t)(((int64_t)kd_tok * p.k_row + (min(4 * (KPB - 1) + kd_run, d_chunks - 1) - 4 * (KPB - 1)) * 8) * (int64_t)sizeof(T));
  // The scalar side of a copy is kept short -- a wavefront issues its instructions in order, and every scalar
  // instruction in front of a copy is time its vector block does not have: the base of the copies is the start
  // of the sequence's keys (one scalar pointer for the whole loop), a tile's and a piece's place go into the
  // lane's 32-bit byte offset (the host sends launches whose keys span more than that to the other kernel), and a
  // piece's place in LDS is its number times 1 KiB.
  constexpr int KW = (KNP + NW - 1) / NW;  // pieces per wavefront
  uint32_t k_off0[KW];
  if constexpr (ROWS) {
#pragma unroll
    for (int i = 0; i < KW; i++) {
      const int q = wave_u + NW * i, r = q / KPB, pi = q % KPB;
      k_off0[i] = (pi == KPB - 1 ? kd_off_last : kd_off) + (uint32_t)(((int64_t)16 * r * p.k_row + 32 * pi) * (int64_t)sizeof(T));
    }
  }
  const T *kp_u = uniform_ptr(kp);
  const T *vp_u = uniform_ptr(vp);
  const uint32_t k_tile_bytes = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((int64_t)BN * p.k_row * (int64_t)sizeof(T)));
  const uint32_t v_tile_bytes = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)((int64_t)BN * p.v_row * (int64_t)sizeof(T)));
  const unsigned lds_wave = (unsigned)__builtin_amdgcn_readfirstlane(
      (int)((unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)smem_raw + (unsigned)wave_u * 1024u));
  auto k_rows_dma = [&](int tile) {
    const int k0 = tile * BN;
    const unsigned dst0 = lds_wave + (unsigned)((tile % NST) * STAGE_ELEMS * (int)sizeof(T));
    const uint32_t tile_off = (uint32_t)tile * k_tile_bytes;
#pragma unroll
    for (int i = 0; i < KW; i++) {
      const int q = wave_u + NW * i;
      if (KNP % NW == 0 || q < KNP) {
        uint32_t off = k_off0[i] + tile_off;
        if (k0 + BN > Lk) {
          const int r = q / KPB, pi = q % KPB;
          int tok = kd_tok, run = kd_run;
          if constexpr (NW == 4 && HDP == 96) {  // (168 registers: the lane number through an opaque copy, as for the values below)
            int l2 = lane;
            asm volatile("" : "+v"(l2));
            tok = l2 & 15;
            run = l2 >> 4;
          }
          const int key = min(k0 + 16 * r + tok, Lk - 1);
          off = (uint32_t)(((int64_t)key * p.k_row + min(4 * pi + run, d_chunks - 1) * 8) * (int64_t)sizeof(T));
        }
        const unsigned dst = dst0 + (unsigned)i * (NW * 1024u);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(dst), "v"(off), "s"(kp_u)
                     : "memory", "m0");
      }
    }
  };
  // W8_ROWS, V: the tile's rows go global -> LDS as they are, [key][HDP elements], in 1 KiB pieces (64 16-byte
  // runs in row order) dealt round the wavefronts; the second product reads its operands from them with the
  // transposing LDS read.  For those reads to be free of bank conflicts -- one covers 64 bytes of each of 4
  // consecutive rows -- run c of row r lies at run c ^ vswz(r) of its row where the row pitch is a multiple of
  // 256 bytes (64-byte groups of runs change places, by the row's low bits); a lane's place in LDS is given by
  // the instruction, so it fetches the run that belongs there.  Runs past d fetch the last real one (rows of the
  // output nobody stores), keys past Lk the last real key (their probabilities are zero).
  constexpr int CPRV = HDP / 8;          // runs per row
  constexpr int VNP = BN * CPRV / 64;    // pieces per tile
  constexpr int VNPW = (VNP + NW - 1) / NW;  // ... per wavefront
  auto vswz = [](int r) -> int { return HDP == 128 ? (r & 3) << 2 : (HDP == 64 ? ((r >> 1) & 1) << 2 : 0); };
  uint32_t vd_off[VNPW];
  if constexpr (ROWS) {
#pragma unroll
    for (int i = 0; i < VNPW; i++) {
      const int u = (wave + NW * i) * 64 + lane;  // the lane's run of the tile, in LDS order
      const int r = u / CPRV, pc = u % CPRV;
      vd_off[i] = (uint32_t)(((int64_t)r * p.v_row + min(pc ^ vswz(r), d_chunks - 1) * 8) * (int64_t)sizeof(T));
    }
  }
  auto v_rows_dma = [&](int tile) {
    const int k0 = tile * BN;
    const unsigned dst0 = lds_wave + (unsigned)(((tile % NST) * STAGE_ELEMS + K_ELEMS) * (int)sizeof(T));
    const uint32_t tile_off = (uint32_t)tile * v_tile_bytes;
#pragma unroll
    for (int i = 0; i < VNPW; i++) {
      const int q = wave_u + NW * i;
      if (VNP % NW == 0 || q < VNP) {
        uint32_t off = vd_off[i] + tile_off;
        if (k0 + BN > Lk) {
          // (the lane number through an opaque copy: hoisted out of the loop, what is derived from it here
          // would hold registers that the loop does not have)
          int l2 = lane;
          asm volatile("" : "+v"(l2));
          const int u = q * 64 + l2;
          const int r = u / CPRV, pc = u % CPRV;
          off = (uint32_t)(((int64_t)min(k0 + r, Lk - 1) * p.v_row + min(pc ^ vswz(r), d_chunks - 1) * 8) * (int64_t)sizeof(T));
        }
        const unsigned dst = dst0 + (unsigned)i * (NW * 1024u);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                     :
                     : "s"(dst), "v"(off), "s"(vp_u)
                     : "memory", "m0");
      }
    }
  };
  auto load_tile = [&](int tile) { load_tile_paged(tile); };
  auto store_tile_paged = [&](int stage) {
    T *ks = smem + stage * STAGE_ELEMS;
    T *vs = ks + K_ELEMS;
#pragma unroll
    for (int i = 0; i < NLOADK; i++) {
      const int u = tid + 512 * i;
      if (K_CHUNKS % 512 == 0 || u < K_CHUNKS) {
        const int r = u / K_PER_BLOCK, rem = u % K_PER_BLOCK;
        *reinterpret_cast<u32x4_t *>(ks + (r * 16 + rem % 16) * TL::KSTR + (rem / 16) * 8) = kst[i];
      }
    }
#pragma unroll
    for (int i = 0; i < NLOADVP; i++) {
      const int u = tid + 512 * i;
      if ((4 * V_PER_BLOCK) % 512 == 0 || u < 4 * V_PER_BLOCK) {
        const int r = u / V_PER_BLOCK, rem = u % V_PER_BLOCK;
        const int drow = rem / 2, half = rem % 2;
        u32x4_t o = vstp[i];
        // Cache tokens past the context hold whatever was there before (possibly NaN, which a zero
        // probability would not neutralise): clear them.
        if (staged_k0 + BN > Lk) {
          const int alive = Lk - (staged_k0 + r * 16 + half * 8);  // keys of this run inside the context
#pragma unroll
          for (int w = 0; w < 4; w++) {
            const int a2 = alive - 2 * w;
            o[w] &= a2 <= 0 ? 0u : (a2 == 1 ? 0xffffu : 0xffffffffu);
          }
        }
        // the run's two groups of 4 keys: groups (2 half, 2 half + 1) of block r -> positions 8 half, 8 half + 4
        // in the order the MFMA operand wants them: [g(8) a(4) b] from [a(8) g(4) b]
        T *row = vs + drow * TL::VTSTR + r * 16;
        *reinterpret_cast<u32x2_t *>(row + half * 4) = u32x2_t{o[0], o[1]};
        *reinterpret_cast<u32x2_t *>(row + 8 + half * 4) = u32x2_t{o[2], o[3]};
      }
    }
  };
  auto store_tile = [&](int stage) { store_tile_paged(stage); };

  // A workgroup has the compute unit to itself, so what it waits for here nobody fills: the loads of Q go
  // out first (nothing else has touched these rows: the longest wait), the block ids and tiles 0 and 1
  // behind them, and Q is turned through stages 2.. while the tiles fly.
  if constexpr (PINGPONG) q_issue();
  if (PAGED && n_tiles > 0) tbl_cur = load_ids(0);
  if constexpr (DMA) {
#pragma unroll
    for (int im = 0; im < IMG; im++) tbl_off[im] = id_to_offset(tbl_cur, im);
    if (n_tiles > 0) dma_tile(0);
    if (n_tiles > 1) {
      if constexpr (NST == 2)
        dma_image(1, 0);
      else
        dma_tile(1);
    }
    clear_image_tails(0, Q_STAGE0 - 1);
    q_finish();
    if (n_tiles > 0) dma_wait(0, NST > 2 && n_tiles > 1);
    __syncthreads();
    if (NST > 3 && n_tiles > 2) dma_tile(2);
    clear_image_tails(Q_STAGE0, NST - 1);  // seen by all after the barrier in front of the loop
  } else if constexpr (ROWS) {
    if (n_tiles > 0) {
      k_rows_dma(0);
      v_rows_dma(0);
    }
    if (n_tiles > 1) {
      k_rows_dma(1);
      if (NST > 2) v_rows_dma(1);
    }
    q_finish();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (NST > 3 && n_tiles > 2) {
      k_rows_dma(2);
      v_rows_dma(2);
    }
  } else {
    if (n_tiles > 0) load_tile(0);
    load_q();
    if (n_tiles > 0) {
      store_tile(0);
      if (n_tiles > 1) load_tile(1);
    }
    __syncthreads();
  }

  // Operand reads.  Staged tiles: K rows and V^T rows with 16 bytes of padding.  Block images: lane c is
  // MFMA row m = [a1 a0 g' b1 b0] and reads token [g' a0 b1 b0] of block a1 of its 32-key half, so that the
  // 8 scores a lane holds for one P.V step belong to 8 consecutive tokens of one block -- the order in which
  // a V row lies in the cache.  Sixteen consecutive lanes then read one whole 256-byte run [chunk][16
  // tokens] of K, and the 32 lanes of a half-wavefront 512 consecutive bytes of V (the DMA places the two
  // 8-token halves of 32 rows one after the other): no padding is needed.
  const int k_lane_off = KIMG ? (c >> 4) * (HDP * 16) + g * 128 + (((c >> 2) & 1) * 8 + ((c >> 3) & 1) * 4 + (c & 3)) * 8
                              : c * TL::KSTR + g * 8;
  const int v_lane_off = DMA ? g * 256 + c * 8 : c * TL::VTSTR + g * 8;
  // W8_ROWS: the transposing read hands lane (g, rh, li) head element 16 rh + li of the 4 keys whose rows its
  // 16-lane group addresses -- source lane s gives 8 bytes of row s / 4: elements 4 (s % 4) .. + 4 of the
  // 16 -- so two reads, at rows 8 g + s / 4 and 4 further, make the 8 keys of a P.V operand.  Element offset
  // of the lane's 8 bytes for output tile dt, first 16-key step:
  int vtr_off[NDT];
#pragma unroll
  for (int dt = 0; dt < NDT; dt++) {
    const int li = lane & 15, rh = (lane >> 4) & 1, r = 8 * g + (li >> 2);
    vtr_off[dt] = r * HDP + ((dt * 4 + 2 * rh + ((li & 3) >> 1)) ^ vswz(r)) * 8 + 4 * (li & 1);
  }
  constexpr int K_HALF = KIMG ? 2 * HDP * 16 : 32 * TL::KSTR;  // elements between the two 32-key halves of a K tile
  constexpr int K_STEP = KIMG ? 256 : 16;                      // ... between contraction steps (16 head elements)
  const f32x16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};

  // S^T = K . Q^T of one tile on its own (used for tile 0): both 32-key halves,
  // LDS reads two contraction steps ahead of the MFMAs that consume them.
  auto phase_qk = [&](int buf, f32x16_t(&s)[2]) {
    const T *ks_base = smem + buf * STAGE_ELEMS;
    auto rd = [&](int kt, int ks) -> vec8 {
      return *reinterpret_cast<const vec8 *>(ks_base + k_lane_off + kt * K_HALF + ks * K_STEP);
    };
    if constexpr (NW == 4 && HDP == 96) {
      // (168 registers: three operands ahead, one at a time, are what fits)
      vec8 kb[4];
#pragma unroll
      for (int n = 0; n < 3; n++) kb[n] = rd(n & 1, n >> 1);
#pragma unroll
      for (int n = 0; n < 2 * KSTEPS; n++) {
        if (n + 3 < 2 * KSTEPS) kb[(n + 3) % 4] = rd((n + 3) & 1, (n + 3) >> 1);
        __builtin_amdgcn_sched_barrier(0);
        s[n & 1] = Mfma32<T>::run(kb[n % 4], qreg[n >> 1], n < 2 ? zero : s[n & 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
      return;
    }
    vec8 ka[3][2];
    ka[0][0] = rd(0, 0);
    ka[0][1] = rd(1, 0);
    if (KSTEPS > 1) {
      ka[1][0] = rd(0, 1);
      ka[1][1] = rd(1, 1);
    }
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) {
      if (ks + 2 < KSTEPS) {
        ka[(ks + 2) % 3][0] = rd(0, ks + 2);
        ka[(ks + 2) % 3][1] = rd(1, ks + 2);
      }
      __builtin_amdgcn_sched_barrier(0);
      s[0] = Mfma32<T>::run(ka[ks % 3][0], qreg[ks], ks == 0 ? zero : s[0]);
      s[1] = Mfma32<T>::run(ka[ks % 3][1], qreg[ks], ks == 0 ? zero : s[1]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Tiles entirely past the diagonal of every row of this wavefront are skipped.
  auto skip_tile = [&](int j) { return (wave_row0 >= Lq) || (p.causal && j * BN > wave_last_row + off); };

  // ---- the pipelined tile loop (staged tiles; block images run the alternating blocks further down) ----
  // Iteration j of a wavefront: the matrix pipe computes S(j+1) = K(j+1).Q^T while
  // the vector ALU turns S(j) into probabilities -- one MFMA is issued, then the
  // few softmax instructions that fit in its shadow, and so on -- then P(j).V(j)
  // runs with the staging of tile j+2 (registers -> LDS) and the loads of tile
  // j+3 in its shadow.  Three LDS buffers: iteration j reads K of (j+1)%3 and V
  // of j%3 and writes (j+2)%3; one barrier per iteration.
  constexpr int NQ = 2 * KSTEPS;   // MFMAs of one S tile: step n = (contraction step n/2, key half n%2)
  constexpr int MAXS = NQ / 4;     // of which the first MAXS shadow the row maximum,
  constexpr int EXPS = NQ - MAXS;  // the rest the exponentials
  constexpr int QK_DEPTH = 3;      // K operands read ahead of their MFMA

  // DO_QK: S(j+1) is wanted (written to sn); the softmax of S(j) (in s) always runs.
  auto qk_softmax = [&](auto do_qk, int j, f32x16_t(&s)[2], f32x16_t(&sn)[2], vec8(&pk)[2][2]) {
    constexpr bool DO_QK = decltype(do_qk)::value;
    const int k0 = j * BN;
    const T *ks_base = smem + ((j + 1) % NST) * STAGE_ELEMS;
    auto rd = [&](int n) -> vec8 {
      return *reinterpret_cast<const vec8 *>(ks_base + k_lane_off + (n & 1) * K_HALF + (n >> 1) * K_STEP);
    };
    vec8 ka[QK_DEPTH + 1];
    if (DO_QK) {
#pragma unroll
      for (int n = 0; n < QK_DEPTH && n < NQ; n++) ka[n] = rd(n);
    }
    auto qk_step = [&](int n) {
      if (DO_QK) {
        if (n + QK_DEPTH < NQ) ka[(n + QK_DEPTH) % (QK_DEPTH + 1)] = rd(n + QK_DEPTH);
        __builtin_amdgcn_sched_barrier(0);
        sn[n & 1] = Mfma32<T>::run(ka[n % (QK_DEPTH + 1)], qreg[n >> 1], (n >> 1) == 0 ? zero : sn[n & 1]);
        __builtin_amdgcn_sched_barrier(0);
      }
    };

    const bool need_mask = (k0 + BN > Lk) || (p.causal && k0 + BN - 1 > wave_row0 + off);
    if (need_mask) {
      const int row = wave_row0 + c;
      int limit = p.causal ? row + off : Lk - 1;
      limit = min(limit, Lk - 1);
#pragma unroll
      for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int i = 0; i < 16; i++) {
          const int key = KIMG ? k0 + kt * 32 + ((i >> 3) & 1) * 16 + g * 8 + ((i >> 2) & 1) * 4 + (i & 3)
                               : k0 + kt * 32 + (i >> 2) * 8 + g * 4 + (i & 3);
          if (key > limit) s[kt][i] = -INFINITY;
        }
    }
    // row maximum in the shadow of the first MAXS MFMAs
    float mx = fmaxf(s[0][0], s[1][0]);
#pragma unroll
    for (int n = 0; n < MAXS; n++) {
      qk_step(n);
#pragma unroll
      for (int i = 16 * n / MAXS; i < 16 * (n + 1) / MAXS; i++)
        if (i > 0) mx = max3(mx, s[0][i], s[1][i]);
    }
    mx = max_across_halves(mx) * p.scale_log2;
    const bool grow = mx > m_run + p.rescale_thr;
    if (__builtin_expect(__any(grow), 0)) {
      const float m_new = grow ? mx : m_run;
      const float alpha = grow ? fast_exp2(m_run - m_new) : 1.0f;
      l_run *= alpha;
#pragma unroll
      for (int dt = 0; dt < NDT; dt++) acc[dt] *= alpha;
      m_run = m_new;
    }
    const float msub = m_run == -INFINITY ? 0.f : m_run;
    const float pmax = fast_exp2(mx - msub);
    float psum = g == 0 ? to_float(from_float<T>(pmax)) - pmax : 0.f;
    // exponentials in the shadow of the remaining MFMAs; value v = (key half, register)
#pragma unroll
    for (int n = 0; n < EXPS; n++) {
      qk_step(MAXS + n);
#pragma unroll
      for (int v = 32 * n / EXPS; v < 32 * (n + 1) / EXPS; v++) {
        const float e = fast_exp2(s[v / 16][v % 16] * p.scale_log2 - msub);
        psum += e;
        pk[v / 16][(v % 16) / 8][v % 8] = from_float<T>(e);
      }
    }
    l_run += psum;
  };

  constexpr int PV_STEPS = NDT * 4;
  f32x16_t s_a[2], s_b[2];
  if constexpr (PINGPONG) {
    // ---- block images and rows: the two wavefronts of a SIMD alternate between the matrix pipe and the vector ALU ----
    // A wavefront that issues MFMAs and vector instructions in turn has its vector instructions held up
    // behind every MFMA that waits for the pipe, and its SIMD mate, doing the same, does not fill the gaps
    // (measured with stamps: the older wavefront of a SIMD needed 3100 cycles per tile and then waited 1600
    // at the barrier for the younger one).  Here a wavefront runs pure blocks instead -- M(t): the 32 MFMAs of
    // P(t-1).V(t-1) and S(t); V(t): the softmax of S(t), then the wait for this wavefront's image of a later
    // tile and the copy of the next one -- and wavefronts 0-3 are half a period ahead of 4-7, so that on
    // every SIMD one wavefront is in an M block while the other is in a V block.
    //   Five stages leave two whole periods between a place becoming free and its tile being needed -- tile T
    // is read in periods T - 1 .. T + 1, its place is that of tile T - 5 -- so both groups wait for tile t + 2
    // and send tile t + 3 in V(t), and one barrier per period is enough (a barrier costs the eight wavefronts
    // some 200 cycles): the groups start a period together, wavefronts 0-3 with V(t), wavefronts 4-7 with
    // M(t), and swap in the middle.
    // Measured on 8 x 4096 tokens from the paged cache: 1.118 -> 1.058 ms with four stages and a barrier per
    // half period, 1.091 -> 1.075 ms from there to five stages and one barrier.
    vec8 pk[2][2];
    auto pv_images = [&](int j) {
      const T *vs_base = smem + (j % NST) * STAGE_ELEMS + K_ELEMS;
      // Step n = (contraction step n / NDT, output tile n % NDT): consecutive MFMAs go to different
      // accumulators, so none waits for the result of the one before it.
      if constexpr (DMA) {
        auto rd = [&](int n) -> vec8 {
          return *reinterpret_cast<const vec8 *>(vs_base + v_lane_off + (n / NDT) * (HDP * 16) + (n % NDT) * 512);
        };
        vec8 va[4];
#pragma unroll
        for (int n = 0; n < 3 && n < PV_STEPS; n++) va[n] = rd(n);
#pragma unroll
        for (int n = 0; n < PV_STEPS; n++) {
          if (n + 3 < PV_STEPS) va[(n + 3) % 4] = rd(n + 3);
          __builtin_amdgcn_sched_barrier(0);
          acc[n % NDT] = Mfma32<T>::run(va[n % 4], pk[(n / NDT) / 2][(n / NDT) % 2], acc[n % NDT]);
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
        // Rows: two transposing reads per operand, written as asm -- the builtin takes no offset, and a
        // register per address is 32 registers -- so the waits for them are written here too (the compiler
        // does not see these reads; what it waits for on its own account only ever waits longer).
        unsigned va_addr[NDT];
        const unsigned vs_lds = (unsigned)(size_t)(__attribute__((address_space(3))) unsigned char *)smem_raw +
                                (unsigned)(((j % NST) * STAGE_ELEMS + K_ELEMS) * (int)sizeof(T));
#pragma unroll
        for (int dt = 0; dt < NDT; dt++) va_addr[dt] = vs_lds + (unsigned)(vtr_off[dt] * (int)sizeof(T));
        u32x2_t lo[4], hi[4];
        auto rd = [&](int n) {
          constexpr int ROW4 = 4 * HDP * (int)sizeof(T);
          asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%3\n\tds_read_b64_tr_b16 %1, %2 offset:%4"
                       : "=&v"(lo[n % 4]), "=&v"(hi[n % 4])
                       : "v"(va_addr[n % NDT]), "n"((n / NDT) * 4 * ROW4), "n"((n / NDT) * 4 * ROW4 + ROW4)
                       : "memory");
        };
#pragma unroll
        for (int n = 0; n < 3 && n < PV_STEPS; n++) rd(n);
#pragma unroll
        for (int n = 0; n < PV_STEPS; n++) {
          if (n + 3 < PV_STEPS) {
            rd(n + 3);
            asm volatile("s_waitcnt lgkmcnt(6)" ::: "memory");
          } else {
            asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(2 * (PV_STEPS - 1 - n)) : "memory");
          }
          __builtin_amdgcn_sched_barrier(0);
          const u32x4_t av = {lo[n % 4][0], lo[n % 4][1], hi[n % 4][0], hi[n % 4][1]};
          acc[n % NDT] = Mfma32<T>::run(bit_cast<vec8>(av), pk[(n / NDT) / 2][(n / NDT) % 2], acc[n % NDT]);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    };
    auto send_keys = [&](int t) {
      if constexpr (DMA)
        dma_image(t, 0);
      else
        k_rows_dma(t);
    };
    auto send_values = [&](int t) {
      if constexpr (DMA)
        dma_image(t, IMG - 1);
      else
        v_rows_dma(t);
    };
    auto m_block = [&](int t) {
      if (t >= 1 && !skip_tile(t - 1)) pv_images(t - 1);
      if (t < n_tiles && !skip_tile(t)) phase_qk(t % NST, s_a);
    };
    // After the softmax: this wavefront's part of tile t + 2, sent a period ago, is waited for, and its part of
    // tile t + 3 follows.
    auto v_block = [&](int t) {
      if (!skip_tile(t)) qk_softmax(std::false_type{}, t, s_a, s_b, pk);
      if constexpr (DMA) {
        if (t + 2 < n_tiles) dma_wait(t + 2, false);
        if (t + 3 < n_tiles) dma_tile(t + 3);
      } else {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wavefront's pieces of tile t + 2
        if (t + 3 < n_tiles) {
          k_rows_dma(t + 3);
          v_rows_dma(t + 3);
        }
      }
    };
    if constexpr (NW == 4) {
      // Four wavefronts, one per SIMD, with other workgroups on the compute unit to fill the pipes.  A period sends a tile first of all
      // and ends when it is there.  Three places: tile j + 2 goes to that of tile j - 1.  Two: in period j the keys of tile j and the
      // values of tile j - 1 have been read for the last time, so the keys of tile j + 2 and the values of tile j + 1 take their places.
      constexpr int V_AHEAD = NST - 1;
      m_block(0);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (DMA && NST > 2 && n_tiles > 1) dma_wait(1, false);
      lds_barrier();
      asm volatile(".p2align 6");
      for (int j = 0; j < n_tiles; j++) {
        if (j + 2 < n_tiles) {
          send_keys(j + 2);
          if (V_AHEAD == 2) send_values(j + 2);
        }
        if (V_AHEAD == 1 && j + 1 < n_tiles) send_values(j + 1);
        if (!skip_tile(j)) qk_softmax(std::false_type{}, j, s_a, s_b, pk);
        m_block(j + 1);
        if (DMA && j + V_AHEAD < n_tiles) dma_wait(j + V_AHEAD, false);
        if (ROWS) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
      }
    } else {
      // The prologue has sent tiles 0, 1 and 2; tiles 0 and 1 have to be complete before the first period.
      const bool second_group = wave_u >= 4;
      if constexpr (DMA) {
        if (!second_group) m_block(0);
        if (n_tiles > 1) dma_wait(1, n_tiles > 2);
      } else {
        if (!second_group) m_block(0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // tiles 1 and 2
      }
      lds_barrier();
      if (!second_group) {
        // The loop starts on a 64-byte boundary: where it happens to fall otherwise moves the time of this
        // kernel by several per cent from one build to the next (1.09 against 1.03 ms on 8 x 4096 tokens for
        // the same instructions at another address).
        asm volatile(".p2align 6");
        for (int j = 0; j < n_tiles; j++) {
          v_block(j);
          m_block(j + 1);
          lds_barrier();
        }
        lds_barrier();  // the other group's last product still reads its tile
      } else {
        asm volatile(".p2align 6");
        for (int j = 0; j < n_tiles; j++) {
          m_block(j);
          v_block(j);
          lds_barrier();
        }
        m_block(n_tiles);
        lds_barrier();
      }
    }
  } else {
    // ---- staged tiles: one software-pipelined loop per wavefront ----
    // P(j).V(j) with the staging for later tiles in its shadow.
    auto pv_stage = [&](bool live, int j, vec8(&pk)[2][2]) {
      const T *vs_base = smem + (j % NST) * STAGE_ELEMS + K_ELEMS;
      // Step n = (contraction step n / NDT, output tile n % NDT): consecutive MFMAs go to different
      // accumulators, so none waits for the result of the one before it.
      auto rd = [&](int n) -> vec8 {
        const int dt = n % NDT, ks = n / NDT, kt = ks / 2, half = ks % 2;
        return *reinterpret_cast<const vec8 *>(vs_base + v_lane_off + dt * 32 * TL::VTSTR + kt * 32 + half * 16);
      };
      if (live) {
        vec8 va[4];
#pragma unroll
        for (int n = 0; n < 3 && n < PV_STEPS; n++) va[n] = rd(n);
#pragma unroll
        for (int n = 0; n < PV_STEPS; n++) {
          if (n + 3 < PV_STEPS) va[(n + 3) % 4] = rd(n + 3);
          __builtin_amdgcn_sched_barrier(0);
          acc[n % NDT] = Mfma32<T>::run(va[n % 4], pk[(n / NDT) / 2][(n / NDT) % 2], acc[n % NDT]);
          __builtin_amdgcn_sched_barrier(0);
          if (n == 1) {
            if (j + 2 < n_tiles) store_tile((j + 2) % 3);
            if (j + 3 < n_tiles) load_tile(j + 3);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      } else {
        if (j + 2 < n_tiles) store_tile((j + 2) % 3);
        if (j + 3 < n_tiles) load_tile(j + 3);
      }
    };

    // S(0) has nothing to hide behind; tile 1 is staged while it runs.
    if (n_tiles > 0 && !skip_tile(0)) phase_qk(0, s_a);
    if (n_tiles > 1) store_tile(1);
    if (n_tiles > 2) load_tile(2);
    lds_barrier();

    auto iteration = [&](int j, f32x16_t(&s)[2], f32x16_t(&sn)[2]) {
      const bool live = !skip_tile(j);
      const bool live_next = j + 1 < n_tiles && !skip_tile(j + 1);
      vec8 pk[2][2];
      if (live) {
        if (live_next)
          qk_softmax(std::true_type{}, j, s, sn, pk);
        else
          qk_softmax(std::false_type{}, j, s, sn, pk);
      }
      pv_stage(live, j, pk);
      lds_barrier();
    };
    for (int j = 0; j < n_tiles; j += 2) {
      iteration(j, s_a, s_b);
      if (j + 1 < n_tiles) iteration(j + 1, s_b, s_a);
    }
  }

  // ---- epilogue ---------------------------------------------------------------
  // The accumulators hold O^T: a lane has 4 consecutive head elements of one row per register quad,
  // which stored directly would be 16-byte pieces of 32 rows per instruction.  Each wavefront turns
  // its 32 x d tile through a private piece of LDS (the tiles are dead: every wavefront is past the
  // last barrier) and writes whole rows, 16 bytes per lane.
  const float l_tot = l_run + __shfl_xor(l_run, 32, 64);
  const float inv = l_tot > 0.f ? 1.0f / l_tot : 0.f;
  constexpr int OSTR = HDP + 8;  // row pitch of the turned tile, elements
  // The thread number passes through an empty asm: the addresses below are then computed here, after the
  // tile loop, instead of before it (where they would have to be kept, and spilled, across the loop).
  int tid_e = tid;
  asm volatile("" : "+v"(tid_e));
  const int lane_e = tid_e & 63, wave_e = tid_e >> 6;
  const int c_e = lane_e & 31, g_e = lane_e >> 5;
  const int hl_e = p.wg_heads_log2;
  const int wave_row0_e = wg_row0 + (hl_e == 0 ? (wave_e < 4 ? wave_e : 11 - wave_e) : wave_e >> hl_e) * 32;
  const int h_e = head0 + (wave_e & ((1 << hl_e) - 1));
  T *op = static_cast<T *>(p.out) + (int64_t)q_begin * p.o_row + (int64_t)h_e * p.o_head;
  T *ost = smem + wave_e * (32 * OSTR);
  if constexpr (STEP::value) {
    if (!whole) {
      const int row = wave_row0_e + c_e;
      if (row < Lq) {
        const int64_t at = ((int64_t)part * p.total_q + q_begin + row) * p.Hq + h_e;
#pragma unroll
        for (int dt = 0; dt < NDT; dt++)
#pragma unroll
          for (int a = 0; a < 4; a++) {
            const int dcol = dt * 32 + a * 8 + g_e * 4;
            f32x4_t r;
#pragma unroll
            for (int i = 0; i < 4; i++) r[i] = acc[dt][a * 4 + i];
            if (dcol < p.d) *reinterpret_cast<f32x4_t *>(p.part_acc + at * p.d + dcol) = r;
          }
        if (g_e == 0) *reinterpret_cast<float2 *>(p.part_ml + 2 * at) = make_float2(m_run, l_tot);
      }
      return;
    }
  }
  if (p.out_f32) {
    // the checking form of the output: straight from the accumulators, 16 bytes per lane
    float *op32 = static_cast<float *>(p.out) + (int64_t)q_begin * p.o_row + (int64_t)h_e * p.o_head;
    const int row = wave_row0_e + c_e;
    if (row < Lq) {
#pragma unroll
      for (int dt = 0; dt < NDT; dt++)
#pragma unroll
        for (int a = 0; a < 4; a++) {
          const int dcol = dt * 32 + a * 8 + g_e * 4;
          if (dcol < p.d) {
            f32x4_t r;
#pragma unroll
            for (int i = 0; i < 4; i++) r[i] = acc[dt][a * 4 + i] * inv;
            *reinterpret_cast<f32x4_t *>(op32 + (int64_t)row * p.o_row + dcol) = r;
          }
        }
    }
    if (p.lse != nullptr && g_e == 0 && row < Lq) {
      const float lse = l_tot > 0.f ? (m_run + __builtin_amdgcn_logf(l_tot)) * kLn2 : INFINITY;
      p.lse[((int64_t)b * p.Hq + h_e) * p.lse_pitch + row] = lse;
    }
    return;
  }
#pragma unroll
  for (int dt = 0; dt < NDT; dt++)
#pragma unroll
    for (int a = 0; a < 4; a++) {
      const int dcol = dt * 32 + a * 8 + g_e * 4;
      T r[4];
#pragma unroll
      for (int i = 0; i < 4; i++) r[i] = from_float<T>(acc[dt][a * 4 + i] * inv);
      *reinterpret_cast<u32x2_t *>(ost + c_e * OSTR + dcol) = *reinterpret_cast<u32x2_t *>(r);
    }
  constexpr int CPRO = HDP / 8;  // 16-byte chunks per row
#pragma unroll
  for (int it = 0; it < (32 * CPRO + 63) / 64; it++) {
    const int idx = it * 64 + lane_e;
    const int r = idx / CPRO, ch = idx % CPRO;
    const int row = wave_row0_e + r;
    if (((32 * CPRO) % 64 == 0 || r < 32) && row < Lq && ch < d_chunks)
      __builtin_nontemporal_store(*reinterpret_cast<const u32x4_t *>(ost + r * OSTR + ch * 8),
                                  reinterpret_cast<u32x4_t *>(op + (int64_t)row * p.o_row + ch * 8));
  }
  if (p.lse != nullptr && g_e == 0 && wave_row0_e + c_e < Lq) {
    const float lse = l_tot > 0.f ? (m_run + __builtin_amdgcn_logf(l_tot)) * kLn2 : INFINITY;
    p.lse[((int64_t)b * p.Hq + h_e) * p.lse_pitch + wave_row0_e + c_e] = lse;
  }
}

}  // namespace
}  // namespace hipattn
