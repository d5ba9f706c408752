// Prefill (variable-length, causal) attention for gfx950.
//
// Replaces flash_attn_varlen_func(q, k, v, max_seqlen_q, cu_seqlens_q, max_seqlen_k, cu_seqlens_k, softmax_scale,
// causal=True, block_table) as nano-vllm calls it for prefill (layers/attention.py:77-83): sequence b owns query
// tokens cu_seqlens_q[b] .. cu_seqlens_q[b+1]-1 of q [Tq, Hq, D] and key tokens 0 .. lk-1, lk = cu_seqlens_k[b+1] -
// cu_seqlens_k[b]; the keys are rows cu_seqlens_k[b] + j of k, v [Tk, Hkv, D], or, with a block table (prefix
// cache, model_runner.py:311-312), cache slot block_table[b][j / block_size] * block_size + j % block_size of the
// paged caches [num_blocks, block_size, Hkv, D]. Query i of a sequence with lq queries sees keys j <= lk - lq + i
// with causal (the mask aligned to the bottom right), all lk keys otherwise. Head h reads kv head h / (Hq / Hkv).
//
// One block (8 waves) per (query tile, sequence, pair of q heads of one kv head): 4 waves and 128 queries per head;
// when Hq / Hkv is odd, one head per block with 8 waves and 256 queries. Wave w of a head owns queries 32w .. 32w+31
// of the tile. The two heads share the K/V tiles (half the K/V traffic of a block per head). Per 64-key tile:
//   1. the K and V tiles go to LDS key-major ([64][D], 16-byte chunks, rows padded);
//   2. S^T [32 keys x 32 queries] = K Q^T per 32-key half with v_mfma_f32_32x32x16_bf16 (K rows from LDS as the A
//      operand, the wave's Q rows from registers as the B operand): lane l holds keys 8 (r / 4) + 4 (l / 32) + r % 4
//      (register r) of query l % 32, so one query's 64 scores sit in lanes l and l ^ 32;
//   3. fp32 online softmax in base 2 per query: the max of the raw scores, then p = 2^(s * scale * log2 e - m) in
//      one FMA and the hardware exp;
//   4. O^T [32 dims x 32 queries] += V^T P^T per 32-dim tile and 16-key step: P (bf16) stays in the registers it was
//      computed in as the B operand, whose 8 k slots of lane l are the keys 4 (l / 32) .. +3 and 8 + 4 (l / 32) ..
//      +3 of the step; the A operand gets the same keys of dim l % 32 from the key-major V tile with two gfx950
//      transpose reads (ds_read_b64_tr_b16, 4 keys each). Each lane keeps one query's O, so the rescale by
//      2^(m_old - m_new) is lane-local.
// A wave's 32 queries use each K and V fragment it reads from LDS twice as often as 16 would, which halves the LDS
// reads per flop; the per-tile work that does not scale with the queries (loads, LDS stores, barriers) is shared by
// twice the flops.
// P is rounded to bf16 for the P.V product (as flash-attn does) and the row sum adds the fp32 p (as flash-attn
// does); scores, softmax and O are fp32; output bf16. The softmax scale must be positive.
// Key splits (with a caller workspace): when the blocks of one pass leave CUs idle and the key ranges are long (a
// prompt chunk over its cached prefix: 2 query tiles x 8 head pairs = 16 blocks streaming thousands of keys each),
// each (query tile, sequence, head group) is cut into key ranges run by separate blocks; each writes its queries'
// (max, sum, O) records and prefill_combine merges them in split order.
#include <algorithm>

#include "decode_attention.h"

namespace nvhip {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kWavesBlock = 8;  // waves per block: 4 per head with two heads, 8 with one
constexpr int kBK = 64;   // keys per tile
constexpr int kThreads = 64 * kWavesBlock;
// queries per block and head (32 per wave)
__host__ __device__ constexpr int block_queries(int heads_per_block) { return 32 * kWavesBlock / heads_per_block; }

struct PrefillArgs {
  uint16_t* out;
  const uint16_t* q;
  const uint16_t* k;  // contiguous [Tk, Hkv, D] rows, or the k cache with a block table
  const uint16_t* v;
  const int32_t* cu_q;
  const int32_t* cu_k;
  const int32_t* bt;  // [num_seqs, max_blocks] or null
  int64_t q_st, q_sh, k_st, v_st, o_st, o_sh;
  int Hkv, G, bs, num_blocks, max_blocks;
  float scale_log2;  // softmax scale * log2(e), > 0
  int causal;
  int qtiles, nhg;  // query tiles per sequence (from max_seqlen_q), head groups (Hq / heads per block)
  int lq_skip;      // sequences with 1 .. lq_skip queries are left to the paged decode kernel
  int splits;       // key ranges per (query tile, sequence, head group): split s takes keys s * split_len ..
  int split_len;    // a multiple of kBK
  int Hq;
  int64_t ws_rows;  // Tq: query rows of one split's records
  // splits > 1: fp32 records merged by prefill_combine -- O [splits, Tq, Hq, D] (unnormalised), then (max, sum)
  // [splits, Tq, Hq, 2]
  float* ws;
  // dec_inline: the blocks of the short sequences (1 .. lq_skip queries) run their paged decode attention
  // themselves (one block per (sequence, kv head), dec: its varlen arguments, one split), concurrently with the
  // prefill tiles, instead of a separate launch before this one
  int dec_inline;
  // dec_extra > 0 (dec.halves): the short sequences' (sequence, kv head) pairs are cut in two; the blocks above
  // run the first halves, dec_extra blocks appended to the grid (one per pair of the call) the second halves
  int dec_extra;
  int plan;       // number of sequences (at most 64) when the blocks find their tile with block_plan, else 0
  int out_lines;  // out 16-byte aligned with strides in whole 16-byte pieces: the output goes out in whole lines
  DecodeArgs dec;
};

// fp32 elements of one (split, query, head) record: O[D] in the O array, max and row sum in the (max, sum) array.
__host__ __device__ constexpr int record_len(int D) { return D + 2; }

// Element offset of key j of sequence b, kv head kvh, in k (v with v_st): a contiguous row, or (PAGED) the cache
// slot of block blk (-1 if the block is not valid).
template <int D, bool PAGED>
__device__ __forceinline__ int64_t key_row(const PrefillArgs& g, int k0s, int j, int blk, int kvh, int64_t st) {
  if constexpr (!PAGED) return int64_t(k0s + j) * st + int64_t(kvh) * D;
  if (blk < 0 || blk >= g.num_blocks) return -1;
  return ((int64_t(blk) * g.bs + j % g.bs) * g.Hkv + kvh) * D;
}

// Which sequence and query tile block `item` of a ragged launch's (sequence, tile) pairs is, for calls of up to 64
// sequences: first the query tiles of the sequences that the prefill kernel takes, the latest (most keys) first across
// all of them, then the sequences left to the decode attention (tile -1), then nothing (false): what the grid, sized
// for the longest sequence, holds beyond that. Every wave computes it from the sequence bounds, one sequence per lane. Without
// it a mixed step's prompt chunk started behind the decode requests' blocks, its last tiles two rounds late, and the
// ends of a ragged batch's grid came between its tiles.
struct Plan {
  int b, qt, q0, lq, k0, lk;
};
__device__ __forceinline__ int nth_bit(uint64_t mask, int n) {  // position of set bit n (it exists)
  const int lane = threadIdx.x % 64;
  const int below = __builtin_amdgcn_mbcnt_hi(uint32_t(mask >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(mask), 0));
  return __builtin_ctzll(__ballot(((mask >> lane) & 1) != 0 && below == n));
}
template <int BQ>
__device__ __forceinline__ bool block_plan(const PrefillArgs& g, int item, Plan& p) {
  const int lane = threadIdx.x % 64;
  const bool in = lane < g.plan;
  const int q0 = in ? g.cu_q[lane] : 0, k0 = in ? g.cu_k[lane] : 0;
  const int lq = (in ? g.cu_q[lane + 1] : 0) - q0, lk = (in ? g.cu_k[lane + 1] : 0) - k0;
  const bool brief = lq >= 1 && lq <= g.lq_skip;
  const int tiles = brief ? 0 : min((lq + BQ - 1) / BQ, g.qtiles);  // < 256
  auto from = [&](int level) {  // tiles at or above this level, of all sequences: the bits of the lanes' counts
    const int n = max(tiles - level, 0);
    int sum = 0;
#pragma unroll
    for (int bit = 0; bit < 8; ++bit) sum += __builtin_popcountll(__ballot((n >> bit) & 1)) << bit;
    return sum;
  };
  const int total = from(0);
  uint64_t mask;
  int n;
  if (item < total) {
    int lo = 0, hi = g.qtiles;  // from(lo) > item >= from(hi)
    while (hi - lo > 1) {
      const int mid = (lo + hi) / 2;
      if (from(mid) > item) lo = mid;
      else hi = mid;
    }
    p.qt = lo;
    n = item - from(lo + 1);
    mask = __ballot(tiles > lo);
  } else {
    p.qt = -1;
    n = item - total;
    mask = __ballot(brief);
    if (n >= __builtin_popcountll(mask)) return false;
  }
  p.b = nth_bit(mask, n);
  p.q0 = __builtin_amdgcn_readlane(q0, p.b), p.lq = __builtin_amdgcn_readlane(lq, p.b);
  p.k0 = __builtin_amdgcn_readlane(k0, p.b), p.lk = __builtin_amdgcn_readlane(lk, p.b);
  return true;
}

// HB q heads of one kv head per block (4 waves each, sharing the K/V tiles in LDS). PLAN: the blocks find their tile with
// block_plan (its own instance: the code of both in one kernel cost small calls without it 0.3-0.5 us).
template <int D, bool PAGED, int HB, bool PLAN>
__global__ __launch_bounds__(kThreads) void prefill_attention_kernel(const PrefillArgs g) {
  constexpr int kBQ = block_queries(HB), kHeadThreads = kThreads / HB;
  constexpr int DC = D / 16;   // 16-wide dim steps of Q.K
  constexpr int DT = D / 32;   // 32-dim output tiles
  constexpr int CPR = D / 8;   // 16-byte chunks per K/V row
  constexpr int KP = D + 8;    // K row pitch (elements)
  // V row pitch: D + 32 elements puts the 4 rows of a transpose read 16 (or 48) banks apart, so the 32 lanes of a
  // half-wave (4 keys x 32 dims) hit 64 distinct banks
  constexpr int VP = D + 32;
  constexpr int STAGE = kBK * (KP + VP);  // elements of one LDS stage (K tile, then V tile)
  // LDS: two K/V tile stages, or (paged) the decode attention's buffers for the blocks of short sequences
  constexpr int DEC_BYTES = PAGED ? decode_lds_bytes(D, 16, false) : 0;
  constexpr int LDS_ELEMS = (2 * STAGE * 2 > DEC_BYTES ? 2 * STAGE * 2 : DEC_BYTES) / 2;
  __shared__ __attribute__((aligned(16))) uint16_t lds[LDS_ELEMS];

  // Block order. The ids are dealt round-robin over the 8 XCDs (block b runs on XCD b % 8) and each XCD starts its
  // blocks in id order as CUs free up. When the groups (sequence, head group) divide evenly, XCD x takes whole
  // groups -- all query tiles of a group read the same K/V, which then stays in one XCD's L2 -- namely groups x,
  // x + 8, x + 16, ..., so that every sequence's head groups are spread over the XCDs (contiguous ranges of groups
  // put a mixed step's prefill chunk, the batch's last sequence, on one XCD), and starts them heaviest query tile
  // (most keys) first across its groups, so that no long tile starts late (longest-first list scheduling; starting
  // one group's tiles before the next group's left a third of the CUs idle at the end of a 4 x 2048-token prefill).
  // Otherwise all groups' tiles are dealt heaviest first.
  // With key splits, the (query tile, split) pairs of a group are its tiles, heaviest (latest query tile, first
  // split) first.
  const int ntile = g.qtiles * g.splits;
  const int nblk = int(gridDim.x) - g.dec_extra, ngrp = nblk / ntile;
  if (int(blockIdx.x) >= nblk) {  // a second half of a short sequence's pair (the whole block: uniform)
    if constexpr (PAGED) {
      const int pair = int(blockIdx.x) - nblk;
      if (g.dec.bs % 32 == 0)
        decode_block<D, 16, true, false, true>(g.dec, 2 * pair + 1, reinterpret_cast<unsigned char*>(lds));
      else
        decode_block<D, 16, false, false, true>(g.dec, 2 * pair + 1, reinterpret_cast<unsigned char*>(lds));
    }
    return;
  }
  int b, hg, qt, split, q0s, lq, k0s, lk;
  if constexpr (PLAN) {  // (no key splits; the head groups divide evenly over the XCDs)
    const int sub = g.nhg / 8, r = blockIdx.x / 8;
    Plan p;
    if (!block_plan<kBQ>(g, r / sub, p)) return;
    hg = r % sub * 8 + int(blockIdx.x) % 8;
    b = p.b, qt = max(p.qt, 0), split = 0, q0s = p.q0, lq = p.lq, k0s = p.k0, lk = p.lk;
  } else {
    int grp, ci;
    if (nblk % 8 == 0 && (nblk / 8) % ntile == 0) {
      const int gx = nblk / 8 / ntile, r = blockIdx.x / 8;
      grp = (r % gx) * 8 + blockIdx.x % 8;
      ci = r / gx;
    } else {
      grp = blockIdx.x % ngrp;
      ci = blockIdx.x / ngrp;
    }
    qt = g.qtiles - 1 - ci / g.splits, split = ci % g.splits;
    b = grp / g.nhg, hg = grp % g.nhg;
    q0s = g.cu_q[b], lq = g.cu_q[b + 1] - q0s;
    k0s = g.cu_k[b], lk = g.cu_k[b + 1] - k0s;
  }
  const int h = hg * HB + int(threadIdx.x) / kHeadThreads, kvh = (hg * HB) / g.G;
  if (lq >= 1 && lq <= g.lq_skip) {  // the paged decode attention takes this sequence (the whole block: b is uniform)
    // one block per (sequence, kv head) runs the decode attention of the pair (the whole block: b, hg, qt uniform)
    if constexpr (PAGED) {
      if (g.dec_inline && (PLAN || qt == g.qtiles - 1) && split == 0 && (hg * HB) % g.G == 0) {
        const int pair = b * g.Hkv + hg * HB / g.G, bid = g.dec.halves ? 2 * pair : pair;
        if (g.dec.bs % 32 == 0) decode_block<D, 16, true, false, true>(g.dec, bid, reinterpret_cast<unsigned char*>(lds));
        else decode_block<D, 16, false, false, true>(g.dec, bid, reinterpret_cast<unsigned char*>(lds));
      }
    }
    return;
  }
  // keys [k_beg, k_stop) of this block: the split's range, cut at the last key its query tile sees
  const int k_beg = split * g.split_len;
  const int k_hi = split == g.splits - 1 ? INT32_MAX : k_beg + g.split_len;  // the last split takes the rest
  const int k_stop = g.causal ? min(min(lk, lk - lq + min(qt * kBQ + kBQ, lq)), k_hi) : min(lk, k_hi);
  if (qt * kBQ >= lq || k_stop <= k_beg) {
    // no keys for this block: zero rows (one pass), or records that say so (the merge then writes zeros)
    const int r = int(threadIdx.x) % kHeadThreads;
    if (qt * kBQ < lq && r < kBQ && qt * kBQ + r < lq) {
      const int64_t row = q0s + qt * kBQ + r;
      if (g.splits > 1) {
        if (row >= g.ws_rows) return;
        const int64_t rec = (int64_t(split) * g.ws_rows + row) * g.Hq + h;
        float* o = g.ws + rec * D;
        for (int d = 0; d < D; ++d) o[d] = 0.0f;
        *reinterpret_cast<f32x2*>(g.ws + int64_t(g.splits) * g.ws_rows * g.Hq * D + 2 * rec) = f32x2{-INFINITY, 0.0f};
      } else {
        uint16_t* o = g.out + row * g.o_st + int64_t(h) * g.o_sh;
        for (int d = 0; d < D; ++d) o[d] = 0;
      }
    }
    return;
  }
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane((tid % kHeadThreads) / 64);
  const int ql = lane % 32, hf = lane / 32;
  const int qi_lane = qt * kBQ + 32 * wave + ql;  // this lane's query (B operand column / O column)

  // Q rows of the wave as the B operand: lane l -> query 32 wave + l % 32, dims 16c + 8 (l / 32) .. +8
  bf16x8_t qf[DC];
  {
    const bool ok = qi_lane < lq;
    const uint16_t* qp = g.q + int64_t(q0s + (ok ? qi_lane : 0)) * g.q_st + int64_t(h) * g.q_sh + 8 * hf;
#pragma unroll
    for (int c = 0; c < DC; ++c) qf[c] = ok ? *reinterpret_cast<const bf16x8_t*>(qp + 16 * c) : bf16x8_t{};
  }
  const int diag = lk - lq;  // query i sees keys <= diag + i
  const int limit_lane = g.causal ? diag + qi_lane : lk - 1;      // last key of this lane's query
  const int wave_q0 = qt * kBQ + 32 * wave;                        // the wave's first query

  f32x16_t o[DT];
#pragma unroll
  for (int t = 0; t < DT; ++t) o[t] = f32x16_t{};
  float m_run = -INFINITY, l_run = 0.0f;

  // 1. a tile's K and V chunks go global -> registers (all loads of a tile issued together; the next tile's loads
  // are issued before this tile's MFMAs) -> LDS. K and V chunk c: key c / CPR, dims (c % CPR) * 8, stored
  // key-major with one 16-byte write. Invalid keys read the first 16 bytes of q and store zeros.
  constexpr int NT = kThreads;              // threads loading the tiles
  constexpr int NL = kBK * CPR / NT;        // chunks per thread per operand
  static_assert(NL >= 1 && NL * NT == kBK * CPR, "tile chunks per thread");
  struct Regs {
    u32x4 k[NL], v[NL];
    uint32_t kok;  // bit i: the key of chunk i is valid (its K and V rows were read)
    bool all;  // every key of the tile is valid (wave-uniform): no zeroing at the LDS store
  };
  const int32_t* bt_row = PAGED ? g.bt + int64_t(b) * g.max_blocks : nullptr;
  // Contiguous keys: this thread's K / V row addresses at key tile 0; tile kt0 adds kt0 rows (a scalar offset).
  const uint16_t* kbase[NL];
  const uint16_t* vbase[NL];
  if constexpr (!PAGED) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int c = tid + i * NT;
      kbase[i] = g.k + int64_t(k0s + c / CPR) * g.k_st + int64_t(kvh) * D + (c % CPR) * 8;
      vbase[i] = g.v + int64_t(k0s + c / CPR) * g.v_st + int64_t(kvh) * D + (c % CPR) * 8;
    }
  }
  // PAGED: block-table entries of this thread's keys in the tile the next gload call loads (the tiles are loaded
  // in order, the last one repeated), fetched one call ahead: the fetch is issued before that call's data loads and
  // retires with them, so no tile's data loads wait for a block-table load (at 4 key tiles per block, a 256-token
  // chunk over 3840 cached keys, that wait was a memory round trip per tile)
  const int last = (k_stop - 1) / kBK * kBK;
  int kblk_nx[NL];
  auto bt_fetch = [&](int kt0) {
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int kj = kt0 + (tid + i * NT) / CPR;
      kblk_nx[i] = kj < lk ? bt_row[kj / g.bs] : 0;
    }
  };
  auto gload = [&](Regs& R, int kt0) {
    R.all = kt0 + kBK <= lk;
    R.kok = 0;
    if constexpr (!PAGED) {
      if (R.all) {  // every row valid: the addresses are the bases plus a per-tile offset
#pragma unroll
        for (int i = 0; i < NL; ++i) {
          R.k[i] = *reinterpret_cast<const u32x4*>(kbase[i] + int64_t(kt0) * g.k_st);
          R.v[i] = *reinterpret_cast<const u32x4*>(vbase[i] + int64_t(kt0) * g.v_st);
        }
        return;
      }
    }
    // block-table entries of this thread's keys (PAGED: fetched by the previous call), then the entries of the
    // tile the next call loads, then every data load back to back
    int kblk[NL];
#pragma unroll
    for (int i = 0; i < NL; ++i) kblk[i] = PAGED ? kblk_nx[i] : 0;
    if constexpr (PAGED) bt_fetch(min(kt0 + kBK, last));
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int c = tid + i * NT;
      const int kj = kt0 + c / CPR;
      const int64_t krow = kj < lk ? key_row<D, PAGED>(g, k0s, kj, kblk[i], kvh, g.k_st) : -1;
      const int64_t vrow = kj < lk ? key_row<D, PAGED>(g, k0s, kj, kblk[i], kvh, g.v_st) : -1;
      R.kok |= uint32_t(krow >= 0) << i;  // krow and vrow are valid together
      R.k[i] = *reinterpret_cast<const u32x4*>(krow >= 0 ? g.k + krow + (c % CPR) * 8 : g.q);
      R.v[i] = *reinterpret_cast<const u32x4*>(vrow >= 0 ? g.v + vrow + (c % CPR) * 8 : g.q);
    }
    if constexpr (PAGED) R.all = false;  // a block-table entry may be invalid
  };
  // every key of the tile at kt0 is valid: the bases plus a per-tile offset (contiguous keys only)
  auto gload_full = [&](Regs& R, int kt0) {
    R.all = true;
    R.kok = 0;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      R.k[i] = *reinterpret_cast<const u32x4*>(kbase[i] + int64_t(kt0) * g.k_st);
      R.v[i] = *reinterpret_cast<const u32x4*>(vbase[i] + int64_t(kt0) * g.v_st);
    }
  };
  auto lstore_full = [&](const Regs& R, int stage) {  // R holds a tile whose keys are all valid
    uint16_t* Ks = lds + stage * STAGE;
    uint16_t* Vs = Ks + kBK * KP;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int c = tid + i * NT;
      *reinterpret_cast<u32x4*>(&Ks[(c / CPR) * KP + (c % CPR) * 8]) = R.k[i];
      *reinterpret_cast<u32x4*>(&Vs[(c / CPR) * VP + (c % CPR) * 8]) = R.v[i];
    }
  };
  auto lstore = [&](const Regs& R, int stage) {
    uint16_t* Ks = lds + stage * STAGE;
    uint16_t* Vs = Ks + kBK * KP;
    const bool all = R.all;
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int c = tid + i * NT;
      const u32x4 zero = u32x4{0, 0, 0, 0};
      const bool ok = all || ((R.kok >> i) & 1);
      *reinterpret_cast<u32x4*>(&Ks[(c / CPR) * KP + (c % CPR) * 8]) = ok ? R.k[i] : zero;
      *reinterpret_cast<u32x4*>(&Vs[(c / CPR) * VP + (c % CPR) * 8]) = ok ? R.v[i] : zero;
    }
  };

  // 2.-4. per tile: S^T of both 32-key halves, one online-softmax step over the tile's 64 keys, O^T += V^T P^T
  // (the p of the second half are computed under the P.V MFMAs of the first). Rescaling is lazy: a query's
  // reference max m_run only moves when a score exceeds it by more than kLazy (base 2), so p <= 2^kLazy; O and the
  // row sum carry the same factor, which cancels in O / sum, and almost every tile after the first skips the O
  // rescale (one wave-uniform branch per tile).
  constexpr float kLazy = 8.0f;
  auto tile = [&](int kt0, int stage) {
    const uint16_t* Ks = lds + stage * STAGE;
    const uint16_t* Vs = Ks + kBK * KP;
    // S^T per 32-key half: lane holds keys kt0 + 32 u + 8 (r / 4) + 4 hf + r % 4 of query qi_lane. All K fragments
    // of the tile are read before the first MFMA, so the MFMAs wait for LDS latency once, not once each.
    bf16x8_t kf[2][DC];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int c = 0; c < DC; ++c)
        kf[u][c] = *reinterpret_cast<const bf16x8_t*>(&Ks[(32 * u + ql) * KP + 8 * hf + 16 * c]);
    f32x16_t s[2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      s[u] = f32x16_t{};
#pragma unroll
      for (int c = 0; c < DC; ++c) s[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[u][c], qf[c], s[u], 0, 0, 0);
    }
    // V^T fragments of both halves (A operands of O^T += V^T P^T): dim 32 t + l % 32, keys 32 u + 16 j + 4 hf .. +3
    // and 32 u + 16 j + 8 + 4 hf .. +3, by transpose reads (lane i of a 16-lane group addresses key i / 4 of the 4,
    // dims 4 (i % 4) .. +3 of the group's 16, and receives dim i of the 4 keys); read here so that they are in flight
    // during the softmax
    const uint16_t* vt0 = Vs + (4 * hf + (lane % 16) / 4) * VP + 16 * (ql / 16) + 4 * (lane % 4);
    u32x4 vf[2][DT][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const uint16_t* vr = vt0 + (32 * u + 16 * j) * VP + 32 * t;
          const u32x2 lo = lds_read_tr16(vr), hi = lds_read_tr16(vr + 8 * VP);
          vf[u][t][j] = u32x4{lo[0], lo[1], hi[0], hi[1]};
        }
    // issue order: the 8 K reads of half 0, then its MFMAs each followed by a K read of half 1, then the MFMAs of
    // half 1 interleaved with the max of half 0 (VALU work under the matrix cores), then the V reads
    __builtin_amdgcn_sched_group_barrier(0x100, DC, 0);
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x100, 4 * DT, 0);
    // Only a tile that reaches past the key count or past the causal limit of the wave's first query needs the
    // mask (wave-uniform test); key offsets within the tile are compile-time constants per register.
    const bool full = kt0 + kBK <= lk && (!g.causal || kt0 + kBK - 1 <= diag + wave_q0);
    const int lim = min(lk - 1, limit_lane) - kt0 - 4 * hf;  // largest visible offset 32 u + 8 (r / 4) + r % 4
    // max of the tile's raw scores (the scale is positive)
    float tmax = -INFINITY;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (!full) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (32 * u + 8 * (r / 4) + r % 4 > lim) s[u][r] = -INFINITY;
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, s[u][r]);
    }
    tmax = pair32_max(tmax) * g.scale_log2;
    const bool move = tmax > m_run + kLazy;  // also true for the first finite max (m_run = -inf)
    if (__ballot(move) != 0) {
      const float alpha = move ? __builtin_amdgcn_exp2f(m_run - tmax) : 1.0f;  // 0 from m_run = -inf
      if (move) m_run = tmax;
      l_run *= alpha;
#pragma unroll
      for (int t = 0; t < DT; ++t) o[t] *= alpha;
    }
    const float m_use = m_run == -INFINITY ? 0.0f : m_run;
    // p = 2^(s * scale_log2 - m) in one FMA and v_exp_f32 (arguments <= kLazy; only results below the fp32 normal
    // range, which flush to 0, differ from exp2f), as bf16 packed per 16-key step in the k-slot order of P.V
    bf16x8_t pf[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float p[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][8 * j + e], g.scale_log2, -m_use));
          l_run += p[e];
        }
        pf[u][j] = __builtin_bit_cast(bf16x8_t, pack8(p));
      }
    // O^T += V^T P^T; the p of half 1 are computed under the MFMAs of half 0
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int t = 0; t < DT; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, vf[u][t][j]), pf[u][j], o[t], 0,
                                                         0, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, 28, 1);
#pragma unroll
    for (int i = 0; i < 2 * DT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 1);
      __builtin_amdgcn_sched_group_barrier(0x002, 4, 1);
    }
  };
  // Two LDS stages: while the waves compute tile i from one, the loads of tile i + 1 (issued a tile earlier) are
  // stored into the other and the loads of tile i + 2 are issued; one barrier per tile. Past the last tile the last
  // one is loaded and stored again, unused (every load is issued unconditionally so the compiler's waits are exact).
  // The first tile is peeled: the loads of tiles 0 and 1 both go out before the first wait, so tile 1's are in
  // flight during the prologue and tile 0 (with one set of tile registers, tile 1's loads went out after tile 0's
  // LDS store and were waited for after a single tile of work).
  {
    Regs A;
    if constexpr (PAGED) bt_fetch(k_beg);
    gload(A, k_beg);
    {
      Regs B;
      gload(B, min(k_beg + kBK, last));
      lstore(A, 0);
      __syncthreads();
      tile(k_beg, 0);
      lstore(B, 1);
    }
    gload(A, min(k_beg + 2 * kBK, last));
    __syncthreads();
    int stage = 1;
    int kt0 = k_beg + kBK;
    if constexpr (!PAGED) {
      // while the tile stored next and the one loaded next are both whole (every key valid), the loop body holds
      // only their loads and stores: the general loader's per-key row arithmetic and the zeroing selects, which the
      // compiler executes on every tile when the two paths share the body, are left to the last tiles
      for (; kt0 < k_stop && min(kt0 + 2 * kBK, last) + kBK <= lk; kt0 += kBK) {
        tile(kt0, stage);
        lstore_full(A, stage ^ 1);
        gload_full(A, min(kt0 + 2 * kBK, last));
        __syncthreads();
        stage ^= 1;
      }
    }
    for (; kt0 < k_stop; kt0 += kBK) {
      tile(kt0, stage);
      lstore(A, stage ^ 1);
      gload(A, min(kt0 + 2 * kBK, last));
      __syncthreads();
      stage ^= 1;
    }
  }

  // row sums over the two lane halves of the query; lane l holds O^T dims 32 t + 8 (r / 4) + 4 hf + r % 4 of query
  // qi_lane
  l_run = pair32_sum(l_run);
  if (g.splits > 1) {
    // this split's records of the wave's queries: the reference max and the row sum, and O unnormalised. O goes out
    // in whole 128-byte lines written through the L2: each half of the dims passes through the wave's own part of
    // the LDS (free after the loop's last barrier), a lane holding dims 32 t + 8 (r / 4) + 4 hf + r % 4 of its query
    // and a store instruction then covering D / 2 consecutive floats of 64 * 16 / (2 D) queries. Stored from the
    // MFMA layout (32-byte pieces of 32 records per instruction, (max, sum) beside O) the records' dirty lines were
    // written back after the last block: a 256-token chunk over 3840 cached keys 34.1 -> 32.2 us, a fresh
    // 2048-token prompt (2 splits) 62.7 -> 59.8 us, 256 over 1792 33.0 -> 29.8 us (whole lines with plain stores:
    // 32.5 / 61.8 / 31.3 us).
    const int nq = min(32, min(lq, int(min<int64_t>(g.ws_rows - q0s, INT32_MAX))) - wave_q0);  // wave-uniform
    if (nq <= 0) return;
    const int64_t rec0 = (int64_t(split) * g.ws_rows + q0s + wave_q0) * g.Hq + h;  // record of the first query
    if (hf == 0 && ql < nq)
      *reinterpret_cast<f32x2*>(g.ws + int64_t(g.splits) * g.ws_rows * g.Hq * D + 2 * (rec0 + int64_t(ql) * g.Hq)) =
          f32x2{m_run, l_run};
    constexpr int HD = D / 2, RP = HD + 4;  // dims per pass, LDS row pitch (floats)
    constexpr int CH = HD / 4, PER = 32 * CH / 64;  // 16-byte chunks per query and pass, per lane and pass
    static_assert(kThreads / 64 * 32 * RP * 4 <= LDS_ELEMS * 2, "record staging exceeds the LDS");
    float* wl = reinterpret_cast<float*>(lds) + (tid / 64) * 32 * RP;
#pragma unroll
    for (int hv = 0; hv < 2; ++hv) {
#pragma unroll
      for (int t = hv * DT / 2; t < (hv + 1) * DT / 2; ++t)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          *reinterpret_cast<f32x4_t*>(wl + ql * RP + 32 * (t - hv * DT / 2) + 8 * rr + 4 * hf) =
              f32x4_t{o[t][4 * rr], o[t][4 * rr + 1], o[t][4 * rr + 2], o[t][4 * rr + 3]};
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int c = lane + 64 * i, qq = c / CH, cc = c % CH;
        const u32x4 x = *reinterpret_cast<const u32x4*>(wl + qq * RP + 4 * cc);
        if (qq < nq) store16_wt(g.ws + (rec0 + int64_t(qq) * g.Hq) * D + hv * HD + 4 * cc, x);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    return;
  }
  const float inv = l_run > 0.0f ? 1.0f / l_run : 0.0f;
  if (g.out_lines) {
    // the wave's 32 output rows pass through its own part of the LDS, so that a store instruction covers whole
    // rows (D bf16 each, 16-byte pieces of 64 * 8 / D queries), written through the L2. Against the rows stored
    // straight from the MFMA layout (8-byte pieces of 32 rows per instruction): 4 x 2048 tokens 82.2 -> 77.3 us
    // (whole lines with plain stores: 78.1), 8 x 512 25.6 -> 21.6 us (23.0), 16 x 256 19.9 -> 15.7 us (17.5); the
    // 256-token mixed step 2170 -> 2160-2167 us per step (plain stores 2155-2205: within its run-to-run spread).
    const int nq = min(32, lq - wave_q0);  // wave-uniform
    if (nq <= 0) return;
    constexpr int RP = D / 2 + 4, CH = D / 8, PER = 32 * CH / 64;  // u32 row pitch, 16-byte pieces per row, per lane
    static_assert(kThreads / 64 * 32 * RP * 4 <= LDS_ELEMS * 2, "output staging exceeds the LDS");
    uint32_t* wl = reinterpret_cast<uint32_t*>(lds) + (tid / 64) * 32 * RP;
#pragma unroll
    for (int t = 0; t < DT; ++t)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr)
        *reinterpret_cast<u32x2*>(wl + ql * RP + 16 * t + 4 * rr + 2 * hf) =
            u32x2{pack_bf16x2(o[t][4 * rr] * inv, o[t][4 * rr + 1] * inv),
                  pack_bf16x2(o[t][4 * rr + 2] * inv, o[t][4 * rr + 3] * inv)};
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    uint16_t* ob = g.out + int64_t(q0s + wave_q0) * g.o_st + int64_t(h) * g.o_sh;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int c = lane + 64 * i, qq = c / CH, cc = c % CH;
      const u32x4 x = *reinterpret_cast<const u32x4*>(wl + qq * RP + 4 * cc);
      if (qq < nq) store16_wt(ob + int64_t(qq) * g.o_st + 8 * cc, x);
    }
    return;
  }
  if (qi_lane >= lq) return;
  uint16_t* op = g.out + int64_t(q0s + qi_lane) * g.o_st + int64_t(h) * g.o_sh + 4 * hf;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int rr = 0; rr < 4; ++rr)
      *reinterpret_cast<u32x2*>(op + 32 * t + 8 * rr) =
          u32x2{pack_bf16x2(o[t][4 * rr] * inv, o[t][4 * rr + 1] * inv),
                  pack_bf16x2(o[t][4 * rr + 2] * inv, o[t][4 * rr + 3] * inv)};
}

// The prefill attention over the paged cache without decode requests (one prompt chunk and its cached prefix, or any
// sequences of a model with more than 16 q heads per kv head), D = 128, with cache blocks of whole key tiles: the grid,
// the query tiles, the key splits and the arithmetic of prefill_attention_kernel, for a block of 4 waves in which a wave
// owns 64 queries.
//
// What bounded prefill_attention_kernel here: every K and V fragment that a wave of 32 queries reads from LDS feeds one
// MFMA (128 bytes per clock and CU, the LDS rate), the K / V tiles pass through registers with per-key row arithmetic,
// and the two waves of a SIMD run the softmax and the matrix products in phase, so they add up (a probe: an MFMA of 32
// clocks leaves room for 4-5 other instructions of its SIMD, and 64 MFMAs and the ~310 others of a tile have to be
// mixed to fit). Here
//   - a fragment read from LDS feeds two MFMAs (64 queries per wave, one wave per SIMD: O and Q in 192 accumulation
//     registers, two tiles' scores in 128 vector registers);
//   - K and V tiles go from memory to LDS without registers (global_load_lds, a wave's instruction brings 4 keys), two
//     tiles ahead; a key tile lies in one cache block, so its address is one scalar table entry. Chunk c of K row r
//     lies at chunk c ^ (r & 15), of V row r at c ^ 4 (r & 3): fragment and transpose reads hit distinct banks;
//   - the stream of a tile is mixed by hand: the scores of the next tile between the probabilities of this one, P.V
//     between the rest of them and the next tile's maxima, one memory load per MFMA behind the barrier.
// The matrix instructions are inline asm, because the compiler's own choice keeps all results in accumulation registers
// and moves the scores back and forth. It does not know their timing, so nothing may read a result, or write an operand
// with a vector instruction, right before or after one: every such pair below lies several MFMAs apart, or behind the
// s_nop fences, and the build measures the distances in the assembly (check_asm.py).
// 2048 queries over 14001 cached keys (16 / 8 heads): 326 -> 249 us with the q/k norm kernel, 0.77 -> 1.0 PFLOP/s (262
// while mask() kept its scalars across the wait: 118 of them spilled); 300 over 4000 39.5 -> 34.2. A form of it for
// contiguous keys, before that, was no faster than prefill_attention_kernel (8192 tokens 257-261 us against 266, 16 x 256
// tokens 19.5 against 16.6), which keeps those.
__device__ const uint32_t kZeroRow[64] = {};  // what the keys of an invalid cache block read

constexpr int kWideThreads = 256;

template <int HB>
__global__ __launch_bounds__(kWideThreads, 1) void prefill_wide_kernel(const PrefillArgs g) {
  constexpr int D = 128, kBQ = block_queries(HB), kHeadThreads = kWideThreads / HB;
  constexpr int NK = 3, NV = 4, TILE = kBK * D * 2;  // LDS slots of K and V tiles, bytes of a tile
  constexpr int LOADS = 8;                           // memory -> LDS loads per wave and event (4 of K, 4 of V)
  __shared__ __attribute__((aligned(1024))) char lds[(NK + NV) * TILE];
  const uint32_t lbase = uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) char*)lds));

  const int ntile = g.qtiles * g.splits, nblk = int(gridDim.x), ngrp = nblk / ntile;
  int grp, ci;
  if (nblk % 8 == 0 && (nblk / 8) % ntile == 0) {
    const int gx = nblk / 8 / ntile, r = blockIdx.x / 8;
    grp = (r % gx) * 8 + blockIdx.x % 8;
    ci = r / gx;
  } else {
    grp = blockIdx.x % ngrp;
    ci = blockIdx.x / ngrp;
  }
  const int qt = g.qtiles - 1 - ci / g.splits, split = ci % g.splits;
  const int b = grp / g.nhg, hg = grp % g.nhg;
  const int h = hg * HB + int(threadIdx.x) / kHeadThreads, kvh = (hg * HB) / g.G;
  const int q0s = g.cu_q[b], lq = g.cu_q[b + 1] - q0s;
  const int lk = g.cu_k[b + 1] - g.cu_k[b];
  const int k_beg = split * g.split_len;
  const int k_hi = split == g.splits - 1 ? INT32_MAX : k_beg + g.split_len;
  const int k_stop = g.causal ? min(min(lk, lk - lq + min(qt * kBQ + kBQ, lq)), k_hi) : min(lk, k_hi);
  if (qt * kBQ >= lq || k_stop <= k_beg) {
    const int r = int(threadIdx.x) % kHeadThreads;
    for (int q = qt * kBQ + r; q < min(qt * kBQ + kBQ, lq); q += kHeadThreads) {
      const int64_t row = q0s + q;
      if (g.splits > 1) {
        if (row >= g.ws_rows) return;
        const int64_t rec = (int64_t(split) * g.ws_rows + row) * g.Hq + h;
        float* o = g.ws + rec * D;
        for (int d = 0; d < D; ++d) o[d] = 0.0f;
        *reinterpret_cast<f32x2*>(g.ws + int64_t(g.splits) * g.ws_rows * g.Hq * D + 2 * rec) = f32x2{-INFINITY, 0.0f};
      } else {
        uint16_t* o = g.out + row * g.o_st + int64_t(h) * g.o_sh;
        for (int d = 0; d < D; ++d) o[d] = 0;
      }
    }
    return;
  }
  const int tid = threadIdx.x, lane = tid % 64, bwave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wave = __builtin_amdgcn_readfirstlane((tid % kHeadThreads) / 64);
  const int ql = lane % 32, hf = lane / 32;
  const int wave_q0 = qt * kBQ + 64 * wave;  // the wave's first query; lane: queries wave_q0 + 32 qh + ql

  bf16x8_t qf[2][8];
#pragma unroll
  for (int qh = 0; qh < 2; ++qh) {
    const int qi = wave_q0 + 32 * qh + ql;
    const bool ok = qi < lq;
    const uint16_t* qp = g.q + int64_t(q0s + (ok ? qi : 0)) * g.q_st + int64_t(h) * g.q_sh + 8 * hf;
#pragma unroll
    for (int c = 0; c < 8; ++c) qf[qh][c] = ok ? *reinterpret_cast<const bf16x8_t*>(qp + 16 * c) : bf16x8_t{};
  }
  const int diag = lk - lq;
  const int nt = (k_stop - k_beg + kBK - 1) / kBK, last = k_beg + (nt - 1) * kBK;

  // loads
  const int32_t* bt_row = g.bt + int64_t(b) * g.max_blocks;
  const uint32_t row_bytes = uint32_t(g.Hkv) * D * 2;
  uint32_t kofs[4], vofs[4];
  const int lr = lane / 16, lc = lane % 16;
  auto offsets = [&](int v_rows, int k_rows) {  // rows of the tiles that exist; past them the last one again (K rows
                                                // there are masked, V rows zeroed by mask())
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int row = 4 * (bwave + 4 * j) + lr;
      kofs[j] = uint32_t(min(row, k_rows - 1)) * row_bytes + ((lc ^ (row & 15)) * 16);
      vofs[j] = uint32_t(min(row, v_rows - 1)) * row_bytes + ((lc ^ ((row & 3) << 2)) * 16);
    }
  };
  offsets(kBK, kBK);
  // Where the K tile loaded next lies, and the V tile, which is the K tile of the event before: first key (the last
  // tile is loaded again past the end), cache block (its table entry fetched an event ahead) and place in it. An invalid
  // block reads 16-byte pieces of kZeroRow: keys and values of zero.
  int k_kt = k_beg, v_kt = k_beg, k_to = 0, v_to = NV - 1;  // (the first event's V tile is not loaded)
  int blk_idx = k_beg / g.bs, blk_ofs = k_beg % g.bs, blk = load_uniform(bt_row + blk_idx);
  int64_t elem = 0;
  uint32_t k_mask = 0, v_mask = 0, k_dst = 0, v_dst = 0;
  uint64_t k_at = 0, v_at = 0;
  const uint64_t zero_row = reinterpret_cast<uint64_t>(kZeroRow);
  auto dma = [&](uint32_t dst, uint32_t ofs, uint64_t p) {
    asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(dst), "v"(ofs), "s"(p) : "memory");
  };
  // One event's loads: next_load() prepares them, load(0 .. 3) issues V's and load(4 .. 7) K's.
  auto next_load = [&]() {
    v_mask = k_mask;
    v_at = v_mask == 0xffffffffu ? reinterpret_cast<uint64_t>(g.v + elem) : zero_row;
    v_dst = lbase + (NK + v_to) * TILE + bwave * 1024;
    k_mask = blk >= 0 && blk < g.num_blocks ? 0xffffffffu : 0xf0u;
    elem = ((int64_t(blk) * g.bs + blk_ofs) * g.Hkv + kvh) * D;
    k_at = k_mask == 0xffffffffu ? reinterpret_cast<uint64_t>(g.k + elem) : zero_row;
    k_dst = lbase + k_to * TILE + bwave * 1024;
    if (k_kt + kBK > lk) offsets(min(kBK, lk - v_kt), lk - k_kt);
    v_to = v_to + 1 == NV ? 0 : v_to + 1;
    k_to = k_to + 1 == NK ? 0 : k_to + 1;
    v_kt = k_kt;
    if (k_kt < last) {
      k_kt += kBK;
      blk_ofs += kBK;
      if (blk_ofs == g.bs) blk_ofs = 0, ++blk_idx;
      blk = load_uniform(bt_row + blk_idx);
    }
  };
  auto load = [&](auto jc) {
    constexpr int j = decltype(jc)::value;
    if constexpr (j < 4) dma(v_dst + j * 4096, vofs[j] & v_mask, v_at);
    else dma(k_dst + (j - 4) * 4096, kofs[j - 4] & k_mask, k_at);
  };
  next_load();
  static_for<4>([&](auto jc) { load(std::integral_constant<int, decltype(jc)::value + 4>{}); });
  next_load();
  static_for<8>([&](auto jc) { load(jc); });
  next_load();
  static_for<8>([&](auto jc) { load(jc); });

  f32x16_t o[4][2];
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int qh = 0; qh < 2; ++qh) o[t][qh] = f32x16_t{};
  auto fence_o = [&]() {
#pragma unroll
    for (int t = 0; t < 4; ++t) asm volatile("s_nop 15" : "+a"(o[t][0]), "+a"(o[t][1]));
  };
  fence_o();
#pragma unroll
  for (int qh = 0; qh < 2; ++qh)
#pragma unroll
    for (int c = 0; c < 8; ++c) asm volatile("s_nop 1" : "+a"(qf[qh][c]));

  float m_run[2] = {-INFINITY, -INFINITY}, l_run[2] = {0.0f, 0.0f}, tmax[2];
  // fragment addresses
  const uint32_t ka = uint32_t(ql) * 256, kx = uint32_t(hf ^ (ql & 15)) << 4;
  const uint32_t va = uint32_t(4 * hf + (lane % 16) / 4) * 256 + (lane % 2) * 8;
  const uint32_t vx = uint32_t((2 * (ql / 16) + (lane % 4) / 2) ^ (((lane % 16) / 4) << 2)) << 4;
  auto read_k = [&](int slot, int u, int c) {
    return *reinterpret_cast<const bf16x8_t*>(lds + slot * TILE + u * 32 * 256 + ka + ((uint32_t(c) << 5) ^ kx));
  };
  auto read_v = [&](int slot, int u, int j, int t) {
    const uint16_t* p = reinterpret_cast<const uint16_t*>(lds + (NK + slot) * TILE + (32 * u + 16 * j) * 256 + va +
                                                          ((uint32_t(t) << 6) ^ vx));
    const u32x2 lo = lds_read_tr16(p), hi = lds_read_tr16(p + 8 * D);
    return __builtin_bit_cast(bf16x8_t, u32x4{lo[0], lo[1], hi[0], hi[1]});
  };
  using Scores = f32x16_t[2][2];  // [u][qh]
  // Masks the scores of the tile at kt0 where it needs it, in front of the barrier that hands out its V rows (slot; one
  // event's loads were issued after them). Behind the last key those are copies of its row, and 0 times an infinity
  // there would be NaN: each wave zeroes what it loaded itself.
  auto mask = [&](Scores& s, int kt0, int slot) {
    if (kt0 + kBK <= lk && (!g.causal || kt0 + kBK - 1 <= diag + wave_q0)) return;
    if (kt0 > last) return;  // the last tile loaded again, unused
#pragma unroll
    for (int qh = 0; qh < 2; ++qh) {
      const int lim = min(lk - 1, g.causal ? diag + wave_q0 + 32 * qh + ql : lk - 1) - kt0 - 4 * hf;
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (32 * u + 8 * (r / 4) + r % 4 > lim) s[u][qh][r] = -INFINITY;
    }
    if (kt0 + kBK > lk) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (4 * (bwave + 4 * j) + lr >= lk - kt0)
          *reinterpret_cast<u32x4*>(lds + (NK + slot) * TILE + j * 4096 + bwave * 1024 + lane * 16) = u32x4{0, 0, 0, 0};
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
  };
  auto max_step = [&](const Scores& s, auto kc) {  // step k of 32: two scores of a query half
    constexpr int k = decltype(kc)::value, qh = k % 2, e = k / 2 * 2;
    const float m = k < 2 ? -INFINITY : tmax[qh];
    tmax[qh] = fmaxf(fmaxf(m, s[e / 16][qh][e % 16]), s[e / 16][qh][e % 16 + 1]);
  };
  auto max_done = [&]() {
#pragma unroll
    for (int qh = 0; qh < 2; ++qh) tmax[qh] = pair32_max(tmax[qh]) * g.scale_log2;
  };
  int k_slot = 0, v_slot = 0;  // K tile of the next scores, V tile of the next P.V
  int kt0 = k_beg;             // tile of the current iteration
  bf16x8_t kf[4];
  auto scores_mfma = [&](Scores& s, auto xc) {  // MFMA x: step n = 2 c + u of query half x % 2
    constexpr int x = decltype(xc)::value, n = x / 2, c = n / 2, u = n % 2, qh = x % 2;
    if constexpr (c == 0)
      asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(s[u][qh]) : "v"(kf[n % 4]), "a"(qf[qh][c]));
    else
      asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(s[u][qh]) : "v"(kf[n % 4]), "a"(qf[qh][c]));
    if constexpr (qh == 1 && n + 4 < 16) kf[n % 4] = read_k(k_slot, (n + 4) % 2, (n + 4) / 2);
  };
  auto first_k = [&]() {
#pragma unroll
    for (int n = 0; n < 4; ++n) kf[n] = read_k(k_slot, n % 2, n / 2);
  };
  auto next_slot = [](int& x, int n) { x = x + 1 == n ? 0 : x + 1; };
  Scores sa, sb;
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * LOADS) : "memory");
  first_k();
  static_for<32>([&](auto xc) { scores_mfma(sa, xc); });
  next_slot(k_slot, NK);
  asm volatile("s_nop 15\n\ts_nop 15" : "+v"(sa[0][0]), "+v"(sa[0][1]), "+v"(sa[1][0]), "+v"(sa[1][1]));
  mask(sa, kt0, v_slot);
  static_for<32>([&](auto kc) { max_step(sa, kc); });
  max_done();
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LOADS) : "memory");
  first_k();
  next_load();
  static_for<8>([&](auto jc) { load(jc); });

  constexpr float kLazy = 8.0f;
  auto iteration = [&](Scores& s, Scores& sn) {
    // move the reference maxima of this tile's scores
    bool move[2];
#pragma unroll
    for (int qh = 0; qh < 2; ++qh) move[qh] = tmax[qh] > m_run[qh] + kLazy;
    if (__ballot(move[0] || move[1]) != 0) {
      float alpha[2];
#pragma unroll
      for (int qh = 0; qh < 2; ++qh) {
        alpha[qh] = move[qh] ? __builtin_amdgcn_exp2f(m_run[qh] - tmax[qh]) : 1.0f;
        if (move[qh]) m_run[qh] = tmax[qh];
        l_run[qh] *= alpha[qh];
      }
      if (kt0 != k_beg) {
        fence_o();
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int qh = 0; qh < 2; ++qh) o[t][qh] *= alpha[qh];
        fence_o();
      }
    }
    float m_use[2];
#pragma unroll
    for (int qh = 0; qh < 2; ++qh) m_use[qh] = m_run[qh] == -INFINITY ? 0.0f : m_run[qh];
    u32x4 pf[2][2][2];  // [u][j][qh]
    auto pair = [&](auto yc) {  // probabilities 2 (y % 4), + 1 of group y / 4
      constexpr int y = decltype(yc)::value, grp8 = y / 4, u = grp8 / 4, j = grp8 / 2 % 2, qh = grp8 % 2, e = y % 4;
      const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][qh][8 * j + 2 * e], g.scale_log2, -m_use[qh]));
      const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][qh][8 * j + 2 * e + 1], g.scale_log2, -m_use[qh]));
      l_run[qh] += p0;
      l_run[qh] += p1;
      uint32_t w = pack_bf16x2(p0, p1);
      asm volatile("" : "+v"(w), "+v"(l_run[qh]));  // here, not where the sums are wanted (the p would stay live)
      pf[u][j][qh][e] = w;
    };
    bf16x8_t vf[4];
    // the next tile's scores over three quarters of this tile's probabilities
    __builtin_amdgcn_sched_barrier(0);
    static_for<32>([&](auto xc) {
      constexpr int x = decltype(xc)::value;
      scores_mfma(sn, xc);
      static_for<24>([&](auto yc) {
        if constexpr (decltype(yc)::value * 32 / 24 == x) pair(yc);
      });
      if constexpr (x >= 28) vf[x - 28] = read_v(v_slot, 0, 0, x - 28);
      __builtin_amdgcn_sched_barrier(0);
    });
    next_slot(k_slot, NK);
    // P.V: MFMA x: step n = (u, j, t) of query half x % 2
    static_for<32>([&](auto xc) {
      constexpr int x = decltype(xc)::value, n = x / 2, u = n / 8, j = n / 4 % 2, t = n % 4, qh = x % 2;
      if constexpr (x == 16) {
        // K(next + 1) and V(next) have landed, and everybody has read K(next) and the V before this one: their slots
        // are free
        asm volatile("" : "+v"(sn[0][0]), "+v"(sn[0][1]), "+v"(sn[1][0]), "+v"(sn[1][1]));
        mask(sn, kt0 + kBK, v_slot + 1 == NV ? 0 : v_slot + 1);
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(LOADS) : "memory");
        next_load();
      }
      if constexpr (x >= 16 && x < 24) load(std::integral_constant<int, x - 16>{});
      asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(o[t][qh]) : "v"(vf[n % 4]), "v"(pf[u][j][qh]));
      if constexpr (qh == 1 && n + 4 < 16) vf[n % 4] = read_v(v_slot, (n + 4) / 8, (n + 4) / 4 % 2, (n + 4) % 4);
      if constexpr (x < 16 && x % 2 == 0) pair(std::integral_constant<int, 24 + x / 2>{});
      if constexpr (x >= 17 && x < 31) {
        static_for<32>([&](auto kc) {
          if constexpr (decltype(kc)::value * 14 / 32 == x - 17) max_step(sn, kc);
        });
        asm volatile("" : "+v"(tmax[0]), "+v"(tmax[1]));
      }
      if constexpr (x == 31) max_done();
      if constexpr (x >= 28) kf[x - 28] = read_k(k_slot, x % 2, (x - 28) / 2);
      __builtin_amdgcn_sched_barrier(0);
    });
    next_slot(v_slot, NV);
    kt0 += kBK;
  };
  // two copies, so that a tile's scores stay in the registers that the matrix cores wrote them to; the last iteration
  // computes scores of a tile loaded again, unused
  for (int left = nt;;) {
    iteration(sa, sb);
    if (--left == 0) break;
    iteration(sb, sa);
    if (--left == 0) break;
  }
  fence_o();
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the LDS is free

#pragma unroll
  for (int qh = 0; qh < 2; ++qh) {
    const int q0 = wave_q0 + 32 * qh, qi_lane = q0 + ql;
    const float l = pair32_sum(l_run[qh]);
    if (g.splits > 1) {
      const int nq = min(32, min(lq, int(min<int64_t>(g.ws_rows - q0s, INT32_MAX))) - q0);  // wave-uniform
      if (nq <= 0) return;
      const int64_t rec0 = (int64_t(split) * g.ws_rows + q0s + q0) * g.Hq + h;
      if (hf == 0 && ql < nq)
        *reinterpret_cast<f32x2*>(g.ws + int64_t(g.splits) * g.ws_rows * g.Hq * D + 2 * (rec0 + int64_t(ql) * g.Hq)) =
            f32x2{m_run[qh], l};
      constexpr int RP = D + 4, CH = D / 4, PER = 32 * CH / 64;
      float* wl = reinterpret_cast<float*>(lds) + bwave * 32 * RP;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          *reinterpret_cast<f32x4_t*>(wl + ql * RP + 32 * t + 8 * rr + 4 * hf) =
              f32x4_t{o[t][qh][4 * rr], o[t][qh][4 * rr + 1], o[t][qh][4 * rr + 2], o[t][qh][4 * rr + 3]};
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int c = lane + 64 * i, qq = c / CH, cc = c % CH;
        const u32x4 x = *reinterpret_cast<const u32x4*>(wl + qq * RP + 4 * cc);
        if (qq < nq) store16_wt(g.ws + (rec0 + int64_t(qq) * g.Hq) * D + 4 * cc, x);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      continue;
    }
    const float inv = l > 0.0f ? 1.0f / l : 0.0f;
    if (g.out_lines) {
      const int nq = min(32, lq - q0);
      if (nq <= 0) return;
      constexpr int RP = D / 2 + 4, CH = D / 8, PER = 32 * CH / 64;
      uint32_t* wl = reinterpret_cast<uint32_t*>(lds) + bwave * 32 * RP;
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int rr = 0; rr < 4; ++rr)
          *reinterpret_cast<u32x2*>(wl + ql * RP + 16 * t + 4 * rr + 2 * hf) =
              u32x2{pack_bf16x2(o[t][qh][4 * rr] * inv, o[t][qh][4 * rr + 1] * inv),
                    pack_bf16x2(o[t][qh][4 * rr + 2] * inv, o[t][qh][4 * rr + 3] * inv)};
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      uint16_t* ob = g.out + int64_t(q0s + q0) * g.o_st + int64_t(h) * g.o_sh;
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int c = lane + 64 * i, qq = c / CH, cc = c % CH;
        const u32x4 x = *reinterpret_cast<const u32x4*>(wl + qq * RP + 4 * cc);
        if (qq < nq) store16_wt(ob + int64_t(qq) * g.o_st + 8 * cc, x);
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      continue;
    }
    if (qi_lane >= lq) continue;
    uint16_t* op = g.out + int64_t(q0s + qi_lane) * g.o_st + int64_t(h) * g.o_sh + 4 * hf;
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr)
        *reinterpret_cast<u32x2*>(op + 32 * t + 8 * rr) =
            u32x2{pack_bf16x2(o[t][qh][4 * rr] * inv, o[t][qh][4 * rr + 1] * inv),
                  pack_bf16x2(o[t][qh][4 * rr + 2] * inv, o[t][qh][4 * rr + 3] * inv)};
  }
}

// Merges the split records of every query of the sequences the prefill kernel took, in split order:
// O = sum_s O_s 2^(m_s - M) / sum_s l_s 2^(m_s - M), M = max_s m_s; a query no split saw (M = -inf) is zero.
// One wave per two (query, head) pairs p0 = 2 w, p0 + 1 (pair = query * Hq + head; records of consecutive pairs are
// adjacent), 4 waves per block (block x: sequence x / per_seq, its waves 4 (x % per_seq) ..): lane s < splits reads
// split s's (max, sum) of both pairs (all at once), the weights come back to the whole wave with readlane, and half
// h of the wave sums pair p0 + h, D / 32 dims per lane (one 16-byte load per split at D = 128), eight splits' loads
// in flight at a time. (One wave per pair, 8-byte loads, four splits at a time: the merge of a 256-token chunk over
// 3840 cached keys, 16 splits, read its 34.6 MB of records at ~5 TB/s.)
template <int D>
__global__ __launch_bounds__(256) void prefill_combine(const PrefillArgs g, int per_seq) {
  constexpr int DPL = D / 32, SB = 8;
  static_assert(DPL == 2 || DPL == 4, "head_dim 64 or 128");
  const int b = blockIdx.x / per_seq;
  const int lane = threadIdx.x % 64, hh = lane / 32;
  const int p0 = ((blockIdx.x % per_seq) * 4 + int(threadIdx.x) / 64) * 2;
  const int q0s = g.cu_q[b], lq = g.cu_q[b + 1] - q0s;
  if (lq <= g.lq_skip) return;  // the decode kernel wrote these rows (or there are none)
  const int64_t rows_left = min<int64_t>(lq, g.ws_rows - q0s);  // queries of the sequence that have records
  const bool ok0 = p0 < rows_left * g.Hq, ok1 = p0 + 1 < rows_left * g.Hq;
  if (!ok0) return;  // the wave's first pair is past the sequence's queries (wave-uniform)
  const int64_t step = g.ws_rows * g.Hq;  // records of one split
  const int64_t rec0 = int64_t(q0s) * g.Hq + p0;
  const float* ml = g.ws + g.splits * step * D + 2 * rec0;  // (max, sum) of pair p0, split 0
  const bool mine = lane < g.splits;  // splits <= 64 (host)
  f32x2 ml0 = {-INFINITY, 0.0f}, ml1 = {-INFINITY, 0.0f};
  if (mine) ml0 = *reinterpret_cast<const f32x2*>(ml + 2 * lane * step);
  if (mine && ok1) ml1 = *reinterpret_cast<const f32x2*>(ml + 2 + 2 * lane * step);
  float M0 = ml0[0], M1 = ml1[0];
#pragma unroll
  for (int off = 32; off >= 1; off /= 2) M0 = fmaxf(M0, __shfl_xor(M0, off)), M1 = fmaxf(M1, __shfl_xor(M1, off));
  const float f0 = M0 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml0[0] - M0);  // 0 for a split that saw nothing
  const float f1 = M1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ml1[0] - M1);
  float den0 = ml0[1] * f0, den1 = ml1[1] * f1;
#pragma unroll
  for (int off = 32; off >= 1; off /= 2) den0 += __shfl_xor(den0, off), den1 += __shfl_xor(den1, off);
  const bool mine_pair = hh == 0 || ok1;
  const float* rp = g.ws + (rec0 + hh) * D + (lane % 32) * DPL;
  float num[DPL] = {};
  for (int sp0 = 0; sp0 < g.splits; sp0 += SB) {
    float v[SB][DPL];
#pragma unroll
    for (int u = 0; u < SB; ++u) {
      const int sp = min(sp0 + u, g.splits - 1);
      if (mine_pair) {
        if constexpr (DPL == 4) {
          const f32x4_t x = *reinterpret_cast<const f32x4_t*>(rp + sp * step * D);
          v[u][0] = x[0], v[u][1] = x[1], v[u][2] = x[2], v[u][3] = x[3];
        } else {
          const f32x2 x = *reinterpret_cast<const f32x2*>(rp + sp * step * D);
          v[u][0] = x[0], v[u][1] = x[1];
        }
      } else {
#pragma unroll
        for (int e = 0; e < DPL; ++e) v[u][e] = 0.0f;
      }
    }
#pragma unroll
    for (int u = 0; u < SB; ++u) {
      if (sp0 + u >= g.splits) break;  // uniform
      const float w0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f0), sp0 + u));
      const float w1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, f1), sp0 + u));
      const float w = hh ? w1 : w0;
#pragma unroll
      for (int e = 0; e < DPL; ++e) num[e] = __builtin_fmaf(v[u][e], w, num[e]);
    }
  }
  if (!mine_pair) return;
  const float den = hh ? den1 : den0;
  const float inv = den > 0.0f ? 1.0f / den : 0.0f;
  const int pr = p0 + hh, i = pr / g.Hq, h = pr % g.Hq;
  uint16_t* o = g.out + int64_t(q0s + i) * g.o_st + int64_t(h) * g.o_sh + (lane % 32) * DPL;
  if constexpr (DPL == 4)
    *reinterpret_cast<u32x2*>(o) =
        u32x2{pack_bf16x2(num[0] * inv, num[1] * inv), pack_bf16x2(num[2] * inv, num[3] * inv)};
  else
    *reinterpret_cast<uint32_t*>(o) = pack_bf16x2(num[0] * inv, num[1] * inv);
}

// Key splits: only when the blocks of one pass (query tiles x sequences x head groups) leave CUs idle and the
// sequences bring long key ranges (a chunk of a prompt over its cached prefix, a single long prompt): aiming at
// ~256 blocks with at least 4 key tiles (256 keys) per split, the longest key range (max_seqlen_k) setting the
// count.
void prefill_split_policy(int64_t blocks, int64_t max_seqlen_k, int& splits, int& split_len) {
  constexpr int64_t kCUs = 256, kMinKeys = 4 * kBK;
  splits = 1;
  split_len = int(std::min<int64_t>(std::max<int64_t>(max_seqlen_k, 1), INT32_MAX / 2));
  if (blocks <= 0 || blocks >= kCUs || max_seqlen_k < 2 * kMinKeys) return;
  const int64_t want = std::min<int64_t>(std::min<int64_t>((kCUs + blocks - 1) / blocks, max_seqlen_k / kMinKeys), 64);
  if (want < 2) return;
  int64_t len = (max_seqlen_k + want - 1) / want;
  len = (len + kBK - 1) / kBK * kBK;
  splits = int((max_seqlen_k + len - 1) / len);
  split_len = int(len);
}

int prefill_heads_per_block(int64_t Hq, int64_t Hkv) { return (Hq / Hkv) % 2 == 0 ? 2 : 1; }

int64_t prefill_workspace_bytes(int64_t num_seqs, int64_t max_seqlen_q, int64_t max_seqlen_k, int64_t Hq,
                                int64_t Hkv, int64_t D, int64_t total_q) {
  const int hb = prefill_heads_per_block(Hq, Hkv);
  const int64_t qtiles = (max_seqlen_q + block_queries(hb) - 1) / block_queries(hb);
  int splits, split_len;
  prefill_split_policy(qtiles * num_seqs * (Hq / hb), max_seqlen_k, splits, split_len);
  if (splits <= 1) return 0;
  const double bytes = double(splits) * double(total_q) * double(Hq) * record_len(int(D)) * sizeof(float);
  if (bytes > double(int64_t(1) << 40)) return 0;  // no split rather than a workspace past 1 TiB
  return int64_t(splits) * total_q * Hq * record_len(int(D)) * int64_t(sizeof(float));
}

// Queries per sequence the paged decode kernel takes in a call with a block table (0: none): sequences with at
// most 16 / G queries, unless the call has one sequence with more (nothing for that kernel then).
int64_t short_queries(int64_t num_seqs, int64_t total_q, int64_t Hq, int64_t Hkv, int64_t max_seqlen_q) {
  const int64_t G = Hq / Hkv;
  if (G > 16 || (num_seqs == 1 && total_q > 16 / G)) return 0;
  return std::min<int64_t>(16 / G, max_seqlen_q);
}

// Workspace: kAttnCounterBytes of counters (the decode attention's in-kernel merge: zero before a call, left
// zero), the prefill kernel's split records, then (16-byte aligned) the short sequences' decode records -- those of
// the paged decode kernel's splits (no longer sequence in the call), or those of the length-balanced pieces that
// the prefill kernel's blocks of the short sequences run (a longer sequence in the call).
int64_t decode_workspace_offset(int64_t prefill_bytes) { return kAttnCounterBytes + (prefill_bytes + 15) / 16 * 16; }

// The short sequences' decode attention inside the prefill launch cuts each (sequence, kv head) pair's context in
// two (halves) for at most kBalanceMaxPairs pairs (the counters): two record blocks of 16 rows per pair.
bool inline_halves(int64_t num_seqs, int64_t Hkv) { return num_seqs * Hkv <= kBalanceMaxPairs; }
int64_t inline_halves_bytes(int64_t num_seqs, int64_t Hkv, int64_t D) {
  return 2 * num_seqs * Hkv * decode_record_stride(16, D, true) * int64_t(sizeof(float));
}

int64_t total_workspace_bytes(int64_t num_seqs, int64_t max_seqlen_q, int64_t max_seqlen_k, int64_t Hq, int64_t Hkv,
                              int64_t D, int64_t total_q) {
  const int64_t pre = prefill_workspace_bytes(num_seqs, max_seqlen_q, max_seqlen_k, Hq, Hkv, D, total_q);
  const int64_t qs = short_queries(num_seqs, total_q, Hq, Hkv, max_seqlen_q);
  int64_t dec = qs > 0 ? paged_decode_varlen_workspace(num_seqs, qs, Hq, Hkv, D) : 0;
  if (qs > 0 && max_seqlen_q > qs && inline_halves(num_seqs, Hkv))
    dec = std::max(dec, inline_halves_bytes(num_seqs, Hkv, D));
  if (pre == 0 && dec == 0) return 0;
  return decode_workspace_offset(pre) + dec;
}

}  // namespace
}  // namespace nvhip

extern "C" int64_t nvhip_prefill_attention_workspace_size(int64_t num_seqs, int64_t max_seqlen_q,
                                                          int64_t max_seqlen_k, int64_t Hq, int64_t Hkv, int64_t D,
                                                          int64_t total_q) {
  if (num_seqs <= 0 || max_seqlen_q <= 0 || max_seqlen_k <= 0 || Hq < 1 || Hkv < 1 || Hq % Hkv != 0 ||
      (D != 64 && D != 128) || total_q <= 0)
    return 0;
  return nvhip::total_workspace_bytes(num_seqs, max_seqlen_q, max_seqlen_k, Hq, Hkv, D, total_q);
}

extern "C" int nvhip_prefill_attention_bf16(void* out, const void* q, const void* k, const void* v,
                                            const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                            int64_t num_seqs, int64_t max_seqlen_q, int64_t max_seqlen_k,
                                            int64_t total_q, int64_t Hq, int64_t Hkv, int64_t D,
                                            int64_t q_stride_token, int64_t q_stride_head, int64_t k_stride_token,
                                            int64_t v_stride_token, int64_t out_stride_token,
                                            int64_t out_stride_head, const int32_t* block_table, int64_t block_size,
                                            int64_t num_blocks, int64_t max_blocks, float scale, int causal,
                                            void* workspace, int64_t workspace_size, void* stream) {
  using namespace nvhip;
  clear_error();
  if (num_seqs < 0 || max_seqlen_q < 0 || max_seqlen_k < 0 || total_q < 0 || Hq < 1 || Hkv < 1)
    return invalid("prefill_attention: bad size");
  if (!(scale > 0.0f) || scale == INFINITY) return invalid("prefill_attention: softmax_scale must be positive");
  if (Hq % Hkv != 0) return invalid("prefill_attention: Hq must be a multiple of Hkv");
  if (D != 64 && D != 128) return invalid("prefill_attention: head_dim must be 64 or 128");
  if (q_stride_head < D || q_stride_token < Hq * q_stride_head || out_stride_head < D ||
      out_stride_token < Hq * out_stride_head || q_stride_head % 8 || q_stride_token % 8 || out_stride_head % 4 ||
      out_stride_token % 4)
    return invalid("prefill_attention: bad q / out strides");
  if (block_table == nullptr && (k_stride_token < Hkv * D || v_stride_token < Hkv * D || k_stride_token % 8 ||
                                 v_stride_token % 8))
    return invalid("prefill_attention: bad k / v strides");
  if (block_table != nullptr && (block_size < 1 || num_blocks < 1 || max_blocks < 1))
    return invalid("prefill_attention: bad block table shape");
  if (num_seqs == 0 || max_seqlen_q == 0 || total_q == 0) return NVHIP_OK;
  if (!out || !q || !k || !v || !cu_seqlens_q || !cu_seqlens_k) return invalid("prefill_attention: null pointer");
  if (!aligned16(q) || !aligned16(k) || !aligned16(v) || reinterpret_cast<uintptr_t>(out) % 8)
    return invalid("prefill_attention: q, k, v must be 16-byte and out 8-byte aligned");
  const int hb = prefill_heads_per_block(Hq, Hkv);  // q heads per block
  const int64_t qtiles = (max_seqlen_q + block_queries(hb) - 1) / block_queries(hb);
  if (qtiles > INT32_MAX || num_seqs > INT32_MAX || num_blocks > INT32_MAX ||
      max_blocks * block_size > INT32_MAX || max_seqlen_k > INT32_MAX / 2)
    return invalid("prefill_attention: size too large");
  PrefillArgs g{};
  g.out = static_cast<uint16_t*>(out);
  g.q = static_cast<const uint16_t*>(q);
  g.k = static_cast<const uint16_t*>(k);
  g.v = static_cast<const uint16_t*>(v);
  g.cu_q = cu_seqlens_q;
  g.cu_k = cu_seqlens_k;
  g.bt = block_table;
  g.q_st = q_stride_token;
  g.q_sh = q_stride_head;
  g.k_st = block_table ? Hkv * D : k_stride_token;
  g.v_st = block_table ? Hkv * D : v_stride_token;
  g.o_st = out_stride_token;
  g.o_sh = out_stride_head;
  g.Hkv = int(Hkv);
  g.G = int(Hq / Hkv);
  g.bs = int(block_size);
  g.num_blocks = int(num_blocks);
  g.max_blocks = int(max_blocks);
  g.scale_log2 = scale * 1.4426950408889634f;
  g.causal = causal ? 1 : 0;
  g.qtiles = int(qtiles);
  g.nhg = int(Hq / hb);
  g.lq_skip = 0;
  g.Hq = int(Hq);
  g.ws_rows = total_q;
  g.out_lines = aligned16(out) && out_stride_token % 8 == 0 && out_stride_head % 8 == 0;
  const int64_t base_blocks = qtiles * num_seqs * (Hq / hb);
  // split the keys over several blocks when the caller gave a large enough workspace
  g.splits = 1;
  g.split_len = int(std::max<int64_t>(max_seqlen_k, 1));
  const int64_t need = prefill_workspace_bytes(num_seqs, max_seqlen_q, max_seqlen_k, Hq, Hkv, D, total_q);
  if (workspace && reinterpret_cast<uintptr_t>(workspace) % 256 != 0)
    return invalid("prefill_attention: workspace must be 256-byte aligned");
  if (need > 0 && workspace && workspace_size >= kAttnCounterBytes + need) {
    prefill_split_policy(base_blocks, max_seqlen_k, g.splits, g.split_len);
    g.ws = reinterpret_cast<float*>(static_cast<char*>(workspace) + kAttnCounterBytes);
  }
  const int64_t blocks = base_blocks * g.splits;
  if (blocks + num_seqs * Hkv > INT32_MAX) return invalid("prefill_attention: size too large");
  const dim3 block(static_cast<unsigned>(kThreads));
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bool paged = block_table != nullptr;
  // With the cache (a mixed step, a prefix-cache chunk), sequences with at most 16 / G queries -- the decode
  // requests of a mixed step -- run in the paged decode kernel, one block per (sequence, kv head) streaming its
  // keys; the prefill kernel's blocks for them return at once.
  const int64_t qs = paged ? short_queries(num_seqs, total_q, Hq, Hkv, max_seqlen_q) : 0;
  if (qs > 0) {
    g.lq_skip = int(qs);
    // its key splits use the part of the workspace after the prefill kernel's records
    const int64_t off = decode_workspace_offset(need);
    float* dws = workspace && workspace_size > off ? reinterpret_cast<float*>(static_cast<char*>(workspace) + off)
                                                   : nullptr;
    // When some sequence has more queries the prefill kernel is launched and its blocks of the short sequences run
    // their decode attention (unsplit) alongside the prefill tiles; otherwise the decode kernel runs alone, its
    // contexts split over blocks with the workspace
    const int64_t G = Hq / Hkv;
    if (max_seqlen_q > g.lq_skip && G * g.lq_skip <= 16) {
      DecodeArgs& d = g.dec;
      d.out = static_cast<uint16_t*>(out), d.q = static_cast<const uint16_t*>(q);
      d.kc = static_cast<const uint16_t*>(k), d.vc = static_cast<const uint16_t*>(v), d.bt = block_table;
      d.q_len = g.lq_skip, d.Hkv = int(Hkv), d.G = int(G), d.bs = int(block_size), d.num_blocks = int(num_blocks);
      d.max_blocks = int(max_blocks);
      d.q_st = q_stride_token, d.q_sh = q_stride_head, d.o_st = out_stride_token, d.o_sh = out_stride_head;
      d.scale_log2 = scale * 1.4426950408889634f, d.causal = causal ? 1 : 0;
      d.splits = 1, d.split_len = int(max_blocks * block_size);
      d.cu_q = cu_seqlens_q, d.cu_k = cu_seqlens_k;
      // each pair's context cut in two when the workspace holds the counters and the halves' records: the pairs
      // stream on twice the CUs (the second halves in blocks appended to the grid, which start as the short
      // sequences' idle query-tile blocks exit -- not in those blocks, which would hold back the long sequence's
      // last tiles), merged inside the launch
      if (inline_halves(num_seqs, Hkv) && dws != nullptr &&
          workspace_size - off >= inline_halves_bytes(num_seqs, Hkv, D)) {
        d.halves = 1, d.num_seqs = int(num_seqs);
        d.counters = static_cast<uint32_t*>(workspace), d.ws = dws;
        d.rec_splits = 2, d.rec_stride = decode_record_stride(16, D, true);
        g.dec_extra = int(num_seqs * Hkv);
      }
      g.dec_inline = 1;
    }
    if (!g.dec_inline) {
      return paged_decode_varlen(static_cast<uint16_t*>(out), static_cast<const uint16_t*>(q),
                                 static_cast<const uint16_t*>(k), static_cast<const uint16_t*>(v), block_table,
                                 cu_seqlens_q, cu_seqlens_k, int(num_seqs), g.lq_skip, int(Hq), int(Hkv), int(D),
                                 int(block_size), int(num_blocks), int(max_blocks), q_stride_token, q_stride_head,
                                 out_stride_token, out_stride_head, scale, causal, dws,
                                 dws ? workspace_size - off : 0, s);
    }
  }
  // prefill_wide_kernel: calls over the paged cache that leave no sequence to the decode attention, with key tiles
  // within cache blocks and enough of them per block. That is one sequence, or several with more than 16 q heads per kv
  // head (32 / 1 heads, us: 4 sequences of 30 .. 900 queries over up to 4000 keys 152 -> 105, 32 one-query sequences of
  // 1000 keys and 500 queries over 3000 189 -> 137), in grid order. Its start costs more: with two heads per block 17
  // queries over 17 keys took 9.0 us against 8.4, 64 over 64 10.3 against 10.4, 128 over 128 13.2 against 14.1; with one
  // (twice the queries) 128 over 128 12.2 against 12.3, 130 over 200 16.4 against 16.1, 256 over 256 17.3 against 19.1.
  const bool wide = paged && D == 128 && g.lq_skip == 0 && block_size % kBK == 0 && Hkv < (int64_t(1) << 16) &&
                    g.split_len >= 4 * kBK / hb;
  // block_plan: lanes for sequences, eighths of the head groups for XCDs. 24 prompts of 30 .. 2100 tokens 259 ->
  // 209-217 us, 48 decode requests and a chunk of 464 queries 87 -> 70, 7 and a chunk of 2000 over 5000 cached keys
  // 486 -> 278 (q/k norm kernel included). It costs a block ~0.5 us and gives nothing where all blocks start at once (a
  // grid of at most one block per CU: 5 prompts of up to 300 tokens 13.8 us without, 14.4 with it) or where the
  // sequences are in its order already (of one length, or nearly: 64 of 1000 .. 1100 tokens 463 without, 476 with it, 8
  // of 500 .. 520 23.4 and 24.5). Of 154 other calls it made 28 slower by 1 .. 6 %, by the luck of the grid order, and
  // 85 faster by 2 .. 71 %.
  const bool ragged = double(total_q) < 0.9 * double(num_seqs) * double(max_seqlen_q);
  g.plan = !wide && ragged && num_seqs <= 64 && g.nhg % 8 == 0 && g.splits == 1 && base_blocks > 256 && qtiles < 256
               ? int(num_seqs)
               : 0;
  const dim3 grid(static_cast<unsigned>(blocks + g.dec_extra));
#define NVHIP_PREFILL_LAUNCH(DD, PG, HBV)                                                                      \
  do {                                                                                                         \
    if (g.plan) hipLaunchKernelGGL((prefill_attention_kernel<DD, PG, HBV, true>), grid, block, 0, s, g);       \
    else hipLaunchKernelGGL((prefill_attention_kernel<DD, PG, HBV, false>), grid, block, 0, s, g);             \
  } while (0)
  if (wide && hb == 2) hipLaunchKernelGGL((prefill_wide_kernel<2>), grid, dim3(kWideThreads), 0, s, g);
  else if (wide) hipLaunchKernelGGL((prefill_wide_kernel<1>), grid, dim3(kWideThreads), 0, s, g);
  else if (hb == 2 && D == 64 && paged) NVHIP_PREFILL_LAUNCH(64, true, 2);
  else if (hb == 2 && D == 64) NVHIP_PREFILL_LAUNCH(64, false, 2);
  else if (hb == 2 && paged) NVHIP_PREFILL_LAUNCH(128, true, 2);
  else if (hb == 2) NVHIP_PREFILL_LAUNCH(128, false, 2);
  else if (D == 64 && paged) NVHIP_PREFILL_LAUNCH(64, true, 1);
  else if (D == 64) NVHIP_PREFILL_LAUNCH(64, false, 1);
  else if (paged) NVHIP_PREFILL_LAUNCH(128, true, 1);
  else NVHIP_PREFILL_LAUNCH(128, false, 1);
#undef NVHIP_PREFILL_LAUNCH
  if (int rc = check_launch("prefill_attention")) return rc;
  if (g.splits == 1) return NVHIP_OK;
  const int64_t per_seq = (max_seqlen_q * Hq + 7) / 8;  // blocks of 4 waves of two (query, head) pairs per sequence
  if (num_seqs * per_seq > INT32_MAX) return invalid("prefill_attention: size too large");
  const dim3 cgrid(static_cast<unsigned>(num_seqs * per_seq));
  if (D == 64) hipLaunchKernelGGL((prefill_combine<64>), cgrid, dim3(256), 0, s, g, int(per_seq));
  else hipLaunchKernelGGL((prefill_combine<128>), cgrid, dim3(256), 0, s, g, int(per_seq));
  return check_launch("prefill_attention (combine)");
}
