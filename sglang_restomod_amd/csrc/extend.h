// What the extend kernels share: their arguments, the work list of row tiles, and the key
// pieces that row tiles are cut into (planning and merge).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"

namespace ma {

// One entry of the work list: sequence in the low 32 bits, row tile in the high 32;
// -1 (sequence -1) past the last tile.
__host__ __device__ constexpr int64_t row_tile_item(int seq, int tile) {
  return (int64_t)(((uint64_t)(uint32_t)tile << 32) | (uint32_t)seq);
}

// Key pieces of row tiles, planned where a batch has too few row tiles to fill the chip or
// to balance over it (plan_pieces below). A piece that is not a whole row tile leaves its
// rows' normalised O and log2 LSE in slot `slot`; extend_merge combines the slots of a tile.
struct ExtendPiece {
  int seq, tile;     // sequence (-1: no piece) and row tile
  int first, count;  // key tiles [first, first + count) of the row tile's range
  int slot;          // partial slot, or -1 when the piece is the whole row tile
  int pad[3];
};
struct ExtendMerge {
  int seq, tile;   // sequence (-1: none) and row tile
  int slot, parts; // its pieces' slots: slot .. slot + parts - 1
};
struct ExtendPieces {
  const ExtendPiece* list;  // the plan kernel's list, or null
  ExtendMerge* merges;      // the cut row tiles, then entries with sequence -1
  int merge_capacity;
  int shares;       // CUs per kv head, or 0
  float slot_cost;  // piece_slot_cost of the kernel
  int capacity;     // pieces per kv head that the list, the grid and the partial slots hold
  float* o;         // [slot][kv head][row of the tile][D] fp32
  float* lse;       // [slot][kv head][row of the tile]
};

struct ExtendArgs {
  const void* q;
  int64_t q_stride_tok, q_stride_head;
  const void* k;
  const void* v;
  int64_t kv_stride_row, kv_stride_head;
  TokenTable tt;
  const int64_t* row_index;
  const int32_t* seq_lens;
  const int32_t* qsl;
  const int32_t* prefix;
  int num_tokens;        // rows of q and out: query rows are clamped into [0, num_tokens)
  int batch, hq, hkv, group;
  // pieces.shares == 0: whole row tiles, from the work list `items` (row_tile_item). Else key
  // pieces: from pieces.list, or where that is null each workgroup plans its own (plan_direct).
  const int64_t* items;
  ExtendPieces pieces;
  int causal, window;
  float scale_log2;
  float v_scale;
  void* out;
  int64_t out_stride_tok, out_stride_head;  // elements of the output dtype
  int out_f32;                              // out holds fp32 (else the query dtype)
  int head_dim;                             // the rows' head dim (<= the kernel's D when padded)
  int chunks;                               // 16-byte chunks of one K/V row at head_dim
};

// Keys [lo, hi) that some row of the bm-row tile starting at row r0 of a sequence may see.
struct KeyRange {
  int lo, hi;
};
__device__ __forceinline__ KeyRange row_tile_keys(int r0, int bm, int ntok, int group, int prefix, int seq,
                                                  int causal, int window) {
  const int t_first = r0 / group;
  const int t_last = min(ntok - 1, (r0 + bm - 1) / group);
  KeyRange k;
  k.lo = window >= 0 ? max(0, prefix + t_first - window) : 0;
  k.hi = causal ? min(seq, prefix + t_last + 1) : seq;
  return k;
}

// ---- key pieces ----
// One workgroup walking a row tile's whole key range leaves compute units idle when the
// batch has few row tiles: a chunk of 1,021 tokens of one prompt at 32 / 8 heads has 128
// workgroups for 256 CUs, four short turns about 50. So a call with at most one row tile
// per CU (by its token count) may have them cut into key pieces. Per call, whole row tiles
// against pieces: that chunk 28,001 tokens into its prompt 782 -> 455 us; 4 turns of 9-130
// tokens over 64-1,500 36.4 -> 26.0 us; 800 tokens at 8 / 1 heads after 8,000 253 -> 60 us.
// Beyond one round of row tiles the pieces gained nothing that their merge did not cost:
// 16 sequences of 300 tokens (75 row tiles, 32 CUs per kv head) 127 us either way.
constexpr int kSplitSlotRounds = 2;  // pieces per CU: a partial takes 128 KB at D = 128 and 256, 256 KB above
constexpr int kSplitMinTiles = 4;    // least key tiles of a piece (a workgroup's start and end cost about 3)
constexpr int kDirectItems = 128;    // row tiles up to which each workgroup plans for itself, two per lane
constexpr int kDirectBatch = 64;     // ... and sequences, one per lane
constexpr int kSplitMaxItems = 1024; // row tiles the plan holds one per thread


// Row tiles of bm rows of a sequence with ntok query tokens.
__device__ __forceinline__ int seq_row_tiles(int ntok, int group, int bm) {
  return ntok > 0 ? (int)(((int64_t)ntok * group + bm - 1) / bm) : 0;
}

// Estimated time, in key tiles, of n pieces of at most `longest` of `all` key tiles on
// `shares` CUs per kv head: the longest piece, or the mean piece times the rounds the
// pieces make, each with a workgroup's start and end, plus the writing and reading back of
// the `split` pieces that leave partials, `slot_cost` for one per CU.
__device__ __forceinline__ float pieces_cost(float all, float n, float longest, float split, float shares,
                                             float slot_cost) {
  constexpr float kStart = 5.f;  // a workgroup's start and end: 6 to 8 us, a key tile 0.9 to 1.9 us
  const float mean = (all + kStart * n) / fmaxf(n, 1.f);
  return fmaxf(longest + kStart, mean * ceilf(n / shares)) + slot_cost * split / shares;
}

// The wave's maximum of values >= 0.
__device__ __forceinline__ int wave_max(int x) {
  x = max(x, dpp0<0x111, 0xf>(x));
  x = max(x, dpp0<0x112, 0xf>(x));
  x = max(x, dpp0<0x114, 0xf>(x));
  x = max(x, dpp0<0x118, 0xf>(x));
  x = max(x, dpp0<0x142, 0xa>(x));
  x = max(x, dpp0<0x143, 0xc>(x));
  return __builtin_amdgcn_readlane(x, 63);
}
// Pieces of at most cap key tiles of a row tile of c (at least one): max(1, ceil(c / cap)),
// exact below 2^24 (a reciprocal, then one step either way).
__device__ __forceinline__ int piece_count(int c, int cap) {
  const int x = c + cap - 1;
  int q = (int)((float)x * __builtin_amdgcn_rcpf((float)cap));
  const int r = x - q * cap;
  q += r >= cap ? 1 : r < 0 ? -1 : 0;
  return max(q, 1);
}

// The piece of list position `w` (per kv head), planned by the wave itself: for batches of
// at most kDirectItems row tiles and kDirectBatch sequences, which then need no plan kernel
// (about 6 us of a call that takes 20). Every wave of every workgroup computes the same plan
// from the same numbers. The first workgroup of kv head 0 lists the cut tiles in `merges`.
template <int BM, int BN>
__device__ __forceinline__ ExtendPiece plan_direct(const ExtendArgs& a, int w, int h) {
  constexpr int kPer = kDirectItems / 64;
  const int lane = lane_id();
  int nt = 0, ntok = 0, seq = 0, prefix = 0;
  if (lane < a.batch) {
    ntok = clamp_query_rows(gptr(a.qsl)[lane], gptr(a.qsl)[lane + 1], a.num_tokens).ntok;
    seq = gptr(a.seq_lens)[lane];
    prefix = a.prefix ? gptr(a.prefix)[lane] : seq - ntok;
    nt = seq_row_tiles(ntok, a.group, BM);
  }
  const int incl = wave_scan(nt);
  const int start = incl - nt;
  const int m = min(__builtin_amdgcn_readlane(incl, 63), min(kDirectItems, a.pieces.capacity));
  // row tiles kPer * lane + x: their sequences and key tiles
  int b[kPer], rt[kPer], c[kPer];
  int cmax = 0, csum = 0;
#pragma unroll
  for (int x = 0; x < kPer; ++x) b[x] = 0;
  for (int s = 1; s < a.batch; ++s) {
    const int first = __builtin_amdgcn_readlane(start, s);
#pragma unroll
    for (int x = 0; x < kPer; ++x)
      if (kPer * lane + x >= first) b[x] = s;
  }
#pragma unroll
  for (int x = 0; x < kPer; ++x) {
    rt[x] = kPer * lane + x - shfl_i(start, b[x]);
    const KeyRange kr = row_tile_keys(rt[x] * BM, BM, shfl_i(ntok, b[x]), a.group, shfl_i(prefix, b[x]),
                                      shfl_i(seq, b[x]), a.causal, a.window);
    c[x] = (kPer * lane + x < m && kr.hi > kr.lo) ? (kr.hi - kr.lo + BN - 1) / BN : 0;
    cmax = max(cmax, c[x]);
    csum += c[x];
  }
  cmax = wave_max(cmax);
  const int all = __builtin_amdgcn_readlane(wave_scan(csum), 63);
  // this lane's pieces at a cap
  int parts[kPer];
  auto cut = [&](int cap) __attribute__((always_inline)) -> int {
    int n = 0;
#pragma unroll
    for (int x = 0; x < kPer; ++x) {
      parts[x] = kPer * lane + x < m ? piece_count(c[x], cap) : 0;
      n += parts[x];
    }
    return n;
  };
  // Three candidates: whole tiles, and the least caps with which the pieces make one and
  // two rounds on the CUs.
  int cap = max(cmax, 1);
  float est = pieces_cost((float)all, (float)m, (float)cmax, 0.f, (float)a.pieces.shares, a.pieces.slot_cost);
#pragma unroll 1
  for (int r = 1; r <= 2; ++r) {
    const int room = min(r * a.pieces.shares, a.pieces.capacity);
    if (m > room || cmax <= kSplitMinTiles) continue;
    int lo = kSplitMinTiles, hi = cmax;  // the least cap whose pieces fit; cmax does
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      const int n = __builtin_amdgcn_readlane(wave_scan(cut(mid)), 63);
      if (n <= room) hi = mid;
      else lo = mid + 1;
    }
    const int n = __builtin_amdgcn_readlane(wave_scan(cut(lo)), 63);
    int split = 0, longest = 0;
#pragma unroll
    for (int x = 0; x < kPer; ++x) {
      split += parts[x] > 1 ? parts[x] : 0;
      longest = max(longest, parts[x] > 0 ? piece_count(c[x], parts[x]) : 0);
    }
    split = __builtin_amdgcn_readlane(wave_scan(split), 63);
    longest = wave_max(longest);
    const float e = pieces_cost((float)all, (float)n, (float)longest, (float)split, (float)a.pieces.shares,
                                a.pieces.slot_cost);
    if (e < est) {
      est = e;
      cap = lo;
    }
  }
  // list position of each tile's first piece: the last tiles come first (in a causal batch
  // the longer ones)
  const int mine = cut(cap);
  const int upto = wave_scan(mine);
  int pos[kPer];
  pos[kPer - 1] = __builtin_amdgcn_readlane(upto, 63) - upto;
#pragma unroll
  for (int x = kPer - 2; x >= 0; --x) pos[x] = pos[x + 1] + parts[x + 1];
  ExtendPiece p;
  p.seq = -1;
  p.tile = p.first = p.count = 0;
  p.slot = -1;
  if (w == 0 && h == 0 && (int)threadIdx.x < 64) {
    int4 MA_GLOBAL* mp = reinterpret_cast<int4 MA_GLOBAL*>(gptr_mut(a.pieces.merges));
    int ncut = 0;
#pragma unroll
    for (int x = 0; x < kPer; ++x) ncut += parts[x] > 1 ? 1 : 0;
    const int upto_cut = wave_scan(ncut);
    int e = upto_cut - ncut;
#pragma unroll
    for (int x = 0; x < kPer; ++x) {
      if (parts[x] > 1 && e < a.pieces.merge_capacity) {
        mp[e].x = b[x];
        mp[e].y = rt[x];
        mp[e].z = pos[x];
        mp[e].w = parts[x];
      }
      e += parts[x] > 1 ? 1 : 0;
    }
    for (int i = __builtin_amdgcn_readlane(upto_cut, 63) + lane; i < a.pieces.merge_capacity; i += 64) mp[i].x = -1;
  }
#pragma unroll
  for (int x = 0; x < kPer; ++x) {
    const uint64_t hit = __builtin_amdgcn_ballot_w64(w >= pos[x] && w < pos[x] + parts[x]);
    if (hit) {
      const int L = __builtin_ctzll(hit);
      const int cx = __builtin_amdgcn_readlane(c[x], L);
      const int np = __builtin_amdgcn_readlane(parts[x], L);
      const int k = w - __builtin_amdgcn_readlane(pos[x], L);
      const int lo = (int)((int64_t)cx * k / np);
      p.seq = __builtin_amdgcn_readlane(b[x], L);
      p.tile = __builtin_amdgcn_readlane(rt[x], L);
      p.first = lo;
      p.count = (int)((int64_t)cx * (k + 1) / np) - lo;
      p.slot = np > 1 ? w : -1;
    }
  }
  return p;
}

// Merge of the row tiles that were cut into key pieces: 1024 / D rows of one tile and kv
// head at a time per workgroup, D / 4 threads per row, four dims each. A running maximum of
// the log2 LSEs rescales the sum of the pieces' normalised O, so one pass reads each piece
// once (four pieces' loads in flight). Pieces in which a row saw no key (LSE -inf) weigh 0.
// The host does not know which tiles are cut, so the grid is one the chip holds at once, and
// its workgroups walk the listed tiles (the list ends at the first empty entry): a workgroup
// for every row set that could be cut cost 9 us where none was (48 sequences at 32 / 32 heads).
constexpr int kMergeGrid = 2048;  // eight workgroups of four waves on each of 256 CUs

template <int D, int kBM, bool QBF16>
__global__ __launch_bounds__(256) void extend_merge(const ExtendArgs args) {
  const ExtendArgs a = args;
  constexpr int kTPR = D / 4;              // threads per row
  constexpr int kRows = 256 / kTPR;        // rows per step of a workgroup
  constexpr int kBlocks = kBM / kRows;     // steps per row tile and kv head
  // where nothing is cut, out before the loop's constants are set up (0.4 us of the call)
  if (cptr(reinterpret_cast<const int*>(a.pieces.merges + (int)blockIdx.x / kBlocks / a.hkv))[0] < 0) return;
  const int d = ((int)threadIdx.x % kTPR) * 4;
  const int64_t pitch = (int64_t)a.hkv * kBM;  // rows of one slot
  const int units = a.pieces.merge_capacity * a.hkv * kBlocks;
  for (int u = (int)blockIdx.x; u < units; u += (int)gridDim.x) {
    const int blk = u % kBlocks;
    const int rest = u / kBlocks;
    const int h = rest % a.hkv;
    const int MA_CONST* e = cptr(reinterpret_cast<const int*>(a.pieces.merges + rest / a.hkv));
    const int b = e[0];
    if (b < 0) return;
    const int rt = e[1], slot = e[2], parts = e[3];
    const QueryRows qr = clamp_query_rows(cptr(a.qsl)[b], cptr(a.qsl)[b + 1], a.num_tokens);
    const int r = blk * kRows + (int)threadIdx.x / kTPR;
    const int R = rt * kBM + r;
    const int t = R / a.group;
    const int g = R - t * a.group;
    if (d >= a.head_dim || t >= qr.ntok) continue;
    const int64_t row0 = ((int64_t)slot * a.hkv + h) * kBM + r;
    const float MA_GLOBAL* lse = gptr(a.pieces.lse) + row0;
    const float MA_GLOBAL* po = gptr(a.pieces.o) + row0 * D + d;
    float m = -INFINITY, w = 0.f;
    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int p = 0; p < parts; ++p) {
      const float l = lse[p * pitch];
      const f32x4 o = *reinterpret_cast<const f32x4 MA_GLOBAL*>(po + p * pitch * D);
      const float m_new = fmaxf(m, l);
      const float base = (m_new == -INFINITY) ? 0.f : m_new;
      const float s_old = __builtin_amdgcn_exp2f(m - base);
      const float s_new = __builtin_amdgcn_exp2f(l - base);
      acc = acc * s_old + o * s_new;
      w = w * s_old + s_new;
      m = m_new;
    }
    const float inv = (w > 0.f) ? a.v_scale / w : 0.f;
    const int64_t off = (int64_t)(qr.tok0 + t) * a.out_stride_tok + (int64_t)(h * a.group + g) * a.out_stride_head + d;
    store_out4<QBF16>(a.out, off, acc, inv, a.out_f32);
  }
}

// Extend above 256 dims (extend_wide.hip): rows per workgroup, keys per tile, and the launch
// of `grid` workgroups on validated arguments.
constexpr int kWideDim = 512;
constexpr int kWideRows = 128;
constexpr int kWideKeys = 32;
hipError_t extend_wide_launch(bool qbf16, int kv, dim3 grid, hipStream_t st, const ExtendArgs& a);

}  // namespace ma
