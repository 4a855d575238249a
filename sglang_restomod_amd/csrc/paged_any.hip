// Paged decode and linear verify at the head dims the tuned kernels do not take: every
// multiple of 16 from 16 to 512 other than 64, 128 and 256 (the reference's paged kernels
// take any head dim, with a default tile configuration and a tuned one for 512:
// sglang_restomod/attention/v100/tilelang/_kernels_paged.py:397-418; above 256 its linear
// verify also runs on the ordinary paged kernel, _paged_adapter.py:612-616), and small
// decodes at every head dim.
//
// A wave computes the scores of 16 query rows (token, GQA head) of one sequence and kv
// head, 16 keys at a time:
//   - scores S^T = K Q^T on 16x16x32 MFMAs (the query's 16-bit type; fp8 K converted),
//     so each lane holds four keys of one row: the B operand of the 16x16x16 fp16 MFMA
//     of O^T += V^T P^T, whose A operand is read transposed (ds_read_b64_tr_b16) from
//     fp16 V rows in LDS,
//   - an online softmax with the tuned kernels' lazy rescale (kLazyRescale).
// The four waves of a workgroup hold the same 16 rows and take a quarter of their 16-key
// tiles each, K straight into operand registers and V through the wave's own LDS rows,
// then merge through LDS.
// The kernel is as wide as the next of 64, 128, 256 and 512: lanes past the head dim
// read the row's last dims again (every load is unconditional), which meet Q's zeros in
// the scores and fill output dims that are never stored.
#include "capi_internal.h"
#include "paged_any.h"

namespace ma {

typedef __attribute__((__vector_size__(4 * sizeof(_Float16)))) _Float16 f16x4;

template <bool FP8>
struct AnyVRaw;  // one V unit (8 elements) as loaded
template <>
struct AnyVRaw<false> {
  typedef u32x4 type;
};
template <>
struct AnyVRaw<true> {
  typedef u32x2 type;
};

// a register buffer index, fixed at compile time
template <int N>
struct AnyIdx {
  static constexpr int v = N;
};

// Two workgroups share a CU where the registers allow it.
template <int DP>
constexpr int any_wg_per_cu() {
  return DP >= 256 ? 1 : 2;
}

template <int DP, bool QBF16, int KV>
__global__ __launch_bounds__(kAnyWaves * 64, any_wg_per_cu<DP>()) void any_kernel(const AnyArgs args) {
  const AnyArgs a = args;  // local copy: the lambdas capture by reference
  constexpr bool kFp8 = (KV == DT_E4M3 || KV == DT_E5M2);
  constexpr int KK = DP / 32;                   // QK MFMA steps
  constexpr int DB = DP / 16;                   // PV MFMA steps, 16 output dims each
  constexpr int kElt = kFp8 ? 1 : 2;            // bytes of one K/V element
  constexpr int kKL = kFp8 ? KK / 2 : KK;       // 16-byte K loads per lane per tile
  constexpr int kRowL = DP * 2 + 32;            // LDS bytes of one fp16 V row, padded: row t
                                                // starts 32 t bytes into a 256-byte bank period
  constexpr int kUnits = DP / 8;                // 8-element V units per row
  constexpr int kUL = kUnits * kAnyKeys / 64;   // V units per lane per tile
  static_assert(kUL >= 1 && (kUnits * kAnyKeys) % 64 == 0, "whole V units per lane");
  static_assert(!kFp8 || KK % 2 == 0, "fp8 K loads cover two QK steps");
  typedef typename AnyVRaw<kFp8>::type VRaw;

  // Decode and verify at the widest head dim with fp16 Q and KV keep Q in LDS (rows padded
  // by 16 bytes so the 16 rows of an operand read fall in different banks): in registers
  // it spilled. bf16 and fp8 KV keep Q in registers (1-3% faster at D=320 and 512 than
  // reading it from LDS every tile).
  constexpr bool kQLds = DP >= 512 && !kFp8 && !QBF16;
  constexpr int kQRow = DP * 2 + 16;
  constexpr int kVBlock = kAnyKeys * kRowL;            // one wave's V rows
  constexpr int kQBlock = kQLds ? kAnyRows * kQRow : 0;  // one wave's Q rows
  constexpr int kSmem = kAnyWaves * (kVBlock + kQBlock);
  // When the four waves split one row block's keys, their partial O meet in the same
  // memory after the loop, kBPR 16-column blocks (1 KiB per wave each) at a time.
  constexpr int kBPR = (DB * kAnyWaves * 1024 <= kSmem) ? DB
                       : (DB / 2 * kAnyWaves * 1024 <= kSmem) ? DB / 2
                       : (DB / 4 * kAnyWaves * 1024 <= kSmem) ? DB / 4 : DB / 8;
  static_assert(kBPR >= 1 && kBPR * kAnyWaves * 1024 <= kSmem, "merge rounds fit the kernel's LDS");
  __shared__ __attribute__((aligned(256))) unsigned char smem[kSmem];
  __shared__ float mrow[kAnyWaves][2][kAnyRows];  // each wave's row max and row sum of p
  int64_t piece_slot = 0;  // decode with pieces > 1: where this workgroup's partial goes

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int c = lane & 15;
  const int j = lane >> 4;
  const int D = a.head_dim;
  const int G = a.group;
  const uint32_t smem_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem;
  const uint32_t lds_base = smem_base + wave * kVBlock;                          // this wave's V rows
  const uint32_t q_base = smem_base + kAnyWaves * kVBlock + wave * kQBlock;      // and Q rows

  // first dim of QK step kk for lane group j (fp8: one 16-byte load covers two steps)
  auto qdim = [&](int kk) -> int {
    if constexpr (kFp8) return (kk >> 1) * 64 + j * 16 + (kk & 1) * 8;
    else return kk * 32 + j * 8;
  };
  const unsigned char MA_GLOBAL* kbase = gptr(reinterpret_cast<const unsigned char*>(a.k));
  const unsigned char MA_GLOBAL* vbase = gptr(reinterpret_cast<const unsigned char*>(a.v));
  const uint32_t row_bytes32 = (uint32_t)(a.kv_stride_row * kElt);  // the hosts check it fits
  const int page_mask = (1 << a.tt.page_shift) - 1;

  // The 16 rows r0 .. r0 + 15 of sequence b, kv head h: the four waves take quarter `split`
  // of their key tiles each, merging at the end.
  auto rows = [&](int b, int h, int r0, int pieces, int split) __attribute__((always_inline)) {
    int tok0, ntok;
    if (a.qsl) {
      const QueryRows qr = clamp_query_rows(cptr(a.qsl)[b], cptr(a.qsl)[b + 1], a.num_tokens);
      tok0 = qr.tok0;
      ntok = qr.ntok;
    } else {
      tok0 = b;
      ntok = b < a.num_tokens ? 1 : 0;
    }
    if (r0 >= ntok * G) return;  // the same for every wave of the workgroup
    const int seq = max(cptr(a.seq_lens)[b], 0);
    const int prefix = a.prefix ? cptr(a.prefix)[b] : seq - ntok;
    const int64_t seq_row = a.row_index ? cptr(a.row_index)[b] : (int64_t)b;
    const int64_t head_off = (int64_t)h * a.kv_stride_head * kElt;

    // this lane's row (column c of every MFMA result)
    const int r = r0 + c;
    const int t = r / G;
    const int g = r - t * G;
    const bool real = t < ntok;
    const int qpos = prefix + t;
    const int lo_r = (real && a.window >= 0) ? max(0, qpos - a.window) : 0;
    const int hi_r = real ? (a.causal ? min(seq, qpos + 1) : seq) : 0;
    u32x4 qv[kQLds ? 1 : KK];
    const uint32_t qa = q_base + c * kQRow + j * 16;
    {
      const uint16_t MA_GLOBAL* qp = gptr(reinterpret_cast<const uint16_t*>(a.q)) +
                                     (int64_t)(tok0 + (real ? t : 0)) * a.q_stride_tok +
                                     (int64_t)(h * G + g) * a.q_stride_head;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) {
        const int d0 = qdim(kk);
        const u32x4 qf = (real && d0 < D) ? *reinterpret_cast<const u32x4 MA_GLOBAL*>(qp + d0) : u32x4{0, 0, 0, 0};
        if constexpr (kQLds) *reinterpret_cast<__attribute__((address_space(3))) u32x4*>((uintptr_t)(qa + kk * 64)) = qf;
        else qv[kk] = qf;
      }
    }
    // keys any of the rows may see
    const int t_first = r0 / G;
    const int t_last = min(ntok - 1, (r0 + kAnyRows - 1) / G);
    const int key_lo = a.window >= 0 ? max(0, prefix + t_first - a.window) : 0;
    const int key_hi = a.causal ? min(seq, prefix + t_last + 1) : seq;
    const int nt = key_hi > key_lo ? (key_hi - key_lo + kAnyKeys - 1) / kAnyKeys : 0;
    // split: this wave's quarter of the workgroup's key piece (pieces x 4 equal shares)
    const int parts = kAnyWaves * pieces;
    const int i_lo = (int)((int64_t)split * nt / parts);
    const int i_hi = (int)((int64_t)(split + 1) * nt / parts);

    float m_run = -INFINITY;
    float lsum = 0.f;  // this lane's share of its row's sum of p (keys 4j .. 4j + 3 of each tile)
    f32x4 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};

    // lane l holds tile i's key l % kAnyKeys: its page, then its slot
    auto key_pos = [&](int i) __attribute__((always_inline)) -> int {
      return min(key_lo + i * kAnyKeys + (lane & (kAnyKeys - 1)), key_hi - 1);
    };
    auto page_load = [&](int i) __attribute__((always_inline)) -> int {
      return gptr(a.tt.table)[seq_row * a.tt.stride + (key_pos(i) >> a.tt.page_shift)];
    };
    // Loads are unconditional, so the compiler's wait counts stay exact (a load behind a
    // branch would make it wait for every load in flight): lanes past the head dim read the
    // row's last dims again. Those finite values meet Q's zeros in the scores and fill
    // output dims that are never stored.
    auto slot_of = [&](int i, int page) __attribute__((always_inline)) -> int {
      return (page << a.tt.page_shift) | (key_pos(i) & page_mask);
    };
    auto load_k = [&](int myslot, u32x4 (&kr)[kKL]) __attribute__((always_inline)) {
      const int kslot = shfl_i(myslot, c);
      const unsigned char MA_GLOBAL* krow = kbase + (uint64_t)(uint32_t)kslot * row_bytes32 + head_off;
#pragma unroll
      for (int x = 0; x < kKL; ++x) {
        const int d0 = min(kFp8 ? x * 64 + j * 16 : x * 32 + j * 8, D - (kFp8 ? 16 : 8));
        kr[x] = *reinterpret_cast<const u32x4 MA_GLOBAL*>(krow + d0 * kElt);
      }
    };
    auto load_v = [&](int myslot, VRaw (&vr)[kUL]) __attribute__((always_inline)) {
#pragma unroll
      for (int x = 0; x < kUL; ++x) {
        const int u = lane + 64 * x;
        const int tr = u / kUnits;
        const int q = min(u - tr * kUnits, D / 8 - 1);
        const int vs = shfl_i(myslot, tr);
        vr[x] = *reinterpret_cast<const VRaw MA_GLOBAL*>(vbase + (uint64_t)(uint32_t)vs * row_bytes32 + head_off + q * 8 * kElt);
      }
    };
    // V units -> fp16 -> this wave's LDS block, row-major with padded rows (the transposed
    // reads take 4 rows of one 32-byte column block per 16 lanes; the padding puts those
    // rows in different banks). Lane-constant base plus an immediate per unit.
    auto write_v = [&](const VRaw (&vr)[kUL]) __attribute__((always_inline)) {
      const uint32_t wa = lds_base + (lane / kUnits) * kRowL + (lane % kUnits) * 16;
#pragma unroll
      for (int x = 0; x < kUL; ++x) {
        u32x4 hv;
        if constexpr (kFp8) {
          hv = cvt8_fp8<KV, false>(vr[x][0], vr[x][1]);
        } else if constexpr (QBF16) {
#pragma unroll
          for (int w = 0; w < 4; ++w)
            hv[w] = pack_f16(__builtin_bit_cast(float, vr[x][w] << 16), __builtin_bit_cast(float, vr[x][w] & 0xffff0000u));
        } else {
          hv = vr[x];
        }
        *reinterpret_cast<__attribute__((address_space(3))) u32x4*>((uintptr_t)(wa + x * (64 / kUnits) * kRowL)) = hv;
      }
    };
    // scores of tile i: lane (c, j) holds keys 4j .. 4j + 3 of row c
    auto scores = [&](const u32x4 (&kr)[kKL]) __attribute__((always_inline)) -> f32x4 {
      f32x4 s = f32x4{0.f, 0.f, 0.f, 0.f};
      if constexpr (kFp8) {
#pragma unroll
        for (int x = 0; x < kKL; ++x) {
          u32x4 k0, k1;
          cvt16_fp8<KV, QBF16>(kr[x], k0, k1);
          s = mfma16t<QBF16>(k0, qv[2 * x], s);
          s = mfma16t<QBF16>(k1, qv[2 * x + 1], s);
        }
      } else {
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
          if constexpr (kQLds) {
            const u32x4 qf = *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>((uintptr_t)(qa + kk * 64));
            s = mfma16t<QBF16>(kr[kk], qf, s);
          } else
            s = mfma16t<QBF16>(kr[kk], qv[kk], s);
        }
      }
      return s;
    };
    // Online softmax of tile i's scores (lane (c, j): keys 4j .. 4j + 3 of row c). Gives p in
    // fp16; `moved` (the same in every lane) says whether some row's exponent base moved, and
    // then `alpha` is the factor the row's earlier O takes (1 for the others). The base moves
    // only when a row's max grew by more than 2^kLazyRescale in p.
    auto softmax = [&](int i, f32x4& s, u32x2& pk, float& alpha, bool& moved) __attribute__((always_inline)) {
      const int kb0 = key_lo + i * kAnyKeys + 4 * j;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (kb0 + e < lo_r || kb0 + e >= hi_r) s[e] = -INFINITY;
      float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
      alpha = 1.f;
      moved = __builtin_amdgcn_ballot_w64((mx - m_run) * a.scale_log2 > kLazyRescale) != 0;
      if (moved) {
        mx = fmaxf(mx, shfl_xor_f(mx, 16));
        mx = fmaxf(mx, shfl_xor_f(mx, 32));
        const float m_new = fmaxf(m_run, mx);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        alpha = __builtin_amdgcn_exp2f((m_run - m_use) * a.scale_log2);
        m_run = m_new;
        lsum *= alpha;
      }
      const float msc = (m_run == -INFINITY ? 0.f : m_run) * a.scale_log2;
      float p[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) p[e] = __builtin_amdgcn_exp2f(s[e] * a.scale_log2 - msc);
      const uint32_t p01 = pack_p16(p[0], p[1]), p23 = pack_p16(p[2], p[3]);
      pk = u32x2{p01, p23};
      // the row sum takes the rounded p, so that most of its rounding cancels in the quotient
      // (fp16 decode of 512 keys: error against float64 4.6e-4 -> 3.0e-4)
      const f16x2 one = {(_Float16)1.f, (_Float16)1.f};
      lsum = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, p01), one, lsum, false);
      lsum = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, p23), one, lsum, false);
    };
    // softmax and PV of tile i (its V in this wave's LDS rows at vt)
    auto finish = [&](int i, f32x4 s, uint32_t vt) __attribute__((always_inline)) {
      float alpha;
      bool moved;
      u32x2 pk;
      softmax(i, s, pk, alpha, moved);
      if (moved) {
#pragma unroll
        for (int db = 0; db < DB; ++db) o[db] *= alpha;
      }
      // O^T[d][row] += V^T[d][key] P^T[key][row], 16 dims per step; the transposed V reads
      // run one batch of kVB steps ahead, as in the scores
      const uint32_t vb = vt + (4 * j + (c >> 2)) * kRowL + (c & 3) * 8;
      constexpr int kVB = DB < 8 ? DB : 8;
      constexpr int kVNB = DB / kVB;
      u32x2 vf[2][kVB];
      auto vfetch = [&](int bb, int sl) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < kVB; ++x)
          vf[sl][x] = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) i16x4*)(uintptr_t)(vb + (bb * kVB + x) * 32)));
      };
      vfetch(0, 0);
#pragma unroll
      for (int bb = 0; bb < kVNB; ++bb) {
        if (bb + 1 < kVNB) vfetch(bb + 1, (bb + 1) & 1);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < kVB; ++x)
          o[bb * kVB + x] = __builtin_amdgcn_mfma_f32_16x16x16f16(
              __builtin_bit_cast(f16x4, vf[bb & 1][x]), __builtin_bit_cast(f16x4, pk), o[bb * kVB + x], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    };

    if (DP <= 128 && i_hi > i_lo) {
      // Up to 128 dims a tile is small and its compute short, so each wave keeps two tiles
      // in flight: step i issues the slot lookup of tile i+3, writes tile i's V to LDS,
      // loads tile i+2 into the buffers tile i-1 has left, and computes tile i. The
      // prologue issues its loads in the steps' order. Tiles past the last are the last
      // again (key positions clamp), so every step issues the same loads on every path.
      u32x4 kq[3][kKL];
      VRaw vq[3][kUL];
      const int pa = page_load(i_lo);
      const int pb = page_load(i_lo + 1);
      load_v(slot_of(i_lo, pa), vq[0]);
      load_k(slot_of(i_lo, pa), kq[0]);
      int pc = page_load(i_lo + 2);
      __builtin_amdgcn_sched_barrier(0);  // the lookup stays ahead of the loads after it
      load_v(slot_of(i_lo + 1, pb), vq[1]);
      load_k(slot_of(i_lo + 1, pb), kq[1]);
      auto step3 = [&](int i, auto cur_t) __attribute__((always_inline)) {
        constexpr int cur = decltype(cur_t)::v;
        constexpr int nx = (cur + 2) % 3;
        const int pn = page_load(i + 3);
        __builtin_amdgcn_sched_barrier(0);
        write_v(vq[cur]);
        const int sn = slot_of(i + 2, pc);
        load_v(sn, vq[nx]);
        load_k(sn, kq[nx]);
        finish(i, scores(kq[cur]), lds_base);
        pc = pn;
      };
      int i = i_lo;
#pragma unroll 1
      for (; i + 2 < i_hi; i += 3) {
        step3(i, AnyIdx<0>{});
        step3(i + 1, AnyIdx<1>{});
        step3(i + 2, AnyIdx<2>{});
      }
      if (i < i_hi) step3(i, AnyIdx<0>{});
      if (i + 1 < i_hi) step3(i + 1, AnyIdx<1>{});
    }
    if (DP > 128 && i_hi > i_lo) {
      // Step i issues the slot lookup of tile i+2, writes tile i's V to LDS and refills the
      // V registers with tile i+1, and loads tile i+1's K (into the other K buffer, or at
      // the widest head dims into the same one once tile i's scores have used it), so every
      // load has a tile's softmax and PV to land in. Tiles past the last are the last again
      // (key positions clamp), so every step issues the same loads on every path.
      constexpr bool kTwoK = DP <= 256;
      u32x4 ka[kKL], kb[kKL];
      VRaw vr[kUL];
      int page1 = page_load(i_lo);
      load_v(slot_of(i_lo, page1), vr);
      load_k(slot_of(i_lo, page1), ka);
      page1 = page_load(i_lo + 1);
      int page2;
      auto step = [&](int i, u32x4 (&kc)[kKL], u32x4 (&kn)[kKL]) __attribute__((always_inline)) {
        page2 = page_load(i + 2);
        write_v(vr);
        const int sn = slot_of(i + 1, page1);
        load_v(sn, vr);
        f32x4 s;
        if constexpr (kTwoK) {
          load_k(sn, kn);
          s = scores(kc);
        } else {
          s = scores(kc);
          load_k(sn, kc);
        }
        finish(i, s, lds_base);
        page1 = page2;
      };
      int i = i_lo;
#pragma unroll 1
      for (; i + 1 < i_hi; i += 2) {
        if constexpr (kTwoK) {
          step(i, ka, kb);
          step(i + 1, kb, ka);
        } else {
          step(i, ka, ka);
          step(i + 1, ka, ka);
        }
      }
      if (i < i_hi) step(i, ka, kTwoK ? kb : ka);
    }

    // normalise and store: row sums first
    float lt = lsum + shfl_xor_f(lsum, 16);
    lt += shfl_xor_f(lt, 32);
    const int64_t off = (int64_t)(tok0 + t) * a.out_stride_tok + (int64_t)(h * G + g) * a.out_stride_head;
    // merge of the four quarters: each O and row sum is relative to its wave's exponent
    // base (its row max, 0 when it saw no key), rescaled to the largest
    if (j == 0) {
      mrow[wave][0][c] = m_run;
      mrow[wave][1][c] = lt;
    }
    __syncthreads();  // every wave is done with its V/Q memory, which the merge reuses
    float mmax = -INFINITY;
#pragma unroll
    for (int u = 0; u < kAnyWaves; ++u) mmax = fmaxf(mmax, mrow[u][0][c]);
    float sc[kAnyWaves];
    float ltot = 0.f;
#pragma unroll
    for (int u = 0; u < kAnyWaves; ++u) {
      const float mu = mrow[u][0][c];
      sc[u] = (mu == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((mu - mmax) * a.scale_log2);
      ltot += mrow[u][1][c] * sc[u];
    }
    const float inv = (ltot > 0.f) ? a.v_scale / ltot : 0.f;
    // one piece of several (pieces > 1): this workgroup's rows normalised over its keys,
    // in fp32, and their log2 LSE, for the merge kernel; every row is written (a row that
    // saw no key gets O = 0 and LSE -inf)
    const bool piece_out = pieces > 1;
    float MA_GLOBAL* po = nullptr;
    if (piece_out) {
      po = gptr_mut(a.part_o) + (int64_t)piece_slot * (16 * DP) + c * DP + 4 * j;
      if (wave == 0 && j == 0)
        gptr_mut(a.part_lse)[(int64_t)piece_slot * 16 + c] =
            (ltot > 0.f) ? __builtin_amdgcn_logf(ltot) + mmax * a.scale_log2 : -INFINITY;
    }
    const float pinv = (ltot > 0.f) ? 1.f / ltot : 0.f;
#pragma unroll
    for (int r = 0; r < DB; r += kBPR) {
#pragma unroll
      for (int blk = 0; blk < kBPR; ++blk)
        *reinterpret_cast<__attribute__((address_space(3))) f32x4*>(
            (uintptr_t)(smem_base + ((wave * kBPR + blk) * 64 + lane) * 16)) = o[r + blk];
      __syncthreads();
      // this wave finishes the round's blocks wave, wave + 4, ...
      for (int blk = wave; blk < kBPR; blk += kAnyWaves) {
        f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < kAnyWaves; ++u)
          acc += *reinterpret_cast<const __attribute__((address_space(3))) f32x4*>(
                     (uintptr_t)(smem_base + ((u * kBPR + blk) * 64 + lane) * 16)) * sc[u];
        if (piece_out)
          *reinterpret_cast<f32x4 MA_GLOBAL*>(po + (r + blk) * 16) = acc * pinv;
        else if (real && (r + blk) * 16 < D)
          store_out4<QBF16>(a.out, off + (r + blk) * 16 + 4 * j, acc, inv, a.out_f32);
      }
      __syncthreads();  // before the next round (or the next row block) reuses the memory
    }
  };

  // workgroup = (kv head, key piece, 16-row block, sequence), kv head fastest; its four waves
  // take the four quarters of its piece of the rows' key tiles. A sequence with more rows
  // than row_blocks blocks (a verify past its hint) has its later blocks taken in turn, whole
  // (the pieces' slots hold row_blocks blocks), by the workgroups of its first piece.
  const int64_t item = blockIdx.x;
  const int h = (int)(item % a.hkv);
  const int64_t rest = item / a.hkv;
  const int piece = (int)(rest % a.pieces);
  const int64_t blk_item = rest / a.pieces;
  const int b = (int)(blk_item / a.row_blocks);
  const int rb = (int)(blk_item - (int64_t)b * a.row_blocks);
  if (b >= a.batch) return;
  piece_slot = (blk_item * a.hkv + h) * a.pieces + piece;
  int rows_b;
  if (a.qsl) rows_b = clamp_query_rows(cptr(a.qsl)[b], cptr(a.qsl)[b + 1], a.num_tokens).ntok * a.group;
  else rows_b = (b < a.num_tokens ? 1 : 0) * a.group;
  int pieces = a.pieces;
#pragma unroll 1
  for (int r0 = rb * kAnyRows; r0 < rows_b; r0 += a.row_blocks * kAnyRows) {
    rows(b, h, r0, pieces, (pieces > 1 ? piece * kAnyWaves : 0) + wave);
    if (piece > 0) return;
    pieces = 1;
  }
}

// Merge of more than kAnyFewPieces key pieces: one workgroup per row of a (sequence, 16-row block,
// kv head). The threads read the pieces' log2 LSEs together; a piece's weight is
// 2^(lse - max), kept in LDS. Then DP / 4 threads, four dims each, read a piece's row, the
// 1024 / DP groups of them every 1024 / DP-th piece, sixteen loads in flight each, and the
// groups' sums meet in LDS. Pieces that saw no key weigh 0. One workgroup per 16 rows with
// eight loads in flight took 156 us on the 352 pieces of one sequence of 22k keys at 8 / 1
// heads and 107 us at D = 256, 12 / 2 heads; this takes 7 us on
// both.
template <int DP, bool QBF16>
__global__ __launch_bounds__(256) void any_merge(const AnyArgs args) {
  const AnyArgs a = args;
  constexpr int kTPR = DP / 4;        // threads of one piece's row
  constexpr int kGroups = 256 / kTPR;
  constexpr int kFlight = 16;
  __shared__ float wt[kAnyMaxPieces];
  __shared__ float red[8];
  __shared__ __attribute__((aligned(16))) f32x4 sum[kGroups][kTPR];
  const int item = (int)blockIdx.x / a.merge_rows;  // (b * row_blocks + rb) * hkv + h
  const int row = (int)blockIdx.x - item * a.merge_rows;
  const int h = item % a.hkv;
  const int blk_item = item / a.hkv;
  const int b = blk_item / a.row_blocks;
  const int rb = blk_item - b * a.row_blocks;
  const int R = rb * kAnyRows + row;
  const int t = R / a.group;
  int tok0 = b, ntok = b < a.num_tokens ? 1 : 0;
  if (a.qsl) {
    const QueryRows qr = clamp_query_rows(cptr(a.qsl)[b], cptr(a.qsl)[b + 1], a.num_tokens);
    tok0 = qr.tok0;
    ntok = qr.ntok;
  }
  if (t >= ntok) return;
  const int np = a.pieces;
  const int64_t slot0 = (int64_t)item * np;
  const float MA_GLOBAL* lse = gptr(a.part_lse) + slot0 * 16 + row;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  // 1. the largest LSE, 2. the weights and their sum
  float lv[kAnyMaxPieces / 256];
  float m = -INFINITY;
#pragma unroll
  for (int k = 0; k < kAnyMaxPieces / 256; ++k) {
    const int p = tid + 256 * k;
    lv[k] = p < np ? lse[(int64_t)p * 16] : -INFINITY;
    m = fmaxf(m, lv[k]);
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) m = fmaxf(m, __shfl_xor(m, d, 64));
  if (lane == 0) red[wave] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float ws = 0.f;
#pragma unroll
  for (int k = 0; k < kAnyMaxPieces / 256; ++k) {
    const int p = tid + 256 * k;
    const float w = lv[k] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(lv[k] - m);
    wt[p] = w;
    ws += w;
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) ws += __shfl_xor(ws, d, 64);
  if (lane == 0) red[4 + wave] = ws;
  __syncthreads();
  ws = (red[4] + red[5]) + (red[6] + red[7]);
  // 3. the weighted sum of the pieces' rows
  const int part = tid % kTPR;
  const int grp = tid / kTPR;
  const float MA_GLOBAL* po = gptr(a.part_o) + slot0 * (16 * DP) + row * DP + part * 4;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int p0 = grp; p0 < np; p0 += kGroups * kFlight) {
    f32x4 o[kFlight];
#pragma unroll
    for (int u = 0; u < kFlight; ++u) {
      const int p = p0 + u * kGroups;
      o[u] = p < np ? *reinterpret_cast<const f32x4 MA_GLOBAL*>(po + (int64_t)p * (16 * DP)) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < kFlight; ++u) {
      const int p = p0 + u * kGroups;
      acc += o[u] * (p < np ? wt[p] : 0.f);
    }
  }
  sum[grp][part] = acc;
  __syncthreads();
  if (grp > 0) return;
#pragma unroll
  for (int k = 1; k < kGroups; ++k) acc += sum[k][part];
  const float inv = (ws > 0.f) ? a.v_scale / ws : 0.f;
  const int64_t off = (int64_t)(tok0 + t) * a.out_stride_tok + (int64_t)(h * a.group + R - t * a.group) * a.out_stride_head;
  if (part * 4 < a.head_dim) store_out4<QBF16>(a.out, off + part * 4, acc, inv, a.out_f32);
}

// The merge of few pieces (kAnyFewPieces): DP / 4 threads per row, four dims each, walk the
// row's pieces, four of them in flight, under a running maximum of the LSEs; 1024 / DP rows of
// any row blocks share a workgroup, without LDS or barriers. A workgroup per row as below took
// 17.6 us per call at D = 64, 32 / 8 heads, e4m3 on 16 sequences of 1,500 keys (four pieces
// each), this 16.4. At 9 to 16 pieces decodes measured the same either way, and verifies 3-8%
// slower than below (4 sequences of 700 keys at D = 512, 16 / 4 heads, bf16 17.6 against 16.5 us).
template <int DP, bool QBF16>
__global__ __launch_bounds__(256) void any_merge_few(const AnyArgs args, int rows_total) {
  const AnyArgs a = args;
  constexpr int kTPR = DP / 4;
  const int u = (int)blockIdx.x * (256 / kTPR) + (int)threadIdx.x / kTPR;  // row of a row block
  const int d = ((int)threadIdx.x % kTPR) * 4;
  if (u >= rows_total || d >= a.head_dim) return;
  const int item = u / a.merge_rows;  // (b * row_blocks + rb) * hkv + h
  const int row = u - item * a.merge_rows;
  const int h = item % a.hkv;
  const int blk_item = item / a.hkv;
  const int b = blk_item / a.row_blocks;
  const int R = (blk_item - b * a.row_blocks) * kAnyRows + row;
  const int t = R / a.group;
  int tok0 = b, ntok = b < a.num_tokens ? 1 : 0;
  if (a.qsl) {
    const QueryRows qr = clamp_query_rows(gptr(a.qsl)[b], gptr(a.qsl)[b + 1], a.num_tokens);
    tok0 = qr.tok0;
    ntok = qr.ntok;
  }
  if (t >= ntok) return;
  const int np = a.pieces;
  const float MA_GLOBAL* lse = gptr(a.part_lse) + (int64_t)item * np * 16 + row;
  const float MA_GLOBAL* po = gptr(a.part_o) + ((int64_t)item * np * 16 + row) * DP + d;
  float m = -INFINITY, w = 0.f;
  f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int p = 0; p < np; ++p) {
    const float l = lse[p * 16];
    const f32x4 o = *reinterpret_cast<const f32x4 MA_GLOBAL*>(po + (int64_t)p * (16 * DP));
    const float m_new = fmaxf(m, l);
    const float base = (m_new == -INFINITY) ? 0.f : m_new;
    const float s_old = __builtin_amdgcn_exp2f(m - base);
    const float s_new = __builtin_amdgcn_exp2f(l - base);
    acc = acc * s_old + o * s_new;
    w = w * s_old + s_new;
    m = m_new;
  }
  const float inv = (w > 0.f) ? a.v_scale / w : 0.f;
  const int64_t off = (int64_t)(tok0 + t) * a.out_stride_tok + (int64_t)(h * a.group + R - t * a.group) * a.out_stride_head + d;
  store_out4<QBF16>(a.out, off, acc, inv, a.out_f32);
}

template <int DP, bool QBF16>
static hipError_t launch_any_q(int kv, dim3 grid, hipStream_t st, const AnyArgs& a) {
  if (kv == DT_E4M3)
    hipLaunchKernelGGL((any_kernel<DP, QBF16, DT_E4M3>), grid, dim3(kAnyWaves * 64), 0, st, a);
  else if (kv == DT_E5M2)
    hipLaunchKernelGGL((any_kernel<DP, QBF16, DT_E5M2>), grid, dim3(kAnyWaves * 64), 0, st, a);
  else
    hipLaunchKernelGGL((any_kernel<DP, QBF16, QBF16 ? DT_BF16 : DT_F16>), grid, dim3(kAnyWaves * 64), 0, st, a);
  return hipGetLastError();
}

template <int DP>
static hipError_t launch_any_d(bool qbf16, int kv, dim3 grid, hipStream_t st, const AnyArgs& a) {
  hipError_t e = qbf16 ? launch_any_q<DP, true>(kv, grid, st, a) : launch_any_q<DP, false>(kv, grid, st, a);
  if (e != hipSuccess || a.pieces <= 1) return e;
  const unsigned rows = grid.x / (unsigned)a.pieces * (unsigned)a.merge_rows;
  if (a.pieces <= kAnyFewPieces) {
    const dim3 fgrid((rows + 1024 / DP - 1) / (1024 / DP));
    if (qbf16) hipLaunchKernelGGL((any_merge_few<DP, true>), fgrid, dim3(256), 0, st, a, (int)rows);
    else hipLaunchKernelGGL((any_merge_few<DP, false>), fgrid, dim3(256), 0, st, a, (int)rows);
    return hipGetLastError();
  }
  const dim3 mgrid(rows);
  if (qbf16) hipLaunchKernelGGL((any_merge<DP, true>), mgrid, dim3(256), 0, st, a);
  else hipLaunchKernelGGL((any_merge<DP, false>), mgrid, dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t any_launch(const AnyArgs& a, int q_dtype, int kv_dtype, int64_t grid_x, hipStream_t st) {
  if (grid_x <= 0) return hipSuccess;
  const dim3 grid((unsigned)grid_x);
  const bool qbf16 = q_dtype == DT_BF16;
  const int d = a.head_dim;
  return d <= 64    ? launch_any_d<64>(qbf16, kv_dtype, grid, st, a)
         : d <= 128 ? launch_any_d<128>(qbf16, kv_dtype, grid, st, a)
         : d <= 256 ? launch_any_d<256>(qbf16, kv_dtype, grid, st, a)
                    : launch_any_d<512>(qbf16, kv_dtype, grid, st, a);
}

}  // namespace ma
