// Prefix-aware paged extend above 256 head dims, for gfx950 (D = 512; other multiples of
// 16 padded up to it). Same rows, masks and work list as the tiled kernel of extend.hip.
//
// At 512 dims a wave cannot keep the output of two 16-row blocks (256 registers), and with
// one block per wave every wave reading all of K and V from LDS costs more LDS time than
// the matrix cores take. So the two products are split differently over the workgroup's
// eight waves (two per SIMD), which own 128 (token, GQA head) rows of one kv head:
//   scores  S^T = K Q^T: wave w takes rows 16 w .. 16 w + 15 over all dims (Q in 64
//           registers) and keeps their softmax state; it reads all of K;
//   output  O^T += V^T P^T: wave w takes dims 64 w .. 64 w + 63 of all 128 rows (O in 128
//           registers); P passes through LDS, and every V element is read once.
// Per 32-key tile the waves read 256 KB of K, 32 KB of V and 64 KB of P from LDS (about
// 1,700 cycles) under 2,048 cycles of MFMA per SIMD; the tile's 32 keys are one 16x16x32
// contraction of the PV product. The kernel before it (four waves of 16 rows, one per SIMD,
// 16-key tiles with 16x16x16 PV MFMAs) took 1,018 us on a batch of 4 (prefixes 0-4,096, 256
// to 2,048 new tokens, 16 / 4 heads, bf16) where this one takes 460 (790 TFLOP/s).
//
// Numerics as in the tiled kernel: K in the query dtype (fp8 converted exactly), V and P in
// fp16 (bf16 V converted as its fragments are read, each by one wave), fp32 accumulation,
// row sums of the rounded P, a row's exponent base moved only when its max has grown by
// more than 2^kLazyRescale in p.
//
// Memory pipeline: K and V tiles travel HBM -> LDS by DMA into two-stage rings (64 KB each).
// Step k: (barrier X) V(k) is issued into the stage that V(k-2) has left; scores of tile k;
// (barrier Y) K(k+2) is issued into the stage that K(k) has left; PV of tile k-1, then the
// softmax of tile k, whose P the next barrier X publishes. Each load has one and a half
// steps to land. Slots are looked up three tiles ahead.

#include <type_traits>

#include "capi_internal.h"
#include "extend.h"

// MA_ASM_PIPELINE: the build verifies the generated code of this file for accesses to
// registers whose inline-assembly loads are still in flight.

namespace ma {

constexpr int kWideWaves = 8;

template <bool QBF16, int KV>
__global__ __launch_bounds__(kWideWaves * 64, 1) void extend_wide_kernel(const ExtendArgs args) {
  const ExtendArgs a = args;  // local copy: the lambdas capture by reference
  constexpr int D = kWideDim;
  constexpr int BM = kWideRows;
  constexpr int BN = kWideKeys;
  constexpr bool kFp8 = (KV == DT_E4M3 || KV == DT_E5M2);
  constexpr bool kConvV = (!kFp8) && QBF16;
  constexpr int kElt = kFp8 ? 1 : 2;
  constexpr int KK = D / 32;                  // QK MFMA steps
  constexpr int KB = BN / 16;                 // 16-key blocks per tile
  constexpr int NRB = BM / 16;                // 16-row blocks of the workgroup
  constexpr int DW = D / kWideWaves;          // output dims per wave
  constexpr int DB = DW / 16;                 // 16-dim blocks of them
  constexpr int kRowB = D * kElt;             // bytes of one K/V row
  constexpr int kKSub = kRowB / 64;           // K DMA blocks (1 KB) per 16-key block
  constexpr int kCPR = kRowB / 16;            // 16-byte chunks per row
  constexpr int kStageB = BN * kRowB;         // bytes of the K (or V) part of a tile
  constexpr int ND = kStageB / 1024 / kWideWaves;  // DMA instructions per wave of K, and of V, per tile
  static_assert(NRB == kWideWaves && KB == 2, "one row block per wave, one 32-key contraction per tile");
  static_assert(ND >= 1 && kKSub % ND == 0, "a wave's K blocks share one key block");

  __shared__ __attribute__((aligned(1024))) unsigned char kring[2][kStageB];
  __shared__ __attribute__((aligned(1024))) unsigned char vring[2][kStageB];
  __shared__ __attribute__((aligned(16))) u32x4 pbuf[2][NRB][64];  // P^T operand fragments
  __shared__ __attribute__((aligned(16))) float abuf[2][BM];       // rescale factors of moved rows
  __shared__ __attribute__((aligned(16))) uint32_t fbuf[2][NRB];   // row block has moved rows

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));  // in scalar registers, with all that derives from it
  const int c = lane & 15;
  const int j = lane >> 4;
  auto qdim = [&](int kk) -> int {  // first dim of QK step kk for lane group j (as in the tiled kernel)
    if constexpr (kFp8) return (kk >> 1) * 64 + j * 16 + (kk & 1) * 8;
    else return kk * 32 + j * 8;
  };

  const int item = (int)blockIdx.x / a.hkv;
  const int h = (int)blockIdx.x - item * a.hkv;
  int b, rt, piece_first = 0, piece_count = -1, piece_slot = -1;
  if (a.pieces.shares > 0) {
    if (a.pieces.list) {
      const int MA_CONST* e = cptr(reinterpret_cast<const int*>(a.pieces.list + item));
      b = e[0];
      rt = e[1];
      piece_first = e[2];
      piece_count = e[3];
      piece_slot = e[4];
    } else {
      const ExtendPiece p = plan_direct<BM, BN>(a, item, h);
      b = p.seq;
      rt = p.tile;
      piece_first = p.first;
      piece_count = p.count;
      piece_slot = p.slot;
    }
    if (b < 0) return;
  } else {
    const int64_t work = cptr(a.items)[item];
    b = (int)(uint32_t)work;
    if (b < 0) return;
    rt = (int)(work >> 32);
  }
  const QueryRows qr = clamp_query_rows(cptr(a.qsl)[b], cptr(a.qsl)[b + 1], a.num_tokens);
  const int tok0 = qr.tok0;
  const int ntok = qr.ntok;
  const int r0 = rt * BM;
  if (r0 >= ntok * a.group) return;
  const int seq = cptr(a.seq_lens)[b];
  const int prefix = a.prefix ? cptr(a.prefix)[b] : seq - ntok;
  const int64_t seq_row = a.row_index ? cptr(a.row_index)[b] : (int64_t)b;

  // ---- Q of this lane's score row (row c of the wave's block) ----
  u32x4 qv[KK];
  {
    const int r = r0 + wave * 16 + c;
    const int t = r / a.group;
    const int g = r - t * a.group;
    const uint16_t MA_GLOBAL* qp = gptr(reinterpret_cast<const uint16_t*>(a.q)) + (int64_t)(tok0 + t) * a.q_stride_tok +
                                   (int64_t)(h * a.group + g) * a.q_stride_head;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
      qv[kk] = (t < ntok && qdim(kk) < a.head_dim) ? *reinterpret_cast<const u32x4 MA_GLOBAL*>(qp + qdim(kk))
                                                   : u32x4{0, 0, 0, 0};
  }
  // waited for here, once (the compiler cannot count the inline-assembly loads below)
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) __asm__ volatile("" : "+v"(qv[kk]));

  // keys any row of the workgroup may see, and the window in which no row needs masking
  const int t_first = r0 / a.group;
  const int t_last = min(ntok - 1, (r0 + BM - 1) / a.group);
  const KeyRange keys = row_tile_keys(r0, BM, ntok, a.group, prefix, seq, a.causal, a.window);
  const int key_lo = keys.lo + piece_first * BN;
  const int key_hi = keys.hi;
  const int full_lo = a.window >= 0 ? max(0, prefix + t_last - a.window) : 0;
  const int full_hi = a.causal ? min(seq, prefix + t_first + 1) : seq;
  const int rest = key_hi > key_lo ? (key_hi - key_lo + BN - 1) / BN : 0;
  const int ntiles = piece_count >= 0 ? min(piece_count, rest) : rest;

  float m_run = -INFINITY;
  float lsum = 0.f;  // this lane's share of its row's sum of the rounded p
  f32x4 o[NRB][DB];
#pragma unroll
  for (int rb = 0; rb < NRB; ++rb)
#pragma unroll
    for (int db = 0; db < DB; ++db) o[rb][db] = f32x4{0.f, 0.f, 0.f, 0.f};

  const unsigned char MA_GLOBAL* kbase = gptr(reinterpret_cast<const unsigned char*>(a.k));
  const unsigned char MA_GLOBAL* vbase = gptr(reinterpret_cast<const unsigned char*>(a.v));
  const uint32_t row_bytes32 = (uint32_t)(a.kv_stride_row * kElt);  // the host checks it fits
  const int64_t head_off = (int64_t)h * a.kv_stride_head * kElt;
  // XOR swizzle of the 16-byte chunks of V row t in LDS (as in the tiled kernel)
  auto swz = [](int t) -> int {
    if constexpr (kFp8) return (t & 3) | ((t >> 2) & 4);
    else return (2 * t) & (kCPR - 2);
  };

  // lane `ln`'s first V^T fragment of the wave's dims, as a byte offset in a V stage
  auto v_first = [&](int ln) __attribute__((always_inline)) -> uint32_t {
    const int lc = ln & 15, lj = ln >> 4;
    if constexpr (kFp8) {
      const int e = lc >> 1;
      const int tr = (e < 4) ? (4 * lj + e) : (16 + 4 * lj + e - 4);
      return tr * kRowB + (((wave * DB) ^ swz(tr)) << 4) + (ln & 1) * 8;
    } else {
      const int tr = 4 * lj + (lc >> 2);
      return tr * kRowB + (((2 * wave * DB + ((ln & 3) >> 1)) ^ swz(tr)) << 4) + (ln & 1) * 8;
    }
  };

  // ---- memory pipeline ----
  auto key_of = [&](int tile) __attribute__((always_inline)) -> int {
    return min(key_lo + min(tile, ntiles - 1) * BN + (lane & (BN - 1)), key_hi - 1);
  };
  auto load_slot = [&](int tile) __attribute__((always_inline)) -> int {
    const int32_t MA_GLOBAL* tp = gptr(a.tt.table) + seq_row * a.tt.stride + (key_of(tile) >> a.tt.page_shift);
    int page;
    __asm__ volatile("global_load_dword %0, %1, off" : "=v"(page) : "v"(tp) : "memory");
    return page;
  };
  auto slot_of = [&](int tile, int page) __attribute__((always_inline)) -> int {
    return (page << a.tt.page_shift) | (key_of(tile) & ((1 << a.tt.page_shift) - 1));
  };
  auto dma = [&](const unsigned char MA_GLOBAL* src, uint32_t lds) __attribute__((always_inline)) {
    const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds);
    __asm__ volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, off" : : "s"(m0), "v"(src) : "memory", "m0");
  };
  // K blocks (kb, sub) = divmod(wave * ND + x, kKSub): lane l -> key 16 kb + (l & 15), chunk 4 sub + j
  auto issue_k = [&](int myslot, int st) __attribute__((always_inline)) {
    const uint32_t kl = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)kring[st];
    int ln = lane;  // redefined per tile, like the V^T addresses: the offsets stay out of the loop's registers
    __asm__ volatile("" : "+v"(ln));
    const int ks = shfl_i(myslot, ((wave * ND) / kKSub) * 16 + (ln & 15));
    const unsigned char MA_GLOBAL* kp = kbase + (uint64_t)(uint32_t)ks * row_bytes32 + head_off;
#pragma unroll
    for (int x = 0; x < ND; ++x) {
      const int blk = wave * ND + x;
      dma(kp + min(4 * (blk % kKSub) + (ln >> 4), a.chunks - 1) * 16, kl + blk * 1024);
    }
  };
  // V rows, row-major, 16-byte chunks XOR-swizzled by row
  auto issue_v = [&](int myslot, int st) __attribute__((always_inline)) {
    const uint32_t vl = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)vring[st];
    int ln = lane;
    __asm__ volatile("" : "+v"(ln));
    constexpr int kRows = 64 / kCPR;  // rows per DMA instruction
#pragma unroll
    for (int x = 0; x < ND; ++x) {
      const int blk = wave * ND + x;
      const int tok = kRows * blk + ln / kCPR;
      const int vs = kRows == 1 ? __builtin_amdgcn_readlane(myslot, blk) : shfl_i(myslot, tok);
      dma(vbase + (uint64_t)(uint32_t)vs * row_bytes32 + head_off + (min((ln % kCPR) ^ swz(tok), a.chunks - 1) << 4),
          vl + blk * 1024);
    }
  };
  auto wait_vm = [&](auto N_) __attribute__((always_inline)) {
    constexpr int N = decltype(N_)::value;
    __asm__ volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
  };
  auto barrier = [&]() __attribute__((always_inline)) { __asm__ volatile("s_barrier" : : : "memory"); };

  // ---- scores of tile k from K stage st: lane (c, j) holds keys 16 kb + 4j .. + 3 of row c ----
  // The K fragments are read kAhead before the MFMAs that use them; without the scheduling
  // barriers the compiler put each read right before its MFMA, which then waited out the LDS
  // latency (576 us on the D = 512 batch, 460 with them and with every wave-uniform value in scalar
  // registers, which ended the spills).
  f32x4 s[KB];
  auto scores = [&](int st) __attribute__((always_inline)) {
    constexpr int kAhead = kFp8 ? 4 : 6;
    constexpr int N = kKSub * KB;
    int ln = lane;
    __asm__ volatile("" : "+v"(ln));
    const unsigned char* kt = kring[st] + ln * 16;
    auto frag = [&](int i) __attribute__((always_inline)) -> u32x4 {  // block kb = i % KB, chunks i / KB
      return *reinterpret_cast<const u32x4*>(kt + ((i % KB) * kKSub + i / KB) * 1024);
    };
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) s[kb] = f32x4{0.f, 0.f, 0.f, 0.f};
    u32x4 kf[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) kf[i] = frag(i);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      const int kb = i % KB, sub = i / KB;
      if constexpr (kFp8) {
        u32x4 k0, k1;
        cvt16_fp8<KV, QBF16>(kf[i % kAhead], k0, k1);
        s[kb] = mfma16t<QBF16>(k0, qv[2 * sub], s[kb]);
        s[kb] = mfma16t<QBF16>(k1, qv[2 * sub + 1], s[kb]);
      } else {
        s[kb] = mfma16t<QBF16>(kf[i % kAhead], qv[sub], s[kb]);
      }
      if (i + kAhead < N) kf[i % kAhead] = frag(i + kAhead);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // ---- softmax of tile k; P, and the factors of rows whose base moved, to LDS half pk ----
  auto softmax = [&](int k, int pk) __attribute__((always_inline)) {
    const int base = key_lo + k * BN;
    int ln = lane;
    __asm__ volatile("" : "+v"(ln));
    if (!(base >= full_lo && base + BN <= full_hi)) {
      // the lane's visible keys, computed again on the few masked tiles: its row's bounds kept
      // through the loop would spill
      const int t = (r0 + wave * 16 + (ln & 15)) / a.group;
      const int qpos = prefix + t;
      const int lo_r = a.window >= 0 ? qpos - a.window : 0;
      const int hi_r = t < ntok ? (a.causal ? min(seq, qpos + 1) : seq) : 0;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int pos = base + kb * 16 + 4 * (ln >> 4) + i;
          if (pos < lo_r || pos >= hi_r) s[kb][i] = -INFINITY;
        }
    }
    float mx = max3f(max3f(s[0][0], s[0][1], s[0][2]), max3f(s[0][3], s[1][0], s[1][1]),
                     max3f(s[1][2], s[1][3], -INFINITY));
    const bool moved = __builtin_amdgcn_ballot_w64((mx - m_run) * a.scale_log2 > kLazyRescale) != 0;
    if (moved) {
      const int sw = ln << 2;  // byte index of the lane for the cross-lane reads
      mx = fmaxf(mx, __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(sw ^ 64, __builtin_bit_cast(int, mx))));
      mx = fmaxf(mx, __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(sw ^ 128, __builtin_bit_cast(int, mx))));
      const float m_new = fmaxf(m_run, mx);
      const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
      const float alpha = __builtin_amdgcn_exp2f((m_run - m_use) * a.scale_log2);
      m_run = m_new;
      lsum *= alpha;
      if (ln < 16) abuf[pk][wave * 16 + ln] = alpha;
    }
    if (ln == 0) fbuf[pk][wave] = moved;
    const float msc = ((m_run == -INFINITY) ? 0.f : m_run) * a.scale_log2;
    u32x4 pf;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb)
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const float p0 = __builtin_amdgcn_exp2f(s[kb][2 * w] * a.scale_log2 - msc);
        const float p1 = __builtin_amdgcn_exp2f(s[kb][2 * w + 1] * a.scale_log2 - msc);
        const uint32_t pw = pack_p16(p0, p1);
        pf[2 * kb + w] = pw;
        // the row sum takes the rounded p, so that rounding cancels in the quotient
        const f16x2 one = {(_Float16)1.f, (_Float16)1.f};
        lsum = __builtin_amdgcn_fdot2(__builtin_bit_cast(f16x2, pw), one, lsum, false);
      }
    pbuf[pk][wave][ln] = pf;
  };
  // ---- O of this wave's dims over tile k: V stage st, P half pk ----
  auto pv = [&](int st, int pk) __attribute__((always_inline)) {
    // The fragments of block db lie at the lane's first one XOR the block (rows start at
    // multiples of the row size, the swizzled chunk below). Redefined per tile: hoisted out
    // of the loop, the blocks' addresses took registers the output needs.
    int ln = lane;
    __asm__ volatile("" : "+v"(ln));
    const uint32_t vl = v_first(ln);
    uint32_t fl = 0;
#pragma unroll
    for (int rb = 0; rb < NRB; rb += 4) {
      const u32x4 f = *reinterpret_cast<const u32x4*>(&fbuf[pk][rb]);
      fl |= f[0] | f[1] | f[2] | f[3];
    }
    const unsigned char* vt = vring[st];
    u32x4 va[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      if constexpr (kFp8) {
        const u32x2 raw = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr8_b64_v2i32(
            (__attribute__((address_space(3))) i32x2*)(vt + (vl ^ (db << 4)))));
        va[db] = cvt8_fp8<KV, false>(raw[0], raw[1]);
      } else {
#pragma unroll
        for (int half = 0; half < 2; ++half) {  // 16 rows on, the swizzle differs in chunk bit 5
          const u32x2 raw = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
              (__attribute__((address_space(3))) i16x4*)(vt + (vl ^ (db << 5) ^ (half << 9)) + half * 16 * kRowB)));
          va[db][2 * half] = raw[0];
          va[db][2 * half + 1] = raw[1];
        }
        if constexpr (kConvV) {
#pragma unroll
          for (int w = 0; w < 4; ++w)
            va[db][w] = pack_f16(__builtin_bit_cast(float, va[db][w] << 16),
                                 __builtin_bit_cast(float, va[db][w] & 0xffff0000u));
        }
      }
    }
    u32x4 pf[2] = {pbuf[pk][0][ln], pbuf[pk][1][ln]};
    if (__builtin_amdgcn_readfirstlane(fl)) {
#pragma unroll
      for (int rb = 0; rb < NRB; ++rb) {
        if (__builtin_amdgcn_readfirstlane(fbuf[pk][rb])) {
          const float al = abuf[pk][rb * 16 + (ln & 15)];
#pragma unroll
          for (int db = 0; db < DB; ++db) o[rb][db] *= al;
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int rb = 0; rb < NRB; ++rb) {  // P fragments two row blocks ahead
#pragma unroll
      for (int db = 0; db < DB; ++db) o[rb][db] = mfma16t<false>(va[db], pf[rb & 1], o[rb][db]);
      if (rb + 2 < NRB) pf[rb & 1] = pbuf[pk][rb + 2][ln];
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // ---- schedule ----
  if (ntiles > 0) {
    int sreg[4];  // slots of tile t in sreg[t % 4]
    sreg[0] = load_slot(0);
    sreg[1] = load_slot(1);
    sreg[2] = load_slot(2);
    wait_vm(std::integral_constant<int, 0>{});
    __asm__ volatile("" : "+v"(sreg[0]), "+v"(sreg[1]), "+v"(sreg[2]));
    issue_k(slot_of(0, sreg[0]), 0);
    issue_k(slot_of(1, sreg[1]), 1);
    // Step k issues, per wave: a slot lookup (tile k+3) and V(k) after barrier X, K(k+2)
    // after barrier Y. Before X it waits for K(k) (newer: the last step's lookup, V and K),
    // before Y for V(k-1) (newer: K(k+1), this step's lookup and V(k)). The lookup that
    // Y's K(k+2) uses was issued a step earlier, before V(k-1), and so has landed. In step
    // 0, K(0)'s wait finds only K(1) newer, and Y's wait covers nothing it needs.
    auto step = [&](auto I_, int k) __attribute__((always_inline)) {
      constexpr int I = decltype(I_)::value;  // k % 4
      if (k == 0) wait_vm(std::integral_constant<int, ND>{});
      else wait_vm(std::integral_constant<int, 1 + 2 * ND>{});
      __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      barrier();  // X
      sreg[(I + 3) & 3] = load_slot(k + 3);
      issue_v(slot_of(k, sreg[I]), I & 1);
      if (k < ntiles) scores(I & 1);
      wait_vm(std::integral_constant<int, 1 + 2 * ND>{});
      __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __asm__ volatile("" : "+v"(sreg[(I + 2) & 3]));
      barrier();  // Y
      issue_k(slot_of(k + 2, sreg[(I + 2) & 3]), I & 1);
      if (k > 0 && k <= ntiles) pv((I + 1) & 1, (I + 1) & 1);
      if (k < ntiles) softmax(k, I & 1);
    };
    auto group = [&]<int... Is>(std::integer_sequence<int, Is...>, int n) __attribute__((always_inline)) {
      (step(std::integral_constant<int, Is>{}, n + Is), ...);
    };
    for (int n = 0; n <= ntiles; n += 4) group(std::make_integer_sequence<int, 4>{}, n);
    wait_vm(std::integral_constant<int, 0>{});  // no DMA may land after the workgroup ends
  }

  // ---- epilogue: row sums meet in LDS, then each wave stores its dims of every row ----
  int ln = lane;
  __asm__ volatile("" : "+v"(ln));
  const int lc = ln & 15;
  float lt = lsum + shfl_xor_f(lsum, 16);
  lt += shfl_xor_f(lt, 32);
  __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  barrier();  // every wave is past its last read of abuf
  if (ln < 16) abuf[0][wave * 16 + lc] = lt;
  __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  barrier();
  if (piece_slot >= 0 && ln < 16 && (r0 + wave * 16 + lc) / a.group < ntok) {
    const int64_t prow = ((int64_t)piece_slot * a.hkv + h) * BM + wave * 16 + lc;
    gptr_mut(a.pieces.lse)[prow] = (lt > 0.f) ? __builtin_amdgcn_logf(lt) + m_run * a.scale_log2 : -INFINITY;
  }
#pragma unroll
  for (int rb = 0; rb < NRB; ++rb) {
    const int R = r0 + rb * 16 + lc;
    const int tr = R / a.group;
    if (tr >= ntok) continue;
    const float l = abuf[0][rb * 16 + lc];
    const int d0 = wave * DW + 4 * (ln >> 4);
    if (piece_slot >= 0) {
      const int64_t prow = ((int64_t)piece_slot * a.hkv + h) * BM + rb * 16 + lc;
      const float inv = (l > 0.f) ? 1.f / l : 0.f;
#pragma unroll
      for (int db = 0; db < DB; ++db)
        if (d0 + db * 16 < a.head_dim)
          *reinterpret_cast<f32x4 MA_GLOBAL*>(gptr_mut(a.pieces.o) + prow * D + d0 + db * 16) = o[rb][db] * inv;
    } else {
      const float inv = (l > 0.f) ? a.v_scale / l : 0.f;
      const int64_t off =
          (int64_t)(tok0 + tr) * a.out_stride_tok + (int64_t)(h * a.group + R - tr * a.group) * a.out_stride_head;
#pragma unroll
      for (int db = 0; db < DB; ++db)
        if (d0 + db * 16 < a.head_dim) store_out4<QBF16>(a.out, off + d0 + db * 16, o[rb][db], inv, a.out_f32);
    }
  }
}

template <bool QBF16>
static hipError_t launch_wide(int kv, dim3 grid, hipStream_t st, const ExtendArgs& a) {
  const dim3 block(kWideWaves * 64);
  if (kv == DT_E4M3)
    hipLaunchKernelGGL((extend_wide_kernel<QBF16, DT_E4M3>), grid, block, 0, st, a);
  else if (kv == DT_E5M2)
    hipLaunchKernelGGL((extend_wide_kernel<QBF16, DT_E5M2>), grid, block, 0, st, a);
  else
    hipLaunchKernelGGL((extend_wide_kernel<QBF16, QBF16 ? DT_BF16 : DT_F16>), grid, block, 0, st, a);
  return hipGetLastError();
}

hipError_t extend_wide_launch(bool qbf16, int kv, dim3 grid, hipStream_t st, const ExtendArgs& a) {
  return qbf16 ? launch_wide<true>(kv, grid, st, a) : launch_wide<false>(kv, grid, st, a);
}

}  // namespace ma
