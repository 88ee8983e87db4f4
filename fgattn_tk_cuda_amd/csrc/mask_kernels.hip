// Threshold-mask pre-pass kernels for gfx950:
//   booleanmask_128          - QK^T sweep -> per-(q-block, key) vote counts
//   booleanmask_to_indexmask - vote mask -> ascending key-index lists (HBM-bound stream)
//   all_index_mask           - identity lists
#include <type_traits>

#include "common.h"
#include "dispatch.h"

namespace spattn {

// ------------------------------------------------------------------------------------
// booleanmask_128.  Reference: include/mask_utils.cuh:131-243.  For q-block I (128 rows)
// and key c the reference counts the 16-row groups W of I with
//   max_{r in W} exp2((s[r,c] - max_q[r]) * sf) / denom[r] > thresh        (:231-238)
// Here the test is done in the log2 domain, which is the same predicate:
//   max_{r in W} (s[r,c] * sf - (max_q[r] * sf + log2 denom[r])) > log2 thresh.
// Pad rows carry denom = -inf (include/maxq_denom.cuh:202-205) and never vote.
//
// One workgroup per q-block, each wave walks its own 32-key blocks; no barrier in the
// sweep.  Scores are S = Q K^T with the query rows as the A operand - held in registers for
// d = 64 (each wave keeps all 128 rows), read from an LDS copy of the tile for d = 128 -
// and the keys as the B operand.  For d = 64 every wave owns an LDS ring of four key
// blocks that HBM -> LDS copies fill three blocks ahead (whole 128-byte rows per copy, the
// swizzle applied by choosing which chunk a lane fetches); for d = 128, where the query
// tile takes the LDS, the keys go HBM -> registers one block ahead.  The accumulator of
// lane (n, g) holds key n against 64 of the 128 query rows.  The test is rewritten once
// more as  s[r,c] - t[r] > 0  with the per-row constant
// t[r] = (log2 thresh + max_q[r] sf + log2 denom[r]) / sf, and -t[r], kept in 64 registers,
// is the C operand of the first multiply of every chain: the matrix unit does the
// subtraction, the vector ALU only takes the maximum of the 8 registers a lane holds of a
// 16-row group (v_max3) and compares it with 0; one exchange with lane n^32 finishes the 8
// votes of a key.  The vote count is stored, not accumulated.
//
// Three output forms (OUT), the sweep is the same:
//   OUT_VOTES   int32 vote count per (128-row q-block, key)         - the reference's mask
//   OUT_BITS128 one bit per (128-row q-block, key): count > 0, 32 keys per stored word,
//               least significant bit first - 1/32 of the bytes, the layout of the mask cache
//   OUT_BITS64  one bit per (64-row q-block, key): the four 16-row groups of each half of the
//               128-row block vote separately; rows 2I and 2I+1 of the output
// A wave holds the votes of 32 consecutive keys in 32 lanes, so a word is one ballot.
// ------------------------------------------------------------------------------------
enum MaskOut : int { OUT_VOTES = 0, OUT_BITS128 = 1, OUT_BITS64 = 2 };

// SPARSE: the sweep restricted to the 64-key blocks of a per-q-block list (ascending ids, e.g. the
// block lists that the threshold of the block maxima gives): a key of a block whose maximum fails
// the test cannot pass it, so every other entry of the mask row is zero and the multiplies of the
// kept blocks give the same votes as the full sweep.  The workgroup first clears its mask row(s),
// then each wave walks every fourth 32-key half block of the listed blocks.
template <int D, int OUT, bool SPARSE>
__global__ __launch_bounds__(256, 2) void booleanmask_kernel(int* __restrict__ mask, const float* __restrict__ max_q,
                                                              const float* __restrict__ denom,
                                                              const uint16_t* __restrict__ q,
                                                              const uint16_t* __restrict__ k, float log2_thresh,
                                                              int mask_stride, int HB, int S, int kv_len, int Sp,
                                                              int SB, float sf, const int* __restrict__ blk_idx,
                                                              const int* __restrict__ blk_cnt, int max_blocks) {
  constexpr int NT = D / 16;
  constexpr int CPR = D / 8;
  constexpr bool Q_REGS = (D == 64);
  __shared__ __attribute__((aligned(16))) unsigned char qs[Q_REGS ? 16 : 128 * D * 2];
  __shared__ __attribute__((aligned(16))) float nthr_l[2][4][16];   // [g][mb][register]
  // d = 64: every wave owns a ring of four 4 KB key blocks, filled by HBM -> LDS copies
  constexpr bool K_RING = Q_REGS;
  constexpr int NSLOT = 4;
  constexpr int KBLK = 32 * D * 2;
  __shared__ __attribute__((aligned(1024))) unsigned char kring[K_RING ? 4 * NSLOT * KBLK : 16];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int ln = lane & 31;
  const int g = lane >> 5;
  const int total = SB * HB;
  const int wg = xcd_remap(blockIdx.x, total);
  const int qb = wg % SB;
  const int bh = wg / SB;
  const size_t head_off = (size_t)bh * S * D;
  const uint16_t* qh = q + head_off;
  const uint16_t* kh = k + head_off;

  // Query rows; rows past S are zero.  In LDS the 16-byte chunk c of row r sits at
  // c ^ swz(r), which spreads one chunk of 16 consecutive rows over all bank groups.
  auto swz = [](int r) -> int { return ((r & 3) << 2) | ((r >> 2) & 3); };
  u32x4 qa[Q_REGS ? 4 : 1][Q_REGS ? NT : 1];
  if constexpr (Q_REGS) {
#pragma unroll
    for (int mb = 0; mb < 4; ++mb) {
      const int row = qb * 128 + 32 * mb + ln;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const u32x4 z = {0, 0, 0, 0};
        qa[mb][t] = (row < S) ? *reinterpret_cast<const u32x4*>(qh + (size_t)row * D + 16 * t + 8 * g) : z;
      }
    }
  } else {
    for (int ch = tid; ch < 128 * CPR; ch += 256) {
      const int r = ch / CPR, c = ch % CPR;
      const int row = qb * 128 + r;
      u32x4 val = {0, 0, 0, 0};
      if (row < S) val = *reinterpret_cast<const u32x4*>(qh + (size_t)row * D + 8 * c);
      *reinterpret_cast<u32x4*>(qs + r * (D * 2) + ((c ^ swz(r)) << 4)) = val;
    }
  }

  // Minus the per-row thresholds on the raw score, gathered through a table in LDS into the
  // registers that start every multiply chain; register 4j+i of block mb in lane half g is query row
  // 32mb + 8j + 4g + i.  Pad rows and rows without keys get -inf and never vote.
  const float inv_sf = 1.f / sf;
  if (tid < 128) {
    const int tg = tid >> 6, tmb = (tid >> 4) & 3, tr = tid & 15;
    const int row = qb * 128 + 32 * tmb + 8 * (tr >> 2) + 4 * tg + (tr & 3);
    float c = -__builtin_huge_valf();
    if (row < S) {
      const float mq = max_q[(size_t)bh * Sp + row];
      const float dn = denom[(size_t)bh * Sp + row];
      if (dn > 0.f) c = -(log2_thresh + (mq * sf + __log2f(dn))) * inv_sf;
    }
    nthr_l[tg][tmb][tr] = c;
  }
  __syncthreads();

  int* mrow = mask + ((size_t)bh * SB + qb) * mask_stride;
  const int nkb = (mask_stride + 31) >> 5;
  // bit outputs: rows of mask_stride / 32 words; with 64-row q-blocks the last 128-row block
  // of a head may have one half only
  const int nq64 = (S + 63) >> 6;
  uint32_t* brow0 = nullptr;
  uint32_t* brow1 = nullptr;
  if constexpr (OUT == OUT_BITS128) {
    brow0 = reinterpret_cast<uint32_t*>(mask) + ((size_t)bh * SB + qb) * (size_t)nkb;
  } else if constexpr (OUT == OUT_BITS64) {
    brow0 = reinterpret_cast<uint32_t*>(mask) + ((size_t)bh * nq64 + 2 * qb) * (size_t)nkb;
    if (2 * qb + 1 < nq64) brow1 = brow0 + nkb;
  }

  // The walk of this workgroup: position j -> 32-key block.  Dense: block j.  Sparse: the two
  // halves of the listed 64-key blocks in list order; positions before the first stand for "no
  // block" (nothing is stored for them), positions past the last repeat the last one (their keys
  // are copied, never multiplied), an id outside the row is replaced by the row's last block.
  typedef const __attribute__((address_space(4))) int* cint_p;
  cint_p lst = nullptr;
  int nseq = nkb;
  if constexpr (SPARSE) {
    const size_t lrow = (size_t)bh * SB + qb;
    int n = ((cint_p)blk_cnt)[lrow];
    n = n < 0 ? 0 : (n > max_blocks ? max_blocks : n);
    nseq = 2 * n;
    lst = (cint_p)(blk_idx + lrow * max_blocks);
    // clear the row(s): 16-byte stores, then every store of the workgroup has reached memory
    // before any wave writes a vote
    const i32x4 z4 = {0, 0, 0, 0};
    if constexpr (OUT == OUT_VOTES) {
      for (int i = tid * 4; i < mask_stride; i += 1024) *reinterpret_cast<i32x4*>(mrow + i) = z4;
    } else {
      for (int i = tid * 4; i < nkb; i += 1024) {
        *reinterpret_cast<i32x4*>(brow0 + i) = z4;
        if (OUT == OUT_BITS64 && brow1 != nullptr) *reinterpret_cast<i32x4*>(brow1 + i) = z4;
      }
    }
    wait_vmcnt<0>();
    __syncthreads();
  }
  auto kb_at = [&](int j) -> int {
    if constexpr (!SPARSE) {
      return j;
    } else {
      if (j < 0) return -1;
      int jj = j < nseq ? j : nseq - 1;
      jj = jj < 0 ? 0 : jj;
      int e = nseq > 0 ? lst[jj >> 1] : 0;
      e = (unsigned)e < (unsigned)(nkb >> 1) ? e : (nkb >> 1) - 1;
      return 2 * e + (jj & 1);
    }
  };

  // Ring layout: key row r of a block at r * 2D bytes, its 16-byte chunk c at c ^ kswz(r),
  // which spreads chunk 2t+g of the 32 rows a half wave reads over all bank groups.  Copy i
  // of a block moves rows 8i .. 8i+7: lane l fills position l of that 1 KB, i.e. fetches the
  // chunk that belongs there, so that every copy reads eight whole rows of HBM.
  auto kswz = [](int r) -> int { return (((r >> 1) & 1) << 2) | ((r >> 2) & 3); };
  lds_cptr kread[K_RING ? NT : 1];     // per-lane read addresses inside slot 0 of this wave
  int krow[K_RING ? 4 : 1];            // per-lane row of copy i inside a block
  uint32_t kcol[K_RING ? 4 : 1];       // byte offset inside that row
  const lds_cptr ring_l = (lds_cptr)kring + __builtin_amdgcn_readfirstlane(wave) * (NSLOT * KBLK);
  const uint32_t ring_base = (uint32_t)(uintptr_t)ring_l;
  if constexpr (K_RING) {
#pragma unroll
    for (int t = 0; t < NT; ++t) kread[t] = ring_l + ln * (D * 2) + (((2 * t + g) ^ kswz(ln)) << 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      krow[i] = 8 * i + (lane >> 3);
      kcol[i] = ((lane & 7) ^ kswz(krow[i])) << 4;
    }
  }
  // Rows past the end re-read the last key, blocks past the end likewise: every block costs
  // the same four copies, which keeps the hand-counted waits valid up to the last block.
  auto issue_keys = [&](int kb, int slot) {
    if constexpr (K_RING) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int key = kb * 32 + krow[i];
        key = key < kv_len ? key : kv_len - 1;
        key = key < 0 ? 0 : key;
        dma16<SPARSE>(kh, (uint32_t)key * (D * 2) + kcol[i],
                      __builtin_amdgcn_readfirstlane(ring_base + slot * KBLK + i * 1024));
      }
    }
  };
  auto slot_addr = [&](int slot) -> uint32_t { return (uint32_t)(slot & (NSLOT - 1)) * KBLK; };
  auto read_keys = [&](int slot, u32x4 (&kf)[NT]) {
    if constexpr (K_RING) {
#pragma unroll
      for (int t = 0; t < NT; ++t) kf[t] = *(SPATTN_LDS const u32x4*)(kread[t] + slot_addr(slot));
    }
  };

  // Keys past the end re-read the last key (their votes are never stored): the loads are
  // unconditional, so the compiler can count them and let a block that was requested one
  // step ahead stay in flight while the current one is multiplied.
  auto load_keys = [&](int kb, u32x4 (&kf)[NT]) {
    int key = kb * 32 + ln;
    key = key < kv_len ? key : kv_len - 1;
    key = key < 0 ? 0 : key;
#pragma unroll
    for (int t = 0; t < NT; ++t) kf[t] = *reinterpret_cast<const u32x4*>(kh + (size_t)key * D + 16 * t + 8 * g);
  };
  // Bits 2mb, 2mb+1 of the result: does any of this lane's 8 rows of the two 16-row groups
  // of block mb lie above its threshold.
  // A float is > 0 exactly when its bit pattern, read as a signed integer, is > 0 (NaNs
  // aside), and integer maxima need no NaN canonicalisation: v_max3_i32, 4 per 8 registers.
  auto group_votes = [&](int mb, const f32x16& s) -> unsigned {
    typedef __attribute__((ext_vector_type(16))) int i32x16;
    const i32x16 si = __builtin_bit_cast(i32x16, s);
    int w0 = si[0], w1 = si[8];
#pragma unroll
    for (int r = 1; r < 8; ++r) {
      w0 = w0 > si[r] ? w0 : si[r];
      w1 = w1 > si[8 + r] ? w1 : si[8 + r];
    }
    return ((w0 > 0 ? 1u : 0u) << (2 * mb)) | ((w1 > 0 ? 1u : 0u) << (2 * mb + 1));
  };

  // Software pipeline over half blocks (a pair of 32-row score blocks = 2 NT multiplies):
  // while the matrix unit multiplies one pair, the vector ALU takes the maxima of the pair
  // before it, a few vector instructions behind every multiply, so that a wave is an even
  // mix of both at every point (two waves that alternate between a multiply-only and a
  // vector-only phase fall into step and leave both units idle in turn).
  // Two accumulator sets alternate: multiplied now, reduced now.  The first multiply of a
  // chain takes the threshold registers as its C operand and writes the set, so nothing has
  // to be initialised.
  constexpr int NACC = 2;
  f32x16 acc[NACC][2];
  f32x16 nthr[4];
#pragma unroll
  for (int mb = 0; mb < 4; ++mb) nthr[mb] = *reinterpret_cast<const f32x16*>(&nthr_l[g][mb][0]);
  unsigned vhold = 0;
  // reload: once a key register set has fed its last multiply of this block it is
  // refilled from the ring slot of the wave's next block.
  auto pair_scores = [&](int p2, u32x4 (&kf)[NT], f32x16 (&a2)[2], bool reload, uint32_t next_lds) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int mb = 2 * p2 + j;
        const int qr = 32 * mb + ln;
        u32x4 a;
        if constexpr (Q_REGS) a = qa[mb][t];
        else a = *reinterpret_cast<const u32x4*>(qs + qr * (D * 2) + (((2 * t + g) ^ swz(qr)) << 4));
        a2[j] = mfma32(a, kf[t], t == 0 ? nthr[mb] : a2[j]);
      }
      if constexpr (K_RING) {
        if (reload) kf[t] = *(SPATTN_LDS const u32x4*)(kread[t] + next_lds);
      }
    }
  };
  auto finish_block = [&](int kb, unsigned votes) {
    // A 16-row group is split over lanes n and n^32: it votes if either half does.
    float lo_, hi_;
    pair_values(__builtin_bit_cast(float, votes), lo_, hi_);   // v_permlane32_swap, no LDS
    votes = __builtin_bit_cast(unsigned, lo_) | __builtin_bit_cast(unsigned, hi_);
    const int key = kb * 32 + ln;   // negative for the block "before the first": nothing is stored
    if constexpr (OUT == OUT_VOTES) {
      if (g == 0 && (unsigned)key < (unsigned)mask_stride) mrow[key] = (key < kv_len) ? __popc(votes) : 0;
    } else {
      // lanes n and n + 32 hold the same votes: the low word of a ballot is the 32 keys
      const bool live = (unsigned)key < (unsigned)kv_len;
      const bool store = lane == 0 && (unsigned)kb < (unsigned)nkb;
      if constexpr (OUT == OUT_BITS128) {
        const uint32_t w = (uint32_t)__ballot(live && votes != 0);
        if (store) brow0[kb] = w;
      } else {
        const uint32_t w0 = (uint32_t)__ballot(live && (votes & 0x0fu) != 0);
        const uint32_t w1 = (uint32_t)__ballot(live && (votes & 0xf0u) != 0);
        if (store) {
          brow0[kb] = w0;
          if (brow1 != nullptr) brow1[kb] = w1;
        }
      }
    }
  };
  // Half H: multiplies pair H&1 of the current block into acc[H % NACC] and reduces the
  // accumulators of the half before; kb_prev: the block before the current one in this wave's walk.
  auto half = [&](auto hc, int kb_prev, u32x4 (&kf)[NT], bool reload, uint32_t next_lds) {
    constexpr int H = decltype(hc)::value;
    constexpr int P = H & 1, A = H % NACC, AP = (H + NACC - 1) % NACC;
    pair_scores(P, kf, acc[A], reload, next_lds);
    const unsigned v = group_votes(2 * (1 - P), acc[AP][0]) | group_votes(2 * (1 - P) + 1, acc[AP][1]);
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, (NT == 4) ? 3 : 2, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (P == 0) finish_block(kb_prev, vhold | v);   // pair 1 of the block before
    else vhold = v;                                          // pair 0 of this block
  };
  // After the last block (its second half went into acc[A]): reduce it and store.
  auto drain = [&](auto ac, int kb) {
    constexpr int A = decltype(ac)::value;
    finish_block(kb, vhold | group_votes(2, acc[A][0]) | group_votes(3, acc[A][1]));
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;

  int j = wave;          // position in the walk; this wave takes every fourth
  acc[1][0] = nthr[2];   // reduced by the very first half; its votes go nowhere
  acc[1][1] = nthr[3];
  if constexpr (K_RING) {
    // The copies of a block go out three of the wave's blocks ahead; the registers of block
    // b+1 are read from the ring during the second half of block b.  Of the vector-memory
    // operations that follow the copies of block b+1 in program order, the 8 copies of the
    // blocks b+2 and b+3 are always there (vote stores may or may not be), hence vmcnt(8).
    u32x4 kf[NT];
    int slot = 0;
    issue_keys(kb_at(j), 0);
    issue_keys(kb_at(j + 4), 1);
    issue_keys(kb_at(j + 8), 2);
    wait_vmcnt<8>();
    read_keys(0, kf);
    auto block = [&](auto h0, auto h1, int jj) {
      issue_keys(kb_at(jj + 12), (slot + 3) & (NSLOT - 1));
      half(h0, kb_at(jj - 4), kf, false, 0u);
      wait_vmcnt<8>();
      half(h1, 0, kf, true, slot_addr(slot + 1));
      slot = (slot + 1) & (NSLOT - 1);
    };
    for (; j < nseq; j += 4) block(I0{}, I1{}, j);
    drain(I1{}, kb_at(j - 4));
    wait_vmcnt<0>();   // no copy may land after the workgroup has given up its LDS
  } else {
    u32x4 k0[NT], k1[NT];
    load_keys(kb_at(j), k0);
    while (j + 4 < nseq) {
      load_keys(kb_at(j + 4), k1);
      half(I0{}, kb_at(j - 4), k0, false, 0u);
      half(I1{}, 0, k0, false, 0u);
      load_keys(kb_at(j + 8), k0);
      half(I0{}, kb_at(j), k1, false, 0u);
      half(I1{}, 0, k1, false, 0u);
      j += 8;
    }
    if (j < nseq) {
      half(I0{}, kb_at(j - 4), k0, false, 0u);
      half(I1{}, 0, k0, false, 0u);
      drain(I1{}, kb_at(j));
    } else {
      drain(I1{}, kb_at(j - 4));
    }
  }
}

template <int D, int OUT>
static void launch_booleanmask(int* mask, float lt, int mask_stride, const float* max_q, const float* denom,
                               const uint16_t* q, const uint16_t* k, int HB, int S, int kv_len, int Sp, int SB, float sf,
                               const int* blk_idx, const int* blk_cnt, int max_blocks, hipStream_t stream) {
  if (blk_idx != nullptr)
    hipLaunchKernelGGL((booleanmask_kernel<D, OUT, true>), dim3(SB * HB, 1, 1), dim3(256), 0, stream, mask, max_q, denom, q,
                       k, lt, mask_stride, HB, S, kv_len, Sp, SB, sf, blk_idx, blk_cnt, max_blocks);
  else
    hipLaunchKernelGGL((booleanmask_kernel<D, OUT, false>), dim3(SB * HB, 1, 1), dim3(256), 0, stream, mask, max_q, denom, q,
                       k, lt, mask_stride, HB, S, kv_len, Sp, SB, sf, nullptr, nullptr, 0);
}

// out_rows: 0 = int32 vote counts; 128 / 64 = bit rows per q-block of that many query rows.
// blk_idx / blk_cnt / max_blocks: optional lists of 64-key blocks per 128-row q-block
// ([B,H,SB,max_blocks] ascending ids, [B,H,SB] counts) that restrict the sweep (see SPARSE above).
hipError_t run_booleanmask(void* out, int out_rows, float thresh, int mask_stride, const float* max_q,
                           const float* denom, const uint16_t* q, const uint16_t* k, int B, int H, int S, int D,
                           int kv_len, float scale, hipStream_t stream, const int* blk_idx, const int* blk_cnt,
                           int max_blocks) {
  const int SB = (S + 127) / 128;
  const int Sp = SB * 128;
  const float sf = kLog2e * scale;
  const float lt = thresh > 0.f ? log2f(thresh) : -__builtin_huge_valf();
  const int total = SB * H * B;
  if (total <= 0) return hipSuccess;
  int* m = static_cast<int*>(out);
  const int HB = H * B;
#define SPATTN_MASK_CASE(DD, OO) \
  launch_booleanmask<DD, OO>(m, lt, mask_stride, max_q, denom, q, k, HB, S, kv_len, Sp, SB, sf, blk_idx, blk_cnt, max_blocks, stream)
  if (D == 128) {
    if (out_rows == 0) SPATTN_MASK_CASE(128, OUT_VOTES);
    else if (out_rows == 128) SPATTN_MASK_CASE(128, OUT_BITS128);
    else if (out_rows == 64) SPATTN_MASK_CASE(128, OUT_BITS64);
    else return hipErrorInvalidValue;
  } else {
    if (out_rows == 0) SPATTN_MASK_CASE(64, OUT_VOTES);
    else if (out_rows == 128) SPATTN_MASK_CASE(64, OUT_BITS128);
    else if (out_rows == 64) SPATTN_MASK_CASE(64, OUT_BITS64);
    else return hipErrorInvalidValue;
  }
#undef SPATTN_MASK_CASE
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------
// booleanmask_to_indexmask.  Reference: include/mask_utils.cuh:273-302 - for each
// (b,h,q-block) row: count = #{c < kv_len : mask[c] > 0}, list = those c, entries past the
// count keep the caller's fill.  The reference appends through one global atomic per key
// (order undefined); here one wave owns one row and streams it as 16-byte vectors with the
// next 8 KB already in flight.  Every kept key is ranked with wave ballots and appended to
// a per-wave LDS ring, which is written out in ascending order 4 KB at a time - no
// atomics, no barrier, full-line stores, and the result is deterministic.  The kernel is
// a pure HBM stream: 4 bytes read per mask entry, 4 bytes written per kept key.
// ------------------------------------------------------------------------------------
constexpr int kCompactUnroll = 8;      // 16-byte loads per lane per step (8 KB per wave)
constexpr int kCompactRing = 2048;     // ints in the per-wave output ring
constexpr int kCompactFlush = 1024;    // ints written out at a time (4 KB bursts)
constexpr int kCompactMaxGrid = 1024;  // workgroups; rows beyond that are taken in further rounds

// Measured on this part: a plain 128 KB-per-wave read stream runs at 6.5 TB/s, the same
// stream with 8 % of its bytes written back at 5.3-5.6 TB/s however the writes are
// grouped; larger bursts are the better end of that range, hence the 4 KB flushes.
__global__ __launch_bounds__(256) void compact_kernel(int* __restrict__ kv_indices, int* __restrict__ kv_num,
                                                      const int* __restrict__ mask, int rows, int mask_stride,
                                                      int kv_len) {
  constexpr int U = kCompactUnroll;
  constexpr int SPAN = 256 * U;        // ints per wave step
  constexpr int QN = kCompactRing;
  constexpr int FL = kCompactFlush;
  static_assert(FL + 256 <= QN && FL % 256 == 0, "a flush must fit the ring next to one more vector of keys");
  __shared__ __attribute__((aligned(16))) int ring[4][QN];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  int* q = ring[wave];
  const int lim = kv_len < mask_stride ? kv_len : mask_stride;
  const int nfull = lim / SPAN;        // steps that lie entirely below lim

  for (int row = blockIdx.x * 4 + wave; row < rows; row += gridDim.x * 4) {
    const int* __restrict__ src = mask + (size_t)row * mask_stride;
    int* __restrict__ dst = kv_indices + (size_t)row * mask_stride;
    int tail = 0;   // keys appended to the ring so far
    int head = 0;   // keys written out so far (a multiple of 256 until the end: whole lines)

    // Ranks the kept keys of one 16-byte vector per lane (keys of lower lanes first, then
    // the lane's own lower keys), appends them to the ring and writes out full bursts.
    auto append = [&](int e0, const bool (&f)[4]) {
      const unsigned long long b0 = __ballot(f[0]), b1 = __ballot(f[1]), b2 = __ballot(f[2]), b3 = __ballot(f[3]);
      int pos = tail;
      pos = __builtin_amdgcn_mbcnt_hi((unsigned)(b0 >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)b0, pos));
      pos = __builtin_amdgcn_mbcnt_hi((unsigned)(b1 >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)b1, pos));
      pos = __builtin_amdgcn_mbcnt_hi((unsigned)(b2 >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)b2, pos));
      pos = __builtin_amdgcn_mbcnt_hi((unsigned)(b3 >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)b3, pos));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (f[i]) q[pos & (QN - 1)] = e0 + i;
        pos += f[i] ? 1 : 0;
      }
      tail += __popcll(b0) + __popcll(b1) + __popcll(b2) + __popcll(b3);
      // fewer than FL keys were pending and at most 256 were added: the ring never wraps
      // onto unwritten keys
      if (tail - head >= FL) {
#pragma unroll
        for (int w = 0; w < FL / 256; ++w)
          *reinterpret_cast<i32x4*>(dst + head + w * 256 + 4 * lane) =
              *reinterpret_cast<const i32x4*>(q + ((head + w * 256 + 4 * lane) & (QN - 1)));
        head += FL;
      }
    };

    i32x4 cur[U], nxt[U];
    auto load = [&](int c, i32x4 (&v)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u)
        v[u] = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(src + c * SPAN + u * 256 + 4 * lane));
    };
    if (nfull > 0) load(0, cur);
    for (int c = 0; c < nfull; ++c) {
      if (c + 1 < nfull) load(c + 1, nxt);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool f[4] = {cur[u][0] > 0, cur[u][1] > 0, cur[u][2] > 0, cur[u][3] > 0};
        append(c * SPAN + u * 256 + 4 * lane, f);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) cur[u] = nxt[u];
    }
    // the ragged rest of the row, entry by entry against lim (mask_stride is a multiple of 4,
    // so a vector that starts below lim stays inside the row)
    for (int e = nfull * SPAN; e < lim; e += 256) {
      const int e0 = e + 4 * lane;
      const i32x4 z = {0, 0, 0, 0};
      const i32x4 v = (e0 < lim) ? *reinterpret_cast<const i32x4*>(src + e0) : z;
      const bool f[4] = {v[0] > 0 && e0 < lim, v[1] > 0 && e0 + 1 < lim, v[2] > 0 && e0 + 2 < lim, v[3] > 0 && e0 + 3 < lim};
      append(e0, f);
    }
    for (; head < tail; head += 64)
      if (head + lane < tail) dst[head + lane] = q[(head + lane) & (QN - 1)];
    if (lane == 0) kv_num[row] = tail;
  }
}

hipError_t run_compact(int* kv_indices, int* kv_num, const int* mask, int rows, int mask_stride, int kv_len,
                       hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  int grid = (rows + 3) / 4;
  if (grid > kCompactMaxGrid) grid = kCompactMaxGrid;
  hipLaunchKernelGGL(compact_kernel, dim3(grid), dim3(256), 0, stream, kv_indices, kv_num, mask, rows, mask_stride, kv_len);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------
// all_index_mask.  Reference: include/utils.cuh:73-93 (host loop + copy): every list is
// 0,1,2,...,mask_stride-1 and every count is seq.  Here a store-only kernel.
// ------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void all_index_kernel(int* __restrict__ kv_indices, int* __restrict__ kv_num,
                                                        int rows, int mask_stride, int seq) {
  const size_t vec_per_row = (size_t)mask_stride / 4;
  const size_t nvec = vec_per_row * rows;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < nvec; i += (size_t)gridDim.x * blockDim.x) {
    const int c = (int)(i % vec_per_row) * 4;
    const i32x4 v = {c, c + 1, c + 2, c + 3};
    reinterpret_cast<i32x4*>(kv_indices)[i] = v;
  }
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < (size_t)rows; i += (size_t)gridDim.x * blockDim.x)
    kv_num[i] = seq;
}

hipError_t run_all_index(int* kv_indices, int* kv_num, int rows, int mask_stride, int seq, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  const size_t nvec = (size_t)mask_stride / 4 * rows;
  size_t blocks = (nvec + 255) / 256;
  if (blocks > 256 * 32) blocks = 256 * 32;
  if (blocks == 0) blocks = 1;
  hipLaunchKernelGGL(all_index_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, kv_indices, kv_num, rows,
                     mask_stride, seq);
  return hipGetLastError();
}

}  // namespace spattn
