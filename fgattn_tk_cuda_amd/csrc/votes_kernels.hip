// Block maxima -> votes per key: the threshold sweep behind a statistics sweep that also wrote the
// per-(row, key block) score maxima.
//
// The reference sweeps Q K^T a second time in full (include/mask_utils.cuh:131-243).  A key can pass
//   exp2((s[r,c] - max_q[r]) sf) / denom[r] > thresh
// only in a key block whose maximum over the row's group passes it, so a workgroup, which owns a 128-row
// q-block and a chunk of keys,
//   1. reads its column of the block maxima (256 bytes per key block) and notes for every 64-key block
//      which of the four 32-row groups hold a row whose maximum lies above its threshold,
//   2. multiplies only those (32-row group, 64-key block) pairs and ORs the votes, a ballot per 32 keys,
//      into a bit row in LDS,
//   3. writes the bits of its chunk: one bit per (q-block, key), the layout of the mask cache
//      (python/spattn/mask_utils.py:421-430).
//
// Split of 2.  A wave keeps the Q rows of R groups in registers (all four at d = 64, two at d = 128) and walks
// its own share of the blocks with an active group among them, 32 keys at a time; it owns a ring of 32-key
// pieces in LDS that it fills itself, so there is no barrier in the walk, and an LDS operand feeds up to R
// multiplies.  Chunks of keys are dealt to the workgroups chunk by chunk, all q-blocks of a head for one
// chunk before the next, so that the K rows that the workgroups of an XCD walk at a time stay near its 4 MB
// of L2.
//
// What bounds it: no one unit.  At 24 x 32760 x 64 with 45 % of the (128-row, 64-key) pairs and 22 % of the
// (32-row, 64-key) pairs active it takes 0.88 ms; without the multiplies 0.65, without the copies 0.80,
// without the walk 0.19.  (The sweep over the listed 64-key blocks that it replaces, all 128 rows of each:
// 1.51 ms behind 0.15 ms for the lists.  6 x 75600 x 128, 29 / 13 %: 1.46 ms; a full sweep takes 8.2 ms.)
// Measured and not taken: the four waves sharing the tiles of a 128-row q-block with a barrier per tile or
// per two tiles, 0.87-1.0 ms and 1.68-1.75 ms.
#include <type_traits>

#include "common.h"
#include "dispatch.h"

namespace spattn {

template <int D>
struct VotesCfg {
  static constexpr int kGroups = (D == 64) ? 4 : 2;            // 32-row groups per wave
  static constexpr int kRowParts = 4 / kGroups;                 // waves along the rows
  static constexpr int kWalkers = 4 / kRowParts;                // waves that share the list of a row part
  static constexpr int kPiece = 32 * D * 2;                     // bytes of 32 keys
  static constexpr int kSlots = (D == 64) ? 4 : 2;              // pieces in a wave's ring: 64 KB per workgroup
  static constexpr int kChunkBlocks = (D == 64) ? 512 : 320;    // 64-key blocks per chunk (4 / 5 MB of K): fewer, and
                                                                // a chunk outgrows L2, more, and the prologue weighs (both measured 2-8 % slower)
};

struct VotesParams {
  uint32_t* bits;            // [HB,SB,stride/32]
  const uint16_t* blockmax;  // [HB,Sp/64,Sp]
  const float* max_q;        // [HB,Sp]
  const float* denom;        // [HB,Sp]
  const uint16_t* q;         // [HB,S,D]
  const uint16_t* k;
  float log2_thresh;         // of the vote
  float log2_thresh_blk;     // of the block test: a little lower, see run_blockmax_votes
  float sf;
  int HB, S, kv_len, Sp, SB, words;
  int nch, ch_blocks;        // chunks per row, 64-key blocks per chunk
};

// v with lane L (or the lane in m0) replaced by the wave-uniform s; the wait states cover a vector-ALU write
// of s, as by a ballot.
template <int L>
__device__ __forceinline__ int write_lane(int s, int v) {
  asm("s_nop 1\n\tv_writelane_b32 %0, %1, %2" : "+v"(v) : "s"(s), "n"(L));
  return v;
}
__device__ __forceinline__ int write_lane_at(int s, int lane, int v) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 1\n\tv_writelane_b32 %0, %1, m0" : "+v"(v) : "s"(s), "s"(lane));
  return v;
}
// Lane U of lo / hi receives the ballot of "row 2 lane or 2 lane + 1 above its threshold" for word U of x.
template <int U, int N>
__device__ __forceinline__ void collect_ballots(const uint32_t (&x)[N], float t0, float t1, int& lo, int& hi) {
  if constexpr (U < N) {
    const float x0 = __builtin_bit_cast(float, x[U] << 16);
    const float x1 = __builtin_bit_cast(float, x[U] & 0xffff0000u);
    const unsigned long long m = __ballot(x0 > t0 || x1 > t1);
    lo = write_lane<U>((int)(unsigned)m, lo);
    hi = write_lane<U>((int)(unsigned)(m >> 32), hi);
    collect_ballots<U + 1, N>(x, t0, t1, lo, hi);
  }
}

template <int D>
__global__ __launch_bounds__(256, 2) void blockmax_votes_kernel(const VotesParams p) {
  using Cfg = VotesCfg<D>;
  constexpr int NT = D / 16;
  constexpr int CPR = D / 8;
  constexpr int ROWB = D * 2;
  constexpr int R = Cfg::kGroups;
  constexpr int RP = Cfg::kRowParts;
  constexpr int TW = Cfg::kWalkers;
  constexpr int PIECE = Cfg::kPiece;
  constexpr int NS = Cfg::kSlots;
  constexpr int LPP = PIECE / 1024;       // 1 KB copies per piece
  constexpr int RPL = 1024 / ROWB;        // rows per copy
  constexpr int CB = Cfg::kChunkBlocks;
  __shared__ __attribute__((aligned(1024))) unsigned char ring_all[4 * NS * PIECE];
  __shared__ uint32_t bits[2 * CB];
  __shared__ uint16_t blist[RP][CB];      // block within the chunk | active groups of the row part << 12
  __shared__ int n_active[RP];
  static_assert(CB <= 4096, "a block number takes 12 bits");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ln = lane & 31;
  const int g = lane >> 5;
  const int rp = wave % RP;
  const int tw = wave / RP;
  // head, then chunk, then q-block: see the top of the file
  const int wg = xcd_remap(blockIdx.x, p.SB * p.nch * p.HB);
  const int qb = wg % p.SB;
  const int hc = wg / p.SB;
  const int bh = hc / p.nch;
  const int J0 = (hc - bh * p.nch) * p.ch_blocks;
  const size_t head_off = (size_t)bh * p.S * D;
  const uint16_t* qh = p.q + head_off;
  const unsigned char* kh = reinterpret_cast<const unsigned char*>(p.k + head_off);
  const int nblk = (p.kv_len + 63) >> 6;
  const int nbc = (nblk - J0) < p.ch_blocks ? (nblk - J0) : p.ch_blocks;   // blocks of this chunk, not positive behind the last

  // The first batch of block maxima (32 key blocks per wave, a lane holds two rows) is requested before
  // anything else: it takes longest to arrive.
  const uint16_t* bm = p.blockmax + (size_t)bh * (p.Sp >> 6) * p.Sp + qb * 128 + 2 * lane;
  uint32_t x[32];
  auto load_maxima = [&](int b) {
#pragma unroll
    for (int u = 0; u < 32; ++u) {
      const int J = J0 + (b + u < nbc ? b + u : nbc - 1);
      x[u] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(bm + (size_t)J * p.Sp));
    }
  };
  if (32 * wave < nbc) load_maxima(32 * wave);

  // Thresholds on the raw score, through a table that overlays the ring: minus the vote threshold of row r
  // (the C operand that starts every multiply chain, as in the full sweep: the same bits), and the block
  // threshold.  Rows past S or without a key never vote.
  float* tab = reinterpret_cast<float*>(ring_all);
  if (tid < 128) {
    const int row = qb * 128 + tid;
    float tv = -__builtin_huge_valf(), tb = __builtin_huge_valf();
    if (row < p.S) {
      const float mq = p.max_q[(size_t)bh * p.Sp + row];
      const float dn = p.denom[(size_t)bh * p.Sp + row];
      const float inv_sf = 1.f / p.sf;
      if (dn > 0.f) {
        tv = -(p.log2_thresh + (mq * p.sf + __log2f(dn))) * inv_sf;
        tb = (p.log2_thresh_blk + (mq * p.sf + __log2f(dn))) * inv_sf;
      }
    }
    tab[tid] = tv;
    tab[128 + tid] = tb;
  }
  for (int i = tid; i < 2 * CB; i += 256) bits[i] = 0;
  if (tid < RP) n_active[tid] = 0;
  // A operands: row 32 (R rp + m) + ln of the q-block, k-step t at chunk 2t + g
  u32x4 qa[R][NT];
#pragma unroll
  for (int m = 0; m < R; ++m) {
    const int row = qb * 128 + 32 * (R * rp + m) + ln;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const u32x4 z = {0, 0, 0, 0};
      qa[m][t] = (row < p.S) ? *reinterpret_cast<const u32x4*>(qh + (size_t)row * D + 16 * t + 8 * g) : z;
    }
  }
  __syncthreads();
  const float tb0 = tab[128 + 2 * lane], tb1 = tab[128 + 2 * lane + 1];

  // ---- 1: active (row group, block) pairs; 32 blocks per wave step, all loads in flight ----
  for (int b = 32 * wave; b < nbc; b += 128) {
    int lo = 0, hi = 0;   // lane u: the ballot of block b + u, rows 2l and 2l + 1 in bit l
    collect_ballots<0, 32>(x, tb0, tb1, lo, hi);
    int act = ((lo & 0xffff) ? 1 : 0) | (((unsigned)lo >> 16) ? 2 : 0) | ((hi & 0xffff) ? 4 : 0) | (((unsigned)hi >> 16) ? 8 : 0);
    if (lane >= 32 || b + lane >= nbc) act = 0;
#pragma unroll
    for (int r = 0; r < RP; ++r) {
      const int mine = (act >> (R * r)) & ((1 << R) - 1);
      const unsigned long long keep = __ballot(mine != 0);
      int base = 0;
      if (lane == 0) base = atomicAdd(&n_active[r], __popcll(keep));   // the order of a list does not matter
      base = __builtin_amdgcn_readfirstlane(base);
      if (mine) blist[r][base + __builtin_amdgcn_mbcnt_lo((unsigned)keep, 0)] = (uint16_t)((b + lane) | (mine << 12));
    }
    if (b + 128 < nbc) load_maxima(b + 128);
  }
  // The compiler waits for its loads of qa here: inside the walk that wait would be one for every copy.
#pragma unroll
  for (int m = 0; m < R; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) asm volatile("" : "+v"(qa[m][t]));
  f32x16 nthr[R];   // register 4j+i of group m: row 32 (R rp + m) + 8j + 4g + i
#pragma unroll
  for (int m = 0; m < R; ++m)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) nthr[m][4 * j + i] = tab[32 * (R * rp + m) + 8 * j + 4 * g + i];
#pragma unroll
  for (int m = 0; m < R; ++m) asm volatile("" : "+v"(nthr[m]));
  __syncthreads();

  // ---- 2: votes of the active pairs ----
  // Piece u of this wave: keys 32 (u & 1) .. of block entry u >> 1 of its share (every TW-th entry of the list
  // of its row part, from tw).  The copies of a piece go out NS pieces ahead; its operands are read from
  // the ring while the piece before it is multiplied.
  const int n = __builtin_amdgcn_readfirstlane(n_active[rp]);
  const int ne = (n - tw + TW - 1) / TW;   // not positive: nothing to do
  const int nu = 2 * ne;
  if (nu > 0) {
    auto swz = [](int r) -> int {
      return D == 128 ? (((r & 3) << 2) | ((r >> 2) & 3)) : ((((r >> 1) & 1) << 2) | ((r >> 2) & 3));
    };
    const uint32_t ring = (uint32_t)(uintptr_t)(lds_cptr)ring_all + wave * (NS * PIECE);
    uint32_t kread[NT];     // operand of k-step t in slot 0
#pragma unroll
    for (int t = 0; t < NT; ++t) kread[t] = ring + ln * ROWB + (((2 * t + g) ^ swz(ln)) << 4);
    uint32_t goff[LPP];     // copy i: lane offset within a piece
#pragma unroll
    for (int i = 0; i < LPP; ++i) {
      const int r = RPL * i + lane / CPR;
      goff[i] = (r < p.kv_len ? r : p.kv_len - 1) * ROWB + (((lane % CPR) ^ swz(r)) << 4);
    }
    // entry u >> 1 for the 64 pieces of a group: lane l holds that of piece u0 + l (past the end: the last one)
    auto entries = [&](int u0) -> int {
      int e = (u0 + lane) >> 1;
      e = e < ne ? e : ne - 1;
      return blist[rp][tw + TW * e];
    };
    int ev = entries(0), ev_next = entries(64);
    auto entry = [&](int i) -> int {   // of piece i of the current group (or of the next)
      return i < 64 ? __builtin_amdgcn_readlane(ev, i) : __builtin_amdgcn_readlane(ev_next, i - 64);
    };
    // Piece i into a slot.  A piece that runs past the last key is copied as the last 32 rows of the sequence
    // (a shorter sequence: from row 0, goff clamps the rows) and its votes are shifted down by what it
    // was moved; what that leaves behind the last key is masked off at the end.
    const int r0_max = p.kv_len > 32 ? p.kv_len - 32 : 0;
    auto first_row = [&](int i) -> int { return (J0 + (entry(i) & 0xfff)) * 64 + 32 * (i & 1); };
    struct PieceLoad {
      const unsigned char* base;
      uint32_t dst;
    };
    auto prepare = [&](int i, int slot) -> PieceLoad {
      const int row0 = first_row(i);
      return PieceLoad{kh + (size_t)(row0 < r0_max ? row0 : r0_max) * ROWB, ring + slot * PIECE};
    };
    auto issue = [&](const PieceLoad& l, int c) { dma16(l.base, goff[c], __builtin_amdgcn_readfirstlane(l.dst + c * 1024)); };
    u32x4 kf[2][NT];
    auto read_piece = [&](int slot, u32x4 (&kd)[NT]) {
#pragma unroll
      for (int t = 0; t < NT; ++t) kd[t] = *(SPATTN_LDS const u32x4*)((lds_cptr)(uintptr_t)kread[t] + slot * PIECE);
    };
#pragma unroll
    for (int j = 0; j < NS; ++j) {
      const PieceLoad l = prepare(j, j);
#pragma unroll
      for (int c = 0; c < LPP; ++c) issue(l, c);
    }
    // pieces past the end repeat the last: the wait counts stay the same
    wait_vmcnt<(NS - 1) * LPP>();
    read_piece(0, kf[0]);

    int words = 0;
    auto piece = [&](auto sc, int i) {   // piece i of the group, in slot S, operands in kf[S & 1]
      constexpr int S = decltype(sc)::value;
      u32x4(&kc)[NT] = kf[S & 1];
      // piece i+1 has landed; the operands of this piece, requested a piece ago, have left its slot
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NS - 2) * LPP) : "memory");
      const PieceLoad next = prepare(i + NS, S);
      read_piece((S + 1) % NS, kf[(S + 1) & 1]);
      const int act = entry(i) >> 12;
      f32x16 acc[2];
      typedef __attribute__((ext_vector_type(16))) int i32x16;
      int top0 = 0, top1 = 0;   // a float is > 0 exactly when its bits are, as an integer
      auto chain = [&](int m) {
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[m & 1] = mfma32(qa[m][t], kc[t], t == 0 ? nthr[m] : acc[m & 1]);
      };
      auto reduce = [&](int m) {
        const i32x16 x = __builtin_bit_cast(i32x16, acc[m & 1]);
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          top0 = top0 > x[r] ? top0 : x[r];
          top1 = top1 > x[r + 8] ? top1 : x[r + 8];
        }
      };
      // The maxima of a chain are taken behind the next chain; the copies go out between the chains (in one
      // burst they queue behind those of the other waves).
#pragma unroll
      for (int m = 0; m < R + 1; ++m) {
        if (m < R && (act & (1 << m))) chain(m);
        if (m < R) {
#pragma unroll
          for (int c = 0; c < LPP / R; ++c) issue(next, m * (LPP / R) + c);
        }
        if (m > 0 && (act & (1 << (m - 1)))) reduce(m - 1);
      }
      const unsigned long long v = __ballot((top0 > top1 ? top0 : top1) > 0);
      const int row0 = first_row(i);
      const uint32_t w = ((uint32_t)v | (uint32_t)(v >> 32)) >> ((row0 < r0_max ? 0 : row0 - r0_max) & 31);
      words = write_lane_at((int)w, i, words);
    };
    for (int u0 = 0; u0 < nu; u0 += 64) {
      const int lim = nu - u0 < 64 ? nu - u0 : 64;   // even
      int i = 0;
      for (; i + NS <= lim; i += NS) {
        piece(std::integral_constant<int, 0>{}, i);
        piece(std::integral_constant<int, 1>{}, i + 1);
        if constexpr (NS == 4) {
          piece(std::integral_constant<int, 2>{}, i + 2);
          piece(std::integral_constant<int, 3>{}, i + 3);
        }
      }
      if (NS == 4 && i < lim) {
        piece(std::integral_constant<int, 0>{}, i);
        piece(std::integral_constant<int, 1>{}, i + 1);
      }
      // lane l: the votes of piece u0 + l
      if (words) atomicOr(&bits[2 * (ev & 0xfff) + (lane & 1)], (uint32_t)words);
      words = 0;
      ev = ev_next;
      ev_next = entries(u0 + 128);
    }
    wait_vmcnt<0>();   // no copy may land after the workgroup has given up its LDS
  }
  __syncthreads();

  // ---- 3: the bits of this chunk; the last chunk also writes the words behind the last key ----
  const bool tail = hc - bh * p.nch == p.nch - 1;
  const int w_end = tail ? p.words - 2 * J0 : 2 * p.ch_blocks;
  const int lim = p.kv_len - J0 * 64;   // keys of this chunk and behind
  uint32_t* dst = p.bits + ((size_t)bh * p.SB + qb) * p.words + 2 * J0;
  for (int w = tid; w < w_end; w += 256) {
    uint32_t x = w < 2 * nbc ? bits[w] : 0u;
    const int left = lim - w * 32;
    if (left < 32) x = left <= 0 ? 0u : (x & ((1u << left) - 1u));
    dst[w] = x;
  }
}

// The block test runs a little below the vote threshold, tau (1 - 1e-3): the statistics sweep rounds a
// score and compares, the vote accumulates s - t in the matrix unit, so a key whose margin is below fp32
// rounding could otherwise sit in a block the (rounded up) maxima leave out.  The blocks this adds
// contribute no votes: the bits equal those of a full threshold sweep.
hipError_t run_blockmax_votes(uint32_t* bits, const uint16_t* blockmax, const float* max_q, const float* denom,
                              const uint16_t* q, const uint16_t* k, float thresh, int mask_stride, int HB, int S, int D,
                              int kv_len, float sf, hipStream_t stream) {
  const int SB = (S + 127) / 128;
  if (SB * HB <= 0) return hipSuccess;
  VotesParams p{};
  p.bits = bits;
  p.blockmax = blockmax;
  p.max_q = max_q;
  p.denom = denom;
  p.q = q;
  p.k = k;
  p.log2_thresh = thresh > 0.f ? log2f(thresh) : -__builtin_huge_valf();
  p.log2_thresh_blk = thresh > 0.f ? log2f((float)((double)thresh * (1.0 - 1e-3))) : -__builtin_huge_valf();
  p.sf = sf;
  p.HB = HB;
  p.S = S;
  p.kv_len = kv_len;
  p.Sp = SB * 128;
  p.SB = SB;
  p.words = mask_stride / 32;
  const int nblk = (kv_len + 63) / 64;
  const int most = D == 128 ? VotesCfg<128>::kChunkBlocks : VotesCfg<64>::kChunkBlocks;
  p.nch = (nblk + most - 1) / most;
  p.ch_blocks = (nblk + p.nch - 1) / p.nch;
  p.nch = (nblk + p.ch_blocks - 1) / p.ch_blocks;   // every chunk holds a key
  const dim3 grid(SB * HB * p.nch);
  if (D == 128) hipLaunchKernelGGL(blockmax_votes_kernel<128>, grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL(blockmax_votes_kernel<64>, grid, dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace spattn
