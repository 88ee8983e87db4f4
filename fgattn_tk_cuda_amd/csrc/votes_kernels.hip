// Block maxima -> votes per key: the threshold sweep behind a statistics sweep that also wrote the
// per-(row, key block) score maxima.
//
// The reference sweeps Q K^T a second time in full (include/mask_utils.cuh:131-243).  A key can pass
//   exp2((s[r,c] - max_q[r]) sf) / denom[r] > thresh
// for row r only in a 64-key block whose maximum for that row passes it.  The key block stands still and the rows come
// to it: a wave holds 64 keys in registers, as the B operand, and takes from a chunk of q-blocks
//   1. the block's maxima of the chunk's rows (contiguous: the maxima lie block by block), of which it keeps one bit
//      per row, "may pass";
//   2. the list of those rows, q-block by q-block, each filled up to a multiple of four with a row of its own;
//   3. the listed rows of Q, sixteen to a tile, copied through a ring in LDS that it fills itself (whole rows, so that
//      the copies coalesce; no barrier) and multiplied with the 64 keys.  In the 16x16 accumulator lanes 16 g .. of
//      register i hold row 4 g + i of the tile, so the ballot of sixteen keys has sixteen bits for each four of rows,
//      and the fours of a tile may belong to different q-blocks (lanes 0..3 shift theirs out of the four ballots: writing
//      them lane by lane took 20 wait states and 40 scalar instructions a tile, 2-5 % of the time);
//   4. the 64 bits of every q-block: one bit per (q-block, key), the layout of the mask cache
//      (python/spattn/mask_utils.py:421-430).
// A chain of 16x16x32 multiplies gives the same bits as the 32x32x16 chain of the full sweep (compared on 1.6 million
// elements, with magnitudes spread over e^8 among them): the votes equal those of the sweep.
//
// Why by rows: at a threshold of 32 mean weights on correlated tokens 45 % of the (q-block, key block) pairs hold an
// active row, 22 % of the (32-row group, key block) pairs, but 4.5 % of the (row, key block) pairs.  Multiplying
// (32-row group, key block) pairs with the rows standing still, as this kernel did before, copied all 64 keys of 45 % of
// the pairs.  What bounds it now: below 5 % of the rows the maxima (5.3 TB/s of them where nothing is active), the
// copies (keys of every wave, listed rows) and the latency of a wave's chain of them, behind that the multiplies next to the
// vector ALU: where every row is listed 0.93 (d = 64) and 1.02 PFLOP/s (d = 128).  Before and after, us, thresholds of
// 1/4, 2, 4, 16, 32, 64 mean weights (67, 31, 22, 8, 4.5, 2.3 % of the rows):
//   24 x 32760 x 64    2576 / 2127 / 1855 / 1200 / 882 / 625    2692 / 1437 / 1085 / 591 / 444 / 353
//   6 x 75600 x 128    7284 / 5925 / 5016 / 3047 / 2172 / 1489  6228 / 3304 / 2456 / 1327 / 1021 / 843
//   16 x 6000 x 128    138 / 122 / 108 / 75 / 56 / 42           117 / 68 / 54 / 34 / 27 / 23
//   96 x 732 x 64      18.3 / 17.7 / 17.4 / 16.2 / 15.3 / 13.9  12.9 / 10.3 / 9.0 / 7.2 / 6.4 / 5.3
//   16 x 400 x 64      7.5 / 7.5 / 7.5 / 7.4 / 7.2 / 6.4        5.2 / 5.0 / 4.9 / 4.6 / 4.7 / 4.6
// Rows that nearly all pass are multiplied faster standing still: below 1/4 of a mean weight the kernel before was ahead on
// long sequences, with every row listed 2485 to 3382 us (24 x 32760 x 64) and 7070 to 7742 (6 x 75600 x 128).
// Measured and not taken: fours replaced by sixteens (every tile of one q-block) 6-14 % slower at d = 128, three ring
// slots 8-30 % slower, the thresholds copied into the list 20 % slower.
#include <type_traits>

#include "common.h"
#include "dispatch.h"

namespace spattn {

template <int D>
struct VotesCfg {
  static constexpr int kTile = 16 * D * 2;                 // bytes of 16 rows
  static constexpr int kSlots = 2;                         // tiles in a wave's ring: a third one costs a workgroup per CU
  static constexpr int kChunk = (D == 64) ? 32 : 16;       // q-blocks per chunk, at most: longer chunks load the keys less
                                                           // often and hold more LDS (thresholds); the other way round
                                                           // measured 11-18 % (d = 64) and 3-8 % (d = 128) slower
  static constexpr int kCap = 32;                          // tiles that a wave lists before it multiplies them
};

struct VotesParams {
  uint32_t* bits;            // [HB,SB,stride/32]
  const uint16_t* blockmax;  // [HB,Sp/64,Sp]
  const float* max_q;        // [HB,Sp]
  const float* denom;        // [HB,Sp]
  const uint16_t* q;         // [HB,S,D]
  const uint16_t* k;
  float log2_thresh;
  float blk_slack;           // how far below its vote threshold a row's block maximum still counts, see run_blockmax_votes
  float sf;
  int HB, S, kv_len, Sp, SB, words;
  int nch, ch_qblocks;       // chunks of rows per head, q-blocks per chunk
  int jgroups;               // groups of four key blocks per head
};

// Exclusive position of a lane's x items in its row of sixteen lanes; total: up to and with this lane.
__device__ __forceinline__ int row_scan(int x, int& total) {
  int v = x;
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);   // row_shr:8
  total = v;
  return v - x;
}

template <int D, int CHUNK>
__global__ __launch_bounds__(256, 3) void blockmax_votes_kernel(const VotesParams p) {
  using Cfg = VotesCfg<D>;
  constexpr int NT = D / 32;              // k-steps
  constexpr int CPR = D / 8;              // 16-byte chunks per row
  constexpr int ROWB = D * 2;
  constexpr int TILE = Cfg::kTile;
  constexpr int NS = Cfg::kSlots;
  constexpr int LPP = TILE / 1024;        // 1 KB copies per tile
  constexpr int CAP = Cfg::kCap;
  constexpr int ROWS = CHUNK * 128;       // rows per chunk, at most
  constexpr int NB = ROWS / 512;          // batches of four q-blocks
  static_assert(NS == 2, "the keys arrive in two halves of the ring's length");
  static_assert(CAP >= 32, "a batch of four q-blocks has up to 32 tiles");
  static_assert(CHUNK <= 64, "a lane writes the votes of one q-block");
  __shared__ __attribute__((aligned(1024))) unsigned char ring_all[4 * NS * TILE];
  __shared__ __attribute__((aligned(16))) float tab[ROWS];                 // minus the vote threshold of a row on its raw score
  __shared__ __attribute__((aligned(16))) uint16_t list_row[4][CAP * 16];  // row within the chunk
  __shared__ unsigned long long votes[4][CHUNK];                           // of a wave's keys, per q-block

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = lane >> 4;
  // head, then chunk of rows, then key blocks: the Q rows of a chunk (1 MB at d = 128) stay in an XCD's L2
  const int wg = xcd_remap(blockIdx.x, p.jgroups * p.nch * p.HB);
  const int jg = wg % p.jgroups;
  const int hc = wg / p.jgroups;
  const int bh = hc / p.nch;
  const int qb0 = (hc - bh * p.nch) * p.ch_qblocks;
  const int nqb = (p.SB - qb0) < p.ch_qblocks ? (p.SB - qb0) : p.ch_qblocks;
  const int row0 = qb0 * 128;
  const int J = 4 * jg + wave;                       // key block
  const int left = p.kv_len - 64 * J;                // its keys and those behind
  const size_t head_off = (size_t)bh * p.S * D;
  const unsigned char* qc = reinterpret_cast<const unsigned char*>(p.q + head_off + (size_t)row0 * D);
  const unsigned char* kh = reinterpret_cast<const unsigned char*>(p.k + head_off);

  // The maxima of the whole chunk are requested before anything else: they take longest to arrive.  Lane l holds
  // rows 512 b + 8 l .. + 7.
  u32x4 x[NB];
  {
    const uint16_t* bm = p.blockmax + ((size_t)bh * (p.Sp >> 6) + (left > 0 ? J : 0)) * p.Sp + row0 + 8 * lane;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const bool in = left > 0 && 512 * b + 8 * lane < 128 * nqb;
      const u32x4 none = {0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u};
      x[b] = in ? __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(bm + 512 * b)) : none;
    }
  }
  // Thresholds: -t[r] is the C operand that starts every multiply chain, as in the full sweep.  Rows past S or
  // without a key never vote.
  {
    constexpr int N = ROWS / 256;
    float mq[N], dn[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int r = row0 + 256 * i + tid;
      const size_t so = (size_t)bh * p.Sp + (r < p.S ? r : row0);
      mq[i] = p.max_q[so];
      dn[i] = p.denom[so];
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const bool ok = row0 + 256 * i + tid < p.S && dn[i] > 0.f;
      const float tv = -(p.log2_thresh + (mq[i] * p.sf + __log2f(dn[i]))) * (1.f / p.sf);
      tab[256 * i + tid] = ok ? tv : -__builtin_huge_valf();
    }
  }
  __syncthreads();

  // ---- 1: one bit per row ----
  constexpr int FW = (NB + 3) / 4;
  uint32_t flags[FW] = {};   // byte b % 4 of word b / 4: rows 512 b + 8 lane + 0..7
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    if (512 * b < 128 * nqb) {
      const f32x4* t = reinterpret_cast<const f32x4*>(tab + 512 * b + 8 * lane);
      const f32x4 t0 = t[0], t1 = t[1];
      uint32_t f = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float lo = __builtin_bit_cast(float, x[b][i] << 16);
        const float hi = __builtin_bit_cast(float, x[b][i] & 0xffff0000u);
        const float a = i < 2 ? t0[2 * (i & 1)] : t1[2 * (i & 1)];
        const float c = i < 2 ? t0[2 * (i & 1) + 1] : t1[2 * (i & 1) + 1];
        f |= (lo + a > p.blk_slack) ? (1u << (2 * i)) : 0u;
        f |= (hi + c > p.blk_slack) ? (2u << (2 * i)) : 0u;
      }
      flags[b / 4] |= f << (8 * (b % 4));
    }
  }
  uint32_t any = 0;
#pragma unroll
  for (int w = 0; w < FW; ++w) any |= flags[w];

  SPATTN_LDS unsigned long long* vw = (SPATTN_LDS unsigned long long*)votes[wave];
  if (lane < CHUNK) vw[lane] = 0;
  if (__ballot(any != 0) != 0) {
    // A copy of a tile: lane h * CPR + pos of copy c fetches chunk pos ^ swz of row LPP h + c, so that the operand
    // reads below (sixteen lanes, one chunk of sixteen rows) cover all sixteen 16-byte bank groups.
    auto swz = [](int r) -> int { return D == 128 ? r : ((r & 1) | ((r >> 2) << 1)); };
    const uint32_t ring = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(lds_cptr)ring_all + wave * (NS * TILE));
    const int h = lane / CPR;
    uint32_t goff[LPP];
#pragma unroll
    for (int c = 0; c < LPP; ++c) goff[c] = (uint32_t)(((lane % CPR) ^ swz(LPP * h + c)) << 4);
    // operand of k-step t in slot 0: this ^ (t << 6)
    const int m = lane & 15;
    const uint32_t rd0 = ring + (m % LPP) * 1024 + (m / LPP) * ROWB + ((g ^ swz(m)) << 4);
    auto read_tile = [&](uint32_t slot, u32x4 (&d)[NT]) {
#pragma unroll
      for (int t = 0; t < NT; ++t) d[t] = *(SPATTN_LDS const u32x4*)((lds_cptr)(uintptr_t)((rd0 + slot) ^ (uint32_t)(t << 6)));
    };
    auto copy = [&](uint32_t off, uint32_t slot, int c) { dma16(qc, off, __builtin_amdgcn_readfirstlane(ring + slot + c * 1024)); };
    // The keys, sixteen at a time like a tile of rows; rows past the last key repeat it, their votes are masked off.
    auto copy_keys = [&](int n, int slot) {
#pragma unroll
      for (int c = 0; c < LPP; ++c) {
        int r = 64 * J + 16 * n + LPP * h + c;
        r = r < p.kv_len ? r : p.kv_len - 1;
        dma16<true>(kh, (uint32_t)r * ROWB + goff[c], __builtin_amdgcn_readfirstlane(ring + (slot * LPP + c) * 1024));
      }
    };
#pragma unroll
    for (int n = 0; n < NS; ++n) copy_keys(n, n);

    const SPATTN_LDS float* ltab = (const SPATTN_LDS float*)tab;
    SPATTN_LDS uint16_t* lrow = (SPATTN_LDS uint16_t*)list_row[wave];
    const int myq = lane >> 4;   // q-block of the batch that this lane's rows belong to
    u32x4 kf[4][NT];
    bool keys_left = true;
    int b = 0;
    for (;;) {
      // ---- 2: list rows until the list is full or the chunk has ended; the keys arrive meanwhile ----
      int ng = 0;   // listed rows, in fours
      bool more = false;
      while (512 * b < 128 * nqb) {
        uint32_t fw = flags[0];
#pragma unroll
        for (int w = 1; w < FW; ++w) fw = (b >> 2) == w ? flags[w] : fw;
        const uint32_t f = (fw >> (8 * (b & 3))) & 0xffu;
        int total;
        const int before = row_scan(__popc(f), total);
        const int n0 = (__builtin_amdgcn_readlane(total, 15) + 3) >> 2;
        const int n1 = (__builtin_amdgcn_readlane(total, 31) + 3) >> 2;
        const int n2 = (__builtin_amdgcn_readlane(total, 47) + 3) >> 2;
        const int n3 = (__builtin_amdgcn_readlane(total, 63) + 3) >> 2;
        const int e0 = ng + n0, e1 = e0 + n1, e2 = e1 + n2, e3 = e2 + n3;
        if (e3 > 4 * CAP) {
          more = true;
          break;
        }
        const int start = myq == 0 ? ng : myq == 1 ? e0 : myq == 2 ? e1 : e2;
        const int end = myq == 0 ? e0 : myq == 1 ? e1 : myq == 2 ? e2 : e3;
        if (e3 > ng) {
          // The last four of a q-block are filled up with one of its listed rows (whichever lane stores last), which only
          // votes again: no row of another q-block, finite or not, is multiplied for this one.
          if (f) {
            const uint16_t first = (uint16_t)(512 * b + 8 * lane + __builtin_ctz(f));
            *(SPATTN_LDS u16x4*)(lrow + 4 * end - 4) = u16x4{first, first, first, first};
          }
          int pos = 4 * start + before;
#pragma unroll
          for (int i = 0; i < 8; ++i)
            if (f & (1u << i)) lrow[pos++] = (uint16_t)(512 * b + 8 * lane + i);
        }
        ng = e3;
        if (b == 0) {
          wait_vmcnt<0>();
#pragma unroll
          for (int n = 0; n < NS; ++n) read_tile(n * TILE, kf[n]);
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
          for (int n = NS; n < 4; ++n) copy_keys(n, n - NS);
        }
        ++b;
      }
      const int nt = (ng + 3) >> 2;
      if (lane < 16 * nt - 4 * ng) lrow[4 * ng + lane] = lrow[4 * ng - 1];   // the last tile: with its last row
      if (keys_left) {
        keys_left = false;
        wait_vmcnt<0>();
#pragma unroll
        for (int n = NS; n < 4; ++n) read_tile((n - NS) * TILE, kf[n]);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
      // ---- 3: multiply the listed tiles ----
      if (nt > 0) {
        // The row lists are written and read by this wave alone, in order: the LDS keeps to it, and the compiler does,
        // as vector types (the entries are read two and four at a time) may alias what was written.
        asm volatile("" ::: "memory");
        struct Load {
          uint32_t off[LPP];
        };
        auto prepare = [&](int i) -> Load {
          i = i < nt ? i : nt - 1;
          Load l;
          uint32_t r[LPP];
          if constexpr (LPP == 4) {
            const u32x2 e = *(const SPATTN_LDS u32x2*)(lrow + 16 * i + 4 * h);
            r[0] = e[0] & 0xffffu, r[1] = e[0] >> 16, r[2] = e[1] & 0xffffu, r[3] = e[1] >> 16;
          } else {
            const u16x2 e = *(const SPATTN_LDS u16x2*)(lrow + 16 * i + 2 * h);
            r[0] = e[0], r[1] = e[1];
          }
#pragma unroll
          for (int c = 0; c < LPP; ++c) l.off[c] = r[c] * ROWB + goff[c];
          return l;
        };
#pragma unroll
        for (int j = 0; j < NS; ++j) {
          const Load l = prepare(j);
#pragma unroll
          for (int c = 0; c < LPP; ++c) copy(l.off[c], j * TILE, c);
        }
        wait_vmcnt<(NS - 1) * LPP>();
        u32x4 qa[2][NT];
        read_tile(0, qa[0]);
        // the C operand of tile i: rows 4 g .. 4 g + 3
        auto read_thr = [&](int i) -> f32x4 {
          i = i < nt ? i : nt - 1;
          const u32x2 e = *(const SPATTN_LDS u32x2*)(lrow + 16 * i + 4 * g);
          return f32x4{ltab[e[0] & 0xffffu], ltab[e[0] >> 16], ltab[e[1] & 0xffffu], ltab[e[1] >> 16]};
        };
        f32x4 thr_next = read_thr(0);
        uint32_t slot = 0;
        auto tile = [&](auto par, int i) {   // tile i, its operands in qa[P]
          constexpr int P = decltype(par)::value;
          const uint32_t next = slot + TILE == NS * TILE ? 0 : slot + TILE;
          // tile i+1 has landed; the operands of this tile have left its slot
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"((NS - 2) * LPP) : "memory");
          const Load l = prepare(i + NS);
          const int qb = (int)lrow[16 * i + 4 * (lane & 3)] >> 7;   // lanes 0..3: q-block of the tile's fours
          const f32x4 thr = thr_next;
          thr_next = read_thr(i + 1);
          read_tile(next, qa[P ^ 1]);
#pragma unroll
          for (int c = 0; c < LPP; ++c) copy(l.off[c], slot, c);
          f32x4 acc[4];
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int n = 0; n < 4; ++n) acc[n] = mfma16(qa[P][t], kf[n][t], t == 0 ? thr : acc[n]);
          // Bit 16 g + j of a ballot: some row of the tile's four g passes for key j of the sixteen.  A listed row has a
          // finite threshold, hence no score that is a NaN (at a threshold of 0, where every row with a key is listed, a
          // score of -inf gives one here as in the full sweep).
          unsigned long long w[4];
#pragma unroll
          for (int n = 0; n < 4; ++n) {
            const i32x4 v = __builtin_bit_cast(i32x4, acc[n]);   // a float is > 0 exactly when its bits are, as an integer
            const int a = v[0] > v[1] ? v[0] : v[1], c = v[2] > v[3] ? v[2] : v[3];
            w[n] = __ballot((a > c ? a : c) > 0);
          }
          // lanes 0..3: the 64 bits of one four
          const int sh = 16 * (lane & 3);
          const uint32_t lo = __builtin_amdgcn_perm((uint32_t)(w[1] >> sh), (uint32_t)(w[0] >> sh), 0x05040100u);
          const uint32_t hi = __builtin_amdgcn_perm((uint32_t)(w[3] >> sh), (uint32_t)(w[2] >> sh), 0x05040100u);
          if (lane < 4) {
            const unsigned long long v = ((unsigned long long)hi << 32) | lo;
            __hip_atomic_fetch_or(vw + qb, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
          }
          slot = next;
        };
        int i = 0;
        for (; i + 2 <= nt; i += 2) {
          tile(std::integral_constant<int, 0>{}, i);
          tile(std::integral_constant<int, 1>{}, i + 1);
        }
        if (i < nt) tile(std::integral_constant<int, 0>{}, i);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
      wait_vmcnt<0>();   // no copy may land in a slot that the next list uses, or after the workgroup has given up its LDS
      if (!more) break;
    }
    wait_vmcnt<0>();
  }
  // ---- 4: the 64 bits of every q-block; keys past the last have none ----
  if (64 * J < 32 * p.words && lane < nqb) {
    const unsigned long long v = left >= 64 ? vw[lane] : left <= 0 ? 0ull : vw[lane] & ((1ull << left) - 1ull);
    *reinterpret_cast<u32x2*>(p.bits + ((size_t)bh * p.SB + qb0 + lane) * p.words + 2 * J) = __builtin_bit_cast(u32x2, v);
  }
}

// q-blocks per chunk.  A wave's tiles are a serial chain, so where the longest chunks leave the chip idle, or in their second
// round, they are cut to what fills the round; `resident` workgroups are on the chip at a time (three per CU at d = 128, by
// registers, four at d = 64, by LDS).  per_chunk: workgroups per chunk of rows.  Longer launches keep whole batches of four
// q-blocks (16 x 12743 x 64 in chunks of 25 instead of 28: 75 -> 82 us).  With chunks of no less than four q-blocks, cut until
// there were four workgroups per CU, and now, us at 1/4, 1, 4, 16, 32 mean weights:
//   16 x 400 x 64      10.6 / 10.2 / 8.7 / 6.6 / 5.5      5.2 / 5.0 / 4.9 / 4.6 / 4.7
//   16 x 512 x 128     14.7 / 14.3 / 12.8 / 9.5 / 7.9     6.1 / 5.9 / 5.7 / 5.2 / 4.9
//   24 x 1000 x 128    13.7 / 12.4 / 10.4 / 7.8 / 6.7     10.4 / 9.4 / 8.4 / 7.0 / 6.4
//   16 x 4096 x 128    66 / 50 / 34 / 22 / 18             58 / 43 / 30 / 18 / 15
//   12 x 7000 x 64     88 / 65 / 42 / 28 / 23             75 / 56 / 38 / 23 / 19
static int votes_chunk(int SB, int most, int resident, long long per_chunk) {
  const int nch = (SB + most - 1) / most;
  const long long rounds = (nch * per_chunk + resident - 1) / resident;
  if (rounds > 2) return ((SB + nch - 1) / nch + 3) / 4 * 4;
  const long long fit = rounds * resident / per_chunk;   // chunks, not fewer than nch
  return fit < SB ? (SB + (int)fit - 1) / (int)fit : 1;
}

// The block test runs a little below the vote threshold, tau (1 - 1e-3): the statistics sweep rounds a
// score and compares, the vote accumulates s - t in the matrix unit, so a key whose margin is below fp32
// rounding could otherwise sit in a block the (rounded up) maxima leave out.  The rows this adds
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
  p.blk_slack = thresh > 0.f ? log2f((float)(1.0 - 1e-3)) / sf : 0.f;
  p.sf = sf;
  p.HB = HB;
  p.S = S;
  p.kv_len = kv_len;
  p.Sp = SB * 128;
  p.SB = SB;
  p.words = mask_stride / 32;
  p.jgroups = (p.words / 2 + 3) / 4;
  p.ch_qblocks = votes_chunk(SB, D == 128 ? VotesCfg<128>::kChunk : VotesCfg<64>::kChunk, (D == 128 ? 3 : 4) * 256,
                             (long long)p.jgroups * HB);
  p.nch = (SB + p.ch_qblocks - 1) / p.ch_qblocks;
  const dim3 grid(p.jgroups * p.nch * HB);
  // short chunks: a quarter to an eighth of the thresholds to make, LDS and maxima to hold (96 x 732 x 64 8.9 -> 7.3 us at 16
  // mean weights, 24 x 1000 x 128 7.5 -> 7.0; a bound read in the one kernel took 2-3 % from the long launches)
  const bool small = p.ch_qblocks <= 4;
  if (D == 128 && small) hipLaunchKernelGGL((blockmax_votes_kernel<128, 4>), grid, dim3(256), 0, stream, p);
  else if (D == 128) hipLaunchKernelGGL((blockmax_votes_kernel<128, VotesCfg<128>::kChunk>), grid, dim3(256), 0, stream, p);
  else if (small) hipLaunchKernelGGL((blockmax_votes_kernel<64, 4>), grid, dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((blockmax_votes_kernel<64, VotesCfg<64>::kChunk>), grid, dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace spattn
