// Dense attention / row-statistics instantiations: q-blocks of 128 rows, and for launches that leave the chip idle with
// those, of 64 rows and of either size with two groups of waves per q-block; of 256 rows for long launches at d = 128.
#include "attn_fwd.h"
#include "dispatch.h"

namespace spattn {

// Four forms with q-blocks of 128 or 64 rows (64: two waves share the rows of a tile and take half of its keys each),
// by one group of four waves or two (which take half of the tiles each).  A q-block is done sooner the more waves share
// it, for more K / V copies per row and a merge; that pays while the q-blocks do not queue.  Measured as time over that
// of the 128-row form by one group, unless said otherwise:
//   64-row q-blocks, up to one per CU (256), both head dims: dense 256 keys 0.89-0.93, 1000 keys 0.73-0.80, 4096 keys
//   0.66-0.73; with statistics 0.70-0.90, statistics only 0.72-0.88;
//   at d = 64 from 768 keys on up to three per CU, what the 40 KB ring and registers allow (768): dense 0.87-0.96, with
//   statistics 0.93-0.98, statistics only 0.89-0.98; at 256 and 512 keys that is 0.93-1.09, behind 768 q-blocks 1.08-1.14.
//   d = 128 is slower (1.02-1.2, with statistics 1.2-1.5: its LDS allows one workgroup per CU) from the second q-block per
//   CU on, except the statistics alone, whose ring is 48 KB, from 768 keys on: 0.90-0.96 up to three per CU, 1.12-1.2 behind.
//   The statistics alone at d = 64 would fit five to a CU and gain 2-6 % from 513 to 640 q-blocks of 128 rows, but a row's
//   denominator would then not have the bits that attention with statistics gives it, nor its mask the same keys.
//   Two groups on 64-row q-blocks, up to one per CU, against one group on them: d = 64 from 12 tiles on 0.72-0.95, 10 and 11
//   0.92-0.99 (8 x 588 with statistics 9.0 -> 8.3 us), 8 and 9 0.99-1.04; d = 128 from 15 on 0.75-1.00 (12 tiles 0.99, 8 tiles
//   1.07-1.13).  Dense with statistics at d = 128 has no LDS for it.
//   Two groups on 128-row q-blocks, up to one per CU, against the best of the other forms: d = 128 from 12 tiles on 0.84-0.95
//   (8 tiles 0.98-1.06); d = 64 from 24 tiles on 0.90-0.98, with statistics from 15 on 0.92-0.96 (below 0.97-1.02).
// 256-row q-blocks by one group of eight waves (d = 128 with V): half of the K / V copies per row, at the power cap
// worth 2-5 % of a full round of one q-block per CU (12 x 32768 5.49 -> 5.28 ms; 2048 keys 2 %, 1024 keys -1, 512 keys -5),
// and a workgroup of its own finishes a CU's last q-block sooner than two do.  A last round that fills up to half of the CUs
// costs it 0-19 % instead (its other form spreads that round over twice as many).  From 32 tiles on with the last round
// empty or more than half full 0.91-0.98; where that is the only round from 22 tiles on 0.90-0.99 (24 x 1715 46.9 -> 42.1 us, 32 x
// 1495 44.6 -> 41.6, with statistics 24 x 1626 46.2 -> 44.0), two rounds of 22-31 tiles 0.97-1.02.  With
// statistics, whose row maxima keep the waves of a workgroup waiting for each other, that holds up to two rounds (0.94-0.99; 12
// x 9000 502 -> 471 us) and from 64 tiles on up to five (68 tiles
// 0.99, 90 and more 0.95-0.98: 12 x 14000 1163 -> 1105, 12 x 20000 2243 -> 2165, 16 x 20400 2968 -> 2905; 36 tiles in three
// rounds 0.98, left to the 128-row form), behind them 0.98-1.03.  Same bits as the 128-row form.
// The other forms add the row sums and outputs of a row in another order: a launch over some heads of a computation
// goes by all of its heads, so that a row's denominator, and with it a key at a threshold, does not depend on the split.
// Between 128 and 256 rows, where no bit changes, it goes by its own q-blocks (3 of 12 heads x 9000 with statistics 142 us
// by its own, 210 by all; 3 of 24 x 5000 77 and 120; 5 of 50 x 2049 36 and 52).
DenseForm dense_form(int D, bool has_v, bool stats, int S, int kv_len, long long launched, long long of_heads) {
  constexpr int kCus = 256;
  const long long heads = of_heads > 0 ? of_heads : launched;
  const long long n64 = heads * ((S + 63) / 64), n128 = heads * ((S + 127) / 128);
  const int tiles = (kv_len + 63) / 64;
  if (n64 <= kCus) return {64, !(D == 128 && has_v && stats) && tiles >= (D == 64 ? 10 : 15) ? 2 : 1};
  if (n128 <= kCus && tiles >= (D == 128 ? 12 : stats ? 15 : 24)) return {128, 2};
  if ((D == 64 || !has_v) && kv_len >= 768 && n64 <= 3 * kCus) return {64, 1};
  if (D == 128 && has_v) {
    const long long n256 = launched * ((S + 255) / 256);
    const long long last = n256 % kCus;
    const bool few = n256 <= 2 * kCus || (tiles >= 64 && n256 <= 5 * kCus);
    if (tiles >= (n256 <= kCus ? 22 : 32) && (last == 0 || last > kCus / 2) && (!stats || few)) return {256, 1};
  }
  return {128, 1};
}

template <int D, bool HAS_V, bool STATS>
static hipError_t run(const AttnParams& p, int heads, hipStream_t stream) {
  const DenseForm f = dense_form(D, HAS_V, STATS, p.S, p.kv_len, (long long)p.B * p.H, heads);
  AttnParams pf = p;
  // the statistics cover the rows up to Sp
  if (f.rows == 64) pf.nqblk = (STATS ? p.Sp : p.S + 63) / 64;
  if (f.rows == 256) pf.nqblk = (p.S + 255) / 256;
  if (f.rows == 64 && f.groups == 2) {
    if constexpr (!(D == 128 && HAS_V && STATS)) return launch_attn_fwd<D, 64, KV_DENSE, HAS_V, STATS, 2>(pf, stream);
  }
  if (f.rows == 64) return launch_attn_fwd<D, 64, KV_DENSE, HAS_V, STATS>(pf, stream);
  if (f.rows == 128 && f.groups == 2) return launch_attn_fwd<D, 128, KV_DENSE, HAS_V, STATS, 2>(pf, stream);
  if (f.rows == 256) {
    if constexpr (D == 128 && HAS_V) return launch_attn_fwd<D, 256, KV_DENSE, HAS_V, STATS>(pf, stream);
  }
  return launch_attn_fwd<D, 128, KV_DENSE, HAS_V, STATS>(p, stream);
}

hipError_t run_attn_dense(const AttnParams& p, int D, bool has_v, bool stats, hipStream_t stream, int heads) {
  if (D == 128) {
    if (has_v && !stats) return run<128, true, false>(p, heads, stream);
    if (has_v && stats) return run<128, true, true>(p, heads, stream);
    if (!has_v && stats) return run<128, false, true>(p, heads, stream);
  } else if (D == 64) {
    if (has_v && !stats) return run<64, true, false>(p, heads, stream);
    if (has_v && stats) return run<64, true, true>(p, heads, stream);
    if (!has_v && stats) return run<64, false, true>(p, heads, stream);
  }
  return hipErrorInvalidValue;
}

template <int D, int QBLK>
static hipError_t prepare() {
  hipError_t e = prepare_attn_fwd<D, QBLK, KV_DENSE, true, false>();
  if (e == hipSuccess) e = prepare_attn_fwd<D, QBLK, KV_DENSE, true, true>();
  if (e == hipSuccess) e = prepare_attn_fwd<D, QBLK, KV_DENSE, false, true>();
  if (e == hipSuccess) e = prepare_attn_fwd<D, QBLK, KV_DENSE, true, false, 2>();
  if constexpr (!(D == 128 && QBLK == 64)) {
    if (e == hipSuccess) e = prepare_attn_fwd<D, QBLK, KV_DENSE, true, true, 2>();
  }
  if (e == hipSuccess) e = prepare_attn_fwd<D, QBLK, KV_DENSE, false, true, 2>();
  return e;
}

hipError_t prepare_attn_dense() {
  hipError_t e = prepare<128, 128>();
  if (e == hipSuccess) e = prepare<128, 64>();
  if (e == hipSuccess) e = prepare<64, 128>();
  if (e == hipSuccess) e = prepare<64, 64>();
  if (e == hipSuccess) e = prepare_attn_fwd<128, 256, KV_DENSE, true, false>();
  if (e == hipSuccess) e = prepare_attn_fwd<128, 256, KV_DENSE, true, true>();
  return e;
}

}  // namespace spattn
