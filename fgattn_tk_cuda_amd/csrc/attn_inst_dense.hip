// Dense attention / row-statistics instantiations: q-blocks of 128 rows, of 64 rows for launches that leave
// the chip idle with 128.
#include "attn_fwd.h"
#include "dispatch.h"

namespace spattn {

// With 64-row q-blocks two waves share the rows of a tile and take half of its keys each: a q-block is done in
// 0.65-0.8 of the time, for twice the K / V copies per row.  That pays while the 64-row q-blocks do not queue:
//   up to one per CU (256), at both head dims: dense 256 keys 1.07-1.13x, 1000 keys 1.25-1.37x, 4096 keys 1.37-1.51x
//   (16 x 512 x 128 11.1 -> 9.6 us, 4 x 4096 x 128 58.9 -> 42.8 us, 4 x 4096 x 64 46.4 -> 30.8 us); with statistics
//   1.11-1.42x (8 x 2048 x 128 34.7 -> 25.5 us), statistics only 1.14-1.38x;
//   at d = 64 from 768 keys on up to three per CU, what its 40 KB ring and registers allow (768): dense 1.04-1.15x
//   (24 x 1536 27.0 -> 23.5 us), with statistics 1.02-1.07x, statistics only 1.02-1.12x.  At 256 and 512 keys that
//   is 0.92-1.08x, behind 768 q-blocks 0.88-0.93x (64 x 1000 21.9 -> 24.3 us).  d = 128 loses 0.81-0.99x (with
//   statistics 0.65-0.83x, its LDS allows one workgroup per CU) from the second q-block per CU on.
// The two forms add the row sums and outputs of a row in another order: a launch over some heads of a computation
// goes by all of its heads, so that a row's denominator, and with it a key at a threshold, does not depend on the split.
static bool small_launch(const AttnParams& p, int D, int heads) {
  constexpr int kCus = 256;
  const long long n64 = (long long)(heads > 0 ? heads : p.B * p.H) * ((p.S + 63) / 64);
  return n64 <= kCus || (D == 64 && p.kv_len >= 768 && n64 <= 3 * kCus);
}

template <int D, bool HAS_V, bool STATS>
static hipError_t run(const AttnParams& p, int heads, hipStream_t stream) {
  if (!small_launch(p, D, heads)) return launch_attn_fwd<D, 128, KV_DENSE, HAS_V, STATS>(p, stream);
  AttnParams p64 = p;
  // the statistics cover the rows up to Sp
  p64.nqblk = (STATS ? p.Sp : p.S + 63) / 64;
  return launch_attn_fwd<D, 64, KV_DENSE, HAS_V, STATS>(p64, stream);
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
  return e;
}

hipError_t prepare_attn_dense() {
  hipError_t e = prepare<128, 128>();
  if (e == hipSuccess) e = prepare<128, 64>();
  if (e == hipSuccess) e = prepare<64, 128>();
  if (e == hipSuccess) e = prepare<64, 64>();
  return e;
}

}  // namespace spattn
