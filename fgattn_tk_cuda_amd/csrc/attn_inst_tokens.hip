// Token-list (gathered) sparse attention instantiations.
#include "attn_fwd.h"
#include "dispatch.h"

namespace spattn {

// A launch that leaves the chip idle is done sooner the more waves share a row: lists of 128-row q-blocks, of either kind, run
// by workgroups of 64 rows, two to a list, up to one of those per CU (256), at d = 64 up to the three per CU that its ring
// and registers allow.  Time over that of the 128-row form, random lists of 8 and 30 % of the keys:
//   d = 64 up to one per CU 0.73-0.95 (8 x 2000 13.3 -> 9.8 us with 10 tiles a list, 8 x 1000 4.2 -> 4.0 with one);
//   d = 64 up to three per CU 0.84-0.98 (12 x 4000 29.3 -> 24.7 us with 19 tiles), but lists of one tile below 1024 keys up to
//   1.04, and block lists below five blocks 0.96-1.10 (theirs are as long as their stride says); behind three per CU 1.03-1.10;
//   d = 128 up to one per CU 0.77-0.97 (8 x 2000 16.8 -> 12.9 us with 10 tiles), lists of one tile 1.01-1.05, which sequences
//   below 768 keys have; from the second per CU on 0.98-1.23.
// The rule looks at the launch alone, not at the counts, which are on the device.  The halves add a row's keys in another
// order: a launch over some heads of a computation goes by all of its heads, so that no bit depends on the split.
bool lists_by_halves(int D, int qblk, bool tokens, long long heads, int S, int kv_len, int idx_stride) {
  if (qblk != 128) return false;
  constexpr long long kCus = 256;
  const long long n64 = heads * ((S + 63) / 64);
  if (D == 128) return n64 <= kCus && kv_len >= 768 && idx_stride >= (tokens ? 256 : 2);
  return n64 <= kCus || (n64 <= 3 * kCus && kv_len >= 1024 && (tokens || idx_stride >= 5));
}

hipError_t run_attn_tokens(const AttnParams& p, int D, int qblk, hipStream_t stream, int heads) {
  if (lists_by_halves(D, qblk, true, heads > 0 ? heads : (long long)p.B * p.H, p.S, p.kv_len, p.idx_stride)) {
    if (D == 128) return launch_attn_fwd<128, 64, KV_TOKENS, true, false, 1, true>(p, stream);
    return launch_attn_fwd<64, 64, KV_TOKENS, true, false, 1, true>(p, stream);
  }
  if (D == 128 && qblk == 128) return launch_attn_fwd<128, 128, KV_TOKENS, true, false>(p, stream);
  if (D == 128 && qblk == 64) return launch_attn_fwd<128, 64, KV_TOKENS, true, false>(p, stream);
  if (D == 64 && qblk == 128) return launch_attn_fwd<64, 128, KV_TOKENS, true, false>(p, stream);
  if (D == 64 && qblk == 64) return launch_attn_fwd<64, 64, KV_TOKENS, true, false>(p, stream);
  return hipErrorInvalidValue;
}

hipError_t prepare_attn_tokens() {
  hipError_t e = prepare_attn_fwd<128, 128, KV_TOKENS, true, false>();
  if (e == hipSuccess) e = prepare_attn_fwd<128, 64, KV_TOKENS, true, false>();
  if (e == hipSuccess) e = prepare_attn_fwd<64, 128, KV_TOKENS, true, false>();
  if (e == hipSuccess) e = prepare_attn_fwd<64, 64, KV_TOKENS, true, false>();
  if (e == hipSuccess) e = prepare_attn_fwd<128, 64, KV_TOKENS, true, false, 1, true>();
  if (e == hipSuccess) e = prepare_attn_fwd<64, 64, KV_TOKENS, true, false, 1, true>();
  return e;
}

}  // namespace spattn
