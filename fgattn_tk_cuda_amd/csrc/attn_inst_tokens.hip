// Token-list (gathered) sparse attention instantiations.
#include "attn_fwd.h"
#include "dispatch.h"

namespace spattn {

// A launch that leaves the chip idle is done sooner the more waves share a row: lists of 128-row q-blocks, of either kind, run
// by workgroups of 64 rows, two to a list, up to one of those per CU (256), at d = 64 up to the three per CU that its ring
// and registers allow.  The workgroups count, not the 64-row blocks: of an odd number of blocks the last list has a second
// workgroup that ends at once, and one workgroup above a CU's share costs 8-29 % (19 x 800 x 128, 266 workgroups: 1.12-1.21).
// Time over that of the 128-row form, lists of threshold masks that keep 4 / 8.5 / 16 % of the keys, and lists of equal length:
//   block lists 0.65-0.80, d = 64 behind one per CU 0.72-0.88 (they are a third of the row and more); equal ones at d = 128
//   1.04-1.07 with one block, 0.96-1.01 with two, 0.93-0.95 with three; at d = 64 up to one per CU 0.97-1.03, 0.91-0.94, 0.88-0.92; in the
//   second per CU 1.06-1.11 with one, 1.02-1.06 with three, 0.98-1.02 with six; in the third 1.04, 0.96-0.98, 0.95;
//   token lists, d = 128: 1.03-1.07 with one tile of 64 keys, 0.96-0.99 with two, 0.94-0.95 with three; at 4 % 1.04-1.05 up to
//   1600 keys, 0.99-1.01 at 2300, 0.93-0.95 at 4000; at 8.5 % and 16 % 0.97 / 0.90 at 1100 and 0.84 / 0.75 at 4000;
//   d = 64 up to one per CU: 0.97-1.00 with one tile, 0.91 with two, 0.89 with three; 4 % 0.97-1.01 up to 1600 keys, 0.90 at 4000;
//   in the second per CU 1.03-1.06 with one to three tiles, 0.99 with four, 0.93-0.97 with six; 4 % 1.04-1.10 up to 2300 keys, 0.99
//   at 4000, 0.88 at 8000; in the third 1.00-1.04 with one, 0.95-0.98 with two and three; 4 % 1.03-1.04 up to 1600 keys, 1.015 at
//   2300, 0.95 at 4000.
// The counts are on the device.  A row of token ids that is shorter than the sequence says how long its lists are; one that holds
// the sequence is taken to hold 4 % of its keys, the sparsest mask, so denser ones in short sequences keep the 128-row form.
// Block lists are taken to be as long as their rows: masks that fill rows of the whole sequence keep a third of the blocks.
// The halves add a row's keys in another order: a launch over some heads of a computation goes by all of its heads, so that no
// bit depends on the split.
bool lists_by_halves(int D, int qblk, bool tokens, long long heads, int S, int kv_len, int idx_stride) {
  if (qblk != 128) return false;
  constexpr long long kCus = 256;
  const int nqblk = (S + 127) / 128;
  const long long wgs = 2 * heads * nqblk;
  const int len = !tokens ? idx_stride : idx_stride < 128 * nqblk ? idx_stride / 128 : (kv_len + 1599) / 1600;   // blocks; tiles
  if (D == 128) return wgs <= kCus && kv_len >= 768 && len >= 2;
  if (wgs <= kCus) return tokens || len >= 2;
  return kv_len >= 1024 && (wgs <= 2 * kCus ? len >= (tokens ? 3 : 7) : wgs <= 3 * kCus && len >= (tokens ? 2 : 5));
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
