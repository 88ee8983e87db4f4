// Block-list sparse attention instantiations (64-key blocks).
#include "attn_fwd.h"
#include "dispatch.h"

namespace spattn {

hipError_t run_attn_blocks(const AttnParams& p, int D, int qblk, hipStream_t stream, int heads) {
  if (lists_by_halves(D, qblk, false, heads > 0 ? heads : (long long)p.B * p.H, p.S, p.kv_len, p.idx_stride)) {
    if (D == 128) return launch_attn_fwd<128, 64, KV_BLOCKS, true, false, 1, true>(p, stream);
    return launch_attn_fwd<64, 64, KV_BLOCKS, true, false, 1, true>(p, stream);
  }
  if (D == 128 && qblk == 128) return launch_attn_fwd<128, 128, KV_BLOCKS, true, false>(p, stream);
  if (D == 128 && qblk == 64) return launch_attn_fwd<128, 64, KV_BLOCKS, true, false>(p, stream);
  if (D == 64 && qblk == 128) return launch_attn_fwd<64, 128, KV_BLOCKS, true, false>(p, stream);
  if (D == 64 && qblk == 64) return launch_attn_fwd<64, 64, KV_BLOCKS, true, false>(p, stream);
  return hipErrorInvalidValue;
}

hipError_t prepare_attn_blocks() {
  hipError_t e = prepare_attn_fwd<128, 128, KV_BLOCKS, true, false>();
  if (e == hipSuccess) e = prepare_attn_fwd<128, 64, KV_BLOCKS, true, false>();
  if (e == hipSuccess) e = prepare_attn_fwd<64, 128, KV_BLOCKS, true, false>();
  if (e == hipSuccess) e = prepare_attn_fwd<64, 64, KV_BLOCKS, true, false>();
  if (e == hipSuccess) e = prepare_attn_fwd<128, 64, KV_BLOCKS, true, false, 1, true>();
  if (e == hipSuccess) e = prepare_attn_fwd<64, 64, KV_BLOCKS, true, false, 1, true>();
  return e;
}

}  // namespace spattn
