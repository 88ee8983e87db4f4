// Bit-packed vote masks for the mask cache.
//
// The reference keeps a cached mask as one bit per key, least significant bit first
// (python/spattn/mask_utils.py:421-439, `pack` / `unpack`), and on every reuse expands it
// with torch ops to an int32 mask that booleanmask_to_indexmask then compacts
// (CompressedBitMaskCache, python/spattn/mask_utils.py:74-98).  Here both directions are
// single kernels:
//   pack_mask_kernel            int32 vote mask -> bits            (reads 4 B per key, writes 1/8 B)
//   packed_to_indexmask_kernel  bits -> ascending index lists      (reads 1/8 B per key, writes 4 B per kept key)
// so that a reuse of a cached mask streams 1/32 of the bytes of the int32 path and never
// materialises the unpacked mask.
#include "common.h"
#include "dispatch.h"

namespace spattn {

// ------------------------------------------------------------------------------------
// pack: bit (c & 7) of byte c >> 3 of a row is set iff mask[row][c] > 0.
// One wave per step of 2048 keys (8 coalesced 16-byte loads per lane, the next step in
// flight).  A lane's four keys give a nibble; three shift-and-or exchanges with the lanes
// 1, 2 and 4 further on assemble the 32 keys of eight neighbouring lanes into one word,
// which every eighth lane stores.
// ------------------------------------------------------------------------------------
constexpr int kPackUnroll = 8;

__global__ __launch_bounds__(256) void pack_mask_kernel(uint32_t* __restrict__ packed, const int* __restrict__ mask,
                                                        int rows, int mask_stride) {
  constexpr int U = kPackUnroll;
  constexpr int SPAN = 256 * U;   // keys per wave step
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int words_per_row = mask_stride >> 5;
  const int nstep = (mask_stride + SPAN - 1) / SPAN;
  for (int row = blockIdx.x * 4 + wave; row < rows; row += gridDim.x * 4) {
    const int* __restrict__ src = mask + (size_t)row * mask_stride;
    uint32_t* __restrict__ dst = packed + (size_t)row * words_per_row;
    i32x4 cur[U], nxt[U];
    auto load = [&](int c, i32x4 (&v)[U]) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e0 = c * SPAN + u * 256 + 4 * lane;
        const i32x4 z = {0, 0, 0, 0};
        v[u] = (e0 < mask_stride) ? __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(src + e0)) : z;
      }
    };
    load(0, cur);
    for (int c = 0; c < nstep; ++c) {
      if (c + 1 < nstep) load(c + 1, nxt);
#pragma unroll
      for (int u = 0; u < U; ++u) {
        uint32_t x = (cur[u][0] > 0 ? 1u : 0u) | (cur[u][1] > 0 ? 2u : 0u) | (cur[u][2] > 0 ? 4u : 0u) |
                     (cur[u][3] > 0 ? 8u : 0u);
        // lanes l + 1, l + 2, l + 4 of the same 16-lane row (row_shl: data moves towards lane 0); only the
        // lanes with l % 8 == 0 use the result, and their partners lie in their own group of eight
        x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x101, 0xf, 0xf, true) << 4;
        x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x102, 0xf, 0xf, true) << 8;
        x |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0x104, 0xf, 0xf, true) << 16;
        const int word = (c * SPAN + u * 256 + 4 * lane) >> 5;
        if ((lane & 7) == 0 && word < words_per_row) dst[word] = x;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) cur[u] = nxt[u];
    }
  }
}

hipError_t run_pack_mask(uint32_t* packed, const int* mask, int rows, int mask_stride, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  int grid = (rows + 3) / 4;
  if (grid > 2048) grid = 2048;
  hipLaunchKernelGGL(pack_mask_kernel, dim3(grid), dim3(256), 0, stream, packed, mask, rows, mask_stride);
  return hipGetLastError();
}

// ------------------------------------------------------------------------------------
// packed bits -> index lists, the fused form of unpack + booleanmask_to_indexmask
// (include/mask_utils.cuh:273-302 for the compaction): per row the keys c < kv_len whose
// bit is set, ascending, counts exact; what lies behind the count is left to the caller or written
// with mask_stride (FILL).
// One wave per row, 2048 keys per step: a lane owns the 32 keys of one word (the words of the next four
// steps are in flight), a lane scan of the popcounts gives its place, it writes its keys into the wave's
// stage in LDS, and the stage leaves as consecutive words.
// What bounds it: without the fill the instructions of the bit loop, as many rounds as the fullest lane has
// keys.  32 keys per lane, four rounds between two branches and no ring bookkeeping: 71 us at 40 x 32760 rows
// (8.5 % of the keys, in runs; 42 MB read, 114 MB written), where 16 keys per lane and 4 KB bursts through a
// ring took 104.  With the fill the 1.34 GB of the lists, 0.28 ms (a plain fill of that size: 0.20 ms; the
// four waves filling one row after the other, staggered starts, 128-byte aligned or non-temporal stores:
// no faster).
template <bool FILL>
__global__ __launch_bounds__(256) void packed_to_indexmask_kernel(int* __restrict__ kv_indices, int* __restrict__ kv_num,
                                                                  const uint32_t* __restrict__ packed, int rows,
                                                                  int mask_stride, int kv_len) {
  constexpr int U = 4;   // steps whose words are in flight
  __shared__ int stage_all[4][2048 + 64];   // and a slot per lane for the rounds in which it has no key left
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int* const stage = stage_all[wave];
  const int lim = kv_len < mask_stride ? kv_len : mask_stride;
  const int words = mask_stride >> 5;
  const int nstep = (lim + 2047) >> 11;

  for (int row = blockIdx.x * 4 + wave; row < rows; row += gridDim.x * 4) {
    const uint32_t* __restrict__ src = packed + (size_t)row * words;
    int* __restrict__ dst = kv_indices + (size_t)row * mask_stride;
    int tail = 0;
    auto load = [&](int c) -> uint32_t {
      const int w = c * 64 + lane;
      return w < words ? src[w] : 0u;
    };
    uint32_t next[U];
#pragma unroll
    for (int u = 0; u < U; ++u) next[u] = load(u);
    for (int c0 = 0; c0 < nstep; c0 += U) {
      uint32_t cur[U];
#pragma unroll
      for (int u = 0; u < U; ++u) cur[u] = next[u];
      if (c0 + U < nstep) {
#pragma unroll
        for (int u = 0; u < U; ++u) next[u] = load(c0 + U + u);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int key0 = ((c0 + u) * 64 + lane) * 32;   // first key of this lane
        const int left = lim - key0;                     // its keys below lim
        uint32_t bits = cur[u];
        if (left < 32) bits = left <= 0 ? 0u : (bits & ((1u << left) - 1u));
        if (__ballot(bits != 0) == 0) continue;          // wave-uniform
        const int own = __popc(bits);
        const int incl = (int)lane_scan((uint32_t)own);
        const int total = __builtin_amdgcn_readlane(incl, 63);
        // four rounds between two branches; a lane without a key left writes its spare slot
        int at = incl - own;
        do {
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            stage[bits ? at : 2048 + lane] = key0 + lowest_bit(bits);
            bits &= bits - 1;
            ++at;
          }
        } while (__ballot(bits != 0) != 0);
        // the stage is the wave's own: its LDS operations are executed in order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int i = lane; i < total; i += 64) dst[tail + i] = stage[i];
        __builtin_amdgcn_wave_barrier();
        tail += total;
      }
    }
    if (lane == 0) kv_num[row] = tail;
    if constexpr (FILL) {   // whole lines from the next 16-byte boundary on
      const int v0 = (tail + 3) & ~3;
      if (lane < v0 - tail) dst[tail + lane] = mask_stride;
      const i32x4 f = {mask_stride, mask_stride, mask_stride, mask_stride};
      for (int i = v0 + 4 * lane; i < mask_stride; i += 256) *reinterpret_cast<i32x4*>(dst + i) = f;
    }
  }
}

hipError_t run_packed_to_indexmask(int* kv_indices, int* kv_num, const uint32_t* packed, int rows, int mask_stride,
                                   int kv_len, bool fill_tail, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  int grid = (rows + 3) / 4;
  if (grid > 65536) grid = 65536;
  if (fill_tail)
    hipLaunchKernelGGL(packed_to_indexmask_kernel<true>, dim3(grid), dim3(256), 0, stream, kv_indices, kv_num, packed, rows,
                       mask_stride, kv_len);
  else
    hipLaunchKernelGGL(packed_to_indexmask_kernel<false>, dim3(grid), dim3(256), 0, stream, kv_indices, kv_num, packed, rows,
                       mask_stride, kv_len);
  return hipGetLastError();
}

}  // namespace spattn
