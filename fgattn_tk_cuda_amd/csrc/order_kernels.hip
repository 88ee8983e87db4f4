// Work order for list-driven attention with very uneven list lengths.
//
// One workgroup per q-block, dispatched in index order, leaves the longest lists to whoever
// happens to get them last: with Zipf-distributed lengths a quarter of the run is spent
// waiting for a few stragglers.  qblock_order_kernel sorts the q-blocks by list length,
// longest first, in quarter-octave classes (stable inside a class, so the order is a function
// of the counts alone); the attention kernels then let workgroup i take q-block order[i].
// Lists whose lengths differ by less than a factor of two keep the default order, in which every XCD works on
// neighbouring q-blocks of one head.  The reference has no counterpart: its grid is fixed
// to (q-block, head, batch) (include/sparseattn_asyncgatherload_padded.cuh:273).
#include <type_traits>

#include "common.h"
#include "dispatch.h"

namespace spattn {

constexpr int kOrderWaves = 16;
constexpr int kOrderSub = 2;                              // bits below the leading one that tell classes apart
constexpr int kOrderClasses = (22 << kOrderSub) + 2;      // 4 per octave up to 2^22 keys, one for longer lists, one for empty ones

// class 0 holds the longest lists
__device__ __forceinline__ int length_class(int c) {
  if (c <= 0) return kOrderClasses - 1;
  const int lg = 31 - __builtin_clz((unsigned)c);            // floor(log2 c), 0..30
  const int below = lg >= kOrderSub ? ((c >> (lg - kOrderSub)) & ((1 << kOrderSub) - 1))
                                    : ((c << (kOrderSub - lg)) & ((1 << kOrderSub) - 1));
  const int fine = (lg << kOrderSub) + below;
  return kOrderClasses - 2 - (fine < kOrderClasses - 2 ? fine : kOrderClasses - 2);
}

// One workgroup; wave w owns a contiguous segment of the counts and goes through it 64 at a time, four of those in flight.
// Lanes of one class find each other by seven ballots, so a class has one LDS add per wave and step, and the place of a count
// is what the classes ahead and the waves before hold plus its lanes before.  What bounds it is the chain of launch, load, three
// barriers and store in short calls, of the steps of a wave in long ones (one thread per segment, tables by thread and a
// serial scan over them: 9.6 us for 36 counts, now 3.5; 511 9.8, now 3.7; 8192 25, now 12.3; 100003 219, now 120).
__global__ __launch_bounds__(64 * kOrderWaves) void qblock_order_kernel(int* __restrict__ order,
                                                                         const int* __restrict__ counts, int n) {
  constexpr int W = kOrderWaves;
  constexpr int U = 4;
  static_assert(kOrderClasses <= 128, "two waves scan the classes, seven bits tell them apart");
  __shared__ int table[kOrderClasses * W];   // [class][wave]: members in that wave's segment, then offsets
  __shared__ int lo_l[W], hi_l[W], first_half;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int steps = (n + 64 * W - 1) / (64 * W);
  const int i0 = wave * steps * 64 + lane;

  // f(index, count, its slot, members of its class in lanes before, and in all lanes; 0 where there is no count)
  auto walk = [&](auto&& f) {
    for (int s = 0; s < steps; s += U) {
      int c[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = i0 + 64 * (s + u);
        c[u] = s + u < steps && i < n ? counts[i] : 0;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (s + u >= steps) break;
        const int i = i0 + 64 * (s + u);
        const int cls = length_class(c[u]);
        unsigned long long same = __ballot(i < n);
#pragma unroll
        for (int b = 0; b < 7; ++b) {
          const unsigned long long m = __ballot((cls >> b) & 1);
          same &= (cls >> b) & 1 ? m : ~m;
        }
        if (i < n) {
          const int before = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(same >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)same, 0));
          f(i, c[u], cls * W + wave, before, (int)__popcll(same));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    }
  };

  for (int e = tid; e < kOrderClasses * W; e += 64 * W) table[e] = 0;
  __syncthreads();
  int lo = 0x7fffffff, hi = 0;
  walk([&](int, int c, int slot, int before, int all) {
    lo = c < lo ? c : lo;
    hi = c > hi ? c : hi;
    if (before == 0) table[slot] += all;
  });
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const int l = __shfl_xor(lo, off, 64), h = __shfl_xor(hi, off, 64);
    lo = l < lo ? l : lo;
    hi = h > hi ? h : hi;
  }
  if (lane == 0) {
    lo_l[wave] = lo;
    hi_l[wave] = hi;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < W; ++w) {
    lo = lo_l[w] < lo ? lo_l[w] : lo;
    hi = hi_l[w] > hi ? hi_l[w] : hi;
  }
  // the longest list less than twice the shortest: little to balance (measured: sorting such
  // lists costs 2 % through the lost locality), keep neighbours together
  if (hi <= 0 || hi < 2 * lo) {
    for (int s = 0; s < steps; ++s)
      if (i0 + 64 * s < n) order[i0 + 64 * s] = xcd_remap(i0 + 64 * s, n);
    return;
  }
  // exclusive prefix sum over the table in storage order; a thread of the first two waves has a class
  int own = 0, upto = 0;
  if (tid < 128) {
    if (tid < kOrderClasses)
#pragma unroll
      for (int w = 0; w < W; ++w) own += table[tid * W + w];
    upto = own;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int t = __shfl_up(upto, off, 64);
      if (lane >= off) upto += t;
    }
    if (tid == 63) first_half = upto;
  }
  __syncthreads();
  if (tid < kOrderClasses) {
    int run = upto - own + (wave == 1 ? first_half : 0);
#pragma unroll
    for (int w = 0; w < W; ++w) {
      const int x = table[tid * W + w];
      table[tid * W + w] = run;
      run += x;
    }
  }
  __syncthreads();
  walk([&](int i, int, int slot, int before, int all) {
    const int at = table[slot];
    order[at + before] = i;
    if (before == all - 1) table[slot] = at + all;
  });
}

// ------------------------------------------------------------------------------------
// The same purpose with an eye on L2.  Sorted over all heads, the q-blocks that an XCD works on at a time come
// from every head, and the key rows they gather share nothing: the sort costs more than the balance gives.
// Workgroups go to the XCDs round robin, so position 8 k + x of an order is the k-th workgroup of XCD x.  Every
// XCD keeps its contiguous share of the q-blocks, in index order by windows of whole heads (at least kWindow
// q-blocks), and inside a window the longest lists go first: one head at a time stays in its L2, lists of like
// length walk the keys in step, and the last window still ends balanced.  Attention in ms, sorted over
// everything / in index order / this: threshold lists 12 x 32760 x 128 0.582 / 0.575 / 0.559, 40 heads 2.00 /
// 1.93 / 1.87, 24 x 32760 x 64 0.696 / 0.685 / 0.671; Zipf lists 32 x 16384 x 128 0.661 / 0.585 / 0.502,
// 32 x 4096 x 128 0.101 / 0.081 / 0.074; 8 x 65536 x 128 5.4 in index order, 4.3 in both others.
// Two exceptions, decided on the counts: where the longest list is more than kTail of the work of one of an
// XCD's 64 workgroup slots, a late window would end with it alone, and the share is one window (Zipf lists
// 24 x 20000 x 64, 0.5 of a slot's work: 0.389 instead of 0.417 ms); and where the shares differ by more than
// kSkew, the sort over everything balances the XCDs (shares within 1.09 of each other still gain by the windows).
// That is also so where no list is twice as long as another: block lists 32 x 16384 x 128, head densities rising by
// 1.8 / 1.4: windows and index order 0.981 / 0.780, sorted 0.846 / 0.731 ms; threshold lists 12 x 32760 x 128, largest
// share 1.28 of the mean: 0.318 and 0.286.  From kCoarse q-blocks on the sort takes quarters of an octave, which keep
// more neighbours together: 40 x 32760 x 128 1.018 -> 0.984 ms, 40 x 75600 x 128 5.12 -> 4.88; up to 7092 q-blocks no
// difference.
// One workgroup per XCD, a wave per window, the sort over everything by one workgroup; classes of an eighth of an
// octave (a sixteenth: no gain) over the seven octaves below the longest list, stable, so the order is a function of
// the counts alone.  What bounds it is the chain of loads and LDS updates of a lane's segment: 6.6 us for 6144
// q-blocks by windows, 16 for 23640, and 15.5 / 42 us for the sort over everything (one wave of one count at a time:
// 47 / 171; qblock_order_kernel: 9 / 32).
// ------------------------------------------------------------------------------------
constexpr int kXcds = 8;
constexpr int kSlotsPerXcd = 64;
constexpr int kWindow = 192;
constexpr float kTail = 0.3f;
constexpr float kSkew = 1.1f;
constexpr int kCoarse = 8192;
constexpr int kSchedSub = 3;
constexpr int kSchedOctaves = 7;
constexpr int kSchedClasses = (kSchedOctaves << kSchedSub) + 4;   // a multiple of 4: a lane reads its table entries 16 bytes at a time

// 0 holds the longest lists; top: floor(log2) of the longest of all; coarse: 1 for quarters of an octave
__device__ __forceinline__ int schedule_class(int c, int top, int coarse) {
  if (c <= 0) return kSchedClasses - 1;
  const int lg = 31 - __builtin_clz((unsigned)c);
  const int below = lg >= kSchedSub ? ((c >> (lg - kSchedSub)) & ((1 << kSchedSub) - 1))
                                    : ((c << (kSchedSub - lg)) & ((1 << kSchedSub) - 1));
  const int cls = ((top - lg) << kSchedSub) + ((1 << kSchedSub) - 1 - below);
  return cls < kSchedClasses - 2 ? cls >> coarse : kSchedClasses - 2;
}

__global__ __launch_bounds__(256) void qblock_schedule_kernel(int* __restrict__ order, const int* __restrict__ counts, int n,
                                                              int per_head) {
  __shared__ __attribute__((aligned(16))) int tables[4][kSchedClasses * 64];   // [wave][class][lane], or all of it [class][thread]
  __shared__ float share_l[kXcds];
  __shared__ int longest_l[4], wave_sum[4];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = blockIdx.x;
  const int per = n / kXcds;

  // the work of every XCD's share and the longest list; a wave takes two shares
  {
    int longest = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int y = 2 * wave + h;
      float sum = 0.f;
      for (int i = y * per + lane; i < (y + 1) * per; i += 512) {
        int c[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) c[u] = i + 64 * u < (y + 1) * per ? counts[i + 64 * u] : 0;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          sum += (float)c[u];
          longest = c[u] > longest ? c[u] : longest;
        }
      }
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
      if (lane == 0) share_l[y] = sum;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int o = __shfl_xor(longest, off, 64);
      longest = o > longest ? o : longest;
    }
    if (lane == 0) longest_l[wave] = longest;
  }
  __syncthreads();
  float total = 0.f, most = 0.f;
#pragma unroll
  for (int y = 0; y < kXcds; ++y) {
    total += share_l[y];
    most = share_l[y] > most ? share_l[y] : most;
  }
  int longest = longest_l[0];
#pragma unroll
  for (int w = 1; w < 4; ++w) longest = longest_l[w] > longest ? longest_l[w] : longest;
  // the sort over everything also classes the up to seven q-blocks behind the shares
  int longest_all = longest;
  for (int i = kXcds * per; i < n; ++i) longest_all = counts[i] > longest_all ? counts[i] : longest_all;
  const int top = 31 - __builtin_clz((unsigned)(longest_all > 0 ? longest_all : 1));
  const bool global = most * kXcds > kSkew * total;
  const int coarse = global && n >= kCoarse ? 1 : 0;
  const bool one_window = (float)longest * kSlotsPerXcd > kTail * share_l[x];

  // Stable counting sort of q-blocks a .. b-1 by class, by one wave or (ALL) by the workgroup; the entry of rank r
  // goes to order[first + r * step].  A lane owns a contiguous segment and has eight of its counts in flight.  A
  // wave's LDS operations execute in order.
  auto sort = [&](auto all, int a, int b, int first, int step) {
    constexpr bool ALL = decltype(all)::value;
    constexpr int L = ALL ? 256 : 64, U = 8;
    const int id = ALL ? (int)threadIdx.x : lane;
    int* const table = tables[ALL ? 0 : wave];
    auto settle = [] {
      if constexpr (ALL) {
        __syncthreads();
      } else {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
    };
    for (int i = 4 * id; i < kSchedClasses * L; i += 4 * L) {
      const i32x4 z = {0, 0, 0, 0};
      *reinterpret_cast<i32x4*>(table + i) = z;
    }
    const int seg = (b - a + L - 1) / L;
    const int i0 = a + id * seg < b ? a + id * seg : b;
    const int i1 = i0 + seg < b ? i0 + seg : b;
    auto walk = [&](auto&& f) {
      for (int i = i0; i < i1; i += U) {
        int c[U];
#pragma unroll
        for (int u = 0; u < U; ++u) c[u] = i + u < i1 ? counts[i + u] : 0;
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (i + u < i1) f(i + u, schedule_class(c[u], top, coarse) * L + id);
      }
    };
    settle();
    walk([&](int, int slot) { table[slot] += 1; });
    settle();
    // exclusive prefix sum in storage order (class-major, lane-minor): lane l scans kSchedClasses entries from
    // l * kSchedClasses on
    int sum = 0;
    i32x4* const own = reinterpret_cast<i32x4*>(table + id * kSchedClasses);
#pragma unroll
    for (int j = 0; j < kSchedClasses / 4; ++j) {
      const i32x4 v = own[j];
      sum += v[0] + v[1] + v[2] + v[3];
    }
    int run = (int)lane_scan((uint32_t)sum) - sum;
    if constexpr (ALL) {
      if (lane == 63) wave_sum[wave] = run + sum;
      __syncthreads();
#pragma unroll
      for (int w = 0; w < 3; ++w) run += w < wave ? wave_sum[w] : 0;
    }
#pragma unroll
    for (int j = 0; j < kSchedClasses / 4; ++j) {
      const i32x4 v = own[j];
      i32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        o[e] = run;
        run += v[e];
      }
      own[j] = o;
    }
    settle();
    walk([&](int i, int slot) {
      const int r = table[slot];
      order[(size_t)first + (size_t)r * step] = i;
      table[slot] = r + 1;
    });
    settle();
  };

  if (global) {
    if (x == 0) sort(std::true_type{}, 0, n, 0, 1);
    return;
  }
  const int end = (x + 1) * per;
  int turn = 0;
  for (int a = x * per; a < end; ++turn) {
    int b = end;
    if (!one_window) {
      b = (a / per_head + 1) * per_head;
      if (b - a < kWindow) b += (kWindow - (b - a) + per_head - 1) / per_head * per_head;
      b = b < end ? b : end;
    }
    if ((turn & 3) == wave) sort(std::false_type{}, a, b, (a - x * per) * kXcds + x, kXcds);
    a = b;
  }
  if (x == 0)
    for (int i = per * kXcds + (int)threadIdx.x; i < n; i += 256) order[i] = i;
}

hipError_t run_qblock_schedule(int* order, const int* counts, int n, int per_head, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(qblock_schedule_kernel, dim3(kXcds), dim3(256), 0, stream, order, counts, n, per_head);
  return hipGetLastError();
}

hipError_t run_qblock_order(int* order, const int* counts, int n, hipStream_t stream) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(qblock_order_kernel, dim3(1), dim3(64 * kOrderWaves), 0, stream, order, counts, n);
  return hipGetLastError();
}

}  // namespace spattn
