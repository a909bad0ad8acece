// Device side of ingestion: the diff of aligned sequences against the reference
// (extractCoverageAndMutationsFromSequence, common/aligned_sequence.cpp:18-122), the per-position
// coverage and symbol counts and the local-reference rule of SequenceColumn::finalize
// (sequence_column.cpp:157-212, vertical_sequence_index.cpp:86-95), and the (chunk, position,
// symbol, row) entries of the vertical index's containers (VerticalSequenceIndex::
// addSymbolsToPositions, vertical_sequence_index.cpp:16-38), radix-sorted.
#include <hip/hip_runtime.h>

#include <hipcub/hipcub.hpp>

#include "kernels.h"

namespace rdb {

namespace {

constexpr uint32_t kDiffWaves = 4;  // rows (one per wavefront) per work-group

__device__ inline uint32_t firstBit(uint64_t m) { return static_cast<uint32_t>(__ffsll(static_cast<long long>(m)) - 1); }

// Bits of the bytes of `x` that are not zero, one per byte.
__device__ inline uint32_t nonzeroBytes(uint32_t x) {
   const uint32_t high = (((x & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | x) & 0x80808080u;
   return (high * 0x00204081u) >> 28;  // bits 7, 15, 23 and 31 side by side; no other product reaches them
}
__device__ inline uint32_t nonzeroBytes(const uint4& x) {
   return nonzeroBytes(x.x) | nonzeroBytes(x.y) << 4 | nonzeroBytes(x.z) << 8 | nonzeroBytes(x.w) << 12;
}
__device__ inline uint32_t byteOf(const uint4& v, uint32_t k) {
   const uint32_t lo = k & 4 ? v.y : v.x, hi = k & 4 ? v.w : v.z;
   return ((k & 8 ? hi : lo) >> (8 * (k & 3))) & 0xFFu;
}
// Bits [lo, hi) of 16; bounds outside them are clipped.
__device__ inline uint32_t bits16(int32_t lo, int32_t hi) {
   const uint32_t a = static_cast<uint32_t>(min(max(lo, 0), 16)), b = static_cast<uint32_t>(min(max(hi, 0), 16));
   return ((1u << b) - 1u) & ~((1u << a) - 1u);
}
__device__ inline uint32_t waveAdd(uint32_t v) {
   for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
   return v;
}
// Sum of v over the lanes below this one; `total` becomes the wavefront's.  Few lanes hold any.
__device__ inline uint32_t lanesBelow(uint32_t v, uint32_t lane, uint32_t& total) {
   uint32_t before = 0;
   total = 0;
   for (uint64_t some = __ballot(v != 0); some; some &= some - 1) {
      const uint32_t src = firstBit(some);
      const uint32_t n = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), static_cast<int>(src)));
      before += lane > src ? n : 0u;
      total += n;
   }
   return before;
}

// One wavefront per row, 1,024 characters a step: each lane compares 16 (one aligned load) with the
// reference's own characters and with the missing character, byte-wise in 32-bit words, and looks up
// only the bytes that match neither, through the character table.  A row differs from the reference in
// few places, so a step is two loads and some 60 operations a lane; the count pass is bound by reading
// the text.  (A character a lane and step, each through the table: 523 us for 8,192 rows of 29,903 and
// 457 us for the write pass; now 75 and 82, of which reading the text at 5.5 TB/s takes 45.)  `j` counts characters of the row, its position is
// offset + j.  Pass 1 (kWrite false) records the covered range, the number of mutations and internal
// missing runs and the first illegal character; pass 2 writes mutations and runs at the row's offsets.
constexpr uint32_t kDiffStep = 64 * 16;
template <bool kWrite>
__global__ __launch_bounds__(64 * kDiffWaves) void diffKernel(DiffBatch d) {
   __shared__ uint8_t lut[256];
   for (uint32_t t = threadIdx.x; t < 256; t += blockDim.x) lut[t] = d.lut[t];
   __syncthreads();
   const uint32_t lane = threadIdx.x & 63;
   const uint32_t r = blockIdx.x * kDiffWaves + (threadIdx.x >> 6);
   if (r >= d.n_rows) return;
   const uint32_t len = static_cast<uint32_t>(d.row_ptr[r + 1] - d.row_ptr[r]);
   const uint32_t row_start = kWrite ? d.start[r] : 0, row_end = kWrite ? d.end[r] : 0;
   if (d.is_null[r] || (kWrite && row_start >= row_end)) {
      if (!kWrite && lane == 0) {
         d.start[r] = 0;
         d.end[r] = 0;
         d.n_mut[r] = 0;
         d.n_run[r] = 0;
         d.err[r] = 0xFFFFFFFFu;
      }
      return;
   }
   const uint32_t off = d.offsets ? d.offsets[r] : 0;
   // lane k's first 16 characters start at the k-th aligned 16 bytes from the row's first character on
   const char* s = d.data + d.row_ptr[r];
   const int32_t skew = static_cast<int32_t>(reinterpret_cast<uintptr_t>(s) & 15);
   const uint32_t miss_word = d.missing_char * 0x01010101u;
   uint64_t mut_w = kWrite ? d.mut_off[r] : 0, run_sw = kWrite ? d.run_off[r] : 0, run_ew = run_sw;
   uint32_t first = 0xFFFFFFFFu, last = 0, n_mut = 0, n_starts = 0, err = 0xFFFFFFFFu;
   uint32_t carry = 0;  // the character before the step's first is missing
   const int32_t n = static_cast<int32_t>(len);
   uint4 next_t, next_c;
   const auto load = [&](int32_t j) {  // (aligned blocks that hold a character of the row, and the reference's there)
      if (j < n) {
         next_t = *reinterpret_cast<const uint4*>(s + j);
         __builtin_memcpy(&next_c, d.ref_text + (static_cast<int32_t>(off) + j), 16);
      }
   };
   next_t = next_c = make_uint4(0, 0, 0, 0);
   load(static_cast<int32_t>(lane * 16) - skew);
   for (int32_t base = -skew; base < n; base += static_cast<int32_t>(kDiffStep)) {
      const int32_t j = base + static_cast<int32_t>(lane * 16);
      const uint4 t = next_t, c = next_c;
      load(j + static_cast<int32_t>(kDiffStep));
      const uint32_t valid = bits16(-j, n - j);
      uint32_t miss = valid & ~nonzeroBytes(make_uint4(t.x ^ miss_word, t.y ^ miss_word, t.z ^ miss_word, t.w ^ miss_word));
      const uint32_t other = valid & ~miss & nonzeroBytes(make_uint4(t.x ^ c.x, t.y ^ c.y, t.z ^ c.z, t.w ^ c.w));
      uint32_t mut = 0, illegal = 0;
      for (uint32_t rest = other; rest; rest &= rest - 1) {
         const uint32_t k = firstBit(rest);
         const uint32_t sym = lut[byteOf(t, k)];
         const uint32_t bit = 1u << k;
         if (sym == 0xFFu) {
            illegal |= bit;
         } else if (sym == d.missing) {
            miss |= bit;
         } else if (sym != lut[byteOf(c, k)]) {
            mut |= bit;
         }
      }
      const uint32_t prev = __shfl_up(miss >> 15, 1, 64);
      const uint32_t before = miss << 1 | (lane == 0 ? carry : prev);  // bit k: character k - 1 is missing
      carry = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(miss >> 15), 63));
      const uint32_t starts = miss & ~before;
      const uint32_t nonmiss = valid & ~miss & ~illegal;
      if constexpr (!kWrite) {
         n_mut += static_cast<uint32_t>(__popc(mut));
         n_starts += static_cast<uint32_t>(__popc(starts));
         if (nonmiss) {
            first = min(first, static_cast<uint32_t>(j + __ffs(static_cast<int>(nonmiss)) - 1));
            last = static_cast<uint32_t>(j + 32 - __clz(static_cast<int>(nonmiss)));
         }
         if (illegal) err = min(err, off + static_cast<uint32_t>(j + __ffs(static_cast<int>(illegal)) - 1));
      } else {
         const uint32_t p = static_cast<uint32_t>(static_cast<int32_t>(off) + j);
         uint32_t total;
         if (__ballot(mut != 0)) {
            uint64_t o = mut_w + lanesBelow(static_cast<uint32_t>(__popc(mut)), lane, total);
            mut_w += total;
            for (uint32_t rest = mut; rest; rest &= rest - 1, ++o) {
               const uint32_t k = firstBit(rest);
               d.mut_pos[o] = p + k;
               d.mut_sym[o] = lut[byteOf(t, k)];
            }
         }
         // internal runs: starts, and ends (the first non-missing character after a run), strictly
         // inside the covered range
         const int32_t p0 = static_cast<int32_t>(p);
         const uint32_t inside = bits16(static_cast<int32_t>(row_start) + 1 - p0, static_cast<int32_t>(row_end) - p0);
         const uint32_t is = starts & inside, ie = nonmiss & before & inside;
         if (__ballot((is | ie) != 0)) {
            uint64_t o = run_sw + lanesBelow(static_cast<uint32_t>(__popc(is)), lane, total);
            run_sw += total;
            for (uint32_t rest = is; rest; rest &= rest - 1) d.run_start[o++] = p + firstBit(rest);
            o = run_ew + lanesBelow(static_cast<uint32_t>(__popc(ie)), lane, total);
            run_ew += total;
            for (uint32_t rest = ie; rest; rest &= rest - 1) d.run_end[o++] = p + firstBit(rest);
         }
      }
   }
   if constexpr (!kWrite) {
      n_mut = waveAdd(n_mut);
      n_starts = waveAdd(n_starts);
      for (int o = 32; o > 0; o >>= 1) {
         first = min(first, static_cast<uint32_t>(__shfl_xor(first, o, 64)));
         last = max(last, static_cast<uint32_t>(__shfl_xor(last, o, 64)));
         err = min(err, static_cast<uint32_t>(__shfl_xor(err, o, 64)));
      }
      if (lane == 0) {
         d.err[r] = err;
         if (first == 0xFFFFFFFFu) {  // nothing covered
            d.start[r] = 0;
            d.end[r] = 0;
            d.n_mut[r] = 0;
            d.n_run[r] = 0;
         } else {
            d.start[r] = off + first;
            d.end[r] = off + last;
            d.n_mut[r] = n_mut;
            d.n_run[r] = n_starts - (first > 0 ? 1u : 0u) - (last < len ? 1u : 0u);
         }
      }
   }
}

// Row i's adaptation keys (see AdaptCount) at mut_ptr[i] + 2 nrun_ptr[i] + 2 i.
__global__ void adaptKeysKernel(AdaptCount a) {
   const DiffRowsDev& R = a.rows;
   const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
   if (i >= R.n_rows) return;
   const uint32_t past = (R.length + 1) << 5;  // sorts after every real key
   uint32_t* k = a.keys + R.mut_ptr[i] + 2 * R.nrun_ptr[i] + 2 * i;
   const bool live = !R.is_null[i];
   const uint32_t s = R.cov_start[i], e = R.cov_end[i];
   const bool cov = live && s < e;
   k[0] = cov ? (s << 5 | kAdaptCodeUp) : past;
   k[1] = cov ? (e << 5 | kAdaptCodeDown) : past;
   k += 2;
   // a null row counts nothing: whatever it lists fills its keys with `past`
   for (uint64_t r = R.nrun_ptr[i]; r < R.nrun_ptr[i + 1]; ++r) {
      *k++ = live ? (R.runs[r] & 0xFFFFu) << 5 | kAdaptCodeDown : past;
      *k++ = live ? (R.runs[r] >> 16) << 5 | kAdaptCodeUp : past;
   }
   for (uint64_t m = R.mut_ptr[i]; m < R.mut_ptr[i + 1]; ++m) *k++ = live ? R.mut_pos[m] << 5 | R.mut_sym[m] : past;
}

// Boundaries of the runs of equal sorted keys: run_start[key] and run_end[key] (count = end - start).
__global__ void adaptRunsKernel(const uint32_t* __restrict__ keys, uint64_t n, uint32_t past, uint32_t* run_start,
                                uint32_t* run_end) {
   const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
   if (i >= n) return;
   const uint32_t k = keys[i];
   if (k >= past) return;
   if (i == 0 || keys[i - 1] != k) run_start[k] = static_cast<uint32_t>(i);
   if (i + 1 == n || keys[i + 1] != k) run_end[k] = static_cast<uint32_t>(i + 1);
}

__device__ inline uint32_t adaptCount(const AdaptCount& a, uint32_t key) { return a.run_end[key] - a.run_start[key]; }

// The adapted local reference, in two kernels over blocks of kRulePositions positions; half a wavefront
// takes a position, a lane per code, so that a position's 32 counts are one line of each array.  The first
// leaves each position's change of coverage and each block's sum of them.  The second adds up the blocks
// before its own and its positions' changes to the coverage; then the reference symbol's count is the
// coverage minus the other symbols' counts, and the local reference is the reference symbol unless
// another symbol's count is strictly larger (the first such symbol with the largest count).  (One
// work-group over all positions, a thread per 30 of them: 1,061 us at 29,903; now 15
// in both.)
constexpr uint32_t kRuleThreads = 256;
constexpr uint32_t kRulePositions = 64;
constexpr uint32_t kRuleAtOnce = kRuleThreads / 32;
static_assert(kAdaptCodeDown < 32, "a lane per code");

__global__ __launch_bounds__(kRuleThreads) void adaptChangesKernel(AdaptCount a) {
   __shared__ int32_t change[kRulePositions];
   const uint32_t L = a.rows.length;
   const uint32_t p0 = blockIdx.x * kRulePositions;
   for (uint32_t k = threadIdx.x / 32; k < kRulePositions; k += kRuleAtOnce) {
      const uint32_t p = p0 + k, code = threadIdx.x & 31;
      const bool event = p < L && (code == kAdaptCodeUp || code == kAdaptCodeDown);
      const int32_t n = event ? static_cast<int32_t>(adaptCount(a, p << 5 | code)) : 0;
      const int32_t up = __shfl(n, kAdaptCodeUp, 32), down = __shfl(n, kAdaptCodeDown, 32);
      if (code == 0) {
         change[k] = up - down;
         if (p < L) a.changes[p] = up - down;
      }
   }
   __syncthreads();
   if (threadIdx.x < 64) {
      int32_t sum = change[threadIdx.x];
      for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
      if (threadIdx.x == 0) a.block_changes[blockIdx.x] = sum;
   }
}

__global__ __launch_bounds__(kRuleThreads) void adaptRuleKernel(AdaptCount a) {
   static_assert(kRulePositions == 64, "a wavefront scans a block's changes");
   __shared__ int32_t part[kRuleThreads / 64];
   __shared__ uint32_t coverage[kRulePositions];
   const DiffRowsDev& R = a.rows;
   const uint32_t L = R.length, nsym = R.n_symbols;
   const uint32_t p0 = blockIdx.x * kRulePositions;
   int32_t sum = 0;
   for (uint32_t b = threadIdx.x; b < blockIdx.x; b += kRuleThreads) sum += a.block_changes[b];
   for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
   if ((threadIdx.x & 63) == 0) part[threadIdx.x / 64] = sum;
   __syncthreads();
   if (threadIdx.x < 64) {
      int32_t at = p0 + threadIdx.x < L ? a.changes[p0 + threadIdx.x] : 0;
      for (uint32_t o = 1; o < 64; o <<= 1) {
         const int32_t v = __shfl_up(at, o, 64);
         if (threadIdx.x >= o) at += v;
      }
      for (uint32_t w = 0; w < kRuleThreads / 64; ++w) at += part[w];
      coverage[threadIdx.x] = static_cast<uint32_t>(at);
      if (p0 + threadIdx.x < L) a.coverage[p0 + threadIdx.x] = static_cast<uint32_t>(at);
   }
   __syncthreads();
   for (uint32_t k = threadIdx.x / 32; k < kRulePositions; k += kRuleAtOnce) {
      const uint32_t p = p0 + k, s = threadIdx.x & 31;
      if (p >= L) continue;  // (the same in all lanes that shuffle with each other)
      const uint32_t current = R.reference[p];
      const bool other = s < nsym && s != current;
      const uint32_t n = other ? adaptCount(a, p << 5 | s) : 0u;
      uint32_t others = n;
      for (int o = 16; o > 0; o >>= 1) others += __shfl_xor(others, o, 32);
      const uint32_t ref_count = coverage[k] - others;
      // the larger count wins, and among equal ones the smaller symbol
      uint32_t best_count = n, best = s;
      for (int o = 16; o > 0; o >>= 1) {
         const uint32_t c2 = __shfl_xor(best_count, o, 32), s2 = __shfl_xor(best, o, 32);
         if (c2 > best_count || (c2 == best_count && s2 < best)) {
            best_count = c2;
            best = s2;
         }
      }
      if (s == 0) a.local_ref[p] = static_cast<uint8_t>(best_count > ref_count ? best : current);
   }
}

// The container entries of one row: its mutations except those to a flipped position's local
// reference symbol; the reference symbol at each flipped position it covers with neither a mutation
// nor a missing run there; and the boundary pseudo-symbols of its covered range and runs (a null
// row, or one that covers nothing: uncovered from position 0).
template <bool kWrite>
__global__ void entriesKernel(EntryBatch e) {
   const DiffRowsDev& R = e.rows;
   const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
   if (i >= R.n_rows) return;
   uint32_t lo = 0, hi = e.n_chunks;  // the chunk c with chunk_offset[c] <= i < chunk_offset[c + 1]
   while (hi - lo > 1) {
      const uint32_t mid = (lo + hi) / 2;
      if (e.chunk_offset[mid] <= i) {
         lo = mid;
      } else {
         hi = mid;
      }
   }
   const uint64_t key_hi = (static_cast<uint64_t>(lo) << 40) | (i - e.chunk_offset[lo]);
   const uint32_t L = R.length, nsym = R.n_symbols;
   const uint64_t w = kWrite ? e.offsets[i] : 0;
   uint32_t n = 0;
   auto push = [&](uint32_t p, uint32_t sym) {
      if constexpr (kWrite) e.keys[w + n] = key_hi | (static_cast<uint64_t>(p) << 24) | (static_cast<uint64_t>(sym) << 16);
      ++n;
   };
   if (R.is_null[i]) {
      push(0, nsym + BND_COV_END);
   } else {
      const bool has_cov = R.cov_start[i] < R.cov_end[i];
      const uint32_t s0 = has_cov ? R.cov_start[i] : 0, e0 = has_cov ? R.cov_end[i] : 0;
      const uint64_t m0 = R.mut_ptr[i], m1 = R.mut_ptr[i + 1];
      const uint64_t r0 = R.nrun_ptr[i], r1 = R.nrun_ptr[i + 1];
      for (uint64_t k = m0; k < m1; ++k) {
         const uint32_t p = R.mut_pos[k];
         if (e.flip_to[p] != 0xFF && R.mut_sym[k] == e.flip_to[p]) continue;
         push(p, R.mut_sym[k]);
      }
      uint64_t mk = m0, rk = r0;  // merge walk: flipped positions, mutations and runs all ascend
      for (uint32_t f = 0; f < e.n_flipped; ++f) {
         const uint32_t p = e.flipped[f];
         if (p < s0) continue;
         if (p >= e0) break;
         while (mk < m1 && R.mut_pos[mk] < p) ++mk;
         while (rk < r1 && (R.runs[rk] >> 16) <= p) ++rk;
         if (mk < m1 && R.mut_pos[mk] == p) continue;
         if (rk < r1 && (R.runs[rk] & 0xFFFFu) <= p) continue;
         push(p, R.reference[p]);
      }
      if (s0 > 0) push(s0, nsym + BND_COV_START);
      if (e0 < L) push(e0, nsym + BND_COV_END);
      for (uint64_t k = r0; k < r1; ++k) {
         push(R.runs[k] & 0xFFFFu, nsym + BND_N_START);
         if ((R.runs[k] >> 16) < L) push(R.runs[k] >> 16, nsym + BND_N_END);
      }
   }
   if constexpr (!kWrite) e.counts[i] = n;
}

}  // namespace

hipError_t launchDiff(const DiffBatch& d, bool write, hipStream_t stream) {
   if (d.n_rows == 0) return hipSuccess;
   const dim3 grid((d.n_rows + kDiffWaves - 1) / kDiffWaves);
   if (write) {
      hipLaunchKernelGGL(diffKernel<true>, grid, dim3(64 * kDiffWaves), 0, stream, d);
   } else {
      hipLaunchKernelGGL(diffKernel<false>, grid, dim3(64 * kDiffWaves), 0, stream, d);
   }
   return hipGetLastError();
}

hipError_t launchAdapt(const AdaptCount& a, void* temp, size_t* temp_bytes, hipStream_t stream) {
   const uint32_t past = (a.rows.length + 1) << 5;
   int end_bit = 1;
   while ((1u << end_bit) <= past) ++end_bit;
   hipcub::DoubleBuffer<uint32_t> buf(a.keys, a.keys_alt);
   if (temp == nullptr) {
      return hipcub::DeviceRadixSort::SortKeys(nullptr, *temp_bytes, buf, static_cast<int>(a.key_count), 0, end_bit,
                                               stream);
   }
   hipError_t err = hipSuccess;
   if (a.rows.n_rows > 0) {
      hipLaunchKernelGGL(adaptKeysKernel, dim3(static_cast<uint32_t>((a.rows.n_rows + 255) / 256)), dim3(256), 0, stream, a);
      if ((err = hipGetLastError()) != hipSuccess) return err;
   }
   if (a.key_count > 0) {
      err = hipcub::DeviceRadixSort::SortKeys(temp, *temp_bytes, buf, static_cast<int>(a.key_count), 0, end_bit, stream);
      if (err != hipSuccess) return err;
      hipLaunchKernelGGL(adaptRunsKernel, dim3(static_cast<uint32_t>((a.key_count + 255) / 256)), dim3(256), 0, stream,
                         buf.Current(), a.key_count, past, a.run_start, a.run_end);
      if ((err = hipGetLastError()) != hipSuccess) return err;
   }
   const uint32_t blocks = (a.rows.length + kRulePositions - 1) / kRulePositions;
   hipLaunchKernelGGL(adaptChangesKernel, dim3(blocks), dim3(kRuleThreads), 0, stream, a);
   if ((err = hipGetLastError()) != hipSuccess) return err;
   hipLaunchKernelGGL(adaptRuleKernel, dim3(blocks), dim3(kRuleThreads), 0, stream, a);
   return hipGetLastError();
}

hipError_t launchEntries(const EntryBatch& e, bool write, hipStream_t stream) {
   if (e.rows.n_rows == 0) return hipSuccess;
   const dim3 grid(static_cast<uint32_t>((e.rows.n_rows + 255) / 256));
   if (write) {
      hipLaunchKernelGGL(entriesKernel<true>, grid, dim3(256), 0, stream, e);
   } else {
      hipLaunchKernelGGL(entriesKernel<false>, grid, dim3(256), 0, stream, e);
   }
   return hipGetLastError();
}

hipError_t scanEntryCounts(const uint32_t* counts, uint64_t* offsets, uint64_t n, void* temp, size_t* temp_bytes,
                           hipStream_t stream) {
   return hipcub::DeviceScan::ExclusiveScan(temp, *temp_bytes, counts, offsets, hipcub::Sum(), uint64_t{0},
                                            static_cast<int>(n), stream);
}

hipError_t sortEntryKeys(uint64_t* keys, uint64_t* keys_alt, uint64_t n, void* temp, size_t* temp_bytes,
                         hipStream_t stream, uint64_t** sorted) {
   hipcub::DoubleBuffer<uint64_t> buf(keys, keys_alt);
   const hipError_t err = hipcub::DeviceRadixSort::SortKeys(temp, *temp_bytes, buf, static_cast<int>(n), 0, 56, stream);
   if (sorted) *sorted = buf.Current();
   return err;
}

}  // namespace rdb
