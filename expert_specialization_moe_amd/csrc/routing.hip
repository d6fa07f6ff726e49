// Routing metadata on the device: top-k expert ids -> the per-expert tensors the grouped operators
// consume, plus the row permutation that packs token rows expert by expert.
//
// The reference builds these on the host with torch/Python in its tests and benchmark
// (counts -> expert_offsets prefix sum: benchmark/benchmark_es_fp8_blockwise_moe.py:44-56,72-88;
// blockscale_offsets = prefix sum of the counts rounded up to 128:
// test/test_es_sm100_mxfp8_blockscaled_grouped_quant.py:42-60).  Here the same integers come out of
// one or two small kernels, so a caller never synchronises with the host between routing and the GEMMs.
//
//   pair p = (token p / topk, choice p % topk), id = topk_ids[p] - first_expert; local if 0 <= id < E
//   counts[e]             = number of local pairs with id == e
//   expert_offsets[e]     = sum of counts[0..e)            (E + 1 entries, the last is the total)
//   blockscale_offsets[e] = sum of align128(counts[0..e))  (E + 1 entries)
//   problem_sizes[e]      = (counts[e], n, k)
//   dst_row[p]            = expert_offsets[id] + (number of local pairs q < p with the same id), or -1
// The rank is by pair index, so the permutation is stable and the result is deterministic.
//
// Pairs are cut into chunks, one workgroup of 16 wavefronts each, a pair per thread (of a chunk longer than 1024 pairs:
// of each 1024 in turn).  A workgroup needs, beside its own pairs, every expert's count over all pairs and over the
// pairs in front of its chunk.  It forms both itself, from the ids (up to kDirectPairs pairs: ONE launch) or from the
// chunks' counts that a first launch wrote: nothing waits for another workgroup, and every workgroup knows the offsets.
// dst_row may be the ids' own buffer.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "permute_rule.h"
#include "wave_scan.h"

namespace esmoe {

constexpr int kRouteThreads = 1024, kRouteWaves = kRouteThreads / 64;
constexpr int kMaxRouteExperts = 1024;   // a thread per expert
constexpr int kMaxChunks = 256;
// Pairs up to which every workgroup counts all ids itself, a pass of LDS atomics over all of them, where the counts cost a
// launch and a pass over [chunks, experts] words.  128 experts, direct against counts: 8192 pairs
// 5.2 / 6.0 us, 16384 pairs 7.1 / 6.1 us, 32768 pairs 11.4 / 6.3 us.
constexpr long kDirectPairs = 8192;

// Lanes of the wavefront that hold the same id as this lane: one ballot per bit of the id instead of one round per
// distinct id (64 pairs over 32 experts are ~25 distinct ids, and a round costs as much as all the ballots together).
// `bits` covers num_experts - 1; lanes with id < 0 get a meaningless mask.
__device__ __forceinline__ unsigned long long lanes_with_same_id(int id, int bits) {
  unsigned long long same = __ballot(id >= 0);
  for (int b = 0; b < bits; b++) {
    const bool bit = (id >> b) & 1;
    const unsigned long long m = __ballot(bit);
    same &= bit ? m : ~m;
  }
  return same;
}
__device__ __forceinline__ int id_bits(int num_experts) { return num_experts > 1 ? 32 - __builtin_clz(num_experts - 1) : 0; }

// Local expert of pair p, or -1 (another rank's expert, or past the last pair).
__device__ __forceinline__ int local_id(int raw, long p, long num_pairs, int first_expert, int num_experts) {
  const unsigned id = (unsigned)raw - (unsigned)first_expert;
  return p < num_pairs && id < (unsigned)num_experts ? (int)id : -1;
}

// Pairs per chunk: 1024, or as many times 1024 as keep the chunks at most kMaxChunks.
__host__ __device__ inline long route_chunk_pairs(long num_pairs) {
  const long per = (num_pairs + kMaxChunks - 1) / kMaxChunks;
  return per <= kRouteThreads ? kRouteThreads : (per + kRouteThreads - 1) / kRouteThreads * kRouteThreads;
}

__global__ void __launch_bounds__(kRouteThreads) route_count_kernel(const int* __restrict__ ids, long num_pairs, int first_expert,
                                                                    int num_experts, long chunk, int* __restrict__ chunk_counts) {
  __shared__ int s_cnt[kMaxRouteExperts];
  const int tid = threadIdx.x;
  s_cnt[tid] = 0;
  __syncthreads();
  const long base = (long)blockIdx.x * chunk;
  for (long off = 0; off < chunk; off += kRouteThreads) {
    const long p = base + off + tid;
    const int id = local_id(p < num_pairs ? ids[p] : 0, p, num_pairs, first_expert, num_experts);
    if (id >= 0) atomicAdd(&s_cnt[id], 1);
  }
  __syncthreads();
  if (tid < num_experts) chunk_counts[(long)blockIdx.x * num_experts + tid] = s_cnt[tid];
}

// One workgroup per chunk.  Counts: kFromChunks from chunk_counts [gridDim.x, num_experts], kFromIds from the ids, kFromWaves from what the
// workgroup's wavefronts find in their own pairs anyway, where it is the only one (up to 1024 pairs; launched with as few wavefronts as
// hold the pairs and the experts).
//
// Latency from end to end (one workgroup per CU, a few thousand pairs): every id is read once per use with eight loads
// in flight, a wavefront's 64 pairs are ranked by ballots once, and the prefix sums run on the vector ALU.  As one
// workgroup that took up to 16384 pairs in dependent rounds, and as three launches past that, 128 experts took 10.5 us at
// 512 pairs (now 2.9), 22.3 at 16384 (6.1), 20.2 at 32768 (6.3), 24.6 at 131072 (8.0).  kFromWaves against a pass of LDS atomics by sixteen
// wavefronts: 8 pairs of 8 experts 3.3 -> 2.6, 128 of 128 3.6 -> 2.9, 512 of 128 3.7 -> 3.05, 1024 of 1024 4.7 -> 4.4.
enum Counts { kFromChunks, kFromIds, kFromWaves };
template <Counts COUNTS>
__global__ void __launch_bounds__(kRouteThreads) route_kernel(const int* ids, long num_pairs, int first_expert,
                                                              int num_experts, long chunk, const int* __restrict__ chunk_counts,
                                                              int n, int k, int* __restrict__ problem_sizes,
                                                              int* __restrict__ expert_offsets, int* __restrict__ blockscale_offsets,
                                                              int* dst_row) {
  __shared__ int s_wave[kRouteWaves][kMaxRouteExperts];   // a wavefront's pairs of every expert, then their first row
  __shared__ int s_before[kMaxRouteExperts];              // pairs of every expert in the chunks in front
  __shared__ int s_rest[kMaxRouteExperts];                // and in this chunk and the ones behind
  __shared__ int s_sum[kRouteWaves][2];
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int E = num_experts, me = blockIdx.x;
  const long base = (long)me * chunk;
  int raw = base + tid < num_pairs ? ids[base + tid] : 0;   // this thread's pair of the chunk's first 1024
  if constexpr (COUNTS != kFromWaves) {
    s_before[tid] = 0;
    s_rest[tid] = 0;
  }
  for (int e = lane; e < E; e += 64) s_wave[w][e] = 0;
  if constexpr (COUNTS != kFromWaves) __syncthreads();   // (the rows of s_wave are their wavefronts' own so far)
  constexpr int kBatch = 8;   // loads in flight
  if constexpr (COUNTS == kFromIds) {
    for (long p0 = 0; p0 < num_pairs; p0 += kBatch * kRouteThreads) {
      int v[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; u++) {
        const long p = p0 + u * kRouteThreads + tid;
        v[u] = p < num_pairs ? ids[p] : 0;
      }
#pragma unroll
      for (int u = 0; u < kBatch; u++) {
        const long first = p0 + u * kRouteThreads;
        if (first >= num_pairs) break;
        const int id = local_id(v[u], first + tid, num_pairs, first_expert, E);
        if (id >= 0) atomicAdd(first < base ? &s_before[id] : &s_rest[id], 1);   // (base is a multiple of 1024)
      }
    }
  } else if constexpr (COUNTS == kFromChunks) {
    // the counts as one flat array: thread t takes the words t, t + 1024, ...
    const int words = (int)gridDim.x * E, mine = me * E;
    for (int i0 = 0; i0 < words; i0 += kBatch * kRouteThreads) {
      int v[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; u++) {
        const int i = i0 + u * kRouteThreads + tid;
        v[u] = i < words ? chunk_counts[i] : 0;
      }
#pragma unroll
      for (int u = 0; u < kBatch; u++) {
        const int i = i0 + u * kRouteThreads + tid;
        if (v[u] != 0) atomicAdd(i < mine ? &s_before[i % E] : &s_rest[i % E], v[u]);
      }
    }
  }
  const int bits = id_bits(E);
  const int waves = COUNTS == kFromWaves ? (int)blockDim.x >> 6 : kRouteWaves;
  int run = 0;   // thread e: next free row of expert e
  for (long off = 0;;) {
    const long p = base + off + tid;
    const int id = local_id(raw, p, num_pairs, first_expert, E);
    // lanes with the same id take consecutive rows in lane order
    const unsigned long long same = lanes_with_same_id(id, bits);
    const int rank = __builtin_popcountll(same & ((1ull << lane) - 1ull));
    if (id >= 0 && rank == 0) s_wave[w][id] = __builtin_popcountll(same);
    __syncthreads();
    int c[kRouteWaves];   // every wavefront's pairs of expert tid
    auto counts = [&] {
#pragma unroll
      for (int i = 0; i < kRouteWaves; i++) c[i] = tid < E && i < waves ? s_wave[i][tid] : 0;
    };
    if (off == 0) {
      // the offsets: prefix sums over the experts, thread = expert
      int before = 0, total = 0;
      if constexpr (COUNTS == kFromWaves) {
        counts();
#pragma unroll
        for (int i = 0; i < kRouteWaves; i++) total += c[i];
      } else {
        before = s_before[tid];
        total = before + s_rest[tid];
      }
      const int padded = (total + 127) & ~127;
      const int so = wave_inclusive_sum(total), sp = wave_inclusive_sum(padded);
      if (lane == 63) {
        s_sum[w][0] = so;
        s_sum[w][1] = sp;
      }
      __syncthreads();
      int o = so - total, bo = sp - padded;
#pragma unroll
      for (int i = 0; i < kRouteWaves; i++) {
        o += i < w ? s_sum[i][0] : 0;
        bo += i < w ? s_sum[i][1] : 0;
      }
      run = o + before;
      if (me == 0 && tid < E) {
        expert_offsets[tid] = o;
        blockscale_offsets[tid] = bo;
        problem_sizes[tid * 3 + 0] = total;
        problem_sizes[tid * 3 + 1] = n;
        problem_sizes[tid * 3 + 2] = k;
        if (tid == E - 1) {
          expert_offsets[E] = o + total;
          blockscale_offsets[E] = bo + padded;
        }
      }
    }
    if (tid < E) {   // its first row of the expert
      if constexpr (COUNTS != kFromWaves) counts();
#pragma unroll
      for (int i = 0; i < kRouteWaves; i++) {
        if (i < waves) s_wave[i][tid] = run;
        run += c[i];
      }
    }
    __syncthreads();
    if (p < num_pairs) dst_row[p] = id >= 0 ? s_wave[w][id] + rank : -1;
    if constexpr (COUNTS == kFromWaves) break;
    off += kRouteThreads;
    if (off >= chunk || base + off >= num_pairs) break;   // the same for the whole workgroup
    raw = base + off + tid < num_pairs ? ids[base + off + tid] : 0;
    __syncthreads();
    for (int e = lane; e < E; e += 64) s_wave[w][e] = 0;   // (rewritten by this wavefront only)
  }
}

// Packs rows for the grouped operators: out[dst_row[p], :] = in[p / topk, :] for every local pair
// (2-byte elements, row_bytes a multiple of 16).  One wavefront moves one row in 1 KB steps.
__global__ void __launch_bounds__(256) permute_rows_kernel(const uint8_t* __restrict__ in, const int* __restrict__ dst_row,
                                                           long num_pairs, int topk, long row_bytes,
                                                           uint8_t* __restrict__ out) {
  typedef int v4i __attribute__((ext_vector_type(4)));
  const long p = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (p >= num_pairs) return;
  const int dst = dst_row[p];
  if (dst < 0) return;
  const uint8_t* src = in + (p / topk) * row_bytes;
  uint8_t* d = out + (long)dst * row_bytes;
  for (long off = (threadIdx.x & 63) * 16; off < row_bytes; off += 4096) {
    v4i v[4];
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (off + u * 1024 < row_bytes) v[u] = __builtin_nontemporal_load((const v4i*)(src + off + u * 1024));
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (off + u * 1024 < row_bytes) __builtin_nontemporal_store(v[u], (v4i*)(d + off + u * 1024));
  }
}

// Pieces of 4096 bytes up to which they are cut in four: half a wavefront per SIMD, so that what counts is how long each takes.  us, as pieces
// of 4096 / 1024 bytes: 1 token x 14 KB x top-8 2.9 / 2.4, 16 x 8 KB 3.5 / 2.6, 64 x 8 KB 3.75 / 3.1, 128 x 8 KB 4.0 / 3.4, 256 x 8 KB 4.5 / 4.4.
constexpr long kPermuteSmall = 512;
constexpr long kMaxPermutePieces = 1L << 22;     // of a launch (2^28 threads; a grid holds fewer than 2^32): larger inputs take several

// The same packing for topk > 1 (at most 64): one wavefront per piece (4096 bytes, or 1024) of a token's row reads it once and
// writes it to every local destination of the token's pairs, where one wavefront per pair would read it topk times.
//
// Bound by the output's bytes.  A wavefront per token walked the pieces one after the other: at 1003 tokens four wavefronts
// per CU, each waiting for memory four times.  Pieces of 1024 bytes are slower in calls of many (1003 tokens x 14336 bytes: 14.6
// against 12.7 us, 2048 x 8192: 27.4 / 24.7).
// Plain stores, where the launch moves more than 60 MB: the packed rows are what the caller quantises next, and what the
// 256 MB cache keeps of them is not fetched from HBM.  Below that they are slower than the non-temporal ones: they leave the
// rows dirty in the eight 4 MB L2s, and the launch's end waits until they are written back.  How many pairs have a local
// destination (under expert parallelism an eighth or so) stands in dst_row alone: every wavefront looks at the same 128
// pairs, in runs of eight spread over the call.  Packing + 1x128 quantisation, plain / hint / as chosen:
//   512 tokens x 14 KB x top-4, 28 MB packed:     21.8 /  17.7 /  17.8 us   2048 x 8 KB x top-8, 1/8 local, 16 MB:  16.4 / 13.3 / 13.2
//   700 x 14 KB x top-4, 38 MB:                   24.6 /  21.1 /  21.1      4096 x 4 KB x top-8, 1/8 local, 16 MB:  16.2 / 11.9 / 12.3
//   1003 x 14 KB x top-8, 110 MB:                 48.5 /  53.8 /  48.5      4096 x 14 KB x top-8, 1/8 local, 56 MB: 36.0 / 37.3 / 36.1
//   4096 x 8 KB x top-8, 256 MB:                 104.8 / 123.3 / 104.8      8192 x 14 KB x top-8, 1/64 local, 14 MB: 17.0 / 14.6 / 14.7
template <int LOADS>   // 16-byte loads in flight per lane, of a piece of LOADS KB
__global__ void __launch_bounds__(256) permute_rows_by_token_kernel(const uint8_t* __restrict__ in,
                                                                    const int* __restrict__ dst_row, uint32_t num_pieces,
                                                                    uint32_t pieces, int topk, long row_bytes, int plain_from,
                                                                    long sample_step, uint8_t* __restrict__ out) {
  typedef int v4i __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63;
  const uint32_t piece = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (piece >= num_pieces) return;
  const uint32_t t = pieces == 1 ? piece : piece / pieces;
  const int mine = lane < topk ? dst_row[(long)t * topk + lane] : -1;   // lane j: destination of the token's pair j
  if (__ballot(mine >= 0) == 0) return;                               // no local pair: the row is not read
  const long off = (long)(piece - t * pieces) * LOADS * 1024 + lane * 16;
  const uint8_t* src = in + (long)t * row_bytes + off;
  v4i v[LOADS];
#pragma unroll
  for (int u = 0; u < LOADS; u++)
    if (off + u * 1024 < row_bytes) v[u] = __builtin_nontemporal_load((const v4i*)(src + u * 1024));
  // (behind the row's loads: the samples come from a cache and are there first)
  bool plain = false;
  if (plain_from <= kPermuteSamples) {
    int sample[kPermuteSamples / 64], local = 0;
#pragma unroll
    for (int u = 0; u < kPermuteSamples / 64; u++) sample[u] = dst_row[(u * 8 + lane / kPermuteRun) * sample_step + lane % kPermuteRun];
#pragma unroll
    for (int u = 0; u < kPermuteSamples / 64; u++) local += __builtin_popcountll(__ballot(sample[u] >= 0));
    plain = local >= plain_from;
  }
  auto store = [&](auto hint) {   // (a loop per form: stores of both kinds in one would be merged into plain ones)
    for (int j = 0; j < topk; j++) {
      const int dst = __builtin_amdgcn_readlane(mine, j);
      if (dst < 0) continue;
      uint8_t* d = out + (long)dst * row_bytes + off;
#pragma unroll
      for (int u = 0; u < LOADS; u++)
        if (off + u * 1024 < row_bytes) {
          if constexpr (decltype(hint)::value) __builtin_nontemporal_store(v[u], (v4i*)(d + u * 1024));
          else *(v4i*)(d + u * 1024) = v[u];
        }
    }
  };
  if (plain) store(std::false_type{}); else store(std::true_type{});
}

}  // namespace esmoe

extern "C" int esmoe_launch_route_metadata(const int* ids, long num_pairs, int first_expert, int num_experts, int n, int k,
                                           int* problem_sizes, int* expert_offsets, int* blockscale_offsets, int* dst_row,
                                           int* chunk_counts, hipStream_t stream) {
  using namespace esmoe;
  const long chunk = route_chunk_pairs(num_pairs);
  const int chunks = num_pairs > 0 ? (int)((num_pairs + chunk - 1) / chunk) : 1;
  // (ids that are overwritten by their rows, dst_row == ids: with several workgroups none may still count from the ids when
  // another writes rows; route_kernel<kFromChunks> reads a pair's id only in the thread that writes its row)
  if (num_pairs <= kRouteThreads) {
    const int threads = ((int)num_pairs > num_experts ? (int)num_pairs + 63 : num_experts + 63) & ~63;
    hipLaunchKernelGGL(route_kernel<kFromWaves>, dim3(1), dim3(threads), 0, stream, ids, num_pairs, first_expert, num_experts,
                       chunk, (const int*)nullptr, n, k, problem_sizes, expert_offsets, blockscale_offsets, dst_row);
    return (int)hipGetLastError();
  }
  if (num_pairs <= kDirectPairs && dst_row != ids) {
    hipLaunchKernelGGL(route_kernel<kFromIds>, dim3(chunks), dim3(kRouteThreads), 0, stream, ids, num_pairs, first_expert, num_experts,
                       chunk, (const int*)nullptr, n, k, problem_sizes, expert_offsets, blockscale_offsets, dst_row);
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL(route_count_kernel, dim3(chunks), dim3(kRouteThreads), 0, stream, ids, num_pairs, first_expert, num_experts,
                     chunk, chunk_counts);
  hipLaunchKernelGGL(route_kernel<kFromChunks>, dim3(chunks), dim3(kRouteThreads), 0, stream, ids, num_pairs, first_expert, num_experts,
                     chunk, chunk_counts, n, k, problem_sizes, expert_offsets, blockscale_offsets, dst_row);
  return (int)hipGetLastError();
}

extern "C" int esmoe_launch_permute_rows(const void* in, const int* dst_row, long num_pairs, int topk, long row_bytes,
                                         void* out, hipStream_t stream) {
  using namespace esmoe;
  if (num_pairs == 0) return 0;
  if (topk > 1 && topk <= 64 && num_pairs % topk == 0) {
    const long tokens = num_pairs / topk;
    const int loads = tokens * ((row_bytes + 4095) / 4096) <= kPermuteSmall ? 1 : 4;
    const long pieces = (row_bytes + loads * 1024 - 1) / (loads * 1024);
    const int plain_from = permute_plain_from(tokens, topk, row_bytes);
    const long step = pieces < kMaxPermutePieces ? kMaxPermutePieces / pieces : 1;   // tokens of a launch
    for (long t = 0; t < tokens; t += step) {
      const long n = tokens - t < step ? tokens - t : step;
      auto kernel = loads == 1 ? permute_rows_by_token_kernel<1> : permute_rows_by_token_kernel<4>;
      hipLaunchKernelGGL(kernel, dim3((unsigned)((n * pieces + 3) / 4)), dim3(256), 0, stream,
                         (const uint8_t*)in + t * row_bytes, dst_row + t * topk, (uint32_t)(n * pieces), (uint32_t)pieces, topk, row_bytes,
                         n * topk >= kPermuteSamples ? plain_from : kPermuteSamples + 1, permute_sample_step(n * topk), (uint8_t*)out);
    }
    return (int)hipGetLastError();
  }
  hipLaunchKernelGGL(permute_rows_kernel, dim3((unsigned)((num_pairs + 3) / 4)), dim3(256), 0, stream, (const uint8_t*)in,
                     dst_row, num_pairs, topk, row_bytes, (uint8_t*)out);
  return (int)hipGetLastError();
}
