// How the row packing of several pairs per token (routing.hip) chooses between plain and non-temporal stores, in plain C++
// so that it is tested on the CPU.
#pragma once

namespace esmoe {

// Bytes a launch moves above which its rows are stored plainly (both sides measured: permute_rows_by_token_kernel).
constexpr long kPlainPermuteBytes = 60L << 20;
// How many pairs have a local destination stands in dst_row alone.  A launch looks at so many of its pairs, in runs spread over
// them (a run of eight is one cache line at most twice); a call with fewer pairs never stores plainly.
constexpr int kPermuteSamples = 128, kPermuteRun = 8;

// Pairs between the starts of two runs: run r covers pairs r * step .. r * step + 7.
inline long permute_sample_step(long num_pairs) { return num_pairs / (kPermuteSamples / kPermuteRun); }

// Samples with a local destination from which the rows are stored plainly; kPermuteSamples + 1: none, no need to look.
// A launch moves the packed rows and the tokens' rows, of which no more are read than are written, so the line is crossed
// by kPlainPermuteBytes less the tokens' rows, or by half of it.
inline int permute_plain_from(long tokens, int topk, long row_bytes) {
  const long pairs = tokens * topk;
  const long line = tokens < kPlainPermuteBytes / 2 / row_bytes ? kPlainPermuteBytes - tokens * row_bytes : kPlainPermuteBytes / 2;
  if (pairs < kPermuteSamples || pairs <= line / row_bytes) return kPermuteSamples + 1;
  return (int)(kPermuteSamples * (double)line / ((double)pairs * (double)row_bytes)) + 1;
}

}  // namespace esmoe
