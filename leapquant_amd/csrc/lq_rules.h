// Host-side launch rules that tests evaluate on the CPU (no HIP in this file).
#pragma once

// Small launches, up to four heads per CU, take the kernels with helper waves (measured figures: lq_step.hip).
static inline bool lq_helper_waves(int N, int HV, int cus) { return (long long)N * HV <= 4ll * cus; }

// Value heads per workgroup of the one-launch KDA decode; 0: the step, then the flush, as two launches.
// A token's key is appended once per key head, by its first value head, and the flush of each of the key head's value
// heads reads it: with the flush in the step's launch, a workgroup therefore holds whole key heads (workgroups of one
// launch are not ordered, and their XCDs' L2s not coherent), so HV = H for one head per workgroup, and HV / H <= 2 for
// two.  Sizes, us per call, two launches -> one, 32 heads, W = 16: B = 48 18.6 -> 16.7, B = 64 21.7 -> 20.0, B = 96 27.9
// -> 27.3, B = 120 32.7 -> 31.7; W = 64, whose units also meet at each chunk's barriers: B = 48 21.9 -> 21.4, B = 64
// 25.6 -> 25.7, B = 96 33.9 -> 35.1.  An odd HV above four heads per CU takes two launches.
static inline int lq_kda_decode_heads(int N, int HV, int H, int L, int cus) {
  const long long heads = (long long)N * HV;
  if (HV == H && lq_helper_waves(N, HV, cus)) return 1;
  if (HV % 2 == 0 && HV / H <= 2 && (heads <= 8ll * cus || (L <= 32 && heads < 16ll * cus))) return 2;
  return 0;
}
