// Host-side launch rules of the decode calls: which form a call takes.  No HIP in this file: tests evaluate it on the CPU.
// Figures are us per call on 256 CUs at K = V = 128 and window 16 unless said otherwise; "in step": all rows at one fill;
// "apart": rows at different fills, one call apart (or, in brackets, at random fills).
#pragma once

// TWO_LAUNCHES: the step, then the persistent flush.  ONE_LAUNCH: the step's workgroups flush the heads they fill, in turn.
// HELPER_WAVES: the same with 256 threads per value head, half of which only flush, so that a workgroup's heads are flushed
// side by side.
enum lq_form { LQ_TWO_LAUNCHES, LQ_ONE_LAUNCH, LQ_HELPER_WAVES };

// The GDN decode.  A second launch costs a call ~2 us also when nothing is due: two launches -> one, in step: GQA 4, B = 24,
// 16 key heads 15.8 -> 12.2, B = 200 77.2 -> 71.0; GQA 1, 32 heads, B = 64 21.0 -> 16.4; (64, 128) at GQA 2, B = 64 13.0 ->
// 10.4; (64, 64) at GQA 1, B = 64 10.9 -> 8.5.  GQA 1 pairs two key heads of a row in a workgroup, so an odd H takes two.
//
// Helper waves up to four heads per CU, where all stay resident.  Without -> with, in step, at 2, 4 and 5 or 6 heads per CU:
// GQA 1, 16 heads 7.4 -> 7.2, 9.5 -> 9.4, 12.3 -> 13.1; GQA 2, 16 key heads 7.1 -> 7.0, 9.3 -> 9.3, 11.5 -> 13.2; GQA 4 with
// conv 12.1 -> 11.9, 13.4 -> 13.1, 17.6 -> 23.9.  Apart they gain more, 4 heads per CU: GQA 1 25.6 -> 17.1, GQA 2 25.1 ->
// 20.4.  GQA 4 without conv has two workgroups of two heads per key head instead, which flush two heads in turn sooner than
// helpers flush four at once: at 1, 2, 3 and 4 heads per CU in step 6.9 | 7.8, 7.2 | 8.1, 8.7 | 8.6, 9.5 | 9.2 with helpers,
// apart 10.1 | 11.3, 14.8 | 16.7, 20.1 | 22.2, 24.9 | 27.6.
//
// The lines for rows in step are the plain entry's.  The deferred entry is for rows that fill their windows on different
// calls, and takes two launches where the flush of a few rows' heads, spread over the CUs, beats flushes in turn behind
// their own step: at GQA 4 with V = 128 when a row is due in about a quarter of the calls (N = L / 4) or more and heads are few
// (up to one per CU; with the conv, whose four heads stay in one workgroup, two): two launches | one, apart, 4 key heads: B = 4
// 10.3 | 9.8, B = 8 13.1 | 14.1, B = 16 19.6 | 22.2 [15.7 | 16.6], B = 24 (1.5 per CU) 23.0 | 22.5; with conv B = 4
// 14.0 | 14.6, B = 16 23.4 | 29.0, B = 32 (2 per CU) 30.3 | 30.8, B = 40 33.1 | 30.9; 16 key heads with conv B = 8 (2 per
// CU) 20.9 | 20.9.  With the conv above four heads per CU: B = 24 38.2 | 43.1, in step 19.4 | 17.6.  At ranks 5 to 8 and
// GQA 4 always, whose 512-thread form flushes two heads at a time: 16 key heads, B = 8 20.9 | 29.3 [18.1 | 23.9], B = 32
// 46.0 | 57.0 [44.5 | 53.5]; in step, which the plain entry's line is drawn by, 10.7 | 10.1 and 20.0 | 17.4.
//
// Large (64, 64) batches at GQA 4 take two launches: the flush there needs more LDS and registers than the step: at 8 rows x
// H per CU 25.2 in two launches | 23.7, at 10 29.8 | 29.0, at 12.5 35.1 | 37.4; with conv at 4 16.6 | 14.3, at 6 20.9 |
// 20.0, at 8 25.2 | 25.6.
static inline lq_form lq_gdn_decode_form(int N, int HV, int H, int K, int V, int R, int L, bool conv, bool deferred,
                                         int cus) {
  const int G = HV / H;
  const long long heads = (long long)N * HV;
  const bool few = heads <= 4ll * cus;
  if (G == 1) {
    if (R > 4 || H % 2 != 0) return LQ_TWO_LAUNCHES;
    return few ? LQ_HELPER_WAVES : LQ_ONE_LAUNCH;
  }
  if (G != 2 && G != 4) return LQ_TWO_LAUNCHES;
  if (R > 4) return G == 4 && deferred ? LQ_TWO_LAUNCHES : LQ_ONE_LAUNCH;
  if (G == 2) return V == 128 && few ? LQ_HELPER_WAVES : LQ_ONE_LAUNCH;
  if (V == 64) return (long long)N * H <= (conv ? 6ll : 10ll) * cus ? LQ_ONE_LAUNCH : LQ_TWO_LAUNCHES;
  const bool often = conv ? 4ll * N >= L : 4ll * N > L;   // a row is due in a quarter of the calls, or in more
  if (deferred && often && heads <= (conv ? 2ll : 1ll) * cus) return LQ_TWO_LAUNCHES;
  if (conv) return few ? LQ_HELPER_WAVES : deferred ? LQ_TWO_LAUNCHES : LQ_ONE_LAUNCH;
  return few && heads > 2ll * cus && !deferred ? LQ_HELPER_WAVES : LQ_ONE_LAUNCH;
}

// Value heads per workgroup of the one-launch KDA decode; 0: the step, then the flush, as two launches.
// A token's key is appended once per key head, by its first value head, and the flush of each of the key head's value
// heads reads it: with the flush in the step's launch, a workgroup therefore holds whole key heads (workgroups of one
// launch are not ordered, and their XCDs' L2s not coherent), so HV = H for one head per workgroup, and HV / H <= 2 for
// two.  Sizes, two launches -> one, 32 heads, in step [at random fills]: windows of one chunk of the step (32 entries), W = 16:
// B = 48 17.5 -> 16.0, B = 64 21.1 -> 19.1 [43.4 -> 36.1], B = 128 33.6 -> 33.0 [56.7 -> 50.5], B = 256 58.7 -> 57.8 [81.2 ->
// 73.0]; W = 32: B = 128 34.6 -> 34.4 [62.0 -> 51.3], B = 256 61.1 -> 60.8 [89.4 -> 75.3]; W = 8: B = 256 63.5 -> 61.9
// [81.8 -> 79.3].  W = 64, whose units also meet at each chunk's barriers, up to eight heads per CU: B = 48 21.9 -> 21.4,
// B = 64 25.6 -> 25.7 [44.1 -> 40.3], B = 96 33.9 -> 35.1.  An odd HV above four heads per CU takes two launches.
static inline int lq_kda_decode_heads(int N, int HV, int H, int L, int cus) {
  const long long heads = (long long)N * HV;
  if (HV == H && heads <= 4ll * cus) return 1;
  if (HV % 2 == 0 && HV / H <= 2 && (L <= 32 || heads <= 8ll * cus)) return 2;
  return 0;
}
