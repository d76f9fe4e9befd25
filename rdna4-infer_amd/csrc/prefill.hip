// Prefill dispatch: the MFMA kernels for head_dim 256 and 16-byte aligned
// buffers (attn_prefill_mfma.hip for f16 K/V, attn_prefill_quant.hip for the
// pairs with a quantized cache); every other shape runs the generic kernel
// with one CTA per (token, kv head) over keys 0..position.
#include <algorithm>
#include <cstdlib>

#include "prefill.hpp"

namespace rd4 {

bool prefill_supported(int kt, int vt, int n_head, int n_head_kv, int head_dim) {
  (void)kt; (void)vt; (void)n_head; (void)n_head_kv; (void)head_dim;
  return true;
}

namespace {

int compute_units() {
  static const int cus = [] {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
      return 0;
    return n;
  }();
  return cus;
}

// Rows per CTA and keys per block of a cache pair's MFMA kernel, and what a CTA
// costs on an MI355X: us per key block, and us before and after its blocks. (The
// f16 kernel's blocks take 2.2 us in a long call on few CUs and 3.2 on all; with a
// few blocks each, first use and masks included, 3.4. The last is taken for all calls:
// it decides where the counts are close, 168 gated queries from position 0 (32.1 us
// in one split, 26.9 in three), and a long call's best count differs little from its
// neighbours.)
struct Shape {
  int rows, keys;
  double block_us, cta_us;
};
Shape shape_of(int kt, int vt) {
  if (kt == F16 && vt == F16) return {192, 64, 3.4, 14.0};
  return {128, 32, 3.0, 14.0};
}
// The merge launch: us of the launch, and bytes of records written and read per us.
constexpr double kMergeUs = 2.0, kMergeBytesPerUs = 5e6;

}  // namespace

// Key splits: a CTA fills a CU, so without them a call runs as many CUs as it
// has row blocks, each over all keys. The count taken is the one of least
// estimated time: the CTAs of one round all run at once; a further round costs a
// whole CTA when the rows see about the same keys (a long prefix), and less when
// they differ (causal rows from position 0, heaviest first); the merge costs its
// launch and the records' traffic. Measured with these constants, calls in a row on one
// cache, no gate, merge included, forced counts of 1 to 64 beside the one taken (us: one split
// / best forced / taken). f16: 201 queries over 1534 keys 63 / 34 / 34, 64 over 8064
// 262 / 38 / 39, 16 over 30016 943 / 43 / 42, 512 over 8192 268 / 123 / 116, 512 over
// 512 32 / 31 / 34, 1000 over 2000 83 / 68 / 68, 168 over 168 21 / 21 / 23, 97 over 397
// 28 / 25 / 26, 700 over 700 39 / 37 / 39; q8_0: 16 over 8016 777 / 37 / 37, 64 over
// 1064 114 / 31 / 31, 512 over 8192 788 / 353 / 341, 512 over 512 62 / 42 / 48, 64 over
// 8064 779 / 64 / 59, 700 over 700 81 / 61 / 76, 900 over 4900 482 / 354 / 482. Over 26
// calls the count taken is within 5% of the best in 20, within 13% in four more; the
// last two of the list (q8_0, a second round of CTAs that costs less than the estimate)
// are 25 and 36% off. These calls have no gate. With one, which an unsplit CTA applies
// at its end and the merge launch in many more waves, short calls gain most: 168 over
// 168 with its gate and stores 42 us in one split, 31 in the count taken, 512 over 512
// 57 and 46; the f16 constants are theirs.
// RD4_PREFILL_KSPLIT forces a count (1: never split).
int prefill_ksplits(const PrefillArgs &p, int kt, int vt, int64_t max_floats) {
  static const int env = [] {
    const char *e = std::getenv("RD4_PREFILL_KSPLIT");
    return e ? std::atoi(e) : 0;
  }();
  const Shape sh = shape_of(kt, vt);
  const int grp = p.n_head / p.n_head_kv;
  const int total = (p.n_q * grp + sh.rows - 1) / sh.rows * p.n_head_kv;
  const int blocks = (p.kmax + sh.keys) / sh.keys;
  const int most = std::min(blocks, kMaxKSplits);
  if (env > 0) return std::max(1, std::min(env, most));
  const int cus = compute_units();
  if (cus <= 0) return 1;
  // mean blocks of a row: consecutive positions up to kmax
  const double mean = (std::max(0, p.kmax - p.n_q + 1) + 0.5 * std::min(p.n_q, p.kmax + 1)) / sh.keys;
  int best = 1;
  double best_us = 0;
  for (int s = 1; s <= most; ++s) {
    const int per = (blocks + s - 1) / s;
    if (s > 1 && (blocks + per - 1) / per != s) continue;  // as many as a smaller count with the same blocks
    if (s > 1 && prefill_part_floats(p, s) > max_floats) break;
    const int64_t ctas = (int64_t)total * s;
    const double one = per * sh.block_us + sh.cta_us;
    const double all = ((double)total * mean * sh.block_us + (double)ctas * sh.cta_us) / cus;
    const double alike = std::min(1.0, std::max(0.0, 2.0 * mean / blocks - 0.5));
    const double even = std::max(one, all);
    double us = even + alike * std::max(0.0, (double)((ctas + cus - 1) / cus) * one - even);
    if (s > 1) us += kMergeUs + (double)prefill_part_floats(p, s) * 4 / kMergeBytesPerUs;
    if (s == 1 || us < best_us) best = s, best_us = us;
    if (ctas > 4 * cus) break;  // more only adds records
  }
  return best;
}
int64_t prefill_part_floats(const PrefillArgs &p, int splits) {
  return (int64_t)splits * p.n_q * p.n_head * (p.head_dim + 2);
}
void prefill_set_ksplits(PrefillArgs &q, int splits, int bn) {
  q.n_ksplit = 1;
  q.ksplit_blocks = 0;
  if (splits <= 1 || !q.part || prefill_part_floats(q, splits) > q.part_floats) return;
  const int blocks = (q.kmax + bn) / bn;
  q.ksplit_blocks = (blocks + splits - 1) / splits;
  q.n_ksplit = (blocks + q.ksplit_blocks - 1) / q.ksplit_blocks;
}

hipError_t prefill_launch(int kt, int vt, const PrefillArgs &p, hipStream_t st) {
  const uintptr_t al = (uintptr_t)p.q | (uintptr_t)p.k | (uintptr_t)p.v | (uintptr_t)p.out |
                       (uintptr_t)p.gate;
  if ((al & 15) == 0 && prefill_mfma_supported(kt, vt, p.n_head, p.n_head_kv, p.head_dim)) {
    static const int dbg = [] { const char *e = std::getenv("RD4_PREFILL_DBG"); return e ? std::atoi(e) : 0; }();
    PrefillArgs q = p;
    q.dbg = dbg;
    return prefill_mfma_launch(q, st);
  }
  // A call with few keys is all launch and first-use latency, and the VALU
  // kernel's is shorter: 16 queries over 16 q8_0 keys 17.2 us there, 18.9 us on
  // the matrix cores; 64 over 64 30.8 against 24.1 us, 512 over 8192 6121
  // against 341 us.
  // (That kernel knows consecutive positions only; no entry point passes others
  // with a quantized cache.)
  if ((al & 15) == 0 && !p.pos && p.kmax >= 24 && prefill_quant_supported(kt, vt, p.n_head, p.n_head_kv, p.head_dim))
    return prefill_quant_launch(kt, vt, p, st);
  AttnArgs a{};
  a.q = (const float *)p.q;
  a.q_f16 = p.q_f16;
  a.k = p.k;
  a.v = p.v;
  a.out = p.out;
  a.gate = p.gate;
  a.pos = p.pos;
  a.t = p.pos0;
  a.kcap = p.kmax + 1;  // keys 0..min(pos[i], kmax), as the reference's tiling bound
  a.n_head = p.n_head;
  a.n_head_kv = p.n_head_kv;
  a.head_dim = p.head_dim;
  a.scale = p.scale;
  a.n_splits = 1;
  return attn_generic_launch(kt, vt, a, p.n_q, st);
}

}  // namespace rd4
