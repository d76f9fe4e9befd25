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
// costs on an MI355X: us per key block, and us before and after its blocks.
struct Shape {
  int rows, keys;
  double block_us, cta_us;
};
Shape shape_of(int kt, int vt) {
  if (kt == F16 && vt == F16) return {192, 64, 3.2, 8.0};
  return {128, 32, 3.4, 8.0};
}

}  // namespace

// A CTA fills a CU, so a call takes ceil(CTAs / CUs) rounds of CTAs. The f16
// kernel's splits: when its row blocks leave CUs idle (the reference engine's
// 512-query chunks: 64 CTAs on 256 CUs), about one CTA per CU, at most 16 and
// at most one per key block. RD4_PREFILL_KSPLIT forces a count (1: never split).
int prefill_ksplits(const PrefillArgs &p, int kt, int vt, int64_t max_floats) {
  static const int env = [] {
    const char *e = std::getenv("RD4_PREFILL_KSPLIT");
    return e ? std::atoi(e) : 0;
  }();
  const Shape sh = shape_of(kt, vt);
  const int grp = p.n_head / p.n_head_kv;
  const int total = (p.n_q * grp + sh.rows - 1) / sh.rows * p.n_head_kv;
  const int blocks = (p.kmax + sh.keys) / sh.keys;
  const int cus = compute_units();
  if (env > 0) return std::max(1, std::min(env, std::min(blocks, 64)));
  if (cus <= 0) return 1;
  if (kt == F16 && vt == F16)
    return std::max(1, std::min((total % 8 == 0 && 2 * total <= cus) ? cus / total : 1, std::min(blocks, 16)));
  int best = 1;
  double best_us = 0;
  for (int s = 1; s <= std::min(blocks, 64); ++s) {
    if (s > 1 && prefill_part_floats(p, s) > max_floats) break;
    const int per = (blocks + s - 1) / s;
    if (s > 1 && (blocks + per - 1) / per != s) continue;
    const int rounds = (total * s + cus - 1) / cus;
    double us = rounds * (per * sh.block_us + sh.cta_us);
    if (s > 1) us += 4.0 + (double)prefill_part_floats(p, s) * 4 / 3.5e6;
    if (s == 1 || us < best_us) best = s, best_us = us;
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
  // against 384 us.
  if ((al & 15) == 0 && p.kmax >= 24 && prefill_quant_supported(kt, vt, p.n_head, p.n_head_kv, p.head_dim))
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
