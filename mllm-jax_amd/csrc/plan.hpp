// plan.hpp -- host-side planning of the fused GRPO loss: argument checks, chunking, the split of
// the d_hidden product, workspace layout, and the tile choices of the sampler's logits product.
//
// Plain C++ (no HIP header, no device code): mj_grpo.hip includes it, and a host-only build under
// the address / undefined-behaviour sanitizers checks it on the CPU -- an indexing mistake here is
// an out-of-bounds access on the GPU.
#pragma once
#include <math.h>
#include <stdarg.h>
#include <stddef.h>
#include <stdint.h>
#include <stdio.h>

#include "../../include/mj_grpo.h"

namespace mj {
namespace host {

inline thread_local char g_err[512] = "";

inline int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

constexpr int kValueRows = 64;             // token rows per workgroup of the value head's weight gradient
constexpr int BM = 256, BN = 256;          // tile of all three contractions
constexpr int64_t kDefaultChunk = 16384;   // tokens whose logits live in the workspace at once
constexpr int kRescueGrid = 256;           // workgroups of the rescue pass (one per CU)

inline int64_t rup(int64_t x, int64_t a) { return (x + a - 1) / a * a; }

struct Plan {
  int64_t N, H, V, chunk, n_pad, ld_z, parts;
  int dh_splits;          // vocab splits of the dHidden product (1 = none)
  int64_t dh_k_per_split;
  // byte offsets into the workspace
  size_t zy, term, eterm, pm, pl, ps, plt, g, ge, hent, state, rs, dead, hs, zt, part, total_fwd, total_bwd;
  // hidden of a chunk in fragment order: behind the regions of a forward pass, which runs without it in a workspace of
  // total_fwd bytes; in `hs` in a backward pass (the logits product is done with it before hs is written)
  size_t hid_frag, total_fwd_frag;
  // token compaction (MJ_GRPO_FLAG_SKIP_MASKED): slot-order copies of the inputs and outputs
  bool compact;
  size_t perm, n_live, hid_p, tgt_p, fin_p[5], fout_p[3], dh_p;
  // value head (mj_grpo_forward_backward_value): laid out behind total_bwd
  size_t v_term, v_dv, v_dv_p, v_part, total_value;
};

// Splits of the dHidden product over the vocab: its (n/256) x (H/256) tiles rarely fill the 256
// CUs in whole rounds, so K = V is cut into the fewest pieces (<= 32) that waste < 4% of a round.
inline int pick_splits(int64_t tiles) {
  int best = 1;
  double best_eff = 0.0;
  for (int s = 1; s <= 32; ++s) {
    const int64_t items = tiles * s, rounds = (items + 255) / 256;
    const double eff = (double)items / (double)(rounds * 256);
    if (eff > best_eff + 1e-9) { best_eff = eff; best = s; }
    if (eff >= 0.96) return s;
  }
  return best;
}

inline int make_plan(const MjGrpoDesc* d, Plan* p) {
  if (d == nullptr) return fail(MJ_GRPO_ERR_NULL, "desc is NULL");
  if (d->n_tokens <= 0 || d->hidden <= 0 || d->vocab <= 0)
    return fail(MJ_GRPO_ERR_SHAPE, "n_tokens/hidden/vocab must be positive (got %lld/%lld/%lld)",
                (long long)d->n_tokens, (long long)d->hidden, (long long)d->vocab);
  // 256 rows of any operand or output must fit one 2 GiB buffer descriptor
  if (d->n_tokens > (1ll << 30) || d->hidden > (1 << 20) || d->vocab > (1 << 21) || d->ld_hidden > (1 << 20) ||
      d->ld_w > (1 << 21) || d->chunk_tokens > (1 << 20))
    return fail(MJ_GRPO_ERR_SHAPE, "shape too large (hidden, ld_hidden <= 2^20; vocab, ld_w <= 2^21; chunk_tokens <= 2^20)");
  if (d->ld_hidden < d->hidden || d->ld_w < d->vocab)
    return fail(MJ_GRPO_ERR_SHAPE, "leading dimension smaller than row length");
  if (d->hidden % 8 || d->vocab % 8 || d->ld_hidden % 8 || d->ld_w % 8)
    return fail(MJ_GRPO_ERR_ALIGN, "hidden, vocab, ld_hidden and ld_w must be multiples of 8");
  if (!(d->temperature > 0.f) || !isfinite(d->temperature))
    return fail(MJ_GRPO_ERR_UNSUPPORTED, "temperature must be positive and finite (got %g)", (double)d->temperature);
  if (d->temperature != 1.0f && d->entropy_coef != 0.f)
    return fail(MJ_GRPO_ERR_UNSUPPORTED, "an entropy bonus needs temperature 1 (got %g)", (double)d->temperature);
  if (d->softcap < 0.f || !isfinite(d->softcap)) return fail(MJ_GRPO_ERR_UNSUPPORTED, "softcap must be >= 0");
  if (d->chunk_tokens < 0) return fail(MJ_GRPO_ERR_SHAPE, "chunk_tokens must be >= 0");
  if (d->flags & ~(uint32_t)(MJ_GRPO_FLAG_DW_ACCUMULATE | MJ_GRPO_FLAG_SFT | MJ_GRPO_FLAG_SKIP_MASKED | MJ_GRPO_FLAG_DW_BF16))
    return fail(MJ_GRPO_ERR_UNSUPPORTED, "unknown bits in flags (0x%x)", d->flags);
  if (!isfinite(d->inv_total_valid_tokens)) return fail(MJ_GRPO_ERR_SHAPE, "inv_total_valid_tokens not finite");
  if (!isfinite(d->entropy_coef) || !isfinite(d->inv_entropy_count) || d->inv_entropy_count < 0.f)
    return fail(MJ_GRPO_ERR_SHAPE, "entropy_coef / inv_entropy_count not finite");
  p->N = d->n_tokens; p->H = d->hidden; p->V = d->vocab;
  int64_t chunk = d->chunk_tokens > 0 ? d->chunk_tokens : kDefaultChunk;
  chunk = rup(chunk, 256);
  if (chunk > p->N) chunk = p->N;
  p->chunk = chunk;
  p->n_pad = rup(chunk, 256);
  p->ld_z = p->V;               // rows of the 16-bit matrix: V % 8 == 0 keeps them 16-byte aligned
  p->parts = 2 * ((p->V + BM - 1) / BM);
  if (d->dhidden_splits > 32) return fail(MJ_GRPO_ERR_SHAPE, "dhidden_splits must be <= 32 (got %u)", d->dhidden_splits);
  p->dh_splits = d->dhidden_splits ? (int)d->dhidden_splits : pick_splits((p->n_pad / BM) * ((p->H + BN - 1) / BN));
  p->dh_k_per_split = rup((p->V + p->dh_splits - 1) / p->dh_splits, 64);
  // pieces are whole 64-wide slices: a small vocabulary has fewer of them than the splits asked for
  p->dh_splits = (int)((p->V + p->dh_k_per_split - 1) / p->dh_k_per_split);
  const size_t frag_bytes = (size_t)p->n_pad * rup(p->H, 64) * 2;   // also of (rs * hidden)^T in whole 16-row blocks
  size_t o = 0;
  auto take = [&](size_t bytes) { size_t at = o; o = (size_t)rup((int64_t)(o + bytes), 256); return at; };
  p->zy = take((size_t)p->N * 4);
  p->term = take((size_t)p->N * 4);
  p->eterm = take((size_t)p->N * 4);
  p->pm = take((size_t)p->parts * p->n_pad * 4);
  p->pl = take((size_t)p->parts * p->n_pad * 4);
  p->ps = take((size_t)p->parts * p->n_pad * 4);
  p->plt = take(d->temperature != 1.0f ? (size_t)p->parts * p->n_pad * 4 : 0);
  p->g = take((size_t)p->n_pad * 4);
  p->ge = take((size_t)p->n_pad * 4);
  p->hent = take((size_t)p->n_pad * 4);
  p->state = take(256);
  p->compact = (d->flags & MJ_GRPO_FLAG_SKIP_MASKED) != 0;
  if (p->compact) {
    p->perm = take((size_t)p->N * 4);
    p->n_live = take(256);
    p->hid_p = take((size_t)p->N * p->H * 2);
    p->tgt_p = take((size_t)p->N * 4);
    for (auto& f : p->fin_p) f = take((size_t)p->N * 4);
    for (auto& f : p->fout_p) f = take((size_t)p->N * 4);
  }
  p->total_fwd = p->hid_frag = o;
  p->total_fwd_frag = (size_t)rup((int64_t)(o + frag_bytes), 256);
  p->dh_p = take(p->compact ? (size_t)p->N * p->H * 2 : 0);
  p->rs = take((size_t)p->n_pad * 4);
  p->dead = take((size_t)p->n_pad / 8);     // one bit per token of a chunk
  p->hs = take(frag_bytes);
  p->zt = take((size_t)p->n_pad * p->ld_z * 2);
  p->part = take(p->dh_splits > 1 ? (size_t)p->dh_splits * p->n_pad * p->H * 4 : 0);
  p->total_bwd = o;
  p->v_term = take((size_t)p->N * 4);
  p->v_dv = take((size_t)rup(p->N, 256) * 4);
  p->v_dv_p = take(p->compact ? (size_t)rup(p->N, 256) * 4 : 0);
  p->v_part = take((size_t)((p->N + kValueRows - 1) / kValueRows) * p->H * 4);
  p->total_value = o;
  return MJ_GRPO_OK;
}

// Whether the logits product reads hidden in fragment order.  The product gains with its size, the pass that writes the
// copy (k_fragment_rows) is a launch of 5 us at the least.  Product without, with, and the pass, us:
//   512 x 896 x 151936   181  176  5.4      1024 x 896 x 151936   324  324  5.4     512 x 1536 x 151936  250  253  5.7
//   512 x 2304 x 152064  343  335  5.4      1024 x 1536 x 151936  479  464  6.8     512 x 4096 x 128256  473  443  6.6
//   4096 x 1536 x 151936 1739 1687  9.8     5005 x 3584 x 152064 4393 4048 14.2     16384 x 3584 x 152064 14489 13073 38
inline bool fragment_hidden(int64_t n, int64_t h, int64_t v) { return (double)n * (double)h * (double)v >= 1.6e11; }

// mj_grpo_forward_noalloc: the plan whose forward workspace fits `scratch_bytes`.  chunk_tokens == 0
// picks the largest chunk (a multiple of 256 tokens, at most 16384) that fits.
inline int noalloc_plan(const MjGrpoDesc* desc, size_t scratch_bytes, MjGrpoDesc* d_out, Plan* p_out) {
  if (desc == nullptr) return fail(MJ_GRPO_ERR_NULL, "desc is NULL");
  MjGrpoDesc d = *desc;
  Plan p;
  int rc;
  if (d.chunk_tokens > 0) {
    if ((rc = make_plan(&d, &p))) return rc;
  } else {
    int64_t lo = 1, hi = (d.n_tokens + 255) / 256;   // in units of 256 tokens
    if (hi > 64) hi = 64;
    d.chunk_tokens = 256;
    if ((rc = make_plan(&d, &p))) return rc;
    while (p.total_fwd <= scratch_bytes && lo < hi) {
      const int64_t mid = (lo + hi + 1) / 2;
      MjGrpoDesc t = d;
      t.chunk_tokens = mid * 256;
      Plan q;
      if ((rc = make_plan(&t, &q))) return rc;
      if (q.total_fwd <= scratch_bytes) { lo = mid; d = t; p = q; } else { hi = mid - 1; }
    }
  }
  if (p.total_fwd > scratch_bytes)
    return fail(MJ_GRPO_ERR_WORKSPACE,
                "this shape needs %zu bytes of forward workspace with %lld-token chunks; the static array holds %zu "
                "(use mj_grpo_forward with a caller workspace)", p.total_fwd, (long long)p.chunk, scratch_bytes);
  *d_out = d;
  *p_out = p;
  return MJ_GRPO_OK;
}

// Sampler's logits product (b rows against the whole vocabulary): batch-row tile and vocab columns
// per work item -- the fewest rounds of resident workgroups (one per CU) whose items are <= 256
// columns wide.  Measured at 3584 x 152064: the 128-row tile beats both a 64-row tile with two
// workgroups per CU (0.25 against 0.23 ms at 64 rows) and, past 128 rows, is beaten by the 256-row
// tile (two 128-row tiles: 0.35 against 0.32 ms at 192 rows).
inline void sample_tiles(int64_t b, int64_t vocab, int* bn_out, int64_t* tiles_n_out, int64_t* tile_rows_out) {
  const int bn = b <= 128 ? 128 : 256;
  const int64_t tiles_n = (b + bn - 1) / bn;
  const int64_t slots = 256;
  int64_t tile_rows = BM;
  for (int64_t rounds = 1; rounds <= 4096; ++rounds) {
    const int64_t per = slots * rounds / tiles_n;            // items along the vocabulary
    if (per == 0) continue;
    const int64_t cols = rup((vocab + per - 1) / per, 8);
    if (cols <= BM) { tile_rows = cols; break; }
  }
  *bn_out = bn;
  *tiles_n_out = tiles_n;
  *tile_rows_out = tile_rows;
}

// The same product for one or two rows (k_logits_few): how many workgroups of at most 256 columns, in which units,
// with how many wavefronts, and in which order they go to the XCDs.  us at hidden 4096 (one row unless it says two):
// the matrix tile, 256-wide workgroups of four wavefronts in plain order whatever the vocabulary, and this rule:
//   65000    83.7  97.5  83.7   rows end inside a memory line (anything but a multiple of 256 bytes), and the
//                               neighbour that needs the other half of it sits on another XCD: kept on one
//   90000   121   141   116    352 workgroups for 256 CUs: some have two, the others wait.  From one round
//   200000  271   297   269    on a whole number of rounds, the columns spread evenly
//   32000    52    65    45    (two rows) half the CUs without a workgroup: up to 256 of at least 64 columns, and eight
//   36000    51    67    53    (two rows) wavefronts each; up to 176 workgroups for two rows, 144 for one
//   40000    53    52          (one row: split 55)
//   152064  221   217   208
//   256000  362   350   353    lines and rounds come out even: plain order (together it is 4 % slower)
// In between (45000 to 65536) 256-wide workgroups are as good as any: 50048 74.6, 64.7, 66.5.
struct FewItems {
  int items, unit, waves;
  bool together;          // neighbouring pieces on one XCD
};
inline FewItems few_items(int64_t b, int64_t vocab, int64_t ld_w) {
  const int64_t full = (vocab + 255) / 256;
  FewItems f = {(int)full, 256, 4, ld_w % 128 != 0};
  if (full > (b == 1 ? 144 : 176) && full <= 256) return f;
  f.unit = f.together ? 32 : 64;
  if (full > 256) f.items = (int)rup(full, 256);
  else {
    f.items = (int)((vocab + 63) / 64);
    if (f.items > 256) f.items = 256;
    f.waves = 8;
  }
  return f;
}

// Segments of a row for the top-k draw: as few as hold the row at kDrawSegment elements each, of even
// length.  segs == 0: the rows are drawn from without them -- short rows (below 4096 elements too few of a
// segment's groups of threads hold any, and one workgroup has a row in registers' reach anyway), rows longer
// than the logits product makes them (kDrawVocabMax; rounding seg_len up to 4 shortens the last segment by
// up to 4 elements per segment: about 500 of the 16384 at this length, all of them at 4096 segments), and launches
// with too many workgroups.
constexpr int kDrawSegment = 16384;
constexpr int64_t kDrawVocabMax = 1 << 21;
struct DrawSegments {
  int segs, seg_len;
  size_t bytes(int64_t b, int k) const { return (size_t)b * segs * k * 8; }     // k 64-bit words per segment
};
inline DrawSegments draw_segments(int64_t b, int64_t vocab) {
  DrawSegments g = {(int)((vocab + kDrawSegment - 1) / kDrawSegment), 0};
  if (b * g.segs > (1ll << 30) || vocab > kDrawVocabMax || vocab < 4096) g.segs = 0;
  else g.seg_len = (int)rup((vocab + g.segs - 1) / g.segs, 4);
  return g;
}

// RMSNorm: whether a matrix's single-use accesses carry the non-temporal hint (mj_norm_kernels.hpp).  From 100 MB
// on: x, dy and dx together are then past the 256 MB Infinity Cache, and what they push out of it costs more than
// finding a matrix there saves.  Kernels of a forward and a backward, us, with the hint and without, inputs in the
// caches / after 1.3 GB of other traffic (that traffic's own time included, as it pays for what is left dirty):
//   38.5 MB (8000 x 2416)  48.3, 44.0 /   -    54.7 MB (8000 x 3584)   63.2, 56.2 /   -
//   82 MB (12000 x 3584)   88.3, 83.4 / 344, 345     96 MB (14000 x 3584)   97.9, 95.6 / 356, 360
//   102.5 MB (15000 x 3584)  102.9, 107.2 / 360, 370   112 MB (16384 x 3584)  113.9, 116.9 / 371, 381
// With a reader of y and a producer of dy in between the sum of all of them differs by less than 1 % either way:
// the hint costs the backward 8 us at 54.7 and 112 MB and the copies around it gain as much.
inline bool norm_streams(int64_t n, int64_t h) { return n * h * 2 > (100ll << 20); }

}  // namespace host
}  // namespace mj
