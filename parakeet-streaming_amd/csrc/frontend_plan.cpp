// Host bookkeeping of one front-end step (pk_fe_plan): the frame counters of
// FeatureExtractor.push / _trim_samples (parakeet/modules/feature_extractor.py:
// 97-151) and the window and cache steps of _run_pre_encode
// (parakeet/engine/model_runner.py:198-234) for every stream of a batch, and the
// device records of pk_fe_step and pk_subsample.  Integer arithmetic only; one
// pass to check and compute, one to commit, so a refused step changes nothing.
// 128 streams: 3 us, against about 110 us for the same in vectorised numpy.

#include <algorithm>
#include <cstdint>
#include <cstdlib>

#include "pk_common.h"

namespace {

int64_t floor_div(int64_t a, int64_t b) { return a / b - ((a % b != 0) && ((a < 0) != (b < 0))); }

struct Step {
  int64_t total, start, n_frames, cached, rows, offset, emitted;
  bool emit;
};

}  // namespace

extern "C" int pk_fe_plan(pk_fe_plan_args* a) {
  pk::clear_error();
  const char* what = "pk_fe_plan";
  if (!a) return pk::fail(PK_ERR_INVALID, "%s: args is NULL", what);
  const int32_t B = a->batch;
  if (B < 0 || a->num_slots < 1 || a->hop < 1 || a->n_fft < 1)
    return pk::fail(PK_ERR_INVALID, "%s: batch %d, slots %d, hop %d, n_fft %d", what, B, a->num_slots, a->hop, a->n_fft);
  a->max_new = a->max_frames = a->max_out = a->out_rows = a->sub_batch = 0;
  if (B == 0) return PK_OK;
  const void* need[] = {a->total, a->emitted, a->offset, a->cached, a->has_cache, a->last_window, a->noise_id,
                        a->slots, a->n_new, a->final_flag, a->fe, a->sub, a->start, a->n_frames, a->n_out, a->out_row};
  for (const void* q : need)
    if (!q) return pk::fail(PK_ERR_INVALID, "%s: an array is NULL", what);
  unsigned char* seen = static_cast<unsigned char*>(std::calloc((size_t)a->num_slots, 1));
  Step* st = static_cast<Step*>(std::malloc(sizeof(Step) * (size_t)B));
  int rc = PK_OK;
  if (!seen || !st) rc = pk::fail(PK_ERR_EXHAUSTED, "%s: out of host memory", what);
  const int64_t hop = a->hop, pad = a->n_fft / 2, lead = (a->n_fft - a->win_length) / 2;
  int64_t over_ring = 0, over_rows = 0;  // the largest ones: what the messages name
  for (int32_t i = 0; rc == PK_OK && i < B; ++i) {
    const int64_t s = a->slots[i];
    if (s < 0 || s >= a->num_slots || seen[s]) {
      rc = pk::fail(PK_ERR_STATE, "slots must be distinct and in range");
      break;
    }
    seen[s] = 1;
    const int64_t n = a->n_new[i];
    const bool fin = a->final_flag[i] != 0;
    Step& t = st[i];
    t.total = a->total[s] + n;
    const int64_t last = fin ? floor_div(t.total, hop) : floor_div(t.total - pad, hop);
    const int64_t off = a->offset[s];
    t.start = std::max(a->emitted[s], off == 0 ? (int64_t)0 : floor_div(off + pad + hop - 1, hop));
    t.emit = n > 0 && (fin || t.total > pad) && t.start <= last;
    t.n_frames = t.emit ? last - t.start + 1 : 0;
    // every sample a frame reads is in the ring and not overwritten by this push
    const int64_t held = t.emit ? t.total - std::max(t.start * hop - pad + lead - 1, (int64_t)0) : n;
    if (held > a->ring_size) over_ring = std::max(over_ring, held);
    t.emitted = t.emit ? last + 1 : a->emitted[s];
    const int64_t keep = std::max((int64_t)0, t.emitted * hop - pad), aligned = floor_div(keep, hop) * hop;
    t.offset = t.emit && keep > off && aligned > off ? aligned : off;
    t.cached = t.emit ? a->cached[s] : 0;
    t.rows = t.cached + t.n_frames;
    if (t.rows > a->mel_rows) over_rows = std::max(over_rows, t.rows);
  }
  if (rc == PK_OK && over_ring)
    rc = pk::fail(PK_ERR_EXHAUSTED, "a push needs %lld samples in the ring (ring_size %lld)", (long long)over_ring, (long long)a->ring_size);
  if (rc == PK_OK && over_rows)
    rc = pk::fail(PK_ERR_EXHAUSTED, "a window of %lld frames exceeds the mel ring (%lld rows)", (long long)over_rows, (long long)a->mel_rows);
  for (int32_t i = 0; rc == PK_OK && i < B; ++i) {
    const int64_t s = a->slots[i];
    const Step& t = st[i];
    pk_fe_stream& f = a->fe[i];
    f.slot = (int32_t)s;
    f.n_new = (int32_t)a->n_new[i];
    f.sample_base = a->total[s];
    f.frame0 = t.emit ? (int32_t)t.start : 0;
    f.n_frames = (int32_t)t.n_frames;
    f.noise_id = a->noise_id[s];
    f.reserved = 0;
    const int64_t drop = a->has_cache[s] ? a->drop : 0;
    const int64_t len = ((t.rows / 2 + 1) / 2 + 1) / 2 + 1;  // after the three stride-2 convolutions
    const int64_t out = t.emit ? std::max(len - drop, (int64_t)0) : 0;
    a->start[i] = t.start;
    a->n_frames[i] = t.n_frames;
    a->n_out[i] = out;
    a->out_row[i] = 0;
    if (out > 0) {
      pk_sub_stream& r = a->sub[a->sub_batch++];
      r.slot = (int32_t)s;
      r.row0 = (int32_t)(t.start - t.cached);
      r.rows = r.length = (int32_t)t.rows;
      r.drop = (int32_t)drop;
      r.n_out = (int32_t)out;
      r.out_row = (int32_t)a->out_rows;
      r.reserved = 0;
      a->out_row[i] = a->out_rows;
      a->out_rows += out;
    }
    a->max_new = i == 0 ? a->n_new[0] : std::max(a->max_new, a->n_new[i]);  // negative: pk_fe_step refuses it
    a->max_frames = std::max(a->max_frames, t.n_frames);
    a->max_out = std::max(a->max_out, out);
    a->total[s] = t.total;
    a->emitted[s] = t.emitted;
    a->offset[s] = t.offset;
    if (t.emit) {
      if (a->cache_size > 0) {
        a->cached[s] = std::min(t.rows, (int64_t)a->cache_size);
        a->has_cache[s] = 1;
      }
      a->last_window[2 * s] = t.start - t.cached;
      a->last_window[2 * s + 1] = t.rows;
    }
  }
  std::free(seen);
  std::free(st);
  return rc;
}
