// fbs_layers.h - the arguments of the layer by layer kernels (fbs_layers.hip), formed by
// fbs_api.cpp: tokens start .. start + len - 1 of `n` sequences' rows; position t of the stretch of
// sequence s is at index s * len + t of every per-position array.
#ifndef UOR_FBS_LAYERS_H
#define UOR_FBS_LAYERS_H

#include <hip/hip_runtime.h>

#include "fbs_device.h"

namespace fbs {

struct LayerArgs {
  uint32_t n, len;
  uint32_t row, start;        // a row's tokens, the stretch's first
  uint32_t taps_high;         // every tap_word of the model lies within +-2^27
  uint32_t turns;             // positions a wavefront of the front kernel takes in turn
  uint64_t len_recip;         // floor(2^32 / len): a position's sequence without a division
  const uint32_t *tokens;     // n * row
  const int64_t *in_state;    // the sessions resumed, as RunArgs' (nullable); a later stretch's are out_*
  const int32_t *in_history;
  const uint32_t *in_position;
  int64_t *out_state;         // the sessions after the tokens (nullable, the three together)
  int32_t *out_history;
  uint32_t *out_position;
  int32_t *status;            // n (a later stretch's sequences keep one that is not 0)
  uint32_t *steps;            // n: the positions before a refused one
  // Per position: the residual stream, the layer's drive, transition (the unit quaternion by the lane
  // weight) and output gate quaternion [d] i32, the window sum and then the moved state at the
  // residual's exponent [d] i64, the keeps [d / 4].
  int32_t *x, *drive, *turn, *gate;
  int64_t *rhs;
  uint32_t *keep;
  // Rows: the query kernel's positions first, first + 1, ... of the stretch; their choices (n * len);
  // each position's query, kept drawers and choice at its place in the rows, and the rows' next-token
  // matches (all nullable; without out_tokens a row's last choice is not made).
  uint32_t first;
  uint32_t *kept;             // a scan's positions * probes
  uint32_t *chosen;
  int32_t *out_query;
  uint32_t *out_kept;
  uint32_t *out_tokens;
  unsigned long long *matches;
};

// fbs_serve.hip
hipError_t launch_fbs_serve_scan(const DevModel &M, const ServeScan &J, uint32_t blocks, hipStream_t stream);
hipError_t launch_fbs_serve_finish(const DevModel &M, const ServeScan &J, hipStream_t stream);

// Whether the kernels' LDS serves the model's shapes.
bool fbs_layers_fit(const DevModel &M);
// Every layer over the positions; `rows`: also the end of the last one (the query kernel's input).
hipError_t launch_fbs_layers(const DevModel &M, const LayerArgs &P, bool rows, hipStream_t stream);
// A.n positions' queries, drawers and choices (S.out_tokens); `cus`: the device's compute units.
hipError_t launch_fbs_layer_query(const DevModel &M, const LayerArgs &P, const RunArgs &A, const ServeScan &S,
                                  uint32_t cus, hipStream_t stream);
// The stretch's choices to out_tokens, and those equal to their row's next token added to *matches.
hipError_t launch_fbs_layer_choices(const LayerArgs &P, hipStream_t stream);

}  // namespace fbs

#endif
