// The prompt of a decode as one pass over all its positions
// (bfp_prefill.hip), instead of one step per position.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "bfp_layer.h"

namespace bfp {

// A pass over positions p0 .. p0 + n - 1 of `batch` sequences: row b*n + j
// is position p0 + j of sequence b.  L holds one layer's weights, KV cache
// and the row activations (L.batch = batch * n rows).
struct PrefillArgs {
  LayerArgs L;
  int batch, n, p0;
  const int *prompt;        // (batch, n_prompt) token ids, device
  int n_prompt, VOCAB;
  const float *embed;       // (VOCAB, D) float32
  double *qf;               // (rows, D) rotated q as float64
  int16_t *hist_m;          // optional: every layer's output, (batch, hist_steps, NL, D)
  int8_t *hist_e;
  int hist_steps;
};

// Most rows of one pass.
constexpr int PF_ROWS = 1024;
// Fewest positions a pass is made for, against the persistent batch-1 decode
// and against a batch's steps.  Calls at SmolLM2's 30 layers with 4 tokens
// generated, ms, pass / steps: batch 1, 3 positions about 3.98 / 3.86, 4 3.99 /
// 4.38, 6 4.00 / 5.43; 2 positions at batch 2 4.99 / 5.16, 5 5.30 / 5.55, 15
// 6.57 / 7.42, 16 7.21 / 8.41, 64 8.36 / 9.16.  (A pass of few rows is 8
// launches a layer whatever their number.)  At D 128 to 1728, 2 to 17 positions
// and 1 to 64 sequences no pass was behind its steps.
constexpr int PF_MIN_PERSIST = 4;
constexpr int PF_MIN = 2;

// Embedding rows of the pass's tokens into L.h_m / L.h_e.
int launch_prefill_embed(const PrefillArgs &a, hipStream_t s);
// One layer over the pass's rows: h in, h out, the cache rows written.
int launch_prefill_layer(const PrefillArgs &a, hipStream_t s);
// Raise the kernels' dynamic-LDS limits (outside any stream capture).
int prepare_prefill_kernels();

}  // namespace bfp
