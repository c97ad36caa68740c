// The streamed small tiles (stream.hip): the experts' grouped products for tiles of at most 64 rows over raw GGUF
// blocks, on the prefill's fp16 activations, and the same for dense rows on bf16 (hi + lo) ones.
#pragma once

#include "common.h"

namespace artlite {

// A launch: for each tile (expert e, sorted rows s0 .. s0 + bm) out[s][n] = sum_k A[row_a(s)][k] W_e[n][k] over fp16 rows
// of A, row_scale[s] = (x, y) as a prefill launch's (experts.h): SwiGLU launches (w[1] set) write h = silu(x g) (x u) y in
// fp16, plain ones fp16 y sum.
struct StreamArgs {
  const uint8_t* w[2];      // weight tensors: (gate, up) or (down, null); expert e at w + e expert_bytes
  int64_t expert_bytes;
  int row_bytes;
  int N, K;                 // output rows per expert, values per row
  int qtype;
  const uint16_t* a;        // A's rows of K values
  const int32_t* row_a;     // per sorted row s: its A row (a token); null: A row s
  const float2* row_scale;  // per sorted row
  int bm;                   // rows of A (tokens for gate / up, pairs for down) of a tile: 16, 32 or (Q4_0, Q4_K, Q8_0) 64
  const int32_t* tiles;     // (expert, first sorted row) per tile of bm rows, sorted rows ascending
  const int32_t* n_tiles;   // the tile count (device)
  int64_t max_tiles;        // grid bound
  int rows;                 // the sorted rows
  uint16_t* h;              // SwiGLU output (row stride N)
  uint16_t* y16;            // plain output (row stride N)
};

// The same for a few dense rows of one matrix over bf16 A (hi + lo planes): SwiGLU launches write h = silu(gate) up as bf16
// hi + lo planes, plain ones fp32.
struct StreamFewArgs {
  const uint8_t* w[2];
  int row_bytes;
  int N, K;
  int qtype;
  const uint16_t* a;      // A's rows of K values (the hi plane)
  const uint16_t* a_lo;   // lo plane (null: A is exactly bf16)
  int rows;
  uint16_t *h_hi, *h_lo;  // SwiGLU output planes (row stride N)
  float* y;               // plain output (row stride N)
};

// whether the streamed tiles take N rows of K values of weights of this type
bool stream_supported(int qtype, int K, int N);

// whether a launch of these takes every item of max_tiles tiles of bm rows
bool stream_fits(int qtype, bool swiglu, int N, int bm, int64_t max_tiles);

// the most rows of a launch of the dense rows (16 a step of the grid's second dimension)
constexpr int STREAM_FEW_ROWS = 65535 * 16;

int launch_stream(const StreamArgs& a, hipStream_t s);
int launch_stream_few(const StreamFewArgs& a, hipStream_t s);

}  // namespace artlite
