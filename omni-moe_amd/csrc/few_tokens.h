// The layer and the shared MLP for a few tokens (few_tokens.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "select.h"

namespace omni {

// 16-bit storage, at most 64 tokens (four matrix tiles of rows)
constexpr int kFewTokens = 64;

struct FewTokens {
  const void *x, *wg, *wu, *wd;
  void *h, *y;                       // h [T,I]
  float* parts;                      // few_tokens_parts_bytes()
  const void* residual = nullptr;    // MLP alone: added to the rounded projection (or NULL)
  int T, H, I;
  // the layer: the router's projection weights, z [T,2r] and its selection (select.lx, ly in z; no batch counts, no statistics out)
  const void *wx = nullptr, *wy = nullptr;
  void* z = nullptr;
  SelectArgs select{};
  // ... and the routed experts that select.gates and select.indices name
  const void *up = nullptr, *down = nullptr;
  int64_t N = 0;
};

bool few_tokens_covers(int64_t T, int64_t H, int64_t I, int dtype);
// ... and with a router of r keys per half and top-k, eval-mode BatchNorm, the gather algorithm's rows
bool few_tokens_covers_layer(int64_t T, int64_t H, int64_t I, int r, int k, int dtype);
size_t few_tokens_parts_bytes(int64_t T, int64_t H, int64_t I);
// rows are fetched 16 bytes at a time: every pointer of `f` (NULL counts as aligned) is
bool few_tokens_aligned(const FewTokens& f);
// launch 3 alone, for any number of tokens (H <= 4096): the experts, and the final add of `splits` parts [splits][T][H] (at most 8) or, with 0, of the rounded rows in y
hipError_t launch_few_back(int dtype, const FewTokens& f, int splits, hipStream_t s);
hipError_t launch_few_tokens(int dtype, const FewTokens& f, hipStream_t s);

}  // namespace omni
