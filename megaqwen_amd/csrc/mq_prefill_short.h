// Interface of the single-launch prefill of short prompts (mq_prefill_short.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "megaqwen_amd.h"
#include "mq_common.h"

namespace mq {
namespace ps {

constexpr int SHORT_MAX_S = 256;  // longest prompt it takes
constexpr int DEAD_WORD = 16;     // word of `sync` that is set once a wait of the launch has given up

struct ShortArgs {
  int S, num_layers, max_seq;
  int groups;  // tasks a column slice's row blocks are dealt to, set by prefill_short_run
  float scale;
  uint64_t place_ticks;  // wait for workgroups on every XCD (0: a single list at once), set likewise
  uint16_t *h, *q, *att, *mid;  // [S, 1024], [S, 2048], [S, 2048], [S, 3072] bf16
  uint16_t *kc, *vc;            // caches, [layers][8][max_seq][128]
  const uint16_t *cos_t, *sin_t;
  uint32_t *sync, *local;  // scratch of 4 KB (tickets, words that cross XCDs) and S x 2 KB (words per XCD)
  uint32_t* err;
  PrefillLayerWeights lw[MAX_LAYERS];
};

}  // namespace ps

// Embedding rows and every layer of a prompt of at most SHORT_MAX_S tokens: h holds the residual
// stream after the last layer, the caches the prompt's K and V rows. `debug`: MQ_DEBUG_PREFILL_* flags.
// MQ_OK or MQ_ERR_HIP.
int prefill_short_run(const int* ids, const uint16_t* embed, const ps::ShortArgs& A, int debug, hipStream_t stream);

}  // namespace mq
