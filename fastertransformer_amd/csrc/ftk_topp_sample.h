// Host side of the top-p step that samples straight from logits (topp_sample_kernels.hip), called by the entry points
// in topp_kernels.hip.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "ftk_sampling.h"

namespace ftk {

struct ToppSampleCall {
    int         dtype;
    void*       workspace;
    size_t      workspace_size;
    const void* logits;
    const void* bias;
    int         vocab_size;
    size_t      vocab_size_padded;
    int         rows;
    // penalties (all null / none: the logits as they are)
    const float* temperatures;
    const float* penalties;
    int          penalty_type;
    const int*   min_lengths;
    const int*   input_lengths;
    const int*   history;
    int          batch_size, step, max_input_length;
    // sampling
    const int*      end_ids;
    bool*           finished;
    int*            sequence_length;
    int*            output_ids;
    float*          cum_log_probs;
    float*          output_log_probs;
    ftk_rng_state*  rng_state;
    const float*    uniform_draws;
    float           max_top_p;
    float*          runtime_top_p;
    const float*    initial_top_p;
    const float*    top_p_decay;
    const float*    top_p_min;
    const int32_t*  top_p_reset_ids;
    const bool*     skip_decode;
};

size_t topp_sample_bytes(int dtype, int rows, int vocab, size_t vocab_padded, bool keeps_y);
bool   topp_sample_covers(int dtype, int rows, int vocab, bool history_penalty);
int    topp_sample_launch(const ToppSampleCall& call, hipStream_t stream);

// non-zero in the test build when a test asked for it: every row takes the whole-row fallback
int topp_force_deep();

}  // namespace ftk
