// Matrix prefill of a bf16 decoder stack: many prompt positions through every layer at once,
// filling the K/V cache the decode worker then continues from.
#pragma once

#include <cstddef>
#include <cstdint>

#include <hip/hip_runtime.h>

#include "tileinfer_amd.h"

namespace tiles {

class MatrixPrefill {
  public:
    // Positions per pass through the layers: the activation buffers hold this many rows.
    static constexpr int kChunkRows = 4096;
    // Or this many, for an object that has seen no longer prompt: 9 MB at Llama-3.2-1B widths instead of
    // 243, so that many contexts with short prompts hold little each.
    static constexpr int kShortRows = TI_MAX_LAUNCH_STEPS;
    // The shortest prompt that takes this path: its kernels read every weight once, in about the time of
    // two worker steps (Llama-3.2-1B: 3 tokens 1.34 ms against 1.97 through the worker, 37 tokens 1.45
    // against 19.2, 2 tokens 1.39 against 1.45; two of its layers alone: 3 tokens 0.68 against 0.77).
    static constexpr int kMinPrompt = 3;
    // Positions up to which the prompt's last token goes through the matrices as well (last_row) and its
    // hidden vector to the LM head, instead of a worker step, which reads every weight again: 0.4-0.5 ms
    // less from 3 tokens (1.34 ms against 1.71) to 1,024 (3.52 against 4.00).  Its attention is one pass
    // over the cache by a block a K/V head, which grows with the position; the worker splits it.
    static constexpr int kLastRowPositions = 1024;

    explicit MatrixPrefill(const ti_worker_program_view& program);
    ~MatrixPrefill();
    MatrixPrefill(const MatrixPrefill&) = delete;
    MatrixPrefill& operator=(const MatrixPrefill&) = delete;

    // Whether a package of this kind can be prefilled with matrices (bf16 decoder stacks).
    static bool supports(const ti_worker_program_view& program);

    // Makes sure of buffers for `count` positions, which enqueue() otherwise does itself.  On failure
    // (TI_* code, no memory) the object is as before.
    int reserve(int count);
    // Enqueues positions [position, position + count) of the prompt whose token ids are at
    // `tokens` (device memory, `count` of them) on `stream`: every layer's K and V rows of those
    // positions go into `kv`.  The positions before `position` must already be in the cache.
    // Returns a TI_* code; the message is in ti_last_error_message().
    int enqueue(hipStream_t stream, void* kv, const ti_token_id* tokens, int position, int count);
    // After enqueue: the rest of the last layer for the last of its positions.  `hidden` receives that
    // position's output of the stack (device memory of this object, good until the next enqueue).
    int last_row(hipStream_t stream, void* kv, int position, const void** hidden);

  private:
    ti_worker_program_view p_;
    struct Buffer {
        void* data = nullptr;  // the partial sums and every activation buffer
        int rows = 0;          // of each
    };
    Buffer short_, long_;  // kept; a short one too when a long one follows, as queued work may use it
    Buffer buffer_;        // the one in use
    int rows_ = 0;  // of the last pass: positions it left in the activation buffers
    int layer(hipStream_t stream, void* kv, int layer, int position, int rows);
    const uint16_t* weights(int layer) const;
    void feed_forward(hipStream_t stream, int layer, int rows, int first_row, const uint16_t* next_norm);
};

} // namespace tiles
