// Where a short convolution over a chunk of a prompt portion finds its inputs.
#pragma once

enum class WindowRow { kBatch, kRing, kNone };

// Token t of a chunk of `count` tokens that begins at position pos0 of a portion that begins at position first_pos; t < 0: tokens in front of the chunk.
// kBatch: the row t behind the chunk's first one; kRing: the ring's entry of position pos0 + t; kNone: zero, and nothing is read: in front of the sequence,
// behind the chunk's tokens, and a chunk without any, whose first row need not be one of its portion.
__host__ __device__ inline WindowRow window_row(int count, int pos0, int first_pos, int t) {
    if (count <= 0 || t >= count || pos0 + t < 0) return WindowRow::kNone;
    return pos0 + t >= first_pos ? WindowRow::kBatch : WindowRow::kRing;
}
