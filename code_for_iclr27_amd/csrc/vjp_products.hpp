// The margin helpers' products with a bf16 weight on matrix cores (vjp_products.hip).
#pragma once

#include "lr_common.hpp"

namespace lr {

constexpr int kProductRows = 8;  // f32 rows of one launch

// out[r * vocab + v] = hidden[r] . weight[v] (+ bias[v]) for `rows` <= kProductRows.
bool takes_head_products(int dtype, int64_t rows, int64_t vocab, int64_t dim);
int launch_head_products(const float* hidden, int64_t rows, const void* weight, const void* bias,
                         int64_t vocab, int64_t dim, float* out, hipStream_t stream);

// Z[block, r, :] = sum over the block's weight rows v of c[r, v] * weight[v], c the competitors'
// softmax (exp(l - M) / S, 0 at the target), for `rows` <= kProductRows.
bool takes_column_products(int dtype, int64_t rows, int64_t vocab, int64_t dim);
int64_t column_product_block_rows(int64_t vocab, int64_t dim);
int launch_column_products(const void* weight, int64_t vocab, int64_t dim, int64_t rows,
                           const float* logits, const float* stats, const int64_t* targets,
                           float* partial, hipStream_t stream);

}  // namespace lr
