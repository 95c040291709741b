// The tiled multi-token products' launches, planes and counts made.
#pragma once

#include "q8_internal.h"

int iris_gemm_row_launch(const GemvArgs& a, hipStream_t stream);
int iris_gemm_fold_launch(const GemvArgs& a, hipStream_t stream);
// The shapes they take, by name (iris_product_route).
void iris_gemm_row_route(const GemvArgs& a, char* name, size_t size);
void iris_gemm_fold_route(const GemvArgs& a, char* name, size_t size);
