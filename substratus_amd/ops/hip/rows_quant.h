// Products of a few rows with GGUF-quantized weights (rows_quant.hip).
#pragma once

#include "rows_gemm.h"

enum class Quant { Q4_0, Q8_0, Q4_K, Q6_K };

bool rows_quant_thin(int m, int n, int k, Quant q, bool paired);
bool rows_quant_takes(int m, int n, int k, Quant q, bool gated);

void launch_rows_quant(bf16_t* y, const bf16_t* x, const void* scales,
                       const unsigned char* qs, int m, int n, int k, Quant q,
                       bool gated, const Heads* heads, const NormOf* norm,
                       const AddTo* add, const Undivided* of,
                       hipStream_t stream);
