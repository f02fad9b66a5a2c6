// Gated output stage: launchers behind the oops_gate_* C entry points.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/oops_amd.h"

namespace oops {

// True when the fused projection kernel serves this geometry and these pointers.
bool gate_projection_ok(const oops_gate_geometry& g, const void* single, const void* weight,
                        const void* attention, const void* gated, const void* logits);

hipError_t launch_gate_projection(const oops_gate_geometry& g, const void* single, const void* weight,
                                  const void* attention, void* gated, void* logits, hipStream_t stream);
hipError_t launch_gate_multiply_forward(const oops_gate_geometry& g, const void* attention, const void* logits,
                                        void* gated, hipStream_t stream);
hipError_t launch_gate_multiply_backward(const oops_gate_geometry& g, const void* attention, const void* logits,
                                         const void* grad, void* grad_attention, void* grad_logits,
                                         hipStream_t stream);

// The whole stage in one pass over its rows (gate_stage.hip); the backward writes row_grad_parts(dtype, rows,
// out_channels, H * D) partials of the output weight's gradient.
bool gate_stage_ok(const oops_gate_geometry& g, int64_t out_channels, int64_t wo_row, const void* single,
                   const void* weight, const void* attention, const void* output_weight);
hipError_t launch_gate_stage_forward(const oops_gate_geometry& g, int64_t out_channels, int64_t wo_row,
                                     const void* single, const void* weight, const void* attention,
                                     const void* output_weight, void* out, void* logits, hipStream_t stream);
hipError_t launch_gate_stage_backward(const oops_gate_geometry& g, int64_t out_channels, int64_t wo_row,
                                      const void* grad, const void* attention, const void* logits,
                                      const void* output_weight, void* grad_attention, void* grad_logits,
                                      float* g_parts, hipStream_t stream);

// d = x w and partials of x^T y in one pass over x and y (gate_stage.hip)
int64_t row_grad_parts(int dtype, int64_t rows, int64_t k, int64_t n);
bool linear_grads_ok(int dtype, int64_t rows, int64_t k, int64_t n, const void* x, int64_t x_row, const void* w,
                     int64_t w_row, const void* y, int64_t y_row, const void* d, int64_t d_row);
hipError_t launch_linear_grads(int dtype, int64_t rows, int64_t k, int64_t n, const void* x, int64_t x_row,
                               const void* w, int64_t w_row, const void* y, int64_t y_row, void* d, int64_t d_row,
                               float* g_parts, hipStream_t stream);

}  // namespace oops
