// Inputs of a captured decode step: the live rows of q, k, v, slots, context lengths
// and block tables copied into the graph's static buffers, the rows up to the graph's
// size padded (replaces run_model's zero fills and row copies, nanovllm/engine/
// model_runner.py:271-280).
//
// As tensor operations this is six fills and six copies, each a launch of ~2 us for a
// few KB to a few MB; here it is one.  Workgroup = one row: its threads stream the
// row's three bf16 pieces (16 bytes per lane) and its block-table entries.  What bounds
// it is the launch.  28 layers, 13 live rows in the graph of 16 (heads 16/8, contexts of
// 100 to 2048 tokens): the whole step went from 654.4 to 634.8 us.
#include "nva_common.h"
#include "nva_kernels.h"

namespace nva {

namespace {

// `n16` 16-byte pieces from src (null: zeros) to dst.
__device__ __forceinline__ void put_row(void* dst, const void* src, int n16) {
  for (int i = threadIdx.x; i < n16; i += blockDim.x)
    st16(static_cast<char*>(dst) + 16 * i, src ? ld16(static_cast<const char*>(src) + 16 * i) : u32x4{0u, 0u, 0u, 0u});
}

__global__ __launch_bounds__(256) void stage_decode_kernel(StageParams p) {
  const int64_t b = blockIdx.x;
  const bool live = b < p.live;
  put_row(p.q_out + b * p.q_elems, live ? p.q + b * p.q_row_stride : nullptr, p.q_elems / 8);
  put_row(p.k_out + b * p.kv_elems, live ? p.k + b * p.k_row_stride : nullptr, p.kv_elems / 8);
  put_row(p.v_out + b * p.kv_elems, live ? p.v + b * p.v_row_stride : nullptr, p.kv_elems / 8);
  const int width = live ? p.width : 0;
  for (int i = threadIdx.x; i < p.out_width; i += blockDim.x)
    p.table_out[b * p.out_width + i] = i < width ? p.table[b * p.table_row_stride + i] : 0;
  if (threadIdx.x == 0) {
    p.slots_out[b] = live ? p.slots[b] : p.pad_slot;
    p.lens_out[b] = live ? p.lens[b] : 0;
  }
}

}  // namespace

hipError_t launch_stage_decode(const StageParams& p, hipStream_t stream) {
  if (p.rows <= 0) return hipSuccess;
  hipLaunchKernelGGL(stage_decode_kernel, dim3(static_cast<unsigned>(p.rows)), dim3(256), 0, stream, p);
  return hipGetLastError();
}

}  // namespace nva
