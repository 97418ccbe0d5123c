// A step's inputs into the static buffers of its captured graph, in one launch:
// up to three tensors and a position (the copies of
// src/solort/model/cuda_graph_executor.py:195-206, :275-283).
//
// Bound: launch latency.  As a copy or fill each these were two to four small
// launches in a row ahead of the replay; here they are one, a workgroup per 4 KB
// of the tensors laid end to end.
// Measured on MI355X, one pass with its inputs: a token through 28 Qwen3-0.6B
// layers 137.7 -> 133.3 us, 36 Qwen3-4B layers 211.3 -> 206.4, a 5-token verify
// 381.8 -> 375.7.
#include "common.h"
#include "capi_internal.h"

namespace solort {

struct StageSeg {
  uint4* dst;
  const uint4* src;
  int64_t bytes;
};

__device__ __forceinline__ int64_t seg_chunks(const StageSeg& s) { return (s.bytes + 15) >> 4; }

__global__ __launch_bounds__(256) void stage_inputs_kernel(StageSeg a, StageSeg b, StageSeg c, int64_t* pos,
                                                           int64_t position) {
  int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i == 0) *pos = position;
  StageSeg s = a;
  if (i >= seg_chunks(s)) {
    i -= seg_chunks(s);
    s = b;
    if (i >= seg_chunks(s)) {
      i -= seg_chunks(s);
      s = c;
      if (i >= seg_chunks(s)) return;
    }
  }
  if (16 * i + 16 <= s.bytes) {
    s.dst[i] = s.src[i];
  } else {  // the tensor's last words
    const uint32_t* from = reinterpret_cast<const uint32_t*>(s.src);
    for (int64_t w = 4 * i; w < s.bytes >> 2; ++w) reinterpret_cast<uint32_t*>(s.dst)[w] = from[w];
  }
}

}  // namespace solort

using namespace solort;

extern "C" int solort_stage_inputs(void* dst0, const void* src0, int64_t bytes0, void* dst1, const void* src1,
                                   int64_t bytes1, void* dst2, const void* src2, int64_t bytes2, int64_t* pos,
                                   int64_t position, solort_stream_t stream) {
  const char* name = "stage_inputs";
  if (!pos || ((uintptr_t)pos & 7u)) return set_error(SOLORT_EINVAL, "%s: pos must be an 8-byte aligned pointer", name);
  const StageSeg seg[3] = {{(uint4*)dst0, (const uint4*)src0, bytes0},
                           {(uint4*)dst1, (const uint4*)src1, bytes1},
                           {(uint4*)dst2, (const uint4*)src2, bytes2}};
  int64_t chunks = 0;
  for (const StageSeg& s : seg) {
    if (s.bytes < 0 || s.bytes % 4 != 0 || s.bytes > ((int64_t)1 << 36))
      return set_error(SOLORT_EINVAL, "%s: bad size %lld (a multiple of 4)", name, (long long)s.bytes);
    if (s.bytes > 0 && (!s.dst || !s.src || !aligned16(s.dst) || !aligned16(s.src)))
      return set_error(SOLORT_EINVAL, "%s: tensors must be non-null and 16-byte aligned", name);
    chunks += (s.bytes + 15) >> 4;
  }
  const int64_t blocks = chunks > 0 ? (chunks + 255) / 256 : 1;
  hipLaunchKernelGGL(stage_inputs_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, seg[0], seg[1],
                     seg[2], pos, position);
  return check_launch(name);
}
