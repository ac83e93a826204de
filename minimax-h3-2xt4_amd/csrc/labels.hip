// AdaLN table row of every row of a DiT forward, from the segments that tile
// the rows. The segments travel in the kernel arguments, so the labels need
// no host-side array, no copy and no wait: built on the host, the copy from
// pageable memory waited for the whole stream, once or twice a layer.
#include "w8a8_host.h"

namespace w8a8 {

constexpr int kLabelSegments = 128;   // per launch (1 KB of arguments)

struct LabelTable {
  int32_t first;                  // first row of the launch
  int32_t count;
  int32_t end[kLabelSegments];    // ascending: segment i covers rows up to end[i]
  int32_t value[kLabelSegments];
};

// One row per thread: a binary search for its segment. Bound by the launch
// (53504 rows write 214 KB).
__global__ __launch_bounds__(256) void segment_labels_kernel(LabelTable t, int32_t* labels) {
  const int32_t row = t.first + (int32_t)(blockIdx.x * 256 + threadIdx.x);
  if (row >= t.end[t.count - 1]) return;
  int lo = 0, hi = t.count - 1;   // the first i with row < end[i]
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (row < t.end[mid]) hi = mid;
    else lo = mid + 1;
  }
  labels[row] = t.value[lo];
}

}  // namespace w8a8

extern "C" int w8a8_segment_labels(const int32_t* ends, const int32_t* values, int64_t count, int32_t* labels,
                                   int64_t rows, void* stream) {
  using namespace w8a8;
  W8A8_REQUIRE(count >= 0 && rows >= 0 && rows < (1LL << 31), "w8a8_segment_labels: bad size");
  if (rows == 0) return W8A8_OK;
  W8A8_REQUIRE(ends && values && labels && ((uintptr_t)labels & 3u) == 0, "w8a8_segment_labels: null or misaligned buffer");
  for (int64_t i = 0; i < count; ++i)
    W8A8_REQUIRE(ends[i] > (i ? ends[i - 1] : 0) && ends[i] <= rows, "w8a8_segment_labels: ends must ascend to rows");
  W8A8_REQUIRE(count > 0 && ends[count - 1] == rows, "w8a8_segment_labels: the segments must cover the rows");
  int32_t first = 0;
  for (int64_t i = 0; i < count; i += kLabelSegments) {
    LabelTable t{};
    t.first = first;
    t.count = (int32_t)(count - i < kLabelSegments ? count - i : kLabelSegments);
    for (int j = 0; j < t.count; ++j) {
      t.end[j] = ends[i + j];
      t.value[j] = values[i + j];
    }
    const int32_t last = t.end[t.count - 1];
    hipLaunchKernelGGL(segment_labels_kernel, dim3((unsigned)((last - first + 255) / 256)), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), t, labels);
    first = last;
  }
  return launch_status("w8a8_segment_labels");
}
