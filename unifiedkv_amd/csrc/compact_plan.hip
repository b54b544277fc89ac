// Page lists of a block-aligned compaction (gfx950): small integer kernels between the selection and
// the page copy, each in place of a chain of elementwise launches.
//
//   ukv_retained_pages    selected middle blocks -> a layer's retained logical pages: the sink's, the
//                         selected ones shifted past it, the window's (core/scheduler.py:762-779)
//   ukv_compact_sources   retained logical pages -> physical source pages of every layer and sequence,
//                         side by side (core/scheduler.py:805-878: the ids a writeback gathers from)
//
// Both are a few KB of latency: the gain is in the launches (nine per sequence for the first, eight for
// the second). Out-of-range entries set a flag in host memory the device can write, which the caller
// reads after synchronising the stream: one wait per call, no copy back.
#include <algorithm>

#include "ukv_common.h"

namespace ukv {

struct RetainedArgs {
  const int32_t* sel;
  int64_t sel_stride;
  int k, n_mid, sink_blocks, obs_first, obs_blocks;
  int32_t* out;  // [layers][sink_blocks + k + obs_blocks]
  int32_t* bad;
};

// grid (column blocks, layers)
__global__ void __launch_bounds__(256) retained_pages_kernel(const RetainedArgs a) {
  const int n = a.sink_blocks + a.k + a.obs_blocks;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  int x = i;
  if (i >= a.sink_blocks + a.k) {
    x = a.obs_first + (i - a.sink_blocks - a.k);
  } else if (i >= a.sink_blocks) {
    x = a.sel[(int64_t)blockIdx.y * a.sel_stride + (i - a.sink_blocks)];
    if (x < 0 || x >= a.n_mid) *a.bad = 1;
    x += a.sink_blocks;
  }
  a.out[(int64_t)blockIdx.y * n + i] = x;
}

constexpr int kSeqsPerLaunch = 64;
struct SourcesArgs {
  const int32_t* keep[kSeqsPerLaunch];  // [layers][n_keep] logical pages
  int64_t keep_stride[kSeqsPerLaunch];
  int n_keep[kSeqsPerLaunch];
  int pages_at[kSeqsPerLaunch];  // the sequence's first entry in pages
  int n_pages[kSeqsPerLaunch];
  int out_at[kSeqsPerLaunch];    // its first column in out
  const int32_t* pages;          // the sequences' physical pages, one after another
  int32_t* out;                  // [layers][out_cols]
  int64_t out_cols;
  int32_t* bad;                  // [sequences of this launch]
};

// grid (column blocks, sequences of this launch, layers)
__global__ void __launch_bounds__(256) compact_sources_kernel(const SourcesArgs a) {
  const int s = blockIdx.y;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= a.n_keep[s]) return;
  const int p = a.keep[s][(int64_t)blockIdx.z * a.keep_stride[s] + i];
  const bool ok = (unsigned)p < (unsigned)a.n_pages[s];
  if (!ok) a.bad[s] = 1;
  a.out[(int64_t)blockIdx.z * a.out_cols + a.out_at[s] + i] = ok ? a.pages[a.pages_at[s] + p] : -1;
}

}  // namespace ukv

using namespace ukv;

extern "C" int ukv_retained_pages(const int32_t* sel, int layers, int64_t sel_layer_stride, int k, int n_mid,
                                  int sink_blocks, int obs_first, int obs_blocks, int32_t* out, int32_t* bad,
                                  ukv_stream_t stream) {
  if (layers < 0 || layers > 65535 || k < 0 || n_mid < 0 || sink_blocks < 0 || obs_first < 0 || obs_blocks < 0)
    return UKV_ERR_INVALID_ARGUMENT;
  const int64_t n = (int64_t)sink_blocks + k + obs_blocks;
  if (layers == 0 || n == 0) return UKV_OK;
  if (n > INT32_MAX - 256 || !out || !bad || (k > 0 && !sel)) return UKV_ERR_INVALID_ARGUMENT;
  const RetainedArgs a{sel, sel_layer_stride, k, n_mid, sink_blocks, obs_first, obs_blocks, out, bad};
  hipLaunchKernelGGL(retained_pages_kernel, dim3((unsigned)((n + 255) / 256), layers), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), a);
  return hipGetLastError() == hipSuccess ? UKV_OK : UKV_ERR_LAUNCH;
}

extern "C" int ukv_compact_sources(const void* const* keep, const int64_t* keep_layer_strides, const int32_t* n_keep,
                                   const int32_t* n_pages, int seqs, int layers, const int32_t* pages, int32_t* out,
                                   int64_t out_cols, int32_t* bad, ukv_stream_t stream) {
  if (seqs < 0 || layers < 0 || layers > 65535 || out_cols < 0) return UKV_ERR_INVALID_ARGUMENT;
  if (seqs == 0 || layers == 0) return UKV_OK;
  if (!keep || !keep_layer_strides || !n_keep || !n_pages) return UKV_ERR_INVALID_ARGUMENT;
  // Everything is checked before the first launch.
  int64_t cols = 0, total = 0;
  for (int s = 0; s < seqs; ++s) {
    if (n_keep[s] < 0 || n_pages[s] < 0 || (n_keep[s] > 0 && !keep[s])) return UKV_ERR_INVALID_ARGUMENT;
    cols += n_keep[s];
    total += n_pages[s];
  }
  if (cols == 0) return UKV_OK;
  if (cols > out_cols || cols > INT32_MAX - 256 || total > INT32_MAX || !out || !bad || (total > 0 && !pages))
    return UKV_ERR_INVALID_ARGUMENT;
  int pages_at = 0, out_at = 0;
  for (int s0 = 0; s0 < seqs; s0 += kSeqsPerLaunch) {
    SourcesArgs a{};
    const int ns = std::min(kSeqsPerLaunch, seqs - s0);
    int widest = 0;
    for (int i = 0; i < ns; ++i) {
      a.keep[i] = static_cast<const int32_t*>(keep[s0 + i]);
      a.keep_stride[i] = keep_layer_strides[s0 + i];
      a.n_keep[i] = n_keep[s0 + i];
      a.n_pages[i] = n_pages[s0 + i];
      a.pages_at[i] = pages_at;
      a.out_at[i] = out_at;
      pages_at += n_pages[s0 + i];
      out_at += n_keep[s0 + i];
      widest = std::max(widest, a.n_keep[i]);
    }
    a.pages = pages;
    a.out = out;
    a.out_cols = out_cols;
    a.bad = bad + s0;
    if (widest > 0)
      hipLaunchKernelGGL(compact_sources_kernel, dim3((widest + 255) / 256, ns, layers), dim3(256), 0,
                         reinterpret_cast<hipStream_t>(stream), a);
    if (hipGetLastError() != hipSuccess) return UKV_ERR_LAUNCH;
  }
  return UKV_OK;
}
