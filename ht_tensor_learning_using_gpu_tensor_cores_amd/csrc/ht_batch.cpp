// Host side of the batched entry point: validation, per-tensor descriptors and output
// layout, work-sorted order, launch-shape autotuning and the hipGraph of the launch.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "ht_engine.h"

using namespace ht;

namespace {

// Checks the tensors and describes each one (items may be null): tree {1},{2,3} in the heap
// numbering 0 = [0,3), 1 = [0,1), 2 = [1,3), 3 = [1,2), 4 = [2,3), whose rank conditions and
// packed layout (ht_output_layout's: U_1 U_3 U_4 B_0 B_2, singular values of nodes 1 to 4)
// are written out here; the general Problem::setup costs ~1 us a tensor.
int describe(int count, const int64_t* dims, const int32_t* ranks, std::vector<BatchItem>* items, int64_t* total,
             int64_t* offsets) {
  int64_t off = 0;
  if (items) items->resize(count);
  for (int b = 0; b < count; ++b) {
    const int64_t* d = dims + 3 * b;
    const int32_t* k = ranks + 5 * b;
    for (int m = 0; m < 3; ++m)
      if (d[m] < 1 || d[m] > BT_NMAX) return HT_ERR_UNSUPPORTED;
    for (int t = 1; t < 5; ++t)
      if (k[t] > BT_RMAX) return HT_ERR_UNSUPPORTED;
    const int64_t rows[5] = {0, d[0], d[1] * d[2], d[1], d[2]}, n = d[0] * d[1] * d[2];
    if (k[0] != 1) return HT_ERR_RANK;
    for (int t = 1; t < 5; ++t)
      if (k[t] < 1 || k[t] > rows[t] || k[t] > n / rows[t]) return HT_ERR_RANK;
    if (k[2] > k[3] * k[4]) return HT_ERR_RANK;
    const int u1 = 0, u3 = u1 + (int)d[0] * k[1], u4 = u3 + (int)d[1] * k[3], b0 = u4 + (int)d[2] * k[4];
    const int b2 = b0 + k[1] * k[2], s1 = b2 + k[3] * k[4] * k[2], s2 = s1 + k[1], s3 = s2 + k[2], s4 = s3 + k[3];
    if (offsets) offsets[b] = off;
    if (items) {
      BatchItem& it = (*items)[b];
      it = BatchItem{0, off, {(int)d[0], (int)d[1], (int)d[2]}, {k[0], k[1], k[2], k[3], k[4]},
                     {-1, u1, -1, u3, u4}, {b0, -1, b2, -1, -1}, {-1, s1, s2, s3, s4}, 0, 0};
    }
    off += s4 + k[4];
  }
  if (total) *total = off;
  return 0;
}

}  // namespace

ht_status ht_batch_output_layout(int32_t count, const int64_t* dims, const int32_t* ranks, int64_t* out_offsets,
                                 int64_t* total) {
  if (count < 1 || !dims || !ranks) return HT_ERR_INVALID_ARG;
  return (ht_status)describe(count, dims, ranks, nullptr, total, out_offsets);
}

ht_status ht_batch_shapes(int32_t count, uint64_t seed, int32_t lo, int32_t hi, int32_t rlo, int32_t rhi,
                          int64_t* dims, int32_t* core) {
  if (count < 1 || !dims || !core || lo < 1 || hi < lo || rlo < 1 || rhi < rlo) return HT_ERR_INVALID_ARG;
  // uniforms of stream 4095, six per tensor: three mode sizes then three Tucker ranks
  for (int b = 0; b < count; ++b)
    for (int m = 0; m < 3; ++m) {
      const double ud = philox_uniform(seed, 4095, (uint64_t)6 * b + m);
      const double ur = philox_uniform(seed, 4095, (uint64_t)6 * b + 3 + m);
      dims[3 * b + m] = std::min<int64_t>(lo + (int64_t)std::floor(ud * (hi - lo + 1)), hi);
      core[3 * b + m] = std::min<int32_t>(rlo + (int32_t)std::floor(ur * (rhi - rlo + 1)), rhi);
    }
  return HT_OK;
}

ht_status ht_generate_batch(ht_handle_t h, int32_t count, const int64_t* dims, const int32_t* core, uint64_t seed,
                            double noise_rel, float* x_dev, const int64_t* x_offsets) {
  if (!h || count < 1 || !dims || !core || !x_dev || !x_offsets || noise_rel < 0) return HT_ERR_INVALID_ARG;
  if (hipSetDevice(h->device) != hipSuccess) return HT_ERR_HIP;
  for (int b = 0; b < count; ++b) {
    const int64_t* d = dims + 3 * b;
    const int32_t* c = core + 3 * b;
    const uint32_t base = 4096u + 16u * (uint32_t)b;
    long nc = 1;
    for (int m = 0; m < 3; ++m) {
      if (d[m] < 1 || c[m] < 1 || c[m] > d[m]) return HT_ERR_INVALID_ARG;
      nc *= c[m];
    }
    std::vector<double> cv(nc);
    for (long i = 0; i < nc; ++i) cv[i] = philox_normal(seed, base, (uint64_t)i);
    std::vector<std::vector<double>> U(3);
    for (int m = 0; m < 3; ++m) U[m] = orthonormal_factor(seed, base + 1 + m, d[m], c[m]);
    ht_status s = generate_from_core(h, 3, d, c, std::move(cv), std::move(U), seed, noise_rel, x_dev + x_offsets[b],
                                     base + 15);
    if (s) return s;
  }
  return HT_OK;
}

ht_status ht_decompose_batched(ht_handle_t h, const float* x, int32_t count, const int64_t* dims,
                               const int32_t* ranks, const int64_t* x_offsets, float* out,
                               const int64_t* out_offsets, double* rel_err, ht_stats* stats) {
  if (!h || !x || !out || count < 1 || !dims || !ranks || !x_offsets || !out_offsets) return HT_ERR_INVALID_ARG;
  if (hipSetDevice(h->device) != hipSuccess) return HT_ERR_HIP;
  std::vector<BatchItem> items;
  int64_t total = 0;
  int s = describe(count, dims, ranks, &items, &total, nullptr);
  if (s) return (ht_status)s;
  std::vector<double> work(count);
  long gsize = 0, bsize = 0;
  int nrows[BT_NMAX + 1] = {};  // eigen problems by number of rows
  for (int b = 0; b < count; ++b) {
    BatchItem& it = items[b];
    it.x_off = x_offsets[b];
    it.out_off = out_offsets[b];
    const double n1 = it.n[0], n2 = it.n[1], n3 = it.n[2];
    work[b] = n1 * n2 * n3 * (n1 + n2 + n3);
    it.g_off = gsize;
    it.u_scr = bsize;
    for (int m = 0; m < 3; ++m) {
      gsize += (long)it.n[m] * it.n[m];
      ++nrows[it.n[m]];
    }
    bsize += batch_basis_size(it.n[0], it.n[1], it.n[2]);
  }
  // largest work first, so that the last work-groups are short
  std::vector<int> order(count);
  std::iota(order.begin(), order.end(), 0);
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return work[a] > work[b]; });
  // eigen problems, most rows first (a counting sort)
  BatchRun r{};
  int at[BT_NMAX + 1], pos = 0;
  for (int n = BT_NMAX; n >= 1; --n) {
    at[n] = pos;
    pos += nrows[n];
    r.eig_count[(n - 1) / 16] += nrows[n];
  }
  order.resize(4 * (size_t)count);
  for (int b = 0; b < count; ++b)
    for (int m = 0; m < 3; ++m) order[count + at[items[b].n[m]]++] = 4 * b + m;
  h->arena.reset();
  r.x = x;
  r.count = count;
  r.out = out;
  BatchItem* itd = (BatchItem*)h->arena.get(sizeof(BatchItem) * count);
  int* ord = (int*)h->arena.get(sizeof(int) * 4 * count);
  double* errd = (double*)h->arena.get(sizeof(double) * count);
  r.gram = (float*)h->arena.get(sizeof(float) * gsize);
  r.basis = (double*)h->arena.get(sizeof(double) * bsize);
  if (!itd || !ord || !errd || !r.gram || !r.basis) return HT_ERR_ALLOC;
  r.items = itd;
  r.order = ord;
  r.eig = ord + count;
  r.rel_err = errd;
  if (hipMemcpyAsync(itd, items.data(), sizeof(BatchItem) * count, hipMemcpyHostToDevice, h->stream) != hipSuccess ||
      hipMemcpyAsync(ord, order.data(), sizeof(int) * order.size(), hipMemcpyHostToDevice, h->stream) != hipSuccess)
    return HT_ERR_HIP;
  // The launch runs from a graph captured for these exact arguments once they come a second
  // time in a row; arguments that change from call to call (a new output each time) are
  // launched as they are, since capturing costs more than the launches it saves.
  std::vector<const void*> bkey = {x, itd, ord, out, errd, r.gram, r.basis, (const void*)(intptr_t)count};
  for (int c = 0; c < BT_CLASSES; ++c) bkey.push_back((const void*)(intptr_t)r.eig_count[c]);
  const bool again = h->bkey == bkey;
  if (!again) {
    if (h->bexec) (void)hipGraphExecDestroy(h->bexec);
    if (h->bgraph) (void)hipGraphDestroy(h->bgraph);
    h->bexec = nullptr;
    h->bgraph = nullptr;
    h->bkey = bkey;
  } else if (!h->bexec) {
    if (hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal) != hipSuccess) return HT_ERR_HIP;
    const int ls = batch_ht_launch(h->stream, r);
    const hipError_t ce = hipStreamEndCapture(h->stream, &h->bgraph);
    if (ls || ce != hipSuccess) return HT_ERR_HIP;
    if (hipGraphInstantiate(&h->bexec, h->bgraph, nullptr, nullptr, 0) != hipSuccess) return HT_ERR_HIP;
  }
  if (hipEventRecord(h->ev[0], h->stream) != hipSuccess) return HT_ERR_HIP;
  if (h->bexec ? hipGraphLaunch(h->bexec, h->stream) != hipSuccess : batch_ht_launch(h->stream, r) != 0)
    return HT_ERR_HIP;
  if (hipEventRecord(h->ev[1], h->stream) != hipSuccess) return HT_ERR_HIP;
  if (rel_err &&
      hipMemcpyAsync(rel_err, errd, sizeof(double) * count, hipMemcpyDeviceToHost, h->stream) != hipSuccess)
    return HT_ERR_HIP;
  if (hipStreamSynchronize(h->stream) != hipSuccess) return HT_ERR_HIP;
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, h->ev[0], h->ev[1]);
  if (stats) {
    std::memset(stats, 0, sizeof(*stats));
    stats->total_ms = ms;
    stats->bytes_x_passes = 4.0;
    stats->eig_calls = 3 * count;
  }
  return HT_OK;
}
