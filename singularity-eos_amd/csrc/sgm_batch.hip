// One closure call as a batch, without a plan: the cells of a plain call are
// sorted by material count and signature on the device and solved by the
// batched kernels (register-resident bins with straggler parking, tails),
// bin bounds and record bases read on the device, so nothing comes back to
// the host. The work arrays come from the context's batch workspaces, or from
// the caller (the server's arena). What bounds a plain call over uneven cells
// is its slowest cell's chain of Newton passes: the plain kernel runs it on one
// lane, behind the wave's cells of other material counts and through every
// repeat of a fixed point. 20,011 uneven cells, RhoT at 1e-10: 96 -> 8.3 ms; 200
// cells 20 -> 1.5 ms; 3,001 cells PT 550 -> 88 ms.
#include "sgm_internal.hpp"

#include <hipcub/hipcub.hpp>

#include <algorithm>

namespace sgm {
// Lanes of a wave that take cells: all 64 once the cells fill `waves` waves
// with them, fewer below, where waves are plentiful and each pass of a wave
// costs the sum of its lanes' material kinds.
int batch_cells_per_wave(long ncell, long waves) {
  int c = 64;
  while (c > 4 && ncell < waves * c) c /= 2;
  return c;
}

namespace {

constexpr int NBIN = BATCH_BINS;  // material counts 2..6
constexpr int BATCH_PARK_AFTER = 20, BATCH_AFTER2 = 4;  // as plans

// From the sorted keys: per material count 2..6 {start, count} and the bin's
// record table (one run per bin: nrec records, or, with nrec 0, a record for
// each of its cells at the cells' own positions); range 0 the cells before them (fewer than 2 materials),
// range 6 those past the register-resident counts.
__global__ void batch_tables_kernel(const unsigned long long *__restrict__ keys, long n,
                                    int method, int nrec, long *__restrict__ range,
                                    BatchBin *__restrict__ bins) {
  __shared__ long pos[NBIN + 1];  // first position with a count of at least k + 2
  const int t = threadIdx.x, max_nm = BinMaxNM(method);
  if (t <= NBIN) {
    const unsigned long long k = (unsigned long long)min(t + 2, max_nm + 1) << 56;
    long lo = 0, hi = n;
    while (lo < hi) {
      const long mid = (lo + hi) >> 1;
      if (keys[mid] < k)
        lo = mid + 1;
      else
        hi = mid;
    }
    pos[t] = lo;
  }
  __syncthreads();
  if (t < NBIN) {
    const long start = pos[t], count = pos[t + 1] - start;
    range[2 * (t + 1)] = start;
    range[2 * (t + 1) + 1] = count;
    bins[t].first = nrec ? t * nrec : (int)start;
    bins[t].records = nrec ? nrec : (int)count;
    long word = 0;
    if (nrec)
      for (int k = 0; k < t; ++k) word += (long)nrec * ParkStride(method, k + 2);
    else
      word = start * ParkStride(method, max_nm);
    bins[t].word = word;
    bins[t].claimed = bins[t].next = bins[t].l2_count = bins[t].l2_next = 0;
  } else if (t == NBIN) {
    range[0] = 0;
    range[1] = pos[0];
    range[2 * NBIN + 2] = pos[NBIN];
    range[2 * NBIN + 3] = n - pos[NBIN];
  }
}

struct Layout {
  size_t keys, keys2, ids, sorted, range, bins, cell_of, rec, tmp, tmp_bytes, total;
};
// nrec: straggler records per bin; 0: one per cell
hipError_t layout(int method, long n, int nrec, Layout &L) {
  size_t o = 0;
  auto take = [&](size_t b) {
    const size_t at = o;
    o += (b + 255) / 256 * 256;
    return at;
  };
  L.keys = take(8 * (size_t)n);
  L.keys2 = take(8 * (size_t)n);
  L.ids = take(4 * (size_t)n);
  L.sorted = take(4 * (size_t)n);
  L.range = take(sizeof(long) * 2 * (NBIN + 2));
  L.bins = take(sizeof(BatchBin) * NBIN);
  const size_t recs = nrec ? (size_t)NBIN * nrec : (size_t)n;
  L.cell_of = take(4 * recs);
  size_t words = 0;  // one record per cell: a bin's start at its cells' positions
  for (int nm = 2; nm <= BinMaxNM(method); ++nm)
    words = nrec ? words + (size_t)ParkStride(method, nm) * nrec
                 : (size_t)ParkStride(method, nm) * n;
  L.rec = take(8 * words);
  size_t b = 0;
  const hipError_t e = hipcub::DeviceRadixSort::SortPairs(
      nullptr, b, (unsigned long long *)nullptr, (unsigned long long *)nullptr, (int *)nullptr,
      (int *)nullptr, (int)n, 0, 64, (hipStream_t) nullptr);
  L.tmp_bytes = b + 16;
  L.tmp = take(L.tmp_bytes);
  L.total = o;
  return e;
}

hipError_t enqueue(int method, const PteArgs &a, const MixParamsDev &P,
                   unsigned long long mod_mask, int nrec, const Layout &L, void *buf,
                   hipStream_t s) {
  char *base = static_cast<char *>(buf);
  auto *keys = (unsigned long long *)(base + L.keys);
  auto *keys2 = (unsigned long long *)(base + L.keys2);
  int *ids = (int *)(base + L.ids), *sorted = (int *)(base + L.sorted);
  long *range = (long *)(base + L.range);
  auto *bins = (BatchBin *)(base + L.bins);
  const int n = (int)a.ncell;
  hipError_t e =
      launch_plan_keys(a.offsets, a.mat_ids, n, a.nnz, keys, ids, s, nullptr, 0, mod_mask);
  if (e != hipSuccess) return e;
  size_t tb = L.tmp_bytes;
  e = hipcub::DeviceRadixSort::SortPairs(base + L.tmp, tb, keys, keys2, ids, sorted, n, 0, 64, s);
  if (e != hipSuccess) return e;
  batch_tables_kernel<<<1, 64, 0, s>>>(keys2, n, method, nrec, range, bins);
  if ((e = hipGetLastError()) != hipSuccess) return e;
  BatchArgs b;
  b.bins = bins;
  b.rec = (double *)(base + L.rec);
  b.cell_of = (int *)(base + L.cell_of);
  b.after = BATCH_PARK_AFTER;
  b.after2 = BATCH_AFTER2;
  e = launch_pte_batch_bins(method, a, P, b, sorted, range, n,
                            batch_cells_per_wave(n, 4L * device_cu_count()), s);
  for (int side = 0; side < 2 && e == hipSuccess; ++side)
    e = launch_pte_list(method, a, P, sorted, n, s, range + (side ? 2 * (NBIN + 1) : 0));
  return e;
}

} // namespace

void BatchWs::release() {
  if (done) {
    (void)hipEventSynchronize(done);
    (void)hipEventDestroy(done);
  }
  if (buf) (void)hipFree(buf);
  *this = BatchWs{};
}

size_t batch_bytes(int method, long n, int nrec) {
  Layout L;
  return layout(method, n, nrec, L) == hipSuccess ? L.total : 0;
}

hipError_t launch_batch(int method, const PteArgs &a, const MixParamsDev &P,
                        unsigned long long mod_mask, int nrec, void *buf, hipStream_t s) {
  Layout L;
  const hipError_t e = layout(method, a.ncell, nrec, L);
  return e != hipSuccess ? e : enqueue(method, a, P, mod_mask, nrec, L, buf, s);
}

namespace {
// allocation and event queries of this call stay out of a capture that the
// same thread holds open on another stream
struct RelaxedCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~RelaxedCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};
} // namespace

hipError_t launch_pte_batch(sgm_ctx *ctx, int method, const PteArgs &a, const MixParamsDev &P,
                            hipStream_t s, bool &taken) {
  taken = false;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) {
    (void)hipGetLastError();
    return hipSuccess;
  }
  const RelaxedCapture relaxed;
  const long chunk = std::min<long>(a.ncell, BATCH_MAX_CELLS);
  Layout L;
  if (layout(method, chunk, 0, L) != hipSuccess) return hipSuccess;
  std::lock_guard<std::mutex> g(ctx->batch_mu);
  // a workspace whose last call was on this stream or has finished, else a
  // new one, else the least recently used; its last call is waited for on the
  // stream in any case
  BatchWs *ws = nullptr, *fresh = nullptr, *oldest = nullptr;
  for (BatchWs &w : ctx->batch) {
    if (!w.done) {
      if (!fresh) fresh = &w;
      continue;
    }
    if (!oldest || w.used < oldest->used) oldest = &w;
    if ((w.last == s || hipEventQuery(w.done) == hipSuccess) && (!ws || w.bytes > ws->bytes))
      ws = &w;
  }
  (void)hipGetLastError();  // a query of unfinished work
  if (!ws) ws = fresh ? fresh : oldest;
  if (!ws->done && hipEventCreateWithFlags(&ws->done, hipEventDisableTiming) != hipSuccess) {
    (void)hipGetLastError();
    ws->done = nullptr;
    return hipSuccess;
  }
  if (ws->bytes < L.total) {
    // growing waits for the last call and for the device (hipFree): a quarter
    // of headroom, so that calls whose cells creep up pay it now and then
    // instead of at every new largest call (79 us of host time against 50, and
    // whatever else the device had in flight)
    const size_t more = std::min(ws->bytes + ws->bytes / 4,
                                 batch_bytes(method, BATCH_MAX_CELLS, 0));
    if (hipEventSynchronize(ws->done) != hipSuccess) return hipSuccess;
    if (ws->buf) (void)hipFree(ws->buf);
    ws->buf = nullptr;
    const size_t sizes[2] = {ws->bytes ? std::max(L.total, more) : L.total, L.total};
    ws->bytes = 0;
    for (size_t want : sizes) {
      if (hipMalloc(&ws->buf, want) == hipSuccess) {
        ws->bytes = want;
        break;
      }
      (void)hipGetLastError();
      ws->buf = nullptr;
    }
    if (!ws->buf) return hipSuccess;  // no room: the plain kernel needs none
  } else if (hipStreamWaitEvent(s, ws->done, 0) != hipSuccess) {
    return hipErrorUnknown;
  }
  ws->last = s;
  ws->used = ++ctx->batch_clock;
  taken = true;
  hipError_t e = hipSuccess;
  const unsigned long long mods = ctx_mod_mask(ctx);
  for (long c0 = 0; c0 < a.ncell && e == hipSuccess; c0 += chunk) {
    PteArgs b = a;
    b.ncell = std::min(chunk, a.ncell - c0);
    b.offsets += c0;
    b.vfrac_tot += c0;
    b.sie_tot += c0;
    if (b.Tnorm) b.Tnorm += c0;
    if (b.conv) b.conv += c0;
    if (b.niter) b.niter += c0;
    if (b.err) b.err += c0;
    if (b.resid) b.resid += c0;
    e = enqueue(method, b, P, mods, 0, L, ws->buf, s);
  }
  const hipError_t er = hipEventRecord(ws->done, s);
  return e != hipSuccess ? e : er;
}

} // namespace sgm
