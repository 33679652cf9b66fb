// TOPK-32 of the LM head for gfx950 as a kernel of its own, over a y32
// vector already in memory: the scan of w4a8_topk_device.h, one wavefront per
// chunk (1024 rows; the first 256), four chunks (a run) per workgroup, one on
// each SIMD.  What bounds it is the chain of dependent lane exchanges and of
// trips through memory.  So a run's lists meet in LDS, only the run's list is
// published, and the list before a run is merged from the earlier runs' by
// all four wavefronts, a quarter each: one trip between workgroups, where a
// wavefront per workgroup and two levels of lists took two (the LM head
// with it, 248,320 x 4096: 102.3 -> 98.1 us).  Workgroups are dispatched in
// run order and a run only waits for lower-numbered runs, which publish
// before they wait, so the waits cannot deadlock.
#include "w4a8_topk_device.h"

namespace w4a8 {

namespace {

using namespace tk;

constexpr int kRun = 4;   // chunks, and wavefronts, of a workgroup
// the earlier runs' lists fall to kRun wavefronts, 16 each at most
constexpr int kMaxChunks = kRun * (16 * kRun + 1);
static_assert(kMaxChunks >= 1 + ((1 << 18) - kTkFirst + kTkRows - 1) / kTkRows &&
              kMaxChunks <= kTopkMaxChunks, "2^18 rows, within the flags");

// Flags (epoch > 0): pub[b] = epoch once run b's list is in part[b]; done[b] =
// 2 epoch + (run b's replay set the overflow bit).  Bit 3 of err: a wait gave
// up.
__global__ __launch_bounds__(64 * kRun) void topk_kernel(const int32_t *y, int64_t n, int nchunks,
                                                         int32_t epoch, uint64_t *part,
                                                         int32_t *flags, int32_t *out,
                                                         int32_t *err, uint32_t spin) {
  __shared__ uint64_t buf[kRun][128];
  __shared__ int32_t rows[kRun][kTkRows];
  __shared__ uint64_t lists[kRun][kTk], before[kRun][kTk];
  __shared__ int32_t over[kRun];
  int32_t *pub = flags, *done = flags + kTopkMaxChunks;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int b = blockIdx.x, c = b * kRun + wave;   // past nchunks: no rows
  const bool up = tk_ror4_up();
  const int64_t s0 = chunk_first(c), end = chunk_end(c, n);
  int32_t yv[kTkPerLane];   // rows s0 + lane + 64 t, loads all in flight
#pragma unroll
  for (int t = 0; t < kTkPerLane; ++t) {
    const int64_t r = s0 + lane + 64 * t;
    yv[t] = r < end ? y[r] : 0;
  }
  const uint64_t own = chunk_top32(yv, rows[wave], buf[wave], s0, end, up, lane);
  if (lane < kTk) lists[wave][lane] = own;
  __syncthreads();
  // all lanes take part in a merge; lanes 32..63 repeat the list
  const uint64_t o0 = lists[0][lane & 31], o1 = lists[1][lane & 31], o2 = lists[2][lane & 31];
  const uint64_t o01 = merge32v(o0, o1, up, lane);
  if (wave == kRun - 1) {
    const uint64_t S = merge32v(o01, merge32v(o2, own, up, lane), up, lane);
    if (lane < kTk) st_coh64(part + (int64_t)b * kTk + lane, S);
    wait_vm();
    if (lane == 0) st_coh32(pub + b, epoch);
  }
  // the list of the earlier chunks of this run ...
  const uint64_t W = wave == 0 ? 0 : wave == 1 ? o0 : wave == 2 ? o01 : merge32v(o01, o2, up, lane);
  // ... and of the earlier runs, a quarter of them per wavefront
  const int per = (b + kRun - 1) / kRun, j0 = min(wave * per, b), cnt = min(per, b - j0);
  bool ok = wait_words(pub + j0, cnt, [epoch](int32_t v) { return v == epoch; }, lane, spin);
  const uint64_t q = top32_lists(part + (int64_t)j0 * kTk, cnt, up, lane);
  if (lane < kTk) before[wave][lane] = q;
  __syncthreads();
  uint64_t pre = W;
  if (b > 0) {
    const uint64_t p01 = merge32v(before[0][lane & 31], before[1][lane & 31], up, lane);
    const uint64_t p23 = merge32v(before[2][lane & 31], before[3][lane & 31], up, lane);
    pre = merge32v(merge32v(p01, p23, up, lane), W, up, lane);
  }
  const int ovf = chunk_replay(pre, rows[wave], s0, end, up, lane);
  if (lane == 0) over[wave] = ovf;
  __syncthreads();
  const int any_run = over[0] | over[1] | over[2] | over[3];
  if (c == nchunks - 1) {
    const uint64_t whole = merge32v(pre, own, up, lane);
    ok = wait_words(done, b, [epoch](int32_t v) { return (v >> 1) == epoch; }, lane, spin) && ok;
    int f = any_run;
    for (int j = lane; j < b; j += 64) f |= ld_coh32(done + j) & 1;
    const bool any = __ballot(f != 0) != 0;
    const int count = n < kTk ? (int)n : kTk;
    if (lane < kTk) {
      const bool live = lane < count;
      out[lane] = live ? tk_val(whole) : 0;
      out[kTk + lane] = live ? (int32_t)tk_row(whole) : 0;
    }
    if (lane == 0) {
      out[2 * kTk] = count;
      out[2 * kTk + 1] = any ? 1 : 0;
    }
  }
  if (wave == 0 && lane == 0) st_coh32(done + b, 2 * epoch + any_run);
  if (!ok && lane == 0) atomicOr(err, 8);
}

}  // namespace

int topk_chunks(int64_t n) {
  using namespace tk;
  return n <= kTkFirst ? 1 : 1 + (int)((n - kTkFirst + kTkRows - 1) / kTkRows);
}

size_t topk_scratch_bytes(int64_t n) {
  return (size_t)(topk_chunks(n) + kTopkMaxChunks / kTopkSuper) * tk::kTk * 8;
}

hipError_t launch_topk32(const int32_t *y, int64_t n, void *scratch, int32_t *flags,
                         int32_t epoch, int32_t *out, int32_t *err, hipStream_t s,
                         uint32_t spin) {
  const int nchunks = topk_chunks(n);
  if (nchunks > kMaxChunks) return hipErrorInvalidValue;
  hipLaunchKernelGGL(topk_kernel, dim3((nchunks + kRun - 1) / kRun), dim3(64 * kRun), 0, s, y, n,
                     nchunks, epoch, (uint64_t *)scratch, flags, out, err,
                     spin ? spin : tk::kTkSpin);
  return hipGetLastError();
}

}  // namespace w4a8
