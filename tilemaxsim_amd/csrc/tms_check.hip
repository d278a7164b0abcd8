// Checks of document bounds on the device, and the entry points that check, score and
// return the verdict: one small kernel before the scoring kernel on the same stream, in
// place of a chain of elementwise passes and host copies. The check also leaves the longest
// scored document's length on the device, where the scoring kernel reads it (the
// zero-padding semantics need it), and there too whether the call is refused, so the host waits
// only for the check's verdict while the scoring kernel runs: PLAID's last stage over 1,024
// packed documents takes 19 us a call against 79, from a residual index of 100,000 documents 23
// against 157.
#include <time.h>

#include <atomic>

#include "tms_check.h"
#include "tms_verdict.h"

namespace tms {

constexpr int kCheckThreads = 1024;
constexpr int kCheckWaves = kCheckThreads / 64;
constexpr int64_t kCheckItems = 2048;  // offsets or pids per workgroup while all of them fit TMS_CHECK_PARTS
constexpr int kScanTiles = TMS_PACKED_SCAN_MAX / kCheckThreads;

__device__ __forceinline__ int64_t wave_max64(int64_t m) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const int64_t x = __shfl_xor(m, o);
    m = x > m ? x : m;
  }
  return m;
}

// The workgroup's maximum length and verdict: parts[blockIdx.x] (when given) for the scoring
// kernel, -1 there if the call is refused (it has a verdict, and it is bad), and the outcome with the check's tag into verdict[blockIdx.x], host memory, which the
// host waits for.
__device__ __forceinline__ void store_verdict(int64_t* word, int64_t tag, bool bad) {
  __hip_atomic_store(word, tag | (bad ? kVerdictBad : kVerdictFine), __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ __forceinline__ void publish(int64_t mx, bool bad, int64_t* parts, int64_t* verdict, int64_t tag) {
  __shared__ int64_t wmax[kCheckWaves];
  __shared__ uint32_t wbad[kCheckWaves];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  mx = wave_max64(mx);
  const uint64_t any = __ballot(bad);
  if (lane == 0) {
    wmax[wid] = mx;
    wbad[wid] = any != 0 ? 1u : 0u;
  }
  __syncthreads();
  if (wid != 0) return;
  mx = wave_max64(lane < kCheckWaves ? wmax[lane] : 0);
  const uint64_t all = __ballot(lane < kCheckWaves && wbad[lane] != 0u);
  if (lane == 0) {
    if (parts) parts[blockIdx.x] = verdict && all != 0 ? -1 : mx;
    if (verdict) store_verdict(verdict + blockIdx.x, tag, all != 0);
  }
}

// Offsets non-decreasing within [0, T] and pids (or null: documents 0 .. B-1) within [0,
// ndocs); the longest of the documents pids names. Bound by the read of the offsets at 16 MB
// (2M documents), by launch and one memory round trip at a few thousand.
__global__ void __launch_bounds__(kCheckThreads) docs_check_kernel(const int64_t* __restrict__ offsets, int64_t ndocs,
                                                                   const int64_t* __restrict__ pids, int64_t B,
                                                                   int64_t T, bool longest, int64_t* parts,
                                                                   int64_t* verdict, int64_t tag) {
  const int64_t first = (int64_t)blockIdx.x * kCheckThreads + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * kCheckThreads;
  bool bad = false;
  int64_t mx = 0;
#pragma unroll 4
  for (int64_t i = first; i < ndocs; i += stride) {
    const int64_t s = offsets[i], e = offsets[i + 1];
    bad |= e < s;
    if (!pids && i < B) mx = e - s > mx ? e - s : mx;
  }
  if (first == 0) bad |= offsets[0] < 0 || offsets[ndocs] > T;
  if (pids) {
#pragma unroll 4
    for (int64_t j = first; j < B; j += stride) {
      const int64_t p = pids[j];
      bad |= p < 0 || p >= ndocs;
      if (ndocs > 0) {
        const int64_t q = p < 0 ? 0 : (p >= ndocs ? ndocs - 1 : p);
        const int64_t len = offsets[q + 1] - offsets[q];
        mx = len > mx ? len : mx;
      }
    }
  }
  publish(longest ? mx : 0, bad, parts, verdict, tag);
}

// Lengths to offsets (B + 1) in one workgroup, with the checks of docs_check_kernel: each
// wave scans its 64 lengths of every 1,024, then the waves' sums are scanned.
__global__ void __launch_bounds__(kCheckThreads) lengths_scan_kernel(const int64_t* __restrict__ lengths, int64_t B,
                                                                     int64_t T, int64_t* __restrict__ offsets,
                                                                     bool longest, int64_t* parts, int64_t* verdict,
                                                                     int64_t tag) {
  __shared__ int64_t sums[kScanTiles * kCheckWaves];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int64_t len[kScanTiles], incl[kScanTiles];
  int64_t mx = 0;
#pragma unroll
  for (int t = 0; t < kScanTiles; t++) {
    const int64_t i = (int64_t)t * kCheckThreads + threadIdx.x;
    len[t] = i < B ? lengths[i] : 0;
  }
#pragma unroll
  for (int t = 0; t < kScanTiles; t++) {
    int64_t x = len[t];
    if ((int64_t)t * kCheckThreads < B) {  // uniform
      mx = x > mx ? x : mx;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int64_t y = __shfl_up(x, o);
        x = (int64_t)((uint64_t)x + (lane >= o ? (uint64_t)y : 0ull));  // wraps as the sum of int64s does
      }
    }
    incl[t] = x;
    if (lane == 63) sums[t * kCheckWaves + wid] = x;
  }
  __syncthreads();
  if (wid == 0) {  // kScanTiles * kCheckWaves / 64 consecutive sums per lane, made exclusive
    constexpr int kPer = kScanTiles * kCheckWaves / 64;
    uint64_t s[kPer], own = 0;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      s[k] = (uint64_t)sums[lane * kPer + k];
      own += s[k];
    }
    uint64_t x = own;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint64_t y = (uint64_t)__shfl_up((int64_t)x, o);
      x += lane >= o ? y : 0ull;
    }
    x -= own;
#pragma unroll
    for (int k = 0; k < kPer; k++) {
      sums[lane * kPer + k] = (int64_t)x;
      x += s[k];
    }
  }
  __syncthreads();
  bool bad = false;
  if (threadIdx.x == 0) offsets[0] = 0;
#pragma unroll
  for (int t = 0; t < kScanTiles; t++) {
    const int64_t i = (int64_t)t * kCheckThreads + threadIdx.x;
    if (i < B) {
      const int64_t e = (int64_t)((uint64_t)incl[t] + (uint64_t)sums[t * kCheckWaves + wid]);
      offsets[i + 1] = e;
      bad |= e < (int64_t)((uint64_t)e - (uint64_t)len[t]) || (i == B - 1 && e > T);
    }
  }
  publish(longest ? mx : 0, bad, parts, verdict, tag);
}

// Codes below K: every code as unsigned, compared with `limit` (K, or 2^(bits - 1) for signed
// codes if that is less, so a negative code is above it). One read of the codes: 16 bytes a
// lane and load, four loads in flight; the unaligned ends go element by element. Bound by
// that read (6.3 TB/s). A scoring call over 1,000 documents x 128 tokens of int32 codes takes
// 16 us with it and 62 with two reductions and two host copies in its place, over 100,000
// documents 276 and 593; of uint8 codes at K = 64 98 and 409.
template <int CB>
__device__ __forceinline__ bool codes_over(const u32x4& x, uint32_t limit) {
  bool over = false;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t w = x[i];
    if constexpr (CB == 4) {
      over |= w >= limit;
    } else if constexpr (CB == 2) {
      over |= (w & 0xffffu) >= limit || (w >> 16) >= limit;
    } else {  // limit <= 255: the top bit of each byte of s is set where (byte & 127) reaches the limit's low part
      const uint32_t low = w & 0x7f7f7f7fu;
      const uint32_t s = low + (limit <= 128u ? 128u - limit : 256u - limit) * 0x01010101u;
      over |= ((limit <= 128u ? s | w : s & w) & 0x80808080u) != 0u;
    }
  }
  return over;
}
template <int CB>
__global__ void __launch_bounds__(kCheckThreads) codes_check_kernel(const uint8_t* __restrict__ codes, int64_t count,
                                                                    uint32_t limit, bool marked, int64_t* verdict,
                                                                    int64_t tag) {
  const int64_t bytes = count * CB;
  int64_t head = (int64_t)((16u - ((uintptr_t)codes & 15u)) & 15u);
  if (head > bytes) head = bytes;
  const int64_t vecs = (bytes - head) / 16;
  const u32x4* __restrict__ body = (const u32x4*)(codes + head);
  const int64_t stride = (int64_t)gridDim.x * kCheckThreads;
  const int64_t first = (int64_t)blockIdx.x * kCheckThreads + threadIdx.x;
  bool bad = false;
  int64_t i = first;
  for (; i + 3 * stride < vecs; i += 4 * stride) {
    u32x4 x[4];
#pragma unroll
    for (int q = 0; q < 4; q++) x[q] = body[i + q * stride];
#pragma unroll
    for (int q = 0; q < 4; q++) bad |= codes_over<CB>(x[q], limit);
  }
  for (; i < vecs; i += stride) bad |= codes_over<CB>(body[i], limit);
  // the ends, fewer than 16 bytes each: one element a thread of the first workgroup
  const int64_t tail = head + vecs * 16, nhead = head / CB;
  if (first < 32) {
    const int64_t e = first < nhead ? first * CB : tail + (first - nhead) * CB;
    if (e + CB <= bytes) {
      uint32_t c;
      if constexpr (CB == 1) c = codes[e];
      else if constexpr (CB == 2) c = *(const uint16_t*)(codes + e);
      else c = *(const uint32_t*)(codes + e);
      bad |= c >= limit;
    }
  }
  if (!marked) {
    publish(0, bad, nullptr, verdict, tag);
  } else if (__ballot(bad) != 0ull && (threadIdx.x & 63) == 0) {
    store_verdict(verdict + 1, tag, true);
  }
}
// After a grid of more workgroups than there are verdict words: the words it wrote are final.
__global__ void check_done_kernel(int64_t* verdict, int64_t tag) { store_verdict(verdict, tag, false); }

static int check_parts(int64_t items) {
  const int64_t g = (items + kCheckItems - 1) / kCheckItems;
  return (int)(g < 1 ? 1 : (g > TMS_CHECK_PARTS ? TMS_CHECK_PARTS : g));
}

// Waits until the check's workgroups have written their verdicts: a spin on host memory,
// which sees them a microsecond or two after the kernel's stores, then short sleeps. Ends
// also when the stream has drained or failed without them.
static int wait_verdict(const char* fn, const int64_t* verdict, int64_t tag, int parts, hipStream_t st) {
  VerdictPoll poll{verdict, parts, tag};
  hipError_t e = hipSuccess;
  const VerdictState s = await_verdict(
      poll, 20000,
      [&]() {
        e = hipStreamQuery(st);
        // neither outcome may surface in a later launch's check: not ready is no error, and a
        // failure is reported here
        if (e != hipSuccess && hipPeekAtLastError() == e) (void)hipGetLastError();
        return e == hipErrorNotReady ? STREAM_BUSY : (e == hipSuccess ? STREAM_DRAINED : STREAM_FAILED);
      },
      []() {
        const timespec nap = {0, 20000};
        nanosleep(&nap, nullptr);
      });
  if (s != VERDICT_PENDING) return s == VERDICT_BAD ? TMS_ERR_BOUNDS : TMS_OK;
  if (e != hipSuccess) (void)hipStreamSynchronize(st);  // the words may go back to their pool after this call
  return fail(TMS_ERR_HIP, "%s: the bounds check did not finish: %s", fn, hipGetErrorString(e));
}

// Refuses a stream under capture (the host cannot wait for a verdict there) and gives the
// check its tag.
static int open_verdict(const char* fn, const int64_t* verdict, hipStream_t st, int64_t& tag) {
  static std::atomic<int64_t> sequence{0};
  tag = 0;
  if (!verdict) return TMS_OK;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  const hipError_t e = hipStreamIsCapturing(st, &cap);
  if (e != hipSuccess) {
    if (hipPeekAtLastError() == e) (void)hipGetLastError();  // reported here, not by a later launch's check
    return fail(TMS_ERR_HIP, "%s: whether the stream is under capture: %s", fn, hipGetErrorString(e));
  }
  if (cap != hipStreamCaptureStatusNone)
    return fail(TMS_ERR_HIP, "%s: the bounds check waits for the GPU and cannot run under stream capture", fn);
  tag = verdict_tag(sequence.fetch_add(1, std::memory_order_relaxed) + 1);
  return TMS_OK;
}

// The launch check of a check kernel. The error it finds may be an older call's and the kernel
// be on its way: its stores are let land before the caller has the words back.
static int check_launched(const char* what, const int64_t* verdict, hipStream_t st) {
  const int rc = check_launch(what);
  if (rc && verdict) (void)hipStreamSynchronize(st);
  return rc;
}

static int refuse(const char* fn, int rc) {
  return rc == TMS_ERR_BOUNDS ? fail(rc, "%s: document bounds or ids out of range", fn) : rc;
}

// The check's outcome first (as when it ran before the scoring call), then the scoring's.
static int close_verdict(const char* fn, const int64_t* verdict, int64_t tag, int parts, hipStream_t st, int scored) {
  if (!verdict) return scored;
  char why[512];
  keep_error(why, sizeof(why));
  const int rc = wait_verdict(fn, verdict, tag, parts, st);
  if (rc) return refuse(fn, rc);
  if (scored) set_error("%s", why);
  return scored;
}

}  // namespace tms

using namespace tms;

extern "C" {

int tms_maxsim_varlen_checked(const void* Qs, int64_t nQ, int64_t nq, int64_t d, const void* D_flat,
                              int64_t total_tokens, const int64_t* offsets, int64_t B, int zero_pad, int dtype,
                              float* out, int64_t* parts, int64_t* verdict, void* stream) {
  const char* fn = "tms_maxsim_varlen_checked";
  if (B < 1 || !offsets) return fail(TMS_ERR_INVALID, "%s: at least one document and its offsets", fn);
  if (zero_pad && !parts) return fail(TMS_ERR_INVALID, "%s: parts is NULL", fn);
  hipStream_t st = (hipStream_t)stream;
  int64_t tag;
  int rc = open_verdict(fn, verdict, st, tag);
  if (rc) return rc;
  const int g = check_parts(B);
  hipLaunchKernelGGL(docs_check_kernel, dim3(g), dim3(kCheckThreads), 0, st, offsets, B, nullptr, B, total_tokens,
                     zero_pad != 0, parts, verdict, tag);
  rc = check_launched("docs_check_kernel", verdict, st);
  if (rc) return rc;
  if (verdict && !parts && (rc = wait_verdict(fn, verdict, tag, g, st))) return refuse(fn, rc);
  rc = varlen_scores(fn, Qs, nQ, nq, d, D_flat, total_tokens, offsets, B, PadLen{0, parts, g, zero_pad != 0}, dtype, out, stream);
  return close_verdict(fn, verdict, tag, g, st, rc);
}

int tms_maxsim_packed_checked(const void* Q, int64_t nq, int64_t d, const void* D_packed, int64_t total_tokens,
                              const int64_t* lengths, int64_t B, int zero_pad, int dtype, float* out, int64_t* offsets,
                              int64_t* parts, int64_t* verdict, void* stream) {
  const char* fn = "tms_maxsim_packed_checked";
  if (B < 1 || !lengths || !offsets) return fail(TMS_ERR_INVALID, "%s: at least one document, its length and offsets", fn);
  if (B > TMS_PACKED_SCAN_MAX) return fail(TMS_ERR_UNSUPPORTED, "%s: more than %d documents", fn, TMS_PACKED_SCAN_MAX);
  if (zero_pad && !parts) return fail(TMS_ERR_INVALID, "%s: parts is NULL", fn);
  hipStream_t st = (hipStream_t)stream;
  int64_t tag;
  int rc = open_verdict(fn, verdict, st, tag);
  if (rc) return rc;
  hipLaunchKernelGGL(lengths_scan_kernel, dim3(1), dim3(kCheckThreads), 0, st, lengths, B, total_tokens, offsets,
                     zero_pad != 0, parts, verdict, tag);
  rc = check_launched("lengths_scan_kernel", verdict, st);
  if (rc) return rc;
  if (verdict && !parts && (rc = wait_verdict(fn, verdict, tag, 1, st))) return refuse(fn, rc);
  rc = varlen_scores(fn, Q, 1, nq, d, D_packed, total_tokens, offsets, B, PadLen{0, parts, 1, zero_pad != 0}, dtype, out, stream);
  return close_verdict(fn, verdict, tag, 1, st, rc);
}

int tms_maxsim_residual_checked(const void* Qs, int64_t nQ, int64_t nq, int64_t d, const void* centroids,
                                int64_t ncent, const void* bucket_weights, int nbits, const int32_t* codes,
                                const uint8_t* residuals, int64_t total_tokens, const int64_t* offsets, int64_t ndocs,
                                const int64_t* pids, int64_t B, int zero_pad, int batched, float* out, int64_t* parts,
                                int64_t* verdict, void* stream) {
  const char* fn = "tms_maxsim_residual_checked";
  if (B < 1 || ndocs < 0 || !offsets) return fail(TMS_ERR_INVALID, "%s: at least one document and the offsets", fn);
  if (!pids && B > ndocs) return fail(TMS_ERR_INVALID, "%s: B=%lld > ndocs=%lld without pids", fn, (long long)B,
                                      (long long)ndocs);
  if (zero_pad && !parts) return fail(TMS_ERR_INVALID, "%s: parts is NULL", fn);
  hipStream_t st = (hipStream_t)stream;
  int64_t tag;
  int rc = open_verdict(fn, verdict, st, tag);
  if (rc) return rc;
  const int g = check_parts(ndocs > B ? ndocs : B);
  hipLaunchKernelGGL(docs_check_kernel, dim3(g), dim3(kCheckThreads), 0, st, offsets, ndocs, pids, B, total_tokens,
                     zero_pad != 0, parts, verdict, tag);
  rc = check_launched("docs_check_kernel", verdict, st);
  if (rc) return rc;
  if (verdict && !parts && (rc = wait_verdict(fn, verdict, tag, g, st))) return refuse(fn, rc);
  rc = residual_scores(fn, Qs, nQ, nq, d, centroids, ncent, bucket_weights, nbits, codes, residuals, total_tokens, offsets,
                       ndocs, pids, B, PadLen{0, parts, g, zero_pad != 0}, batched != 0, out, stream);
  return close_verdict(fn, verdict, tag, g, st, rc);
}

// verdict[TMS_CHECK_PARTS - 1] is the host's: the check's tag with the words to wait for, 0 of
// them for a marked grid (word 0 says that it is done, word 1 that a code was out of range).
int tms_codes_check(const void* codes, int64_t count, int code_bytes, int64_t K, int64_t* verdict, void* stream) {
  const char* fn = "tms_codes_check";
  if (count < 1 || K < 0 || !codes || !verdict) return fail(TMS_ERR_INVALID, "%s: bad size or NULL pointer", fn);
  if (code_bytes != 1 && code_bytes != 2 && code_bytes != 4)
    return fail(TMS_ERR_INVALID, "%s: code_bytes must be 1, 2 or 4, got %d", fn, code_bytes);
  if ((uintptr_t)codes % code_bytes) return fail(TMS_ERR_INVALID, "%s: misaligned codes", fn);
  hipStream_t st = (hipStream_t)stream;
  int64_t tag;
  int rc = open_verdict(fn, verdict, st, tag);
  if (rc) return rc;
  const int64_t top = code_bytes == 1 ? 256 : (code_bytes == 2 ? 32768 : (int64_t)1 << 31);
  verdict[TMS_CHECK_PARTS - 1] = tag | 1;
  if (K >= top && code_bytes == 1) {  // every byte is a code
    verdict[0] = tag | kVerdictFine;
    return TMS_OK;
  }
  const uint32_t limit = (uint32_t)(K < top ? K : top);
  // up to 32 MiB the workgroups' own words will do; more bytes want more workgroups
  const int64_t bytes = count * code_bytes, want = (bytes + 16 * kCheckThreads * 4 - 1) / (16 * kCheckThreads * 4);
  const bool marked = bytes > ((int64_t)32 << 20);
  const int64_t most = marked ? 512 : TMS_CHECK_PARTS - 1;
  const int g = (int)(want < most ? want : most);
  verdict[TMS_CHECK_PARTS - 1] = tag | (marked ? 0 : g);
  const uint8_t* p = (const uint8_t*)codes;
  if (code_bytes == 1)
    hipLaunchKernelGGL(codes_check_kernel<1>, dim3(g), dim3(kCheckThreads), 0, st, p, count, limit, marked, verdict, tag);
  else if (code_bytes == 2)
    hipLaunchKernelGGL(codes_check_kernel<2>, dim3(g), dim3(kCheckThreads), 0, st, p, count, limit, marked, verdict, tag);
  else
    hipLaunchKernelGGL(codes_check_kernel<4>, dim3(g), dim3(kCheckThreads), 0, st, p, count, limit, marked, verdict, tag);
  if (marked) hipLaunchKernelGGL(check_done_kernel, dim3(1), dim3(1), 0, st, verdict, tag);
  return check_launched("codes_check_kernel", verdict, st);
}

int tms_codes_verdict(const int64_t* verdict, void* stream) {
  const char* fn = "tms_codes_verdict";
  if (!verdict) return fail(TMS_ERR_INVALID, "%s: NULL pointer", fn);
  const int64_t mark = verdict[TMS_CHECK_PARTS - 1], tag = mark & ~(int64_t)0xff;
  const int parts = (int)(mark & 0xff);
  int rc = wait_verdict(fn, verdict, tag, parts > 0 ? parts : 1, (hipStream_t)stream);
  if (rc == TMS_OK && parts == 0 && __atomic_load_n(verdict + 1, __ATOMIC_ACQUIRE) == (tag | kVerdictBad))
    rc = TMS_ERR_BOUNDS;
  return rc == TMS_ERR_BOUNDS ? fail(rc, "%s: codes out of range", fn) : rc;
}

}  // extern "C"
