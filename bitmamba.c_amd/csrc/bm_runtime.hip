// Runtime of the BitLinear backend: lifecycle, weight registry, the
// dispatch-table entry points (host pointers, synchronous) and the
// device-pointer entry points.
//
// Threading: like the reference's Metal backend (src/metal/bm_metal.c:93-95)
// every entry point serializes on one process-wide mutex; the reference calls
// the dispatch-table kernels from its main thread only (src/block.c:362-370,
// src/model.c:1225, 1259).
#include <stdarg.h>
#include <stdlib.h>
#include <string.h>

#include <immintrin.h>

#include <chrono>
#include <mutex>
#include <new>
#include <unordered_map>
#include <vector>

#include "bm_common.h"
#include "bm_dev.h"
#include "bm_hip.h"
#include "bm_bit2.h"


static thread_local char g_err[512];

extern "C" void bm_set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

extern "C" const char* bm_hip_last_error(void) { return g_err; }

// Scratch of the allocation-free entry point bm_hip_bitlinear_noalloc_dev:
// a file-scope device array (each GPU holds its own copy until the process
// ends).  In host code `scratch` names a host-side stand-in, never device
// memory: kernels and copies get the address that hipGetSymbolAddress
// returns at set-up (Backend::scratch_dev).
constexpr size_t kScratchBytes = (size_t)8 << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

namespace bm {

// up to three runs of bytes at the same offsets of a device buffer and of
// mapped host memory, in slices of `slice` bytes, a block each
struct HostSlices {
  size_t off[3], bytes[3], slice;
  int first[3];  // the run's first block
};

__global__ __launch_bounds__(256) void k_to_host(HostSlices h, const uint8_t* __restrict__ src,
                                                 uint8_t* __restrict__ dst,
                                                 unsigned* __restrict__ flags, unsigned seq) {
  const int b = blockIdx.x;
  const int i = b >= h.first[2] ? 2 : (b >= h.first[1] ? 1 : 0);
  const size_t at = (size_t)(b - h.first[i]) * h.slice;
  const size_t n = min(h.slice, h.bytes[i] - at), base = h.off[i] + at;
  const uint8_t* __restrict__ p = src + base;
  uint8_t* __restrict__ q = dst + base;
  if (((uintptr_t)p | (uintptr_t)q) % 16 == 0) {
    const size_t n16 = n / 16;
#pragma unroll 4
    for (size_t k = threadIdx.x; k < n16; k += 256) ((uint4*)q)[k] = ((const uint4*)p)[k];
    for (size_t k = 16 * n16 + threadIdx.x; k < n; k += 256) q[k] = p[k];
  } else {
    for (size_t k = threadIdx.x; k < n; k += 256) q[k] = p[k];
  }
  // each wave waits for its own stores (the barrier does not), then the
  // release writes back what L2 holds of them before the word
  __asm__ __volatile__("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (threadIdx.x == 0)
    __hip_atomic_store(flags + b, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace bm

namespace {

constexpr int kMaxDevices = 16;

// calls whose inputs and outputs fit here skip the DMA copies: the kernels
// read x from, and write their results to, mapped host memory
constexpr size_t kZeroCopyMax = 256 * 1024;

struct DevBuf {
  void* ptr = nullptr;
  size_t bytes = 0;
  void* dev = nullptr;  // device address of a mapped host buffer
};

struct Registered {
  void* dev = nullptr;
  size_t bytes = 0;
};

struct Backend {
  std::mutex mu;
  bool ready = false;
  int device = 0;
  hipStream_t stream = nullptr;
  // weights and float vectors of registered model images, by host address
  // (an image registered with bm_hip_set_mmap must not change afterwards)
  std::unordered_map<const void*, Registered> packed;
  std::unordered_map<const void*, Registered> floats;
  // the last image bm_hip_set_mmap registered: the batch context's tensors
  // must lie inside it
  const uint8_t* mmap_base = nullptr;
  size_t mmap_size = 0;
  // grow-on-demand device scratch for the host-pointer entry points; d_w
  // and d_g receive tensors that belong to no registered image, per call
  DevBuf d_x, d_out, d_act, d_scale, d_w, d_g;
  // pinned host staging (copies), and mapped coherent host memory that
  // the kernels of small calls read and write directly
  DevBuf h_stage, h_zc;
  // device address of `scratch` on each device the library set up
  void* scratch_dev[kMaxDevices] = {};
  // one-launch calls at one token: the blocks' completion words (mapped
  // host memory) and the last sequence number handed out
  DevBuf h_flag;
  unsigned seq = 0;
};

// completion words of the one-launch path: one per block, which covers
// the 50257-row LM heads (786 blocks at K = 1024, 1571 at K = 2048)
constexpr int kDropInMaxBlocks = 2048;

Backend& B() {
  static Backend* b = new Backend();  // intentionally leaked: no static dtor
  return *b;
}

[[noreturn]] void die(const char* what) {
  fprintf(stderr, "Fatal: HIP BitLinear backend: %s: %s\n", what, g_err);
  exit(1);
}

bool ensure_dev(DevBuf& b, size_t bytes) {
  if (b.bytes >= bytes && b.ptr) return true;
  if (b.ptr) (void)hipFree(b.ptr);
  b.ptr = nullptr;
  b.bytes = 0;
  size_t want = bytes < 4096 ? 4096 : bytes + bytes / 4;
  BM_HIP_CHECK_RET(hipMalloc(&b.ptr, want), false);
  b.bytes = want;
  return true;
}

bool ensure_pinned(DevBuf& b, size_t bytes) {
  if (b.bytes >= bytes && b.ptr) return true;
  if (b.ptr) (void)hipHostFree(b.ptr);
  b = DevBuf{};
  size_t want = bytes < 65536 ? 65536 : bytes + bytes / 4;
  void* p = nullptr;
  BM_HIP_CHECK_RET(hipHostMalloc(&p, want, hipHostMallocMapped | hipHostMallocCoherent), false);
  void* d = nullptr;
  if (hipHostGetDevicePointer(&d, p, 0) != hipSuccess) {
    (void)hipHostFree(p);
    bm_set_error("hipHostGetDevicePointer failed");
    return false;
  }
  b.ptr = p;
  b.dev = d;
  b.bytes = want;
  return true;
}

bool ensure_mapped(DevBuf& b, size_t bytes) {
  if (b.bytes >= bytes && b.ptr) return true;
  if (b.ptr) (void)hipHostFree(b.ptr);
  b = DevBuf{};
  void* p = nullptr;
  BM_HIP_CHECK_RET(hipHostMalloc(&p, kZeroCopyMax, hipHostMallocMapped | hipHostMallocCoherent),
                   false);
  void* d = nullptr;
  if (hipHostGetDevicePointer(&d, p, 0) != hipSuccess) {
    (void)hipHostFree(p);
    bm_set_error("hipHostGetDevicePointer failed");
    return false;
  }
  b.ptr = p;
  b.dev = d;
  b.bytes = kZeroCopyMax;
  return bytes <= kZeroCopyMax;
}

// the completion words of the one-launch path, made once (zeroed)
bool ensure_dropin(Backend& b) {
  if (b.h_flag.ptr) return true;
  const size_t bytes = sizeof(unsigned) * kDropInMaxBlocks;
  void* p = nullptr;
  BM_HIP_CHECK_RET(hipHostMalloc(&p, bytes, hipHostMallocMapped | hipHostMallocCoherent), false);
  void* d = nullptr;
  if (hipHostGetDevicePointer(&d, p, 0) != hipSuccess) {
    (void)hipHostFree(p);
    bm_set_error("hipHostGetDevicePointer failed");
    return false;
  }
  memset(p, 0, bytes);
  b.h_flag.ptr = p;
  b.h_flag.dev = d;
  b.h_flag.bytes = bytes;
  return true;
}

// the next sequence number (never 0, the words' initial value; when the
// counter wraps the words are cleared first)
unsigned next_seq(Backend& b) {
  if (++b.seq == 0) {
    memset(b.h_flag.ptr, 0, b.h_flag.bytes);
    b.seq = 1;
  }
  return b.seq;
}

// Whether words[0..n) all hold seq.  The CPU reads mapped coherent memory
// without caching it (~30 ns per load whatever its width), so the words
// are compared 8 (AVX2) or 4 (SSE2) per load: 786 words take ~3 us instead
// of ~23 us one by one.
__attribute__((target("avx2"))) bool all_published_avx2(const unsigned* w, int n, unsigned seq) {
  const __m256i want = _mm256_set1_epi32((int)seq);
  int i = 0;
  for (; i + 8 <= n; i += 8) {
    const __m256i v = _mm256_load_si256((const __m256i*)(w + i));
    if (_mm256_movemask_epi8(_mm256_cmpeq_epi32(v, want)) != -1) return false;
  }
  for (; i < n; ++i)
    if (__atomic_load_n(w + i, __ATOMIC_ACQUIRE) != seq) return false;
  return true;
}

bool all_published_sse2(const unsigned* w, int n, unsigned seq) {
  const __m128i want = _mm_set1_epi32((int)seq);
  int i = 0;
  for (; i + 4 <= n; i += 4) {
    const __m128i v = _mm_load_si128((const __m128i*)(w + i));
    if (_mm_movemask_epi8(_mm_cmpeq_epi32(v, want)) != 0xffff) return false;
  }
  for (; i < n; ++i)
    if (__atomic_load_n(w + i, __ATOMIC_ACQUIRE) != seq) return false;
  return true;
}

bool all_published(const unsigned* w, int n, unsigned seq) {
  static const bool avx2 = __builtin_cpu_supports("avx2");
  const bool r = avx2 ? all_published_avx2(w, n, seq) : all_published_sse2(w, n, seq);
  __atomic_thread_fence(__ATOMIC_ACQUIRE);  // the results are read after the words
  return r;
}

// Waits until every block of the one-launch kernel has published `seq` (a
// stream synchronization costs ~5 us more than the kernel's own completion
// writes take to arrive): the blocks finish about in launch order, so the
// last block's word is polled alone, then all words are checked with wide
// loads.  After ~2 s of polling it falls back to synchronizing the stream,
// which reports a failed kernel.
hipError_t wait_flags(const unsigned* flags, int n, unsigned seq, hipStream_t s) {
  const auto t0 = std::chrono::steady_clock::now();
  for (unsigned i = 1;; ++i) {
    if (__atomic_load_n(flags + n - 1, __ATOMIC_ACQUIRE) == seq && all_published(flags, n, seq))
      return hipSuccess;
    if ((i & 4095) == 0 && std::chrono::steady_clock::now() - t0 > std::chrono::seconds(2)) break;
  }
  const hipError_t e = hipStreamSynchronize(s);
  if (e != hipSuccess) return e;
  if (all_published(flags, n, seq)) return hipSuccess;
  bm_set_error("a kernel finished without publishing every block's completion word");
  return hipErrorUnknown;
}

bool init_locked(Backend& b) {
  if (b.ready) return true;
  int n = 0;
  if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) {
    bm_set_error("no HIP device");
    return false;
  }
  hipDeviceProp_t prop;
  BM_HIP_CHECK_RET(hipGetDeviceProperties(&prop, 0), false);
  if (strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
    bm_set_error("device 0 is %s, the library targets gfx950 only", prop.gcnArchName);
    return false;
  }
  BM_HIP_CHECK_RET(hipSetDevice(0), false);
  BM_HIP_CHECK_RET(hipStreamCreateWithFlags(&b.stream, hipStreamNonBlocking), false);
  b.device = 0;
  // with device 0 current: the address of its copy of `scratch`
  void* sp = nullptr;
  BM_HIP_CHECK_RET(hipGetSymbolAddress(&sp, HIP_SYMBOL(scratch)), false);
  b.scratch_dev[0] = sp;
  b.ready = true;
  return true;
}

}  // namespace

namespace bm {

// Host -> device copies of caller memory go through pinned staging of the
// library's own (two 4 MiB halves used in turn, each reused once the copy
// out of it has completed): the runtime then never pins, registers or
// tracks the caller's pages, which may be a mapped model file that other
// threads of the caller read at the same time, and the source may be
// reused as soon as the call returns.
hipError_t upload(void* dst, const void* src, size_t bytes, hipStream_t s) {
  constexpr size_t kHalf = (size_t)4 << 20;
  static std::mutex mu;
  static uint8_t* stage = nullptr;
  static hipEvent_t done[2];
  static bool pending[2];
  std::lock_guard<std::mutex> lk(mu);
  if (!stage) {
    void* p = nullptr;
    hipError_t e = hipHostMalloc(&p, 2 * kHalf, hipHostMallocDefault);
    if (e != hipSuccess) return e;
    for (int k = 0; k < 2; ++k) {
      e = hipEventCreateWithFlags(&done[k], hipEventDisableTiming);
      if (e != hipSuccess) return e;
      pending[k] = false;
    }
    stage = (uint8_t*)p;
  }
  int k = 0;
  for (size_t off = 0; off < bytes; off += kHalf, k ^= 1) {
    const size_t n = bytes - off < kHalf ? bytes - off : kHalf;
    if (pending[k]) {
      const hipError_t e = hipEventSynchronize(done[k]);
      if (e != hipSuccess) return e;
      pending[k] = false;
    }
    memcpy(stage + k * kHalf, (const uint8_t*)src + off, n);
    hipError_t e = hipMemcpyAsync((uint8_t*)dst + off, stage + k * kHalf, n,
                                  hipMemcpyHostToDevice, s);
    if (e == hipSuccess) e = hipEventRecord(done[k], s);
    if (e != hipSuccess) return e;
    pending[k] = true;
  }
  return hipSuccess;
}

}  // namespace bm

namespace {

// Copies a packed tensor to an aligned device buffer and rewrites code 11.
const uint8_t* register_packed(Backend& b, const uint8_t* host, size_t bytes) {
  auto it = b.packed.find(host);
  if (it != b.packed.end() && it->second.bytes >= bytes) return (const uint8_t*)it->second.dev;
  if (it != b.packed.end()) {
    (void)hipFree(it->second.dev);
    b.packed.erase(it);
  }
  void* d = nullptr;
  BM_HIP_CHECK_RET(hipMalloc(&d, bytes ? bytes : 1), nullptr);
  BM_HIP_CHECK_RET(bm::upload(d, host, bytes, b.stream), nullptr);
  BM_HIP_CHECK_RET(bm::launch_canonicalize((uint8_t*)d, bytes, b.stream), nullptr);
  BM_HIP_CHECK_RET(hipStreamSynchronize(b.stream), nullptr);
  b.packed[host] = Registered{d, bytes};
  return (const uint8_t*)d;
}

// Device copy of a packed tensor for one call: the registered copy when the
// tensor belongs to a registered image, else a fresh upload into d_w (host
// memory outside an image may be reused for other data at any time, so it
// is never cached).
const uint8_t* packed_for_call(Backend& b, const uint8_t* host, size_t bytes) {
  auto it = b.packed.find(host);
  if (it != b.packed.end() && it->second.bytes >= bytes) return (const uint8_t*)it->second.dev;
  if (!ensure_dev(b.d_w, bytes ? bytes : 1)) return nullptr;
  BM_HIP_CHECK_RET(bm::upload(b.d_w.ptr, host, bytes, b.stream), nullptr);
  BM_HIP_CHECK_RET(bm::launch_canonicalize((uint8_t*)b.d_w.ptr, bytes, b.stream), nullptr);
  BM_HIP_CHECK_RET(hipStreamSynchronize(b.stream), nullptr);
  return (const uint8_t*)b.d_w.ptr;
}

const float* floats_for_call(Backend& b, const float* host, size_t count) {
  const size_t bytes = count * sizeof(float);
  auto it = b.floats.find(host);
  if (it != b.floats.end() && it->second.bytes >= bytes) return (const float*)it->second.dev;
  if (!ensure_dev(b.d_g, bytes ? bytes : 4)) return nullptr;
  BM_HIP_CHECK_RET(bm::upload(b.d_g.ptr, host, bytes, b.stream), nullptr);
  BM_HIP_CHECK_RET(hipStreamSynchronize(b.stream), nullptr);
  return (const float*)b.d_g.ptr;
}

const float* register_floats(Backend& b, const float* host, size_t count) {
  const size_t bytes = count * sizeof(float);
  auto it = b.floats.find(host);
  if (it != b.floats.end() && it->second.bytes >= bytes) return (const float*)it->second.dev;
  if (it != b.floats.end()) {
    (void)hipFree(it->second.dev);
    b.floats.erase(it);
  }
  void* d = nullptr;
  BM_HIP_CHECK_RET(hipMalloc(&d, bytes ? bytes : 4), nullptr);
  BM_HIP_CHECK_RET(bm::upload(d, host, bytes, b.stream), nullptr);
  BM_HIP_CHECK_RET(hipStreamSynchronize(b.stream), nullptr);
  b.floats[host] = Registered{d, bytes};
  return (const float*)d;
}

void bitlinear_check(int n, const struct tensor* w) {
  // BITLINEAR_CHECK (src/bitmamba.h:219-231)
  if (n != w->cols) {
    fprintf(stderr, "Fatal: bitlinear dim mismatch n=%d vs cols=%d\n", n, w->cols);
    exit(1);
  }
  if (!w->is_bitnet) {
    fprintf(stderr, "Fatal: bitlinear requires packed BitNet weights\n");
    exit(1);
  }
}

// results from here on are copied to `out` past the CPU's caches, as one large
// memcpy does by itself and one per slice does not: 2048 tokens, 1024 -> 4192
// (34 MB) 2.47 -> 2.00 ms (2.35 with one copy command and one memcpy), 1280
// tokens (21 MB) 1.30 against 1.28, 1024 (17 MB) 1.02 against 1.07
constexpr size_t kStreamedBytes = (size_t)24 << 20;

struct OutPart {
  size_t off, bytes;  // the same offset in the device buffer and the stage
};

// memcpy past the caches
void copy_streamed(uint8_t* d, const uint8_t* s, size_t n) {
  const size_t head = (16 - ((uintptr_t)d & 15)) & 15;
  if (n < head + 64) {
    memcpy(d, s, n);
    return;
  }
  memcpy(d, s, head);
  size_t i = head;
  for (; i + 64 <= n; i += 64) {
    const __m128i a = _mm_loadu_si128((const __m128i*)(s + i));
    const __m128i b = _mm_loadu_si128((const __m128i*)(s + i + 16));
    const __m128i c = _mm_loadu_si128((const __m128i*)(s + i + 32));
    const __m128i e = _mm_loadu_si128((const __m128i*)(s + i + 48));
    _mm_stream_si128((__m128i*)(d + i), a);
    _mm_stream_si128((__m128i*)(d + i + 16), b);
    _mm_stream_si128((__m128i*)(d + i + 32), c);
    _mm_stream_si128((__m128i*)(d + i + 48), e);
  }
  memcpy(d + i, s + i, n - i);
  _mm_sfence();
}

// The results of a host-pointer call: a kernel copies them to the stage (the
// caller's `out` first, part 0) in slices, a block each, and publishes every
// slice, so that the CPU copies one to `out` while the next ones travel; no
// copy commands, events or stream wait.  Bound by the bus and the CPU's one
// copying thread: 256 tokens, K = 1024 -> 4192 (4.3 MB of results) 330 -> 258
// us per call against one copy command, a wait and one copy by the CPU; copy
// commands in 512 KiB pieces with an event each were no faster than that.
hipError_t results_to_host(Backend& b, const OutPart (&part)[3], uint8_t* out, uint8_t* hs,
                           const uint8_t* dev, hipStream_t s) {
  // 64 KiB slices, more where that would take more blocks than words
  size_t slice = 64 * 1024, total = 0;
  for (const OutPart& p : part) total += p.bytes;
  while ((total + slice - 1) / slice + 3 > (size_t)kDropInMaxBlocks) slice *= 2;
  bm::HostSlices hsl{};
  int blocks = 0;
  for (int i = 0; i < 3; ++i) {
    hsl.off[i] = part[i].off;
    hsl.bytes[i] = part[i].bytes;
    hsl.first[i] = blocks;
    blocks += (int)((part[i].bytes + slice - 1) / slice);
  }
  hsl.slice = slice;
  const unsigned seq = next_seq(b);
  hipLaunchKernelGGL(bm::k_to_host, dim3(blocks), dim3(256), 0, s, hsl, dev,
                     (uint8_t*)b.h_stage.dev, (unsigned*)b.h_flag.dev, seq);
  hipError_t e = hipGetLastError();
  const bool streamed = part[0].bytes >= kStreamedBytes;
  const unsigned* flags = (const unsigned*)b.h_flag.ptr;
  for (int k = 0; k < blocks && e == hipSuccess; ++k) {
    e = wait_flags(flags + k, 1, seq, s);
    const size_t off = (size_t)k * slice;
    if (e == hipSuccess && off < part[0].bytes) {
      const size_t bytes = part[0].bytes - off < slice ? part[0].bytes - off : slice;
      if (streamed)
        copy_streamed(out + off, hs + part[0].off + off, bytes);
      else
        memcpy(out + off, hs + part[0].off + off, bytes);
    }
  }
  return e;
}

// Host-pointer batch BitLinear: quantize + product on the device, results
// copied back.  Any HIP failure is fatal (never zero outputs silently).
void host_bitlinear(const float* x, int M, int n, const uint8_t* packed, int rows, int cols,
                    float w_scale, const float* norm_w, float* out, float* x_norm_buf,
                    int8_t* x_quant, int quant_stride) {
  Backend& b = B();
  std::lock_guard<std::mutex> lk(b.mu);
  if (!init_locked(b)) die("init");
  if (M <= 0) return;
  const size_t wbytes = (size_t)rows * (size_t)((cols + 3) / 4);
  const uint8_t* dW = packed_for_call(b, packed, wbytes);
  const float* dG = floats_for_call(b, norm_w, (size_t)n);
  if (!dW || !dG) die("weight upload");

  const size_t xbytes = (size_t)M * n * sizeof(float);
  const size_t obytes = (size_t)M * rows * sizeof(float);
  const size_t qbytes = (size_t)M * n;
  const size_t abytes = (size_t)M * bm::act_row_bytes(n);
  // the results, [out | x_norm | int8] at 256-byte aligned offsets, the same in
  // the device buffer and the pinned stage
  const size_t o_norm = bm::align_up(obytes, 256), o_q = o_norm + bm::align_up(xbytes, 256);
  const size_t iobytes = o_q + qbytes;
  if (!ensure_dev(b.d_out, iobytes) || !ensure_dev(b.d_act, abytes) ||
      !ensure_dev(b.d_scale, (size_t)M * 4))
    die("scratch allocation");
  if (!ensure_pinned(b.h_stage, xbytes > iobytes ? xbytes : iobytes)) die("pinned staging");
  if (!ensure_dropin(b)) die("completion words");

  // small calls: [x | out | x_norm | int8] in mapped host memory, no copies
  const size_t o_x = bm::align_up(iobytes, 256);
  const bool zc = o_x + xbytes <= kZeroCopyMax && ensure_mapped(b.h_zc, o_x + xbytes);
  uint8_t* hs = zc ? (uint8_t*)b.h_zc.ptr : (uint8_t*)b.h_stage.ptr;
  uint8_t* dio = zc ? (uint8_t*)b.h_zc.dev : (uint8_t*)b.d_out.ptr;
  // the quantizers up to n = 8192 read x once: straight from the stage (258
  // against 284 us per call of 256 tokens with a copy command); beyond, one
  // that reads it three times, from a device copy
  const bool copy_x = !zc && n > 8192;
  if (copy_x && !ensure_dev(b.d_x, xbytes)) die("scratch allocation");
  const float* dx = zc       ? (const float*)(dio + o_x)
                    : copy_x ? (const float*)b.d_x.ptr
                             : (const float*)b.h_stage.dev;
  hipStream_t s = b.stream;
  hipError_t e = hipSuccess;
  bool out_done = false;
  memcpy(zc ? hs + o_x : hs, x, xbytes);
  if (copy_x) e = hipMemcpyAsync(b.d_x.ptr, hs, xbytes, hipMemcpyHostToDevice, s);
  const bool generic = bm::product_needs_generic(M, cols);
  const int nblk = M == 1 && bm::rows_fit(n) ? bm::dropin_blocks(rows, n) : 0;
  if (zc && nblk > 0 && nblk <= kDropInMaxBlocks && ensure_dropin(b)) {
    // one token on mapped memory: RMSNorm, int8 and the GEMV in one launch
    // whose blocks publish their completion to the host
    const unsigned seq = next_seq(b);
    if (e == hipSuccess)
      e = bm::launch_dropin(dx, n, dG, dW, rows, w_scale, (float*)dio, (float*)(dio + o_norm),
                            (int8_t*)(dio + o_q), (unsigned*)b.h_flag.dev, seq, s);
    if (e == hipSuccess) e = wait_flags((const unsigned*)b.h_flag.ptr, nblk, seq, s);
  } else {
    if (e == hipSuccess)
      e = bm::launch_quantize(dx, M, n, n, dG, (float*)(dio + o_norm), (int8_t*)(dio + o_q), n,
                              (float*)b.d_scale.ptr, generic ? nullptr : (uint8_t*)b.d_act.ptr,
                              s);
    if (e == hipSuccess) {
      if (generic)
        e = bm::launch_generic((const int8_t*)(dio + o_q), n, (const float*)b.d_scale.ptr, M, dW,
                               rows, cols, w_scale, dio, bm::MODE_STORE, s, zc);
      else
        e = bm::launch_product((const uint8_t*)b.d_act.ptr, (const float*)b.d_scale.ptr, M, dW,
                               rows, cols, w_scale, true, dio, bm::MODE_STORE, s);
    }
    if (e == hipSuccess && !zc) {
      // x_norm leaves for the last token only
      const size_t last = o_norm + (size_t)(M - 1) * n * sizeof(float);
      const OutPart part[3] = {{0, obytes}, {last, x_norm_buf ? (size_t)n * 4 : 0},
                               {o_q, x_quant ? qbytes : 0}};
      e = results_to_host(b, part, (uint8_t*)out, hs, dio, s);
      out_done = e == hipSuccess;
    }
    if (e == hipSuccess && !out_done) e = hipStreamSynchronize(s);
  }
  if (e != hipSuccess) {
    bm_set_error("%s", hipGetErrorString(e));
    die("bitlinear");
  }
  if (!out_done) memcpy(out, hs, obytes);
  // x_norm_buf is a single n-vector reused per token: the last token stays
  if (x_norm_buf)
    memcpy(x_norm_buf, hs + o_norm + (size_t)(M - 1) * n * sizeof(float), (size_t)n * 4);
  if (x_quant)
    for (int m = 0; m < M; ++m)
      memcpy(x_quant + (size_t)m * quant_stride, hs + o_q + (size_t)m * n, (size_t)n);
}

}  // namespace

// ---------------------------------------------------------------------------
// Lifecycle
// ---------------------------------------------------------------------------
extern "C" bool bm_hip_init(void) {
  Backend& b = B();
  std::lock_guard<std::mutex> lk(b.mu);
  return init_locked(b);
}

extern "C" bool bm_hip_available(void) {
  Backend& b = B();
  std::lock_guard<std::mutex> lk(b.mu);
  return b.ready;
}

extern "C" bool bm_hip_set_mmap(const void* base, size_t size) {
  Backend& b = B();
  std::lock_guard<std::mutex> lk(b.mu);
  if (!init_locked(b)) return false;
  b.mmap_base = (const uint8_t*)base;
  b.mmap_size = size;
  bm_bit2_view_t v;
  if (bm_bit2_parse(base, size, &v) != 0) {
    // not a BIT2 image: tensors are uploaded lazily on first use
    return true;
  }
  // what the table's entries read: the packed BitLinear weights and their
  // norms (in_proj.norm, out_proj.norm, lm_head.norm) and norm_f; not the
  // embedding (vocab x d_model floats the decode reads on the CPU) nor the
  // SSM parameters
  const int first_tail = 1 + BM_L_COUNT * v.n_layers;
  for (int i = 0; i < v.n_tensors; ++i) {
    const bm_bit2_tensor_t* t = &v.tensors[i];
    const int which = (i - 1) % BM_L_COUNT;
    const bool norm = i >= first_tail ||
                      (i >= 1 && (which == BM_L_IN_NORM || which == BM_L_OUT_NORM));
    if (t->is_bitnet) {
      if (!register_packed(b, t->packed, (size_t)t->rows * (size_t)((t->cols + 3) / 4))) {
        bm_bit2_view_free(&v);
        return false;
      }
    } else if (norm && !register_floats(b, t->data, t->n_elements)) {
      bm_bit2_view_free(&v);
      return false;
    }
  }
  bm_bit2_view_free(&v);
  return true;
}

extern "C" void bm_hip_cleanup(void) {
  Backend& b = B();
  std::lock_guard<std::mutex> lk(b.mu);
  if (!b.ready) return;
  (void)hipStreamSynchronize(b.stream);
  for (auto& kv : b.packed) (void)hipFree(kv.second.dev);
  for (auto& kv : b.floats) (void)hipFree(kv.second.dev);
  b.packed.clear();
  b.floats.clear();
  b.mmap_base = nullptr;
  b.mmap_size = 0;
  for (DevBuf* d : {&b.d_x, &b.d_out, &b.d_act, &b.d_scale, &b.d_w, &b.d_g}) {
    if (d->ptr) (void)hipFree(d->ptr);
    *d = DevBuf{};
  }
  for (DevBuf* h : {&b.h_stage, &b.h_zc, &b.h_flag}) {
    if (h->ptr) (void)hipHostFree(h->ptr);
    *h = DevBuf{};
  }
  (void)hipStreamDestroy(b.stream);
  b.stream = nullptr;
  b.ready = false;
}

// ---------------------------------------------------------------------------
// Dispatch-table entry points
// ---------------------------------------------------------------------------
extern "C" float hip_rms_norm(const float* x, int size, const float* weight, float* out) {
  Backend& b = B();
  std::lock_guard<std::mutex> lk(b.mu);
  if (!init_locked(b)) die("init");
  const float* dG = floats_for_call(b, weight, (size_t)size);
  const size_t xbytes = (size_t)size * sizeof(float);
  // out and max|out| leave in one copy: [out | max]
  if (!dG || !ensure_dev(b.d_x, xbytes) || !ensure_dev(b.d_out, xbytes + 16) ||
      !ensure_pinned(b.h_stage, xbytes + 16))
    die("rms_norm scratch");
  uint8_t* hs = (uint8_t*)b.h_stage.ptr;
  uint8_t* dio = (uint8_t*)b.d_out.ptr;
  memcpy(hs, x, xbytes);
  hipStream_t s = b.stream;
  hipError_t e = hipMemcpyAsync(b.d_x.ptr, hs, xbytes, hipMemcpyHostToDevice, s);
  if (e == hipSuccess)
    e = bm::launch_rms_norm((const float*)b.d_x.ptr, size, dG, (float*)dio,
                            (float*)(dio + xbytes), s);
  if (e == hipSuccess) e = hipMemcpyAsync(hs, dio, xbytes + 4, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    bm_set_error("%s", hipGetErrorString(e));
    die("rms_norm");
  }
  memcpy(out, hs, xbytes);
  float mx;
  memcpy(&mx, hs + xbytes, 4);
  return mx;
}

extern "C" void hip_bitlinear_forward(const float* x, int n, const struct tensor* w,
                                      const struct tensor* norm_w, float* out, float* x_norm_buf,
                                      int8_t* x_quant_buf) {
  bitlinear_check(n, w);
  host_bitlinear(x, 1, n, w->packed_data, w->rows, w->cols, w->scale, norm_w->data, out,
                 x_norm_buf, x_quant_buf, n);
}

extern "C" void hip_bitlinear_forward_batch(const float* x_batch, int n_tokens, int n,
                                            const struct tensor* w, const struct tensor* norm_w,
                                            float* out_batch, float* x_norm_buf,
                                            int8_t* x_quant_batch, int quant_stride) {
  bitlinear_check(n, w);
  host_bitlinear(x_batch, n_tokens, n, w->packed_data, w->rows, w->cols, w->scale, norm_w->data,
                 out_batch, x_norm_buf, x_quant_batch, quant_stride);
}

extern "C" void bm_hip_bitlinear_forward_batch(const float* x_batch, int n_tokens, int n,
                                               const uint8_t* packed_data, int rows, int cols,
                                               float w_scale, const float* norm_weight,
                                               float* out_batch, float* x_norm_buf,
                                               int8_t* x_quant_batch, int quant_stride) {
  if (n != cols) {
    fprintf(stderr, "Fatal: bitlinear dim mismatch n=%d vs cols=%d\n", n, cols);
    exit(1);
  }
  host_bitlinear(x_batch, n_tokens, n, packed_data, rows, cols, w_scale, norm_weight, out_batch,
                 x_norm_buf, x_quant_batch, quant_stride);
}

extern "C" bool bm_hip_register(bm_hip_dispatch_t* t) {
  if (!t || !bm_hip_init()) return false;
  t->rms_norm = (void*)&hip_rms_norm;
  t->bitlinear_forward = (void*)&hip_bitlinear_forward;
  t->bitlinear_forward_batch = (void*)&hip_bitlinear_forward_batch;
  t->bitlinear_prepare = nullptr;
  t->bitlinear_row_worker = nullptr;
  t->name = "hip";
  return true;
}

// ---------------------------------------------------------------------------
// Batch context (src/metal/bm_metal.h:57-99, src/metal/bm_metal.c:610-960):
// persistent activation buffers, BitLinear and residual steps encoded
// without running, and one submit that runs them in order.  Metal shares
// its buffers with the CPU; here each buffer is a device buffer with a
// pinned host copy, the pointer bm_hip_batch_ptr returns.  A submit copies
// to the device what its steps read before any of them writes it (the
// host copy then holds the caller's latest values), runs the steps on one
// stream, copies back what they wrote, and waits: at every submit boundary
// the host copies are what Metal's shared buffers would hold.  Every buffer
// region a step touches starts at the buffer's first float (n_tokens rows
// of the step's width), so what a submit reads and writes is a prefix.
// ---------------------------------------------------------------------------
struct bm_hip_batch_ctx {
  struct Op {
    bool residual;
    int src, dst, input_dim, rows, cols, count;
    float w_scale;
    const uint8_t* dW;
    const float* dG;
  };
  int n_tokens = 0, d_model = 0, max_proj = 0, d_inner = 0, quant_stride = 0;
  size_t width[4] = {};  // floats per token of X, PROJ, Y, OUT
  float* host[4] = {};
  float* dev[4] = {};
  uint8_t* act = nullptr;  // activation workspace, scales, int8 rows
  float* scale = nullptr;
  int8_t* xq = nullptr;
  std::vector<Op> ops;
};

namespace {

void batch_free(bm_hip_batch_ctx_t* c) {
  for (int i = 0; i < 4; ++i) {
    if (c->host[i]) (void)hipHostFree(c->host[i]);
    if (c->dev[i]) (void)hipFree(c->dev[i]);
  }
  if (c->act) (void)hipFree(c->act);
  if (c->scale) (void)hipFree(c->scale);
  if (c->xq) (void)hipFree(c->xq);
  delete c;
}

}  // namespace

extern "C" bm_hip_batch_ctx_t* bm_hip_batch_begin(int n_tokens, int d_model, int max_proj,
                                                  int d_inner, int quant_stride) {
  Backend& b = B();
  std::lock_guard<std::mutex> lk(b.mu);
  if (!b.ready) {
    bm_set_error("batch_begin: backend not initialized (bm_hip_init)");
    return nullptr;
  }
  if (n_tokens <= 0 || d_model <= 0 || max_proj <= 0 || d_inner <= 0 || quant_stride < 0) {
    bm_set_error("batch_begin: invalid dimensions (n_tokens=%d d_model=%d max_proj=%d "
                 "d_inner=%d)", n_tokens, d_model, max_proj, d_inner);
    return nullptr;
  }
  auto* c = new (std::nothrow) bm_hip_batch_ctx_t();
  if (!c) return nullptr;
  c->n_tokens = n_tokens;
  c->d_model = d_model;
  c->max_proj = max_proj;
  c->d_inner = d_inner;
  c->quant_stride = quant_stride;
  const size_t widths[4] = {(size_t)d_model, (size_t)max_proj, (size_t)d_inner, (size_t)d_model};
  const int kmax = d_model > d_inner ? d_model : d_inner;
  bool ok = true;
  for (int i = 0; i < 4 && ok; ++i) {
    c->width[i] = widths[i];
    const size_t bytes = (size_t)n_tokens * widths[i] * sizeof(float);
    ok = hipHostMalloc((void**)&c->host[i], bytes, hipHostMallocDefault) == hipSuccess &&
         hipMalloc((void**)&c->dev[i], bytes) == hipSuccess;
    if (ok) memset(c->host[i], 0, bytes);
  }
  ok = ok && hipMalloc((void**)&c->act, (size_t)n_tokens * bm::act_row_bytes(kmax)) == hipSuccess &&
       hipMalloc((void**)&c->scale, (size_t)n_tokens * sizeof(float)) == hipSuccess &&
       hipMalloc((void**)&c->xq, (size_t)n_tokens * kmax) == hipSuccess;
  if (!ok) {
    bm_set_error("batch_begin: allocation failed (n_tokens=%d)", n_tokens);
    batch_free(c);
    return nullptr;
  }
  return c;
}

extern "C" float* bm_hip_batch_ptr(bm_hip_batch_ctx_t* ctx, int buf_id) {
  if (!ctx || buf_id < BM_HIP_BUF_X || buf_id > BM_HIP_BUF_OUT) return nullptr;
  return ctx->host[buf_id];
}

extern "C" bool bm_hip_encode_bitlinear(bm_hip_batch_ctx_t* ctx, int src_id, int input_dim,
                                        const uint8_t* packed_data, int rows, int cols,
                                        float w_scale, const float* norm_weight, int dst_id) {
  if (!ctx || !packed_data) return false;
  if ((src_id != BM_HIP_BUF_X && src_id != BM_HIP_BUF_Y) ||
      (dst_id != BM_HIP_BUF_PROJ && dst_id != BM_HIP_BUF_OUT))
    return false;
  if (cols % 16 != 0) {
    fprintf(stderr, "[HIP] encode: cols=%d not multiple of 16\n", cols);
    return false;
  }
  Backend& b = B();
  std::lock_guard<std::mutex> lk(b.mu);
  if (!b.mmap_base) return false;
  const uint8_t* w_ptr = packed_data;
  const uint8_t* n_ptr = (const uint8_t*)norm_weight;
  const uint8_t* mmap_end = b.mmap_base + b.mmap_size;
  if (w_ptr < b.mmap_base || n_ptr < b.mmap_base || w_ptr >= mmap_end || n_ptr >= mmap_end) {
    fprintf(stderr, "[HIP] encode: pointer outside mmap region\n");
    return false;
  }
  const size_t weight_bytes = (size_t)rows * (size_t)((cols + 3) / 4);
  const size_t norm_bytes = (size_t)input_dim * sizeof(float);
  if (rows <= 0 || input_dim <= 0 || weight_bytes > (size_t)(mmap_end - w_ptr) ||
      norm_bytes > (size_t)(mmap_end - n_ptr)) {
    fprintf(stderr, "[HIP] encode: tensor data exceeds mmap region\n");
    return false;
  }
  // beyond Metal's checks: the norm covers the product's columns, and the
  // rows fit the buffers (Metal's kernels would run past them)
  if (input_dim != cols || (size_t)input_dim > ctx->width[src_id] ||
      (size_t)rows > ctx->width[dst_id]) {
    fprintf(stderr, "[HIP] encode: input_dim=%d cols=%d rows=%d do not fit the batch buffers\n",
            input_dim, cols, rows);
    return false;
  }
  const uint8_t* dW = register_packed(b, packed_data, weight_bytes);
  const float* dG = register_floats(b, norm_weight, (size_t)input_dim);
  if (!dW || !dG) return false;
  ctx->ops.push_back(bm_hip_batch_ctx_t::Op{false, src_id, dst_id, input_dim, rows, cols, 0,
                                            w_scale, dW, dG});
  return true;
}

extern "C" void bm_hip_encode_residual(bm_hip_batch_ctx_t* ctx, int count) {
  if (!ctx) return;
  if (count < 0 || (size_t)count > (size_t)ctx->n_tokens * ctx->width[BM_HIP_BUF_X]) {
    fprintf(stderr, "[HIP] encode_residual: count=%d exceeds the batch buffers\n", count);
    return;
  }
  ctx->ops.push_back(bm_hip_batch_ctx_t::Op{true, BM_HIP_BUF_OUT, BM_HIP_BUF_X, 0, 0, 0, count,
                                            0.0f, nullptr, nullptr});
}

extern "C" void bm_hip_submit_and_wait(bm_hip_batch_ctx_t* ctx) {
  if (!ctx) return;
  Backend& b = B();
  std::lock_guard<std::mutex> lk(b.mu);
  // floats of each buffer to copy in (read before this submit writes them)
  // and to copy back (written)
  size_t in[4] = {}, out[4] = {}, written[4] = {};
  auto reads = [&](int id, size_t n) {
    if (n > written[id] && n > in[id]) in[id] = n;
  };
  auto writes = [&](int id, size_t n) {
    if (n > written[id]) written[id] = n;
    if (n > out[id]) out[id] = n;
  };
  const size_t T = (size_t)ctx->n_tokens;
  for (const auto& op : ctx->ops) {
    if (op.residual) {
      reads(BM_HIP_BUF_X, (size_t)op.count);
      reads(BM_HIP_BUF_OUT, (size_t)op.count);
      writes(BM_HIP_BUF_X, (size_t)op.count);
    } else {
      reads(op.src, T * op.input_dim);
      writes(op.dst, T * op.rows);
    }
  }
  hipStream_t s = b.stream;
  hipError_t e = hipSuccess;
  for (int i = 0; i < 4 && e == hipSuccess; ++i)
    if (in[i])
      e = hipMemcpyAsync(ctx->dev[i], ctx->host[i], in[i] * sizeof(float), hipMemcpyHostToDevice,
                         s);
  for (const auto& op : ctx->ops) {
    if (e != hipSuccess) break;
    if (op.residual) {
      e = bm::launch_residual_add(ctx->dev[BM_HIP_BUF_X], ctx->dev[BM_HIP_BUF_OUT],
                                  (size_t)op.count, s);
      continue;
    }
    // each token's row of the source: RMSNorm + int8 (src/kernel.c:72-129,
    // 356-386), then the blocked product (src/kernel.c:388-447)
    const int M = ctx->n_tokens, n = op.input_dim;
    const bool generic = bm::product_needs_generic(M, op.cols);
    e = bm::launch_quantize(ctx->dev[op.src], M, n, n, op.dG, nullptr, generic ? ctx->xq : nullptr,
                            n, ctx->scale, generic ? nullptr : ctx->act, s,
                            !generic && bm::product_reads_nibbles(M, op.rows, op.cols));
    if (e != hipSuccess) break;
    if (generic)
      e = bm::launch_generic(ctx->xq, n, ctx->scale, M, op.dW, op.rows, op.cols, op.w_scale,
                             ctx->dev[op.dst], bm::MODE_STORE, s);
    else
      e = bm::launch_product(ctx->act, ctx->scale, M, op.dW, op.rows, op.cols, op.w_scale, true,
                             ctx->dev[op.dst], bm::MODE_STORE, s);
  }
  for (int i = 0; i < 4 && e == hipSuccess; ++i)
    if (out[i])
      e = hipMemcpyAsync(ctx->host[i], ctx->dev[i], out[i] * sizeof(float), hipMemcpyDeviceToHost,
                         s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  ctx->ops.clear();
  if (e != hipSuccess) {
    bm_set_error("%s", hipGetErrorString(e));
    fprintf(stderr, "[HIP] Batch submit error: %s\n", hipGetErrorString(e));
  }
}

extern "C" void bm_hip_batch_end(bm_hip_batch_ctx_t* ctx) {
  if (!ctx) return;
  Backend& b = B();
  std::lock_guard<std::mutex> lk(b.mu);
  if (b.stream) (void)hipStreamSynchronize(b.stream);
  batch_free(ctx);
}

// ---------------------------------------------------------------------------
// Device memory helpers
// ---------------------------------------------------------------------------
extern "C" void* bm_hip_malloc(size_t bytes) {
  if (!bm_hip_init()) return nullptr;
  void* p = nullptr;
  BM_HIP_CHECK_RET(hipMalloc(&p, bytes ? bytes : 1), nullptr);
  return p;
}

extern "C" void bm_hip_free(void* dev) {
  if (dev) (void)hipFree(dev);
}

extern "C" int bm_hip_memcpy_h2d(void* dev, const void* host, size_t bytes) {
  BM_HIP_CHECK_RET(hipMemcpy(dev, host, bytes, hipMemcpyHostToDevice), -1);
  return 0;
}

extern "C" int bm_hip_memcpy_d2h(void* host, const void* dev, size_t bytes) {
  BM_HIP_CHECK_RET(hipMemcpy(host, dev, bytes, hipMemcpyDeviceToHost), -1);
  return 0;
}

extern "C" int bm_hip_memset(void* dev, int value, size_t bytes) {
  BM_HIP_CHECK_RET(hipMemset(dev, value, bytes), -1);
  return 0;
}

extern "C" int bm_hip_synchronize(void) {
  BM_HIP_CHECK_RET(hipDeviceSynchronize(), -1);
  return 0;
}

static hipStream_t stream_or_default(void* s) {
  return s ? (hipStream_t)s : B().stream;
}

extern "C" int bm_hip_canonicalize_dev(uint8_t* packed, size_t bytes, void* stream) {
  if (!bm_hip_init()) return -1;
  BM_HIP_CHECK_RET(bm::launch_canonicalize(packed, bytes, stream_or_default(stream)), -1);
  return 0;
}

// ---------------------------------------------------------------------------
// Device-pointer kernels
// ---------------------------------------------------------------------------
extern "C" size_t bm_hip_act_bytes(int M, int n) {
  if (M <= 0 || n <= 0) return 0;
  return (size_t)M * bm::act_row_bytes(n);
}

extern "C" size_t bm_hip_i8_act_bytes(int M, int K) { return bm_hip_act_bytes(M, K); }

static int quantize_dev(const float* x, int M, int n, int x_stride, const float* norm_w,
                        float* x_norm, int8_t* x_quant, int quant_stride, float* scale_x,
                        void* act, void* stream, bool fast) {
  if (!bm_hip_init()) return -1;
  if (M < 0 || n <= 0 || x_stride < n || !x || !norm_w || !scale_x ||
      (x_quant && quant_stride < n)) {
    bm_set_error("quantize: invalid arguments (M=%d n=%d x_stride=%d)", M, n, x_stride);
    return -2;
  }
  if (act && n % 16 != 0) {
    bm_set_error("quantize: activation workspace needs n %% 16 == 0 (n=%d)", n);
    return -2;
  }
  BM_HIP_CHECK_RET(bm::launch_quantize(x, M, n, x_stride, norm_w, x_norm, x_quant, quant_stride,
                                       scale_x, (uint8_t*)act, stream_or_default(stream), true,
                                       fast),
                   -1);
  return 0;
}

extern "C" int bm_hip_quantize_dev(const float* x, int M, int n, int x_stride,
                                   const float* norm_w, float* x_norm, int8_t* x_quant,
                                   int quant_stride, float* scale_x, void* act, void* stream) {
  return quantize_dev(x, M, n, x_stride, norm_w, x_norm, x_quant, quant_stride, scale_x, act,
                      stream, false);
}

extern "C" int bm_hip_quantize_fast_dev(const float* x, int M, int n, int x_stride,
                                        const float* norm_w, float* x_norm, int8_t* x_quant,
                                        int quant_stride, float* scale_x, void* act,
                                        void* stream) {
  return quantize_dev(x, M, n, x_stride, norm_w, x_norm, x_quant, quant_stride, scale_x, act,
                      stream, true);
}

extern "C" int bm_hip_bitlinear_act_dev(const void* act, const float* scale_x, int M,
                                        const uint8_t* packed, int N, int K, float w_scale,
                                        int canonical, float* out, void* stream) {
  if (!bm_hip_init()) return -1;
  if (M < 0 || N <= 0 || K <= 0 || !act || !scale_x || !packed || !out) {
    bm_set_error("bitlinear_act: invalid arguments");
    return -2;
  }
  if (bm::product_needs_generic(M, K)) {
    bm_set_error("bitlinear_act: K=%d needs the int8 path (bm_hip_bitlinear_dev)", K);
    return -2;
  }
  BM_HIP_CHECK_RET(bm::launch_product((const uint8_t*)act, scale_x, M, packed, N, K, w_scale,
                                      canonical != 0, out, bm::MODE_STORE,
                                      stream_or_default(stream)),
                   -1);
  return 0;
}

extern "C" int bm_hip_bitlinear_dev(const float* x, int M, int K, const float* norm_w,
                                    const uint8_t* packed, int N, float w_scale, int canonical,
                                    float* out, int8_t* x_quant, int quant_stride, float* scale_x,
                                    void* act, void* stream) {
  if (!bm_hip_init()) return -1;
  if (M < 0 || N <= 0 || K <= 0 || !x || !norm_w || !packed || !out || !x_quant || !scale_x ||
      quant_stride < K) {
    bm_set_error("bitlinear: invalid arguments");
    return -2;
  }
  hipStream_t s = stream_or_default(stream);
  const bool generic = bm::product_needs_generic(M, K);
  if (!generic && !act) {
    bm_set_error("bitlinear: act workspace required");
    return -2;
  }
  if (M == 1 && canonical && bm::rows_fit(K)) {
    // one token: the fused single-launch kernel of the decode (RMSNorm and
    // int8 prologue in every block, block 0 writing x_quant and scale_x)
    BM_HIP_CHECK_RET(bm::launch_rows_dev(x, K, norm_w, packed, N, w_scale, out, x_quant, scale_x,
                                         s),
                     -1);
    return 0;
  }
  BM_HIP_CHECK_RET(bm::launch_quantize(x, M, K, K, norm_w, nullptr, x_quant, quant_stride, scale_x,
                                       generic ? nullptr : (uint8_t*)act, s),
                   -1);
  if (generic)
    BM_HIP_CHECK_RET(bm::launch_generic(x_quant, quant_stride, scale_x, M, packed, N, K, w_scale,
                                        out, bm::MODE_STORE, s),
                     -1);
  else
    BM_HIP_CHECK_RET(bm::launch_product((const uint8_t*)act, scale_x, M, packed, N, K, w_scale,
                                        canonical != 0, out, bm::MODE_STORE, s),
                     -1);
  return 0;
}

extern "C" int bm_hip_ternary_gemm_i32_dev(const int8_t* xq, int M, int ldx,
                                           const uint8_t* packed, int N, int K, int canonical,
                                           int32_t* out, void* act, void* stream) {
  if (!bm_hip_init()) return -1;
  if (M < 0 || N <= 0 || K <= 0 || ldx < K || !xq || !packed || !out) {
    bm_set_error("ternary_gemm_i32: invalid arguments");
    return -2;
  }
  hipStream_t s = stream_or_default(stream);
  if (bm::product_needs_generic(M, K)) {
    BM_HIP_CHECK_RET(bm::launch_generic(xq, ldx, nullptr, M, packed, N, K, 0.0f, out,
                                        bm::MODE_I32, s),
                     -1);
    return 0;
  }
  if (!act) {
    bm_set_error("ternary_gemm_i32: act workspace required");
    return -2;
  }
  if (M == 1 && bm::rows_i8_fit(K)) {
    // one token: one launch, the block turns the int8 row into split
    // nibbles itself (the workspace stays unused)
    BM_HIP_CHECK_RET(bm::launch_rows_i8(xq, M, ldx, K, packed, N, canonical != 0, out, s), -1);
    return 0;
  }
  {
    // few tokens: one launch that reads the int8 rows itself
    const hipError_t e = bm::launch_small_i8(xq, M, ldx, K, packed, N, canonical != 0, out, s);
    if (e == hipSuccess) return 0;
    if (e != hipErrorNotSupported) {
      bm_set_error("%s", hipGetErrorString(e));
      return -1;
    }
  }
  BM_HIP_CHECK_RET(bm::launch_prep_i8(xq, M, ldx, K, (uint8_t*)act,
                                      bm::product_reads_nibbles(M, N, K), s),
                   -1);
  BM_HIP_CHECK_RET(bm::launch_product((const uint8_t*)act, nullptr, M, packed, N, K, 0.0f,
                                      canonical != 0, out, bm::MODE_I32, s),
                   -1);
  return 0;
}

// Quantize + product like bm_hip_bitlinear_dev, with the workspace (per-token
// scale, activation workspace or int8 copy) in the file-scope scratch array
// instead of caller or library allocations: no hipMalloc, hipFree or other
// allocating call, so callers that cannot allocate (code under stream
// capture, serving loops) can use it.  Calls that overlap on one GPU share
// the array and race.
extern "C" int bm_hip_bitlinear_noalloc_dev(const float* x, int M, int K, const float* norm_w,
                                            const uint8_t* packed, int N, float w_scale,
                                            int canonical, float* out, void* stream) {
  Backend& b = B();
  uint8_t* base = nullptr;
  hipStream_t s = nullptr;
  {
    std::lock_guard<std::mutex> lk(b.mu);
    if (!b.ready) {
      bm_set_error("bitlinear_noalloc: call bm_hip_init first (this entry point allocates "
                   "nothing, the stream and scratch address included)");
      return -1;
    }
    base = (uint8_t*)b.scratch_dev[b.device];
    s = stream ? (hipStream_t)stream : b.stream;
  }
  if (M < 1 || N <= 0 || K <= 0 || !x || !norm_w || !packed || !out || !base) {
    bm_set_error("bitlinear_noalloc: invalid arguments (M=%d N=%d K=%d)", M, N, K);
    return -2;
  }
  const bool generic = bm::product_needs_generic(M, K);
  // [scale_x (M floats) | activation workspace, or the int8 copy for K the
  // products cover only through the generic kernel]
  const size_t o_work = bm::align_up((size_t)M * 4, 256);
  const size_t work = generic ? (size_t)M * (size_t)K : (size_t)M * bm::act_row_bytes(K);
  const size_t need = o_work + work;
  if (need > kScratchBytes) {
    bm_set_error("bitlinear_noalloc: M=%d K=%d needs %zu bytes of scratch, the limit is %zu",
                 M, K, need, kScratchBytes);
    return -2;
  }
  float* sc = (float*)base;
  uint8_t* wk = base + o_work;
  BM_HIP_CHECK_RET(bm::launch_quantize(x, M, K, K, norm_w, nullptr, generic ? (int8_t*)wk : nullptr,
                                       K, sc, generic ? nullptr : wk, s),
                   -1);
  if (generic)
    BM_HIP_CHECK_RET(bm::launch_generic((const int8_t*)wk, K, sc, M, packed, N, K, w_scale, out,
                                        bm::MODE_STORE, s),
                     -1);
  else
    BM_HIP_CHECK_RET(bm::launch_product(wk, sc, M, packed, N, K, w_scale, canonical != 0, out,
                                        bm::MODE_STORE, s),
                     -1);
  return 0;
}

extern "C" size_t bm_hip_noalloc_scratch_bytes(void) { return kScratchBytes; }

// ---------------------------------------------------------------------------
// Timing and calibration helpers (no reference counterpart)
// ---------------------------------------------------------------------------
extern "C" void* bm_hip_stream(void) {
  if (!bm_hip_init()) return nullptr;
  return (void*)B().stream;
}

extern "C" void* bm_hip_event_create(void) {
  if (!bm_hip_init()) return nullptr;
  hipEvent_t e = nullptr;
  BM_HIP_CHECK_RET(hipEventCreate(&e), nullptr);
  return (void*)e;
}

extern "C" void bm_hip_event_destroy(void* ev) {
  if (ev) (void)hipEventDestroy((hipEvent_t)ev);
}

extern "C" int bm_hip_event_record(void* ev, void* stream) {
  BM_HIP_CHECK_RET(hipEventRecord((hipEvent_t)ev, stream_or_default(stream)), -1);
  return 0;
}

extern "C" float bm_hip_event_elapsed_ms(void* start, void* stop) {
  float ms = -1.0f;
  if (hipEventSynchronize((hipEvent_t)stop) != hipSuccess) return -1.0f;
  if (hipEventElapsedTime(&ms, (hipEvent_t)start, (hipEvent_t)stop) != hipSuccess) return -1.0f;
  return ms;
}

namespace bm {
__global__ void k_copy16(const uint4* __restrict__ src, uint4* __restrict__ dst, size_t n) {
  for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x)
    dst[i] = src[i];
}
}  // namespace bm

namespace bm {
// int8 MFMA ceiling: each wave runs `iters` rounds of 16 v_mfma_i32_32x32x32_i8
// on four accumulators.  Operands are fixed small integers (ternary = 0) or,
// like the prefill GEMM's, hashed int8 activations against codes 0..2
// (ternary = 1): the sustained rate depends on the data (clock under load).
__global__ __launch_bounds__(256) void k_mfma_peak(int iters, int ternary, int* __restrict__ sink) {
  v16i acc[2][2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][b][v] = 0;
  v4i opa[2][4], opb[2][4];
  uint32_t z = (threadIdx.x + 1) * 2654435761u ^ (blockIdx.x + 1) * 40503u;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        z ^= z << 13;
        z ^= z >> 17;
        z ^= z << 5;
        const uint32_t w = z;
        z ^= z << 13;
        z ^= z >> 17;
        z ^= z << 5;
        uint32_t c = z & 0x03030303u;
        c -= (c >> 1) & (c & 0x01010101u);  // code 3 -> 2
        opa[a][q][e] = ternary ? (int)w : (int)(threadIdx.x + e);
        opb[a][q][e] = ternary ? (int)c : (int)(q + a);
      }
  for (int i = 0; i < iters; ++i) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          acc[mt][nt] =
              __builtin_amdgcn_mfma_i32_32x32x32_i8(opa[mt][q], opb[nt][q], acc[mt][nt], 0, 0, 0);
  }
  int r = 0;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) r ^= acc[a][b][0] ^ acc[a][b][15];
  if (r == 0x5eed5eed) sink[0] = r;  // keeps the MFMAs live
}
}  // namespace bm

extern "C" int bm_hip_mfma_peak_dev(int blocks, int iters, int ternary, int* sink, void* stream) {
  if (!bm_hip_init()) return -1;
  if (blocks < 1 || iters < 1) {
    bm_set_error("mfma_peak: blocks and iters must be positive");
    return -2;
  }
  hipLaunchKernelGGL(bm::k_mfma_peak, dim3(blocks), dim3(256), 0, stream_or_default(stream), iters,
                     ternary, sink);
  BM_HIP_CHECK_RET(hipGetLastError(), -1);
  return 0;
}

extern "C" int bm_hip_copy_dev(void* dst, const void* src, size_t bytes, void* stream) {
  if (!bm_hip_init()) return -1;
  if (bytes % 16 || ((uintptr_t)dst | (uintptr_t)src) % 16) {
    bm_set_error("copy: 16-byte sizes and alignment only");
    return -2;
  }
  const size_t n = bytes / 16;
  int blocks = (int)((n + 255) / 256);
  if (blocks > 8192) blocks = 8192;
  if (blocks < 1) blocks = 1;
  hipLaunchKernelGGL(bm::k_copy16, dim3(blocks), dim3(256), 0, stream_or_default(stream),
                     (const uint4*)src, (uint4*)dst, n);
  BM_HIP_CHECK_RET(hipGetLastError(), -1);
  return 0;
}
