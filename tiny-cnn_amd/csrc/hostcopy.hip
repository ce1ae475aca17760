// hostcopy.hip — small copies between pageable host memory and the device.
//
// The runtime's copy of a small pageable buffer is a staging copy, a blit kernel and a wait for
// the stream, and the wait keeps the host from queueing what comes next. Here the buffer goes
// through a ring of pinned pieces that a kernel of one workgroup reads (or writes) over the bus,
// and the same kernel leaves the piece's turn in pinned memory behind its data: an upload waits
// for nothing but a free piece, and a download polls that word instead of waiting for the stream.
// us a call, runtime / here: upload of 1 KB 16 / 6, 12 KB 19 / 7, 48 KB 26 / 10, 64 KB 13 / 11;
// download of 1 KB 22 / 12, 12 KB 30 / 20, 48 KB 12 / 23. (From some tens of kilobytes on the
// runtime maps the caller's pages and copies without staging: the limits lie there.)
#include <atomic>
#include <cstring>
#include <mutex>

#include "common.h"

namespace tdh {
namespace {

constexpr int HC_THREADS   = 1024;
constexpr size_t HC_PIECE  = 64 * 1024;  // a workgroup moves it with four 16-byte accesses a thread
constexpr size_t HC_MAX_DOWN = 16 * 1024;
constexpr int HC_PIECES    = 16;

struct Ring {
  char *data = nullptr;       // [HC_PIECES][HC_PIECE], pinned
  uint32_t *turn = nullptr;   // turn[i]: the last turn of piece i whose kernel has run
  uint32_t issued[HC_PIECES] = {};
  int next = 0;
};
Ring g_ring;
std::mutex g_ring_mutex;  // (callers on several threads: a download keeps its piece until its data has left it)

// dst and src share the alignment of `word` bytes (16, 4 or 1)
template <typename W>
__device__ __forceinline__ void copy_words(void *dst, const void *src, const uint32_t bytes) {
  const uint32_t n = bytes / sizeof(W);
  W *d       = static_cast<W *>(dst);
  const W *s = static_cast<const W *>(src);
  for (uint32_t i = threadIdx.x; i < n; i += HC_THREADS) d[i] = s[i];
  const uint32_t done = n * sizeof(W);
  if (done + threadIdx.x < bytes)
    static_cast<char *>(dst)[done + threadIdx.x] = static_cast<const char *>(src)[done + threadIdx.x];
}

__global__ void __launch_bounds__(HC_THREADS)
host_copy_kernel(void *dst, const void *src, const uint32_t bytes, const bool down, uint32_t *turn, const uint32_t value) {
  const uintptr_t at = reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(src);
  if (at % 16 == 0)
    copy_words<uint4>(dst, src, bytes);
  else if (at % 4 == 0)
    copy_words<uint32_t>(dst, src, bytes);
  else
    copy_words<char>(dst, src, bytes);
  // Of an upload the host waits only for the piece to have been read, which the barrier says; what a
  // download has written must be there before the word.
  if (down) __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(turn, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

int ring_ready() {
  if (g_ring.data) return TDH_OK;
  Ring r;
  void *d = nullptr, *t = nullptr;
  if (hipHostMalloc(&d, HC_PIECES * HC_PIECE, hipHostMallocDefault) != hipSuccess ||
      hipHostMalloc(&t, HC_PIECES * sizeof(uint32_t), hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    if (d) (void)hipHostFree(d);
    return set_error(TDH_ERR_OOM, "cannot allocate pinned memory for host copies");
  }
  r.data = static_cast<char *>(d);
  r.turn = static_cast<uint32_t *>(t);
  std::memset(r.turn, 0, HC_PIECES * sizeof(uint32_t));
  g_ring = r;
  return TDH_OK;
}

// Polls until the kernel of the piece's last turn has run; after a while it waits for the stream
// instead, which also reports an error of the device.
int wait_piece(int i) {
  const std::atomic<uint32_t> *word = reinterpret_cast<const std::atomic<uint32_t> *>(g_ring.turn + i);
  for (int spin = 0; spin < (1 << 16); ++spin)
    if (word->load(std::memory_order_acquire) == g_ring.issued[i]) return TDH_OK;
  TDH_HIP(hipStreamSynchronize(ctx().stream));
  return TDH_OK;
}

// the next piece, free to be written
int take_piece(int *piece) {
  TDH_TRY(ring_ready());
  *piece      = g_ring.next;
  g_ring.next = (g_ring.next + 1) % HC_PIECES;
  return wait_piece(*piece);
}

int launch_piece(void *dst, const void *src, size_t bytes, bool down, int i) {
  const uint32_t value = ++g_ring.issued[i];
  TDH_LAUNCH(host_copy_kernel, dim3(1), dim3(HC_THREADS), 0, ctx().stream, dst, src, static_cast<uint32_t>(bytes), down,
             g_ring.turn + i, value);
  TDH_LAUNCH_CHECK();
  return TDH_OK;
}

}  // namespace

// What the runtime's copy would look at, and a kernel that is handed an address does not: whether it is
// memory of this device, and whether the whole copy lies in that allocation. An address that is
// nothing of the kind is left to the runtime's copy.
static int kernel_may_copy(const void *device, size_t bytes, bool *may) {
  *may = false;
  hipPointerAttribute_t attr;
  if (hipPointerGetAttributes(&attr, device) != hipSuccess) {
    (void)hipGetLastError();
    return TDH_OK;
  }
  if (attr.type != hipMemoryTypeDevice || attr.device != ctx().device) return TDH_OK;
  hipDeviceptr_t base = nullptr;
  size_t size         = 0;
  if (hipMemGetAddressRange(&base, &size, const_cast<void *>(device)) != hipSuccess) {
    (void)hipGetLastError();
    return TDH_OK;
  }
  const size_t at = static_cast<size_t>(static_cast<const char *>(device) - static_cast<const char *>(base));
  if (at > size || bytes > size - at)
    return set_error(TDH_ERR_INVALID, "a copy of %zu bytes reaches past the end of its allocation (%zu bytes at %zu)", bytes,
                     size, at);
  *may = true;
  return TDH_OK;
}
int host_copy_up_applies(const void *device, size_t bytes, bool *applies) {
  *applies = false;
  return bytes <= HC_PIECE ? kernel_may_copy(device, bytes, applies) : TDH_OK;
}
int host_copy_down_applies(const void *device, size_t bytes, bool *applies) {
  *applies = false;
  return bytes <= HC_MAX_DOWN ? kernel_may_copy(device, bytes, applies) : TDH_OK;
}

int host_copy_up(void *dst, const void *src, size_t bytes) {
  std::lock_guard<std::mutex> lock(g_ring_mutex);
  int i = 0;
  TDH_TRY(take_piece(&i));
  std::memcpy(g_ring.data + i * HC_PIECE, src, bytes);
  return launch_piece(dst, g_ring.data + i * HC_PIECE, bytes, /*down=*/false, i);
}

int host_copy_down(void *dst, const void *src, size_t bytes) {
  std::lock_guard<std::mutex> lock(g_ring_mutex);
  int i = 0;
  TDH_TRY(take_piece(&i));
  TDH_TRY(launch_piece(g_ring.data + i * HC_PIECE, src, bytes, /*down=*/true, i));
  TDH_TRY(wait_piece(i));
  std::memcpy(dst, g_ring.data + i * HC_PIECE, bytes);
  return TDH_OK;
}

void host_copy_release() {
  std::lock_guard<std::mutex> lock(g_ring_mutex);
  if (g_ring.data) (void)hipHostFree(g_ring.data);
  if (g_ring.turn) (void)hipHostFree(g_ring.turn);
  g_ring = Ring();
}

}  // namespace tdh
