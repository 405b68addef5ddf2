// hes_transfer.hpp -- a state on its way to the host: structure-of-arrays rows
// on the device, one state after another (component fastest) in host memory.
//
// A copy into pageable memory runs at the rate of one host thread that copies
// out of the runtime's staging memory and takes the page faults of a fresh
// array (9 GB/s; 47 to 52 ms for 2^22 cells of 14 components, whose 400 Rusanov
// steps take 72; 10.5 ms as here, 45 GB/s).  A large state is therefore cut into pieces, and several
// threads each let a kernel write a piece into page-locked memory of their
// own, in the host's order, and copy it out.
#pragma once
#include <hip/hip_runtime.h>
#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <thread>

#include "hes_host.hpp"

namespace hes {

// Cells [first, first + cells) of the rows Q in the host's order into out
// (device or page-locked host memory), a block per GATHER_CELLS of them by way
// of LDS, so that both sides move whole lines.
constexpr int GATHER_CELLS = 128, GATHER_BLOCK = 256;
static __global__ __launch_bounds__(GATHER_BLOCK) void k_gather(const double* __restrict__ Q,
                                                               double* __restrict__ out, int nc,
                                                               long long first, long long cells,
                                                               long long pitch) {
  extern __shared__ double tile[];
  const long long c0 = (long long)blockIdx.x * GATHER_CELLS;
  const int here = (int)(cells - c0 < GATHER_CELLS ? cells - c0 : GATHER_CELLS);
  const int c = threadIdx.x % GATHER_CELLS;
  if (c < here)
    for (int r = threadIdx.x / GATHER_CELLS; r < nc; r += GATHER_BLOCK / GATHER_CELLS)
      tile[c * nc + r] = __builtin_nontemporal_load(Q + r * pitch + first + c0 + c);
  __syncthreads();
  for (int t = threadIdx.x; t < here * nc; t += GATHER_BLOCK) out[c0 * nc + t] = tile[t];
}

inline hipError_t gather(const double* Q, double* out, int nc, long long first, long long cells,
                         long long pitch, hipStream_t s) {
  hipLaunchKernelGGL(k_gather, dim3((unsigned)((cells + GATHER_CELLS - 1) / GATHER_CELLS)),
                     dim3(GATHER_BLOCK), sizeof(double) * GATHER_CELLS * nc, s, Q, out, nc, first,
                     cells, pitch);
  return hipGetLastError();
}

// Page-locked pieces of memory with a stream each, for the threads of large
// downloads; those of one download are kept for the next.
struct Piece {
  static constexpr size_t BYTES = 4 << 20;
  int dev = 0;
  char* p = nullptr;
  hipStream_t stream = nullptr;
};
inline constexpr int DOWNLOAD_THREADS = 8;
using KeptPieces = Kept<Piece, DOWNLOAD_THREADS>;
inline KeptPieces& pieces() {
  static KeptPieces p;
  static_assert(std::is_trivially_destructible<KeptPieces>::value, "outlives the runtime's own end");
  return p;
}
inline void piece_free(Piece& b) {
  if (b.stream) (void)hipStreamDestroy(b.stream);
  if (b.p) (void)hipHostFree(b.p);
}
inline hipError_t piece_take(int dev, Piece* b) {
  if (pieces().take(dev, b)) return hipSuccess;
  b->dev = dev;
  hipError_t e = hipHostMalloc((void**)&b->p, Piece::BYTES);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
  if (e != hipSuccess) {
    piece_free(*b);
    *b = Piece();
  }
  return e;
}
inline void piece_give(Piece& b, bool keep) {
  if (!keep || !pieces().give(b)) piece_free(b);
}

// From this size on a download is shared by threads: below it their start and
// the pieces' faults cost what they save.
constexpr size_t DOWNLOAD_SHARED_MIN = 6 << 20;

// Cells [first, first + cells) of the rows into `out` by way of a space's memory.
inline hipError_t download_plain(const double* Q, double* out, int nc, long long first,
                                 long long cells, long long pitch) {
  const size_t bytes = sizeof(double) * (size_t)nc * (size_t)cells;
  Space s;
  hipError_t e = space_take(&s);
  if (e != hipSuccess) return e;
  const bool small = bytes <= Space::HOST;
  if (!small) e = space_device(s, bytes);
  double* at = (double*)(small ? s.host : s.device);
  if (e == hipSuccess) e = gather(Q, at, nc, first, cells, pitch, s.stream);
  if (e == hipSuccess && !small) e = hipMemcpyAsync(out, at, bytes, hipMemcpyDeviceToHost, s.stream);
  const hipError_t es = hipStreamSynchronize(s.stream);
  if (e == hipSuccess) e = es;
  if (e == hipSuccess && small) std::memcpy(out, at, bytes);
  space_give(s, e == hipSuccess);
  return e;
}

// The n states of rows Q (written by work that has been waited for) into `out`.
inline hipError_t download_state(const double* Q, double* out, int nc, long long n,
                                 long long pitch) {
  const size_t bytes = sizeof(double) * (size_t)nc * (size_t)n;
  if (bytes < DOWNLOAD_SHARED_MIN) return download_plain(Q, out, nc, 0, n, pitch);
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  // cells of a piece: a share of a small state, a whole piece of a large one
  const size_t piece = std::max<size_t>(std::min(Piece::BYTES, bytes / DOWNLOAD_THREADS), 1 << 20);
  const long long per = (long long)(piece / (sizeof(double) * nc));
  const long long parts = (n + per - 1) / per;
  std::atomic<long long> next{0};
  std::atomic<int> failed{(int)hipSuccess};
  // page_locked: a thread without a piece leaves its share to the others
  auto work = [&](bool page_locked) {
    Piece b;
    hipError_t we = hipSetDevice(dev);
    if (we == hipSuccess && page_locked && piece_take(dev, &b) != hipSuccess) {
      (void)hipGetLastError();
      return;
    }
    while (we == hipSuccess && failed.load() == (int)hipSuccess) {
      const long long k = next.fetch_add(1);
      if (k >= parts) break;
      const long long c0 = k * per, cells = std::min(per, n - c0);
      if (!page_locked) {
        we = download_plain(Q, out + c0 * nc, nc, c0, cells, pitch);
        continue;
      }
      we = gather(Q, (double*)b.p, nc, c0, cells, pitch, b.stream);
      const hipError_t es = hipStreamSynchronize(b.stream);
      if (we == hipSuccess) we = es;
      if (we == hipSuccess)
        std::memcpy(out + c0 * nc, b.p, sizeof(double) * (size_t)nc * (size_t)cells);
    }
    if (we != hipSuccess) failed.store((int)we);
    if (b.p) piece_give(b, we == hipSuccess);
  };
  std::thread threads[DOWNLOAD_THREADS - 1];
  try {
    for (long long k = 1; k < std::min<long long>(DOWNLOAD_THREADS, parts); ++k)
      threads[k - 1] = std::thread(work, true);
  } catch (const std::exception&) {  // fewer threads share the work
  }
  work(true);
  for (std::thread& t : threads)
    if (t.joinable()) t.join();
  work(false);  // what is left when no thread had a piece
  return (hipError_t)failed.load();
}

}  // namespace hes
