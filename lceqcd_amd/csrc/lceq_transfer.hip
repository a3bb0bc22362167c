// lceq_transfer.hip -- link and Higgs fields between the caller's host arrays
// (the reference's COMMON layout, include/lceq.h) and the device layout
// (field_offset).  The reordering runs on the device, in kernels that read or
// write pinned host memory directly; the host only copies between the pinned
// slots and the caller's array, in several threads where the field is large.
//
// What bounds it is the host side: a 64^3 link field is 25 MB, 0.5 ms over
// the bus, but a fresh host array costs a page fault per 4 KiB, which one
// thread takes at a few GB/s.  Reordering on the host (a strided pass over a
// second, zero-filled array) and copying from pageable memory took 3.9 ms
// for the links and the Higgs field of 64^3.
#include <string.h>

#include <algorithm>
#include <exception>
#include <mutex>
#include <new>
#include <thread>

#include "../../include/lceq.h"
#include "lceq_internal.hpp"

namespace lceq {
namespace {

// Rows are the host array's sites in order, row = cls * n + s.  Links: one
// thread per 16-byte half, so that a wave touches one contiguous KiB of the
// host array and two contiguous runs of the device halves.
template <bool GET>
__global__ __launch_bounds__(256) void k_links_host(double2* __restrict__ dev,
                                                    double2* __restrict__ host, unsigned n,
                                                    unsigned npad, unsigned row0, unsigned halves) {
  unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i >= halves) return;
  unsigned row = row0 + (i >> 1), cls = row / n, s = row - cls * n;
  size_t d = (size_t)(2 * cls + (i & 1)) * npad + s;
  if (GET)
    host[i] = dev[d];
  else
    dev[d] = host[i];
}

// Higgs triples: one thread per component
template <bool GET>
__global__ __launch_bounds__(256) void k_higgs_host(double* __restrict__ dev,
                                                    double* __restrict__ host, unsigned n,
                                                    unsigned npad, unsigned row0, unsigned values) {
  unsigned i = blockIdx.x * 256 + threadIdx.x;
  if (i >= values) return;
  unsigned k = i / 3, c = i - 3 * k, row = row0 + k, cls = row / n, s = row - cls * n;
  size_t d = field_offset(3, (int)cls, (int)c, s, npad);
  if (GET)
    host[i] = dev[d];
  else
    dev[d] = host[i];
}

// Pinned slots of one transfer: two per worker, so that a worker copies one
// slot while the device fills or drains its other one.
constexpr int MAX_WORKERS = 8;
constexpr int SLOTS = 2 * MAX_WORKERS;
constexpr size_t SLOT_BYTES = 1536 << 10;  // whole rows of 32 and of 24 bytes
constexpr size_t MIN_CHUNK = SLOT_BYTES / 2;

}  // namespace

// Pinned blocks not in use stay allocated for the next lattice, batch or transfer
// on their device, up to KEEP of each kind (121 MiB) while a lattice or batch
// exists and LEFT (one of each, 26 MiB) when none does, so that a program that
// makes lattices one after the other does not allocate them each time: the driver
// unmaps a freed block behind the call, and the next lattice's allocations wait for
// it.  A life with the links read and written, in us, with pageable copies, with
// blocks freed with the last lattice, and as here: 8^3 154-246 213-291 193-227,
// 16^3 202-260 225-343 244-261, 24^3 411-752 1530-2400 1080-1290, 40^3 2700-2910
// 915-980 800-885.
struct Pinned {
  int device, kind;
  char* host;
  hipEvent_t ev[SLOTS];  // EVENTS of them
};

namespace {

constexpr size_t PINNED_BYTES[PINNED_KINDS] = {PINNED_RESULTS_BYTES, 2 * MIN_CHUNK,
                                               SLOTS * SLOT_BYTES};
constexpr int EVENTS[PINNED_KINDS] = {0, 2, SLOTS};
constexpr int KEEP[PINNED_KINDS] = {16, 16, 4}, LEFT[PINNED_KINDS] = {1, 1, 1}, KEEP_MOST = 16;
std::mutex g_mu;
Pinned* g_idle[PINNED_KINDS][KEEP_MOST];
int g_nidle[PINNED_KINDS];
int g_users = 0;

void pinned_free(Pinned* P) {
  for (hipEvent_t e : P->ev)
    if (e) (void)hipEventDestroy(e);
  if (P->host) (void)hipHostFree(P->host);
  delete P;
}

}  // namespace

Pinned* pinned_take(int device, int kind) {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    for (int i = g_nidle[kind] - 1; i >= 0; --i)
      if (g_idle[kind][i]->device == device) {
        Pinned* P = g_idle[kind][i];
        g_idle[kind][i] = g_idle[kind][--g_nidle[kind]];
        return P;
      }
  }
  Pinned* P = new (std::nothrow) Pinned();
  if (!P) return nullptr;
  P->device = device;
  P->kind = kind;
  bool ok = hipHostMalloc((void**)&P->host, PINNED_BYTES[kind], hipHostMallocDefault) == hipSuccess;
  for (int i = 0; ok && i < EVENTS[kind]; ++i)
    ok = hipEventCreateWithFlags(&P->ev[i], hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();  // reported here, not by the next launch
    pinned_free(P);
    return nullptr;
  }
  return P;
}

void pinned_give(Pinned* P) {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_nidle[P->kind] < (g_users > 0 ? KEEP : LEFT)[P->kind]) {
      g_idle[P->kind][g_nidle[P->kind]++] = P;
      return;
    }
  }
  pinned_free(P);
}

void* pinned_host(Pinned* P) { return P->host; }

namespace {

struct Transfer {
  hipStream_t stream;
  int device;
  double *dev, *host;
  int64_t ld;
  unsigned n, npad;
  int ncomp;
  bool get;
  unsigned rows, rows_per_slot;
  size_t slot_bytes;
  int chunks, workers;
  Pinned* stage;
};

// copy between the slot and the caller's array: row r of the field is at
// host[((r / n) * ld + r % n) * ncomp]
void host_copy(const Transfer& t, char* slot, unsigned row0, unsigned rows) {
  const size_t rb = (size_t)t.ncomp * sizeof(double);
  while (rows) {
    unsigned cls = row0 / t.n, s = row0 - cls * t.n;
    unsigned k = t.ld == (int64_t)t.n ? rows : std::min(rows, t.n - s);
    char* h = reinterpret_cast<char*>(t.host) + ((size_t)cls * t.ld + s) * rb;
    if (t.get)
      memcpy(h, slot, k * rb);
    else
      memcpy(slot, h, k * rb);
    slot += k * rb;
    row0 += k;
    rows -= k;
  }
}

hipError_t launch_slot(const Transfer& t, char* slot, unsigned row0, unsigned rows) {
  unsigned units = rows * (t.ncomp == 4 ? 2 : 3);
  dim3 grid((units + 255) / 256), blk(256);
  double2 *d2 = reinterpret_cast<double2*>(t.dev), *h2 = reinterpret_cast<double2*>(slot);
  double* h1 = reinterpret_cast<double*>(slot);
  if (t.ncomp == 4) {
    if (t.get)
      hipLaunchKernelGGL(k_links_host<true>, grid, blk, 0, t.stream, d2, h2, t.n, t.npad, row0, units);
    else
      hipLaunchKernelGGL(k_links_host<false>, grid, blk, 0, t.stream, d2, h2, t.n, t.npad, row0, units);
  } else {
    if (t.get)
      hipLaunchKernelGGL(k_higgs_host<true>, grid, blk, 0, t.stream, t.dev, h1, t.n, t.npad, row0, units);
    else
      hipLaunchKernelGGL(k_higgs_host<false>, grid, blk, 0, t.stream, t.dev, h1, t.n, t.npad, row0, units);
  }
  return hipGetLastError();
}

// chunks w, w + workers, ... in order through the worker's two slots
hipError_t run_worker(const Transfer& t, int w) {
  hipError_t e = hipSuccess;
  int prev = -1;
  auto rows_of = [&](int c) {
    return std::min(t.rows_per_slot, t.rows - (unsigned)c * t.rows_per_slot);
  };
  auto slot_of = [&](int c) { return 2 * w + ((c / t.workers) & 1); };
  auto finish = [&](int c) {  // wait for chunk c's kernel
    return t.chunks > 1 ? hipEventSynchronize(t.stage->ev[slot_of(c)])
                        : hipStreamSynchronize(t.stream);
  };
  for (int c = w; c < t.chunks && e == hipSuccess; c += t.workers) {
    int k = slot_of(c);
    char* slot = t.stage->host + (size_t)k * t.slot_bytes;
    unsigned row0 = (unsigned)c * t.rows_per_slot;
    if (!t.get) {
      int before = c - 2 * t.workers;  // the slot's previous chunk
      if (before >= 0 && (e = finish(before)) != hipSuccess) break;
      host_copy(t, slot, row0, rows_of(c));
    }
    if ((e = launch_slot(t, slot, row0, rows_of(c))) != hipSuccess) break;
    // a lone chunk is waited for through its stream: an event's record and
    // wait cost 8 us more, which shows in the smallest transfers
    if (t.chunks > 1 && (e = hipEventRecord(t.stage->ev[k], t.stream)) != hipSuccess) break;
    if (t.get && prev >= 0) {
      if ((e = finish(prev)) != hipSuccess) break;
      host_copy(t, t.stage->host + (size_t)slot_of(prev) * t.slot_bytes,
                (unsigned)prev * t.rows_per_slot, rows_of(prev));
    }
    prev = c;
  }
  if (t.get && prev >= 0 && e == hipSuccess) {
    if ((e = finish(prev)) != hipSuccess) return e;
    host_copy(t, t.stage->host + (size_t)slot_of(prev) * t.slot_bytes,
              (unsigned)prev * t.rows_per_slot, rows_of(prev));
  }
  return e;
}

}  // namespace

void transfer_user(int change) {
  Pinned* drop[PINNED_KINDS * KEEP_MOST];
  int ndrop = 0;
  {
    std::lock_guard<std::mutex> lock(g_mu);
    g_users += change;
    for (int k = 0; g_users == 0 && k < PINNED_KINDS; ++k)
      while (g_nidle[k] > LEFT[k]) drop[ndrop++] = g_idle[k][--g_nidle[k]];
  }
  while (ndrop) pinned_free(drop[--ndrop]);
}

int transfer_field(hipStream_t stream, int device, const Geom& g, double* dev, double* host,
                   int64_t ld, int ncomp, int nclass, bool get) {
  Transfer t;
  t.stream = stream;
  t.device = device;
  t.dev = dev;
  t.host = host;
  t.ld = ld;
  t.n = (unsigned)g.n;
  t.npad = (unsigned)g.npad;
  t.ncomp = ncomp;
  t.get = get;
  t.rows = (unsigned)nclass * t.n;
  // a chunk per worker, within a slot and not below half of one; a second
  // worker from four chunks (3 MiB) on.  Measured, links in us a download
  // (host array already touched): 16^3 30 with one chunk and worker, 41 with
  // two; 24^3 65 against 93 with two workers; 48^3 350 either way; 160^3
  // 12.2, 10.2 and 8.5 ms with slots of 384, 768 and 1536 KiB.
  const size_t rb = (size_t)ncomp * sizeof(double);
  unsigned share = (t.rows + MAX_WORKERS - 1) / MAX_WORKERS;
  t.rows_per_slot = std::min((unsigned)(SLOT_BYTES / rb), std::max((unsigned)(MIN_CHUNK / rb), share));
  t.slot_bytes = t.rows_per_slot * rb;
  t.chunks = (int)((t.rows + t.rows_per_slot - 1) / t.rows_per_slot);
  t.workers = std::min(MAX_WORKERS, std::max(1, t.chunks / 2));
  int current = device;
  if (hipGetDevice(&current) == hipSuccess && current != device) (void)hipSetDevice(device);
  // one worker's chunks are MIN_CHUNK, and it has two slots
  t.stage = pinned_take(device, t.workers > 1 ? PINNED_LARGE : PINNED_SMALL);
  if (!t.stage) {
    if (current != device) (void)hipSetDevice(current);
    return set_error(LCEQ_ERR_HIP, "no pinned memory for a field transfer");
  }
  hipError_t err[MAX_WORKERS] = {};
  std::thread th[MAX_WORKERS];
  for (int w = 1; w < t.workers; ++w) {
    try {
      th[w] = std::thread([&t, &err, w] {
        err[w] = hipSetDevice(t.device);
        if (err[w] == hipSuccess) err[w] = run_worker(t, w);
      });
    } catch (const std::exception&) {
      err[w] = run_worker(t, w);  // no thread to be had: its chunks here
    }
  }
  err[0] = run_worker(t, 0);
  for (int w = 1; w < t.workers; ++w)
    if (th[w].joinable()) th[w].join();
  // after a put the slots are free, and an error surfaces, once the stream is
  // idle; after an error no kernel may still use them
  hipError_t e = hipSuccess;
  for (int w = 0; w < t.workers; ++w)
    if (e == hipSuccess) e = err[w];
  if (!get || e != hipSuccess) {
    hipError_t es = hipStreamSynchronize(stream);
    if (e == hipSuccess) e = es;
  }
  if (current != device) (void)hipSetDevice(current);
  pinned_give(t.stage);
  if (e != hipSuccess)
    return set_error(LCEQ_ERR_HIP, "field transfer failed: %s", hipGetErrorString(e));
  return LCEQ_OK;
}

}  // namespace lceq
