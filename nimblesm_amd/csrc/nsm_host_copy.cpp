// nsm_host_copy.cpp -- device memory into a caller's pageable host memory.
//
// hipMemcpy stages such a copy without overlap, and into fresh memory (a
// result array just allocated) it reaches 10-14 GB/s where the link moves 57:
// the 51.5 MB node field of the 128^3 cube took 5.0 ms.  Here the copy goes
// in chunks through pinned slots; while the host empties one (about 40 us per
// MB, the page faults of fresh memory included), the device fills the next
// ones.  A kernel writes the slots: a copy-engine transfer and its event cost
// about 20 us per chunk.
//
// Memory past the allocator's mmap threshold (32 MB) is fresh every time, and
// its page faults alone take one thread most of the copy, so from kShared on
// helper threads take chunks too, each through two slots of its own.  A new
// thread may first wait a scheduler tick (4 ms) for a CPU, so nobody waits for
// one: chunks are claimed one at a time, the caller carries whatever the
// helpers do not, and a helper that starts late finds none left.
// Into fresh memory, hipMemcpy / here: 2.8 MB 188 / 133 us, 6.6 MB 456 / 277,
// 15 MB 1.04 / 0.62 ms, 21.9 MB 1.49 / 0.86, 32 MB 2.20 / 1.24, 45 MB 4.32 /
// 1.34, 51.5 MB 5.04 / 1.49; into memory the caller keeps, 2.8 MB 154 / 112
// us, 21.9 MB 1.19 / 0.56 ms, 51.5 MB 2.95 / 1.30.  (Host to device the
// runtime already reaches 29-37 GB/s: those copies stay with it.)
//
// Memory that the device can write itself (pinned by the caller, managed, or
// device memory) gets one copy at the link's rate instead; through the slots
// it took twice that: 2.8 MB 58 / 118 us, 15 MB 271 / 625 us, 51.5 MB 0.91 /
// 1.30 ms.  Asking for the kind of memory takes 0.4 us.
#include "nsm_host_copy.h"

#include "nsm_copy_plan.h"
#include "nsm_kernels.h"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <new>
#include <thread>

namespace nsm {
namespace {

// pinned slots of one copy at a time
struct Ring {
  int        device = -1, slots = 0;
  size_t     bytes  = 0;
  char*      base   = nullptr;
  hipEvent_t done[kMaxSlots] = {};
};

// Idle rings: at most kIdle (at most 18 MB each), the largest of those given
// back, since a small ring is soon made again; released with the last holder.
constexpr int kIdle = 2;
struct Pool {
  std::mutex m;
  int        holders = 0, idle = 0;
  Ring*      ring[kIdle];
};
// never destroyed: copies may still run while the process ends
Pool& pool()
{
  static Pool* p = new Pool;
  return *p;
}

void destroy(Ring* r)
{
  for (hipEvent_t e : r->done)
    if (e) (void)hipEventDestroy(e);
  if (r->base) (void)hipHostFree(r->base);
  delete r;
}

Ring* take(int device, const CopyPlan& plan)
{
  const int    slots = plan.slots();
  const size_t bytes = plan.pinned();
  {
    Pool&                       p = pool();
    std::lock_guard<std::mutex> lk(p.m);
    for (int i = 0; i < p.idle; i++)
      if (p.ring[i]->device == device && p.ring[i]->slots >= slots && p.ring[i]->bytes >= bytes) {
        Ring* r   = p.ring[i];
        p.ring[i] = p.ring[--p.idle];
        return r;
      }
  }
  Ring* r = new (std::nothrow) Ring;
  if (!r) return nullptr;
  r->device = device;
  r->slots  = slots;
  r->bytes  = bytes;
  bool ok   = hipHostMalloc((void**)&r->base, bytes, hipHostMallocDefault) == hipSuccess;
  for (int i = 0; i < slots; i++)
    ok = ok && hipEventCreateWithFlags(&r->done[i], hipEventDisableTiming) == hipSuccess;
  if (ok) return r;
  (void)hipGetLastError();
  destroy(r);
  return nullptr;
}

void give_back(Ring* r)
{
  const auto smaller = [](const Ring* a, const Ring* b) { return a->bytes < b->bytes; };
  {
    Pool&                       p = pool();
    std::lock_guard<std::mutex> lk(p.m);
    if (p.holders > 0 && p.idle < kIdle) {
      p.ring[p.idle++] = r;
      return;
    }
    if (p.holders > 0) {
      Ring*& least = *std::min_element(p.ring, p.ring + kIdle, smaller);
      if (least->bytes < r->bytes) std::swap(least, r);
    }
  }
  destroy(r);
}

// One copy, shared by the caller and its helpers.  A helper counts itself
// active before it claims a chunk, so once every chunk is claimed and nobody
// is active, nobody touches the ring or the caller's memory again.
struct Copy {
  Ring*               ring;
  CopyPlan            plan;
  hipStream_t         stream;
  char*               dst;
  const char*         src;
  size_t              bytes, chunks;
  std::atomic<size_t> next{0};
  std::atomic<int>    active{0}, error{hipSuccess};

  // a chunk to carry, or `chunks` when none is left or the copy has failed
  size_t claim()
  {
    if (error.load() != hipSuccess) return chunks;
    return std::min(next.fetch_add(1), chunks);
  }
};

// Carries chunks through slots [slot0, slot0 + n) until none is left.
void carry(Copy& c, int slot0, int n)
{
  size_t     held[kMaxOwnSlots];  // chunk in each slot, in the order of the slots
  int        first = 0, count = 0;
  hipError_t e     = hipSuccess;
  const size_t chunk = c.plan.chunk;
  const auto   size  = [&](size_t k) { return std::min(chunk, c.bytes - k * chunk); };
  const auto fill  = [&] {  // the next chunk into the slot after the last held one
    const size_t k = c.claim();
    if (k >= c.chunks) return false;
    const int i = (first + count) % n;
    launch_copy_out((const double*)(c.src + k * chunk), (double*)(c.ring->base + (size_t)(slot0 + i) * chunk),
                    (int)(size(k) / sizeof(double)), c.stream);
    e = hipGetLastError();
    if (e == hipSuccess) e = hipEventRecord(c.ring->done[slot0 + i], c.stream);
    held[i] = k;
    count++;
    return e == hipSuccess;
  };
  bool more = true;
  while (more && count < n) more = fill();
  while (count > 0 && e == hipSuccess) {
    const int i = first;
    if ((e = hipEventSynchronize(c.ring->done[slot0 + i])) != hipSuccess) break;
    std::memcpy(c.dst + held[i] * chunk, c.ring->base + (size_t)(slot0 + i) * chunk, size(held[i]));
    first = (first + 1) % n;
    count--;
    if (more) more = fill();
  }
  if (e != hipSuccess) c.error.store(e);
}

hipError_t plain(hipStream_t stream, void* dst, const void* src, size_t bytes)
{
  const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream);
  const hipError_t d = hipStreamSynchronize(stream);
  return e != hipSuccess ? e : d;
}

// whether the runtime copies to dst without staging
bool direct(const void* dst)
{
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, dst) != hipSuccess) {
    (void)hipGetLastError();  // unknown to the runtime: pageable
    return false;
  }
  return a.type != hipMemoryTypeUnregistered;
}

hipError_t staged(int device, hipStream_t stream, char* dst, const char* src, size_t bytes, Ring* ring,
                  const CopyPlan& plan)
{
  const std::shared_ptr<Copy> c(
      new Copy{ring, plan, stream, dst, src, bytes, (bytes + plan.chunk - 1) / plan.chunk});
  try {
    for (int h = 0; h < plan.helpers; h++)
      std::thread([c, h, device] {
        c->active.fetch_add(1);
        if (c->next.load() < c->chunks) {
          const hipError_t e = hipSetDevice(device);
          if (e == hipSuccess)
            carry(*c, c->plan.own + h * kHelperSlots, kHelperSlots);
        }
        c->active.fetch_sub(1);
      }).detach();
  } catch (const std::exception&) {
    // no further thread: the caller carries the rest
  }
  carry(*c, 0, plan.own);
  while (c->active.load() > 0) std::this_thread::yield();
  return (hipError_t)c->error.load();
}

}  // namespace

hipError_t device_to_host(int device, hipStream_t stream, double* dst, const double* src, size_t count)
{
  const size_t bytes = count * sizeof(double);
  if (bytes < kStaged || direct(dst)) return plain(stream, dst, src, bytes);
  const CopyPlan plan = copy_plan(bytes);
  Ring* const    ring = take(device, plan);
  if (!ring) return plain(stream, dst, src, bytes);
  hipError_t e;
  try {
    e = staged(device, stream, (char*)dst, (const char*)src, bytes, ring, plan);
  } catch (const std::exception&) {  // no memory for the shared record: nothing was started
    e = plain(stream, dst, src, bytes);
  }
  // after an error a transfer may still be in flight
  if (e != hipSuccess) (void)hipStreamSynchronize(stream);
  give_back(ring);
  return e;
}

void host_copy_hold()
{
  std::lock_guard<std::mutex> lk(pool().m);
  pool().holders++;
}

void host_copy_release()
{
  Ring* drop[kIdle];
  int   n = 0;
  {
    Pool&                       p = pool();
    std::lock_guard<std::mutex> lk(p.m);
    if (--p.holders == 0)
      while (p.idle > 0) drop[n++] = p.ring[--p.idle];
  }
  for (int i = 0; i < n; i++) destroy(drop[i]);
}

}  // namespace nsm
