// zr_transfer.hpp -- per-particle arrays between the caller's memory (the
// reference's particle-major layout) and the engine's structure of arrays.
// Included by zr_engine.hip inside its anonymous namespace, after zr_engine.
//
// A pageable copy of fresh host memory runs at 9-10 GB/s here (one thread,
// page faults included) where the link carries 57 GB/s from pinned memory, and
// every call allocated and freed its device scratch.  So the arrays of a call,
// taken as one stream of doubles, are cut into windows of 4 MiB; up to eight
// threads, the caller among them, each take the next window, have it packed by
// a kernel into a device buffer of their own, copied to a pinned buffer of
// their own, and copy that to the caller's pages (uploads the other way
// round).  A call of one window has the kernel store into the pinned buffer
// and no thread is made.  2.1M particles (403 MB) down: 40 -> 11 ms.
//
// The pinned buffers are the process's (at most 32 MiB, made as needed, freed
// with the last engine); a transfer holds their lock, so that engines in
// several threads take turns on the link.  Device buffers and events belong to
// the engine.

constexpr uint64_t kWindow = uint64_t(1) << 19;  // doubles

struct PinnedPool {
  std::mutex lock;
  int engines = 0;
  void* buf[kIoThreads] = {};
};
PinnedPool g_pinned;

void pinned_acquire()
{
  std::lock_guard<std::mutex> hold(g_pinned.lock);
  ++g_pinned.engines;
}
void pinned_release()
{
  std::lock_guard<std::mutex> hold(g_pinned.lock);
  if (--g_pinned.engines > 0) return;
  for (auto& b : g_pinned.buf) {
    if (b) (void)hipHostFree(b);
    b = nullptr;
  }
}

// elements [begin, begin + count) of the particle-major array with nc
// components; place: the engine's place of each of the caller's particles
// (null: the same)
__global__ __launch_bounds__(256) void k_pack(const double* __restrict__ soa, double* __restrict__ out, uint64_t begin,
                                              uint32_t count, uint32_t nc, int64_t stride,
                                              const uint32_t* __restrict__ place)
{
  const uint32_t k = blockIdx.x * 256u + threadIdx.x;
  if (k >= count) return;
  const uint64_t t = begin + k;
  const uint32_t i = (uint32_t)(t / nc), c = (uint32_t)(t - (uint64_t)i * nc);
  out[k] = soa[c * stride + (place ? place[i] : i)];
}
__global__ __launch_bounds__(256) void k_unpack(double* __restrict__ soa, const double* __restrict__ in,
                                                uint64_t begin, uint32_t count, uint32_t nc, int64_t stride)
{
  const uint32_t k = blockIdx.x * 256u + threadIdx.x;
  if (k >= count) return;
  const uint64_t t = begin + k;
  const uint32_t i = (uint32_t)(t / nc), c = (uint32_t)(t - (uint64_t)i * nc);
  soa[c * stride + i] = in[k];
}
__global__ __launch_bounds__(256) void k_places(uint32_t n, const uint32_t* __restrict__ uid, uint32_t* __restrict__ place)
{
  const uint32_t k = blockIdx.x * 256u + threadIdx.x;
  if (k < n) place[uid[k]] = k;
}

struct HostArray {
  double* host;  // null: skipped
  double* dev;   // nc rows of n
  int nc;
};

struct TransferJob {
  zr_engine* e;
  const HostArray* items;
  int count;
  bool to_host;
  int device;
  uint64_t total;
  const uint32_t* place;
  std::atomic<uint64_t> next{ 0 };
  std::atomic<int> error{ 0 };
};

// f(item, first element, count, offset in the window) for the items' parts in
// window w
template <class Fn>
void window_parts(const TransferJob& J, uint64_t w, Fn f)
{
  const uint64_t lo = w * kWindow, hi = lo + kWindow < J.total ? lo + kWindow : J.total;
  uint64_t at = 0;
  for (int q = 0; q < J.count; ++q) {
    const uint64_t len = J.items[q].host ? (uint64_t)J.e->n * (uint64_t)J.items[q].nc : 0u;
    const uint64_t a = lo > at ? lo : at, b = hi < at + len ? hi : at + len;
    if (a < b) f(J.items[q], a - at, (uint32_t)(b - a), a - lo);
    at += len;
  }
}
uint64_t window_size(const TransferJob& J, uint64_t w)
{
  return (w + 1) * kWindow < J.total ? kWindow : J.total - w * kWindow;
}
void pack_window(TransferJob& J, uint64_t w, double* out)
{
  window_parts(J, w, [&](const HostArray& a, uint64_t begin, uint32_t m, uint64_t off) {
    k_pack<<<blocks_for(m, 256), 256, 0, J.e->stream>>>(a.dev, out + off, begin, m, (uint32_t)a.nc, J.e->n, J.place);
  });
}
void unpack_window(TransferJob& J, uint64_t w, const double* in)
{
  window_parts(J, w, [&](const HostArray& a, uint64_t begin, uint32_t m, uint64_t off) {
    k_unpack<<<blocks_for(m, 256), 256, 0, J.e->stream>>>(a.dev, in + off, begin, m, (uint32_t)a.nc, J.e->n);
  });
}
void copy_window(const TransferJob& J, uint64_t w, double* buf)
{
  window_parts(J, w, [&](const HostArray& a, uint64_t begin, uint32_t m, uint64_t off) {
    if (J.to_host)
      memcpy(a.host + begin, buf + off, (size_t)m * sizeof(double));
    else
      memcpy(buf + off, a.host + begin, (size_t)m * sizeof(double));
  });
}

// one thread's share, with its own buffers; HIP errors are left in J.error
void transfer_worker(TransferJob* J, int t)
{
  zr_engine* e = J->e;
  double* const pin = static_cast<double*>(g_pinned.buf[t]);
  double* const dev = e->io_dev + (size_t)t * kWindow;
  hipError_t st = hipSetDevice(J->device);
  bool inflight = false;
  const uint64_t windows = (J->total + kWindow - 1) / kWindow;
  while (st == hipSuccess && J->error.load() == 0) {
    const uint64_t w = J->next.fetch_add(1);
    if (w >= windows) break;
    const size_t bytes = window_size(*J, w) * sizeof(double);
    if (J->to_host) {
      pack_window(*J, w, dev);
      st = hipGetLastError();
      if (st == hipSuccess) st = hipMemcpyAsync(pin, dev, bytes, hipMemcpyDeviceToHost, e->stream);
      if (st == hipSuccess) st = hipEventRecord(e->io_ev[t], e->stream);
      if (st == hipSuccess) st = hipEventSynchronize(e->io_ev[t]);
      if (st == hipSuccess) copy_window(*J, w, pin);
    } else {
      if (inflight) st = hipEventSynchronize(e->io_ev[t]);
      if (st != hipSuccess) break;
      copy_window(*J, w, pin);
      st = hipMemcpyAsync(dev, pin, bytes, hipMemcpyHostToDevice, e->stream);
      if (st == hipSuccess) {
        unpack_window(*J, w, dev);
        st = hipGetLastError();
      }
      if (st == hipSuccess) st = hipEventRecord(e->io_ev[t], e->stream);
      inflight = st == hipSuccess;
    }
  }
  if (inflight) st = hipEventSynchronize(e->io_ev[t]);
  if (st != hipSuccess) J->error.store((int)st);
}

// in_place_order: the arrays are in the engine's current order of particles
// (downloads; the adjoints stay in the caller's)
int transfer_arrays(zr_engine* e, const HostArray* items, int count, bool to_host, bool in_place_order)
{
  TransferJob J;
  J.e = e;
  J.items = items;
  J.count = count;
  J.to_host = to_host;
  J.place = nullptr;
  J.total = 0;
  for (int q = 0; q < count; ++q)
    if (items[q].host) J.total += (uint64_t)e->n * (uint64_t)items[q].nc;
  if (J.total == 0) return ZR_OK;
  ZR_HIP(e, hipGetDevice(&J.device));
  std::lock_guard<std::mutex> hold(g_pinned.lock);
  const uint64_t windows = (J.total + kWindow - 1) / kWindow;
  int threads = windows < (uint64_t)kIoThreads ? (int)windows : kIoThreads;
  for (int t = 0; t < threads; ++t) {
    if (!g_pinned.buf[t])
      ZR_HIP(e, hipHostMalloc(&g_pinned.buf[t], kWindow * sizeof(double),
                              hipHostMallocPortable | hipHostMallocCoherent));
  }
  if (to_host && in_place_order && e->permuted) {
    // the sort's key array (8 bytes per particle, written again before every
    // use) holds the inverse of uid
    uint32_t* const place = reinterpret_cast<uint32_t*>(e->keys);
    k_places<<<blocks_for((uint64_t)e->n, 256), 256, 0, e->stream>>>((uint32_t)e->n, e->uid, place);
    ZR_LAUNCH_CHECK(e);
    J.place = place;
  }
  if (windows == 1) {
    double* const pin = static_cast<double*>(g_pinned.buf[0]);
    if (to_host) {
      pack_window(J, 0, pin);
      ZR_LAUNCH_CHECK(e);
      int rc = sync_counts(e);
      if (rc) return rc;
      copy_window(J, 0, pin);
    } else {
      copy_window(J, 0, pin);
      unpack_window(J, 0, pin);
      ZR_LAUNCH_CHECK(e);
      ZR_HIP(e, hipStreamSynchronize(e->stream));
    }
    return ZR_OK;
  }
  if (e->io_threads < threads) {
    dfree(e->io_dev);
    e->io_threads = 0;
    ZR_HIP(e, dev_malloc(e, &e->io_dev, (size_t)threads * kWindow * sizeof(double)));
    e->io_threads = threads;
  }
  for (int t = 0; t < threads; ++t)
    if (!e->io_ev[t]) ZR_HIP(e, hipEventCreateWithFlags(&e->io_ev[t], hipEventDisableTiming));
  std::vector<std::thread> team;
  try {
    team.reserve((size_t)threads);
    for (int t = 1; t < threads; ++t) team.emplace_back(transfer_worker, &J, t);
  } catch (...) {  // fewer threads: the ones there are take every window
  }
  transfer_worker(&J, 0);
  for (auto& th : team) th.join();
  if (J.error.load() != 0)
    return fail(e, ZR_ERR_HIP, std::string("particle transfer: ") + hipGetErrorString((hipError_t)J.error.load()));
  return ZR_OK;
}
