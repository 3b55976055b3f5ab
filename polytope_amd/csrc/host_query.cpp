// Host-buffer ray queries (ptx_intersect_closest).  The rays go to HBM and the
// hits come back through pinned host slots.  Up to four host threads each
// take a contiguous share of the caller's arrays and copy it chunk by chunk
// into their two slots while the DMA engine moves the chunk copied before, so
// the caller's pageable memory is read and written at host-memory speed and
// the link runs at the pinned DMA rate (about 57 GB/s each way on MI355X,
// against 28 GB/s host-to-device and 16 GB/s device-to-host for copies from
// pageable memory).  Chunks are 2 MiB: each copy call costs about 18 us that
// the DMA does not hide, so 1 MiB and 512 KiB chunks were slower.  A large call
// runs in parts: the kernel (the device query's, QueryLaunch) is launched on a
// part once its rays are resident, while the next part's go up and the hits of
// the one before come back.
#include "host_query.h"

#include <sched.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "scene.h"

namespace ptx {

HostQueryStaging::~HostQueryStaging() {
   (void)hipSetDevice(ordinal);
   for (hipEvent_t &e : events)
      if (e) (void)hipEventDestroy(e);
   for (uint32_t i = 0; i < kMaxParts; i++) {
      if (sent[i]) (void)hipEventDestroy(sent[i]);
      if (done[i]) (void)hipEventDestroy(done[i]);
   }
   if (up) (void)hipStreamDestroy(up);
   if (down) (void)hipStreamDestroy(down);
   if (pinned) (void)hipHostFree(pinned);
   if (d_buf) (void)hipFree(d_buf);
}

namespace {

constexpr size_t kSlot = HostQueryStaging::kSlotBytes;
// Rays of a part, at least, and parts a worker sends before the first comes
// back.  2^20 + 17 rays on 327,680 faces: 1.84 ms in one part, 1.49 in four of
// 2^18 (one or three ahead: 1.72 and 1.51), 2.00 in eight of 2^17, whose copies
// and launches cost more than the overlap gives; the link needs 0.88 both ways.
// With counters, whose kernel steps over binary records, parts gain as much: 2^19
// rays 1.35 ms in one part and 1.27 in two, 2^20 2.19 and 1.85, 2^22 7.44 and 5.70.
constexpr uint32_t kPartRays = 1u << 18;
constexpr uint32_t kAhead = 2;

// Host threads for one call: half the cores this process may run on, at most
// kMaxWorkers (four threads copy pageable to pinned memory at 60-75 GB/s,
// past what the link takes; eight gave no more).
uint32_t host_workers() {
   cpu_set_t cs;
   CPU_ZERO(&cs);
   unsigned c = sched_getaffinity(0, sizeof cs, &cs) == 0 ? unsigned(CPU_COUNT(&cs)) : std::thread::hardware_concurrency();
   return std::clamp<uint32_t>(c / 2, 1u, HostQueryStaging::kMaxWorkers);
}

// Worker w's share of the spans: bytes [total * w / workers, total * (w + 1) /
// workers) of their concatenation, cut at the spans' ends and every kSlot
// bytes.
std::vector<Piece> share(const std::vector<Span> &spans, uint32_t w, uint32_t workers) {
   size_t total = 0;
   for (const Span &a : spans) total += a.bytes;
   const size_t lo = total / workers * w + total % workers * w / workers;
   const size_t hi = total / workers * (w + 1) + total % workers * (w + 1) / workers;
   std::vector<Piece> out;
   size_t base = 0;
   for (const Span &a : spans) {
      const size_t b0 = std::max(lo, base), b1 = std::min(hi, base + a.bytes);
      for (size_t off = b0; off < b1; off += kSlot)
         out.push_back(Piece{a.host + (off - base), a.dev + (off - base), std::min(kSlot, b1 - off)});
      base += a.bytes;
   }
   return out;
}

// The host spans that go up before a part's launch and the device spans that
// come back after it.
struct Part {
   std::vector<Span> in, out;
};

// State one call's workers share.  The calling thread launches a part
// (`between`) once every worker has queued its copies; a worker queues a part's
// copies up, then copies the part before it back.  A failed step ends the call:
// the rest is skipped.  A call of one part copies on the launch's stream, a
// call of several on the staging's own, one for each direction.
struct HostCall {
   HostQueryStaging *st;
   hipStream_t stream;
   int ordinal;
   uint32_t workers = 1;
   std::vector<Part> parts;
   std::mutex mu;
   std::condition_variable cv;
   uint32_t arrived[HostQueryStaging::kMaxParts] = {};
   uint32_t launched = 0;             // parts whose hits may be waited for
   bool stop = false;
   std::string error;

   bool several() const { return parts.size() > 1; }
   void fail(const std::string &m) {
      std::lock_guard<std::mutex> lock(mu);
      if (error.empty()) error = m;
      stop = true;
      cv.notify_all();
   }
   bool ok(hipError_t e, const char *what) {
      if (e == hipSuccess) return true;
      (void)hipGetLastError();
      fail(std::string(what) + ": " + hipGetErrorString(e));
      return false;
   }
   // slot and event k of a worker's two in one direction
   char *slot(uint32_t w, uint32_t back, uint32_t k) const {
      return st->pinned + (4 * size_t(w) + 2 * back + (k & 1)) * kSlot;
   }
   hipEvent_t event(uint32_t w, uint32_t back, uint32_t k) const { return st->events[4 * w + 2 * back + (k & 1)]; }

   // Worker w's share of a part going up: copy a piece into a slot, then queue
   // its DMA; a slot is refilled once the DMA that read it has finished.  used:
   // pieces this worker has sent in the call.
   bool send(uint32_t w, const Part &part, uint32_t &used) {
      const hipStream_t s = several() ? st->up : stream;
      for (const Piece &p : share(part.in, w, workers)) {
         const uint32_t k = used++;
         if (k >= 2 && !ok(hipEventSynchronize(event(w, 0, k)), "hipEventSynchronize")) return false;
         std::memcpy(slot(w, 0, k), p.host, p.len);
         if (!ok(hipMemcpyAsync(p.dev, slot(w, 0, k), p.len, hipMemcpyHostToDevice, s), "hipMemcpyAsync")) return false;
         if (!ok(hipEventRecord(event(w, 0, k), s), "hipEventRecord")) return false;
      }
      return true;
   }

   // Worker w's share of a part coming back: the DMA of piece k + 1 is queued
   // before piece k is copied out of its slot.
   bool receive(uint32_t w, uint32_t c) {
      const std::vector<Piece> ps = share(parts[c].out, w, workers);
      if (ps.empty()) return true;
      hipStream_t s = stream;
      if (several()) {
         s = st->down;
         if (!ok(hipEventSynchronize(st->done[c]), "hipEventSynchronize")) return false;
      }
      auto queue = [&](uint32_t k) {
         return ok(hipMemcpyAsync(slot(w, 1, k), ps[k].dev, ps[k].len, hipMemcpyDeviceToHost, s), "hipMemcpyAsync") &&
                ok(hipEventRecord(event(w, 1, k), s), "hipEventRecord");
      };
      if (!queue(0)) return false;
      for (uint32_t k = 0; k < ps.size(); k++) {
         if (k + 1 < ps.size() && !queue(k + 1)) return false;
         if (!ok(hipEventSynchronize(event(w, 1, k)), "hipEventSynchronize")) return false;
         std::memcpy(ps[k].host, slot(w, 1, k), ps[k].len);
      }
      return true;
   }

   void worker(uint32_t w) {
      if (!ok(hipSetDevice(ordinal), "hipSetDevice")) return;
      uint32_t used = 0;
      // up to kAhead parts go up before the first comes back
      for (uint32_t c = 0; c < parts.size() + kAhead; c++) {
         if (c < parts.size()) {
            if (!send(w, parts[c], used)) return;
            std::lock_guard<std::mutex> lock(mu);
            arrived[c]++;
            cv.notify_all();
         }
         if (c < kAhead) continue;
         {
            std::unique_lock<std::mutex> lock(mu);
            cv.wait(lock, [&] { return stop || launched > c - kAhead; });
            if (stop) return;
         }
         if (!receive(w, c - kAhead)) return;
      }
   }

   // Launches part c behind its rays.
   template <class F>
   int launch(uint32_t c, F &between) {
      if (!several()) return between(c);
      if (!ok(hipEventRecord(st->sent[c], st->up), "hipEventRecord") ||
          !ok(hipStreamWaitEvent(stream, st->sent[c], 0), "hipStreamWaitEvent"))
         return PTX_ERR_HIP;
      if (const int rc = between(c)) return rc;
      return ok(hipEventRecord(st->done[c], stream), "hipEventRecord") ? PTX_OK : PTX_ERR_HIP;
   }

   // The whole call on the calling thread and up to `workers` threads.
   template <class F>
   int run(F between) {
      size_t in_bytes = 0, out_bytes = 0;
      for (const Part &p : parts) {
         for (const Span &a : p.in) in_bytes += a.bytes;
         for (const Span &a : p.out) out_bytes += a.bytes;
      }
      const size_t pieces = (std::max(in_bytes, out_bytes) + kSlot - 1) / kSlot;
      workers = uint32_t(std::min<size_t>(host_workers(), std::max<size_t>(1, pieces)));
      int rc = PTX_OK;
      if (workers == 1) {
         uint32_t used = 0;
         for (uint32_t c = 0; c < parts.size() + kAhead && rc == PTX_OK && !stop; c++) {
            if (c < parts.size() && send(0, parts[c], used)) rc = launch(c, between);
            if (c >= kAhead && rc == PTX_OK && !stop) receive(0, c - kAhead);
         }
      } else {
         std::vector<std::thread> ts;
         ts.reserve(workers);
         try {
            for (uint32_t w = 0; w < workers; w++) ts.emplace_back([this, w] { worker(w); });
         } catch (const std::exception &) {
            fail("could not start the host copy threads");
         }
         for (uint32_t c = 0; c < parts.size(); c++) {
            {
               std::unique_lock<std::mutex> lock(mu);
               cv.wait(lock, [&] { return stop || arrived[c] == workers; });
               if (stop) break;
            }
            rc = launch(c, between);
            std::lock_guard<std::mutex> lock(mu);
            if (rc == PTX_OK) launched = c + 1;
            else stop = true;
            cv.notify_all();
            if (stop) break;
         }
         for (std::thread &th : ts) th.join();
      }
      // every queued copy has finished before the slots serve another call
      hipError_t se = several() ? hipStreamSynchronize(st->up) : hipSuccess;
      const hipError_t ss = hipStreamSynchronize(stream), sd = several() ? hipStreamSynchronize(st->down) : hipSuccess;
      if (se == hipSuccess) se = ss != hipSuccess ? ss : sd;
      if (!error.empty()) return set_error(PTX_ERR_HIP, error);
      if (rc != PTX_OK) return rc;
      if (se != hipSuccess) {
         (void)hipGetLastError();
         return set_error(PTX_ERR_HIP, std::string("hipStreamSynchronize: ") + hipGetErrorString(se));
      }
      return PTX_OK;
   }
};

int ensure_staging(ptx_device *dev, size_t need) {
   if (!dev->host_query) {
      dev->host_query = std::make_unique<HostQueryStaging>();
      dev->host_query->ordinal = dev->ordinal;
   }
   HostQueryStaging &st = *dev->host_query;
   if (!st.ready) {
      // what an earlier failed call made is kept and not made again
      if (!st.pinned)
         PTX_HIP_TRY(hipHostMalloc(reinterpret_cast<void **>(&st.pinned), 4 * HostQueryStaging::kMaxWorkers * kSlot,
                                   hipHostMallocDefault));
      for (hipEvent_t &e : st.events)
         if (!e) PTX_HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
      for (uint32_t i = 0; i < HostQueryStaging::kMaxParts; i++)
         for (hipEvent_t *e : {&st.sent[i], &st.done[i]})
            if (!*e) PTX_HIP_TRY(hipEventCreateWithFlags(e, hipEventDisableTiming));
      for (hipStream_t *s : {&st.up, &st.down})
         if (!*s) PTX_HIP_TRY(hipStreamCreateWithFlags(s, hipStreamNonBlocking));
      st.ready = true;
   }
   if (need > st.d_cap) {
      if (st.d_buf) PTX_HIP_TRY(hipFree(st.d_buf));
      st.d_buf = nullptr;
      st.d_cap = 0;
      PTX_HIP_TRY(hipMalloc(reinterpret_cast<void **>(&st.d_buf), need));
      st.d_cap = need;
   }
   return PTX_OK;
}

size_t round_up(size_t b) { return (b + 255) & ~size_t(255); }

}  // namespace

int intersect_host(ptx_scene *s, const float *rays, uint32_t n, ptx_hit *hits, ptx_ray_counters *counters) {
   ptx_device *dev = s->dev;
   const size_t b_rays = round_up(size_t(n) * 24), b_hits = round_up(size_t(n) * sizeof(ptx_hit));
   const size_t b_cnt = counters ? round_up(size_t(n) * sizeof(ptx_ray_counters)) : 0;
   if (int rc = ensure_staging(dev, b_rays + b_hits + b_cnt)) return rc;
   HostQueryStaging &st = *dev->host_query;
   HostCall call;
   call.st = &st;
   call.stream = dev->stream;
   call.ordinal = dev->ordinal;
   char *d_hits = st.d_buf + b_rays, *d_cnt = counters ? d_hits + b_hits : nullptr;
   const uint32_t np = std::clamp<uint32_t>(n / kPartRays, 1u, HostQueryStaging::kMaxParts);
   // parts of whole batches, the last one taking the rest
   const uint32_t each = n / np & ~63u;
   auto first = [&](uint32_t c) { return size_t(c) * each; };
   auto count = [&](uint32_t c) { return c + 1 < np ? each : n - (np - 1) * each; };
   for (uint32_t c = 0; c < np; c++) {
      const size_t f = first(c), m = count(c);
      Part p;
      p.in.push_back(Span{reinterpret_cast<char *>(const_cast<float *>(rays + 6 * f)), st.d_buf + f * 24, m * 24});
      p.out.push_back(Span{reinterpret_cast<char *>(hits + f), d_hits + f * sizeof(ptx_hit), m * sizeof(ptx_hit)});
      if (counters)
         p.out.push_back(Span{reinterpret_cast<char *>(counters + f), d_cnt + f * sizeof(ptx_ray_counters),
                              m * sizeof(ptx_ray_counters)});
      call.parts.push_back(std::move(p));
   }
   // one scratch for all parts, which run one after another: given back between
   // them it made the next launch wait for the one before
   const ptx_tuning t = tuning_of(dev);
   QueryLaunch q(s, n, d_cnt != nullptr, false, t);
   if (int rc = q.take_scratch(call.stream)) return rc;
   const int rc = call.run([&](uint32_t c) {
      const size_t f = first(c);
      return q.launch(reinterpret_cast<const float *>(st.d_buf + f * 24), count(c),
                      reinterpret_cast<ptx_hit *>(d_hits) + f,
                      d_cnt ? reinterpret_cast<ptx_ray_counters *>(d_cnt) + f : nullptr, nullptr, call.stream);
   });
   const int free_rc = q.give_scratch(call.stream);
   return rc ? rc : free_rc;
}

int download_host(ptx_device *dev, hipStream_t stream, const std::vector<Span> &spans) {
   if (int rc = ensure_staging(dev, 0)) return rc;
   HostCall call;
   call.st = dev->host_query.get();
   call.stream = stream;
   call.ordinal = dev->ordinal;
   call.parts.push_back(Part{{}, spans});
   return call.run([](uint32_t) { return int(PTX_OK); });
}

}  // namespace ptx
