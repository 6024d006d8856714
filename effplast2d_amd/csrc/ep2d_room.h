// ep2d_room.h -- which handles and batches of this process are at work on a
// device, and which handles may run resident (ep2d_resident.hip) side by side.
#pragma once

#include <algorithm>
#include <chrono>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "ep2d_internal.h"

namespace ep2d {

// What one handle, or batch, has on a device.  Its fields are the room's while the
// handle is in it.
struct RoomUser {
  hipStream_t stream = nullptr;      // its work
  unsigned half = 0, whole = 0;      // its resident tiles (0, 0: it has no such shape)
  const unsigned* told = nullptr;    // pinned words a resident run writes when it ends
  unsigned run = 0;                  // the resident run it has in flight (0: none)
  bool atWork = false;               // other work may be in flight
  bool held = false;                 // its stream must not be asked (a capture is on),
                                     // or need not be (a batch in a step)
  std::thread::id thread;            // the thread it was last used by, and when;
  std::chrono::steady_clock::time_point used, asked;  // when its stream was last asked
};

// While a stream is being captured, waiting for another stream, or asking it, is
// refused and ends the capture; a thread in the relaxed mode may do both.  For
// the library's own streams, of which none is being captured then.
class RelaxedCapture {
 public:
  RelaxedCapture() { on_ = hipThreadExchangeStreamCaptureMode(&mode_) == hipSuccess; }
  ~RelaxedCapture() {
    if (on_) (void)hipThreadExchangeStreamCaptureMode(&mode_);
  }
  RelaxedCapture(const RelaxedCapture&) = delete;
  RelaxedCapture& operator=(const RelaxedCapture&) = delete;

 private:
  hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
  bool on_ = false;
};

// The words: the last run that has completed, and how a run failed (0: none did).
inline bool run_ended(const unsigned* told, unsigned run) {
  return __atomic_load_n(told, __ATOMIC_ACQUIRE) == run ||
         __atomic_load_n(told + 1, __ATOMIC_ACQUIRE) != 0;
}

// The handles and batches of this process on one device.
class DeviceRoom {
 public:
  static constexpr size_t kQueues = 4;  // HIP's default (GPU_MAX_HW_QUEUES)
  static DeviceRoom& of(int device) {
    // never destroyed: handles may outlive static objects
    static std::mutex* m = new std::mutex;
    static auto* rooms = new std::map<int, DeviceRoom>;
    const std::lock_guard<std::mutex> lock(*m);
    return (*rooms)[device];
  }
  void join(RoomUser* u) {
    const std::lock_guard<std::mutex> lock(m_);
    users_.push_back(u);
  }
  // (its work is done: the stream is idle)
  void leave(RoomUser* u) {
    const std::lock_guard<std::mutex> lock(m_);
    users_.erase(std::remove(users_.begin(), users_.end(), u), users_.end());
  }
  // Before work of `me` is enqueued: 0 if the resident run `run` (0: none) may be
  // launched, else the handles at work, `me` among them (counted to 3).  It may
  // be if it fits the device beside the resident tiles of the others that can
  // run at once with it, the largest: the process has kQueues hardware queues,
  // and launches of streams that share one run one after another.  The launch
  // itself counts exactly.
  // Resident tiles keep their CUs for the whole run, so beside work that is not
  // resident (a batch, a larger grid) they take a quarter of the device at most.
  // A batch of 20 split 1024^2 (124 ms a pass alone) beside a handle that runs
  // intervals of 500 iterations: FP64 128^2 (48 CUs) resident 142 ms a pass and
  // 2.7 ms an interval, on the chains 134 and 11; FP64 512^2 (240 CUs) resident
  // 612 and 3.2, on the chains 139 and 16 (on tiles, each iteration a launch,
  // 151 and 15).
  int enter(RoomUser* me, unsigned run, unsigned cus) {
    const std::lock_guard<std::mutex> lock(m_);
    touch(me);
    int n = 1;
    bool all = run != 0, shared = false;
    std::vector<const RoomUser*> at;
    for (RoomUser* u : users_) {
      if (run == 0 && n >= 3) break;
      if (u == me || !busy(*u, *me)) continue;
      n++;
      at.push_back(u);
      shared = shared || u->half + u->whole == 0;
    }
    if (at.size() >= kQueues)
      std::sort(at.begin(), at.end(), [](const RoomUser* a, const RoomUser* b) {
        return a->half + 2 * a->whole > b->half + 2 * b->whole;
      });
    unsigned half = me->half, whole = me->whole;
    for (size_t k = 0; k < std::min(at.size(), kQueues - 1); k++) {
      half += at[k]->half;
      whole += at[k]->whole;
    }
    all = all && (shared ? half + whole <= cus / 4 : resident_fits(cus, half, whole));
    // (a run that is turned down leaves those before it in the entry; the other
    // kernels' launches, run 0, come when the handle has none in flight)
    if (all || run == 0) me->run = run;
    if (run == 0) me->atWork = true;
    return all ? 0 : n;
  }
  // Before launches that do not depend on the others'.
  void work(RoomUser* me) {
    const std::lock_guard<std::mutex> lock(m_);
    touch(me);
    me->run = 0;
    me->atWork = true;
  }
  // The stream of `me` has been waited for.
  void idle(RoomUser* me) {
    const std::lock_guard<std::mutex> lock(m_);
    touch(me);
    me->run = 0;
    me->atWork = false;
  }
  // A batch's step.
  void work(RoomUser* me, bool on) {
    const std::lock_guard<std::mutex> lock(m_);
    me->atWork = me->held = on;
  }
  void hold(RoomUser* me, bool on) {
    const std::lock_guard<std::mutex> lock(m_);
    me->held = on;
  }

 private:
  // Whether u is at work, seen from `me`, which has just been touched.  A stream
  // takes about 5 us to answer, as long as a short call takes, so it is asked
  // only so often.  A handle that another thread used a moment ago counts as at
  // work between its calls too: 4 FP64 handles of 512^2 on a thread each, 40
  // iterations and a residual a call, took 220 us a call while each went
  // resident whenever the others were between calls (on tiles 151, on chains
  // for several throughout 130).  Handles of one thread, waited for in turn, do
  // not see each other.
  static bool busy(RoomUser& u, const RoomUser& me) {
    using std::chrono::microseconds;
    if (u.run != 0 && run_ended(u.told, u.run)) u.run = 0;
    if (u.atWork && !u.held && me.used - u.asked >= microseconds(300)) {
      u.asked = me.used;
      const RelaxedCapture relaxed;
      if (hipStreamQuery(u.stream) == hipSuccess) u.atWork = false;
      else (void)hipGetLastError();
    }
    return u.run != 0 || u.atWork ||
           (u.thread != me.thread && me.used - u.used < microseconds(2000));
  }
  static void touch(RoomUser* me) {
    me->thread = std::this_thread::get_id();
    me->used = std::chrono::steady_clock::now();
  }
  std::mutex m_;
  std::vector<RoomUser*> users_;
};

}  // namespace ep2d
