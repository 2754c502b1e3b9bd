// Which decode call of this process has the resident launch of a device (host only).
//
// Two resident launches that each held part of the CUs would wait for CUs the other holds
// until their polls run out, so a device has one turn, held from the first launch of a call
// until everything it launched has finished.  The turn is this process's: launches of
// processes that share a device were measured to run one process at a time (two processes,
// 945 calls each in 8 s, no wait ran out), and where they do not, the polls end it.
#pragma once
#include <atomic>
#include <functional>
#include <utility>

namespace mlg {

// A decode call that never takes the launch (a batch, beam search) while it runs.  A resident
// launch beside it holds more than half of the CUs and polls: sentences one by one in one
// context and batches of 16 in another took 5.2 and 14.1 ms per call, against 9.0 and 12.4 with
// the per-layer launches, 1322 sentences per second instead of 1408.  So none starts meanwhile.
// (Single sentences from 2, 3 and 4 contexts: 283, 327 and 349 per second with the resident
// launch for one of them at a time, 230, 294 and 340 without.)
class OtherDecode {
  public:
    explicit OtherDecode(int device) : device_(device) { count(device_).fetch_add(1, std::memory_order_relaxed); }
    OtherDecode(const OtherDecode &) = delete;
    OtherDecode &operator=(const OtherDecode &) = delete;
    ~OtherDecode() { count(device_).fetch_sub(1, std::memory_order_relaxed); }
    static bool running(int device) { return count(device).load(std::memory_order_relaxed) > 0; }

  private:
    static std::atomic<int> &count(int device) {
        static std::atomic<int> n[64];
        return n[device & 63];
    }
    int device_;
};

class ResidentTurn {
  public:
    // drain: waits for everything the call has launched
    ResidentTurn(int device, std::function<void()> drain) : device_(device), drain_(std::move(drain)) {}
    ResidentTurn(const ResidentTurn &) = delete;
    ResidentTurn &operator=(const ResidentTurn &) = delete;
    ~ResidentTurn() {  // a call that fails on the way still has launches on the stream
        if (taken_) drain_();
        done();
    }
    bool take() {
        return taken_ = !OtherDecode::running(device_) && !turn(device_).exchange(true, std::memory_order_acquire);
    }
    // the call's launches have finished
    void done() {
        if (taken_) turn(device_).store(false, std::memory_order_release);
        taken_ = false;
    }

  private:
    static std::atomic<bool> &turn(int device) {
        static std::atomic<bool> t[64];
        return t[device & 63];
    }
    int device_;
    std::function<void()> drain_;
    bool taken_ = false;
};

}  // namespace mlg
