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
    bool take() { return taken_ = !turn(device_).exchange(true, std::memory_order_acquire); }
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
