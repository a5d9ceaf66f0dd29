// Admission of resident grids to one device's CUs, in the order asked. Host code without HIP.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <cstdint>
#include <deque>
#include <mutex>

namespace hoefem {

// A launch takes a place in the line and gets its CUs when it is at the front and they are free. Without the
// order, launches that need few CUs could pass one that needs most of them for ever (a solve of 240 work-groups
// beside threads that step small scenes).
class CuLine {
public:
    // The work-groups of a launch are dealt to the XCDs in turn, the first to the same one each time, and one that
    // finds its XCD full waits there although others have room. A launch is therefore charged the same number of
    // CUs on every XCD, the most that any of them gets: launches of 82, 82 and 90 work-groups (254) would put 34 on
    // an XCD of 32 CUs.
    static constexpr int XCDS = 8;
    static int charge(int wgs) { return (wgs + XCDS - 1) / XCDS * XCDS; }

    explicit CuLine(int cus) : cus_(cus), free_(cus) {}
    int cus() const { return cus_; }

    uint64_t enter() {
        std::lock_guard<std::mutex> lock(mu_);
        line_.push_back(++last_);
        return last_;
    }
    // n CUs (at most cus()) for the holder of the place, who thereby leaves the line; false, with the place kept: not
    // yet (never with wait)
    bool take(uint64_t place, int n, bool wait) {
        std::unique_lock<std::mutex> lock(mu_);
        auto ready = [&] { return line_.front() == place && free_ >= n; };
        if (wait)
            cv_.wait(lock, ready);
        else if (!ready())
            return false;
        line_.pop_front();
        free_ -= n;
        cv_.notify_all();  // the next one may fit beside it
        return true;
    }
    // n more CUs for a launch that has its place behind it, if they are free and nobody waits
    bool take_more(int n) {
        std::lock_guard<std::mutex> lock(mu_);
        if (!line_.empty() || free_ < n) return false;
        free_ -= n;
        return true;
    }
    void leave(uint64_t place) {
        std::lock_guard<std::mutex> lock(mu_);
        line_.erase(std::remove(line_.begin(), line_.end(), place), line_.end());
        cv_.notify_all();
    }
    void give(int n) {
        std::lock_guard<std::mutex> lock(mu_);
        free_ += n;
        cv_.notify_all();
    }

private:
    const int cus_;
    int free_;
    uint64_t last_ = 0;
    std::deque<uint64_t> line_;
    std::mutex mu_;
    std::condition_variable cv_;
};

}  // namespace hoefem
