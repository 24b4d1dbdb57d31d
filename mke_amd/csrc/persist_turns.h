// Which persistent launches (persist.hip) of a process run at the same time on
// one device: as many as are sure to be resident together.  Two that each
// held half of the CUs would wait for each other until they give up.
#pragma once
#include <algorithm>
#include <condition_variable>
#include <mutex>

namespace phg {

// Workgroups go round the 8 XCDs and round each XCD's four shader engines, so
// a launch puts at most every 32nd of its workgroups on one engine, whichever
// it begins with.  An engine has 8 CUs and a workgroup needs one at most:
// launches fit together while their workgroups, counted in 32s, are no more
// than the device's CUs in 32s.  The threads that wait take their turns in
// the order in which they came, so a launch that needs the whole device is
// not passed for ever by small ones.  Level-4 solves (22 workgroups) of 2 and
// 4 threads: 6,800 and 13,150 a second, with one turn for the whole device 3,430.
class PersistTurns {
    std::mutex mu;
    std::condition_variable cv;
    int most, used = 0;
    unsigned long next = 0, now = 0;

    int units(int workgroups) const { return std::min((workgroups + 31) / 32, most); }
    bool fits(int workgroups) const { return used + units(workgroups) <= most; }

public:
    explicit PersistTurns(int cus) : most(std::max(1, cus / 32)) {}
    bool try_enter(int workgroups)
    {
        std::lock_guard<std::mutex> l(mu);
        if (next != now || !fits(workgroups)) return false;
        used += units(workgroups);
        return true;
    }
    void enter(int workgroups)
    {
        std::unique_lock<std::mutex> l(mu);
        const unsigned long mine = next++;
        cv.wait(l, [&] { return mine == now && fits(workgroups); });
        ++now;
        used += units(workgroups);
        cv.notify_all();  // the next one may fit too
    }
    void leave(int workgroups)
    {
        std::lock_guard<std::mutex> l(mu);
        used -= units(workgroups);
        cv.notify_all();
    }
};

}  // namespace phg
