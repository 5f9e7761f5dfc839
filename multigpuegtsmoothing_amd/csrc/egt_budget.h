// Places on a GPU that launches of this process may count on at once (host-only, no HIP: the CPU tests compile it with
// g++).
//
// A launch whose workgroups wait for one another needs all of them on the GPU together. Two such launches that fit
// one by one but not side by side can each hold places that the other waits for; each takes its workgroups from the
// device's budget first, so those that run together fit together.
#pragma once
#include <map>
#include <mutex>

namespace egt {

class TileBudget {
public:
    // Takes `tiles` of the device's `capacity`; false, with nothing taken, when fewer are left.
    bool take(int device, int tiles, int capacity) {
        std::lock_guard<std::mutex> lock(mu);
        int& u = used[device];
        if (tiles > capacity - u) return false;
        u += tiles;
        return true;
    }
    void give(int device, int tiles) {
        std::lock_guard<std::mutex> lock(mu);
        used[device] -= tiles;
    }

private:
    std::mutex mu;
    std::map<int, int> used;
};

// A share of a budget, given back at the end of the scope.
class TileShare {
public:
    TileShare(TileBudget& b, int device, int tiles, int capacity)
        : b_(b), device_(device), tiles_(tiles), taken_(b.take(device, tiles, capacity)) {}
    ~TileShare() {
        if (taken_) b_.give(device_, tiles_);
    }
    TileShare(const TileShare&) = delete;
    TileShare& operator=(const TileShare&) = delete;
    explicit operator bool() const { return taken_; }

private:
    TileBudget& b_;
    int device_, tiles_;
    bool taken_;
};

}  // namespace egt
