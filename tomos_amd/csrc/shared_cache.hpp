// A few kept objects by key, shared with the calls that use them: the batched
// solvers' instantiated graphs.  A call holds its share until it has
// synchronized, so that an object which another thread's insert evicts
// meanwhile is destroyed only when no call runs it any more.
#pragma once

#include <cstddef>
#include <memory>
#include <mutex>
#include <utility>
#include <vector>

namespace tomos_hip {

template <class Key, class T>
class SharedCache {
public:
    explicit SharedCache(size_t most) : most_(most) {}

    std::shared_ptr<T> find(const Key& k) {
        std::lock_guard<std::mutex> lock(mu_);
        for (const auto& e : kept_)
            if (e.first == k) return e.second;
        return nullptr;
    }
    // The oldest entry leaves when there are `most`.
    void insert(const Key& k, std::shared_ptr<T> object) {
        std::shared_ptr<T> evicted;  // released outside the lock
        std::lock_guard<std::mutex> lock(mu_);
        if (kept_.size() >= most_) {
            evicted = std::move(kept_.front().second);
            kept_.erase(kept_.begin());
        }
        kept_.emplace_back(k, std::move(object));
    }

private:
    size_t most_;
    std::mutex mu_;
    std::vector<std::pair<Key, std::shared_ptr<T>>> kept_;
};

}  // namespace tomos_hip
