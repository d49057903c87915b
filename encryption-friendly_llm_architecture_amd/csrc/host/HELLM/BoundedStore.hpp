// What is prepared per weight and kept: entries by key, the oldest given up for a new one once their costs would pass a limit.
#pragma once
#include <cstdint>
#include <deque>
#include <map>
#include <utility>

namespace HELLM {

template <class Key, class Entry>
class BoundedStore {
public:
    explicit BoundedStore(uint64_t limit) : limit_(limit) {}
    // stays where it is until the next makeRoom(), keep() or clear()
    const Entry *find(const Key &key) const {
        auto it = entries_.find(key);
        return it == entries_.end() ? nullptr : &it->second.first;
    }
    // gives up what an entry of this cost has to replace: in front of an allocation, which then finds the memory
    void makeRoom(uint64_t cost) {
        while (!order_.empty() && cost_ + cost > limit_) drop(order_.front());
    }
    // an entry that costs more than the limit is kept alone
    const Entry &keep(const Key &key, Entry entry, uint64_t cost = 1) {
        drop(key);
        makeRoom(cost);
        order_.push_back(key);
        cost_ += cost;
        return entries_.emplace(key, std::make_pair(std::move(entry), cost)).first->second.first;
    }
    void clear() {
        entries_.clear();
        order_.clear();
        cost_ = 0;
    }
    uint64_t cost() const { return cost_; }

private:
    void drop(const Key key) {   // (by value: the key may be one of order_)
        auto it = entries_.find(key);
        if (it == entries_.end()) return;
        cost_ -= it->second.second;
        entries_.erase(it);
        for (auto o = order_.begin(); o != order_.end(); ++o)
            if (!(*o < key) && !(key < *o)) {
                order_.erase(o);
                break;
            }
    }
    uint64_t limit_, cost_ = 0;
    std::map<Key, std::pair<Entry, uint64_t>> entries_;
    std::deque<Key> order_;
};

}  // namespace HELLM
