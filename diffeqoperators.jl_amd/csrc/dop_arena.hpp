// dop_arena.hpp -- the memory of a server's resident requests: a first-fit allocator over device
// allocations ("segments") made as requests need them, `budget` bytes in all at most.
//
// One allocation of the whole budget per server cost small bursts more than their steps: of a
// 2 GiB budget 0.3 ms to make and 0.45 ms to free at best, and now and then 40 to 1260 ms to make
// or 43 to 57 ms to free, for bursts of 1.5 to 6 ms (two to twelve requests of 64^2 to 600^2).  A
// segment is as large as the requests known when it is made, so a burst has one, and a long stream
// that needs it has the whole budget in one.
#pragma once
#include <algorithm>
#include <cstddef>
#include <iterator>
#include <map>
#include <vector>

namespace dop {

constexpr size_t kArenaAlign = 256;
inline size_t arena_round(size_t n) { return (n + kArenaAlign - 1) / kArenaAlign * kArenaAlign; }

// Mem: char* get(size_t) (null: no memory) and void put(char*, size_t)
template <typename Mem>
class Arena {
public:
    ~Arena() { clear(); }
    void init(size_t budget) { budget_ = budget; }

    // Memory for n bytes (the budget at most) in one segment, when there is none yet.
    void reserve(size_t n)
    {
        if (total_ == 0 && n > 0) (void)grow(std::min(arena_round(n), budget_));
    }

    // n bytes, or null when they do not fit now (always after a release, and when nothing is
    // allocated only if memory is short).  want(): bytes that the caller expects to need soon.
    template <typename F>
    char* alloc(size_t n, const F& want)
    {
        n = arena_round(n);
        if (char* p = carve(n)) return p;
        if (short_) return nullptr;
        // (pieces too small, all of them empty: the budget in one piece from now on)
        const bool whole = used_ == 0 && total_ > 0 && budget_ - total_ < n;
        if (whole) clear();
        if (n > budget_ - total_) return nullptr;
        // at least what is there already: live submissions make few segments
        const size_t most = whole ? budget_ : std::max(std::max(arena_round(want()), total_), n);
        if (!grow(std::min(most, budget_ - total_)) && !grow(n)) {
            if (used_ == 0) clear();
            if (used_ > 0 || !grow(n)) {
                short_ = used_ > 0;   // asked again after a release
                return nullptr;
            }
        }
        return carve(n);
    }
    void release(char* p, size_t n)
    {
        n = arena_round(n);
        used_ -= n;
        short_ = false;
        for (Segment& s : segs_) {
            if (p < s.base || p >= s.base + s.size) continue;
            auto it = s.free.emplace((size_t)(p - s.base), n).first;
            auto nx = std::next(it);
            if (nx != s.free.end() && it->first + it->second == nx->first) {
                it->second += nx->second;
                s.free.erase(nx);
            }
            if (it != s.free.begin()) {
                auto pv = std::prev(it);
                if (pv->first + pv->second == it->first) {
                    pv->second += it->second;
                    s.free.erase(it);
                }
            }
            return;
        }
    }
    // Gives all memory back (nothing may be resident).
    void clear()
    {
        for (Segment& s : segs_) mem_.put(s.base, s.size);
        segs_.clear();
        total_ = used_ = 0;
    }
    size_t used() const { return used_; }
    size_t total() const { return total_; }

private:
    struct Segment {
        char* base;
        size_t size;
        std::map<size_t, size_t> free;
    };
    char* carve(size_t n)
    {
        for (Segment& s : segs_) {
            for (auto it = s.free.begin(); it != s.free.end(); ++it) {
                if (it->second < n) continue;
                const size_t at = it->first, rest = it->second - n;
                s.free.erase(it);
                if (rest) s.free[at + n] = rest;
                used_ += n;
                return s.base + at;
            }
        }
        return nullptr;
    }
    bool grow(size_t size)
    {
        char* p = mem_.get(size);
        if (!p) return false;
        segs_.push_back({p, size, {{0, size}}});
        total_ += size;
        return true;
    }
    Mem mem_;
    std::vector<Segment> segs_;
    size_t budget_ = 0, total_ = 0, used_ = 0;
    bool short_ = false;
};

}  // namespace dop
