// The last plans a thread computed, by the extents they are for. Choosing a plan evaluates some fifty estimates, 1 to 3 us of host work; a
// program's layers have the same extents in every step, and a small product is over on the GPU before its next call is enqueued.
#ifndef NZHIP_PLAN_CACHE_H
#define NZHIP_PLAN_CACHE_H

#include <cstdint>
#include <cstring>

namespace nzhip {

// Key: a plain struct without padding, compared byte by byte. Direct-mapped, 64 entries.
template <typename Key, typename Plan>
class PlanCache {
public:
    // the entry of a key; `known` says whether it holds that key's plan, otherwise the caller fills it
    Plan& at(const Key& key, bool& known) {
        uint64_t h = 1469598103934665603ull;
        uint64_t words[sizeof(Key) / 8];
        static_assert(sizeof(Key) % 8 == 0, "whole words");
        std::memcpy(words, &key, sizeof(Key));
        for (uint64_t w : words) h = (h ^ w) * 1099511628211ull;
        Entry& e = entries_[(h ^ (h >> 29)) & 63];
        known = e.used && std::memcmp(&e.key, &key, sizeof(Key)) == 0;
        if (!known) {
            std::memcpy(&e.key, &key, sizeof(Key));
            e.used = true;
        }
        return e.plan;
    }

private:
    struct Entry {
        Key key;
        Plan plan;
        bool used = false;
    };
    Entry entries_[64];
};

}  // namespace nzhip

#endif
