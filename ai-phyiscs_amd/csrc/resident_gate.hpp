// SPDX-License-Identifier: Apache-2.0
//
// Which one-launch solves of a device may be in flight together.
#pragma once

#include <algorithm>
#include <cstddef>
#include <vector>

namespace chysx_amd {

constexpr int kXcds = 8;

// A workgroup of a one-launch solve keeps a compute unit while it waits for
// the rest of its instance to start, and an XCD is given every 8th workgroup
// of a launch and no other.  Launches in flight on several streams must leave
// at least one compute unit of every XCD that no waiting workgroup can hold;
// then each of them comes to run in the end, in any order.  Otherwise each can
// hold what the others need, until the start-up agreement gives up after half
// a second.
//
// gate_weight: the compute units of one XCD that the waiting workgroups of a
// launch can hold.  by_start: places in the order of starting, where only part
// of one instance waits; by number, an XCD that is ahead can be full of them.
// None where every instance is a single workgroup.
inline int gate_room(int cus) { return std::max(0, cus / kXcds - 1); }
inline int gate_weight(int wgs, int max_cluster, bool by_start, int cus) {
    if (max_cluster <= 1) return 0;
    const int w = by_start ? std::min(max_cluster - 1, (wgs + kXcds - 1) / kXcds) : gate_room(cus);
    return std::min(w, gate_room(cus));
}

// The launches in flight, one entry per problem: a problem's own launches
// follow each other, and its event is recorded behind each.  A launch that
// does not fit beside the others waits for the oldest of them.  An entry then
// also stands for those that its launch waits for: they and it are not under
// way together, so it weighs the most that can be of them, and the entries'
// weights never add up to more than the room.
//
// (One after the other for all launches of more than 8 workgroups an instance,
// and no order for the rest, let a 512 x 512 cloth and a batch of small ones
// block each other; and a rule that spared launches on the stream of the one
// before knew streams by their handles, which are used again.)
template <class Event>
class GateBook {
public:
    // The events that a launch of `owner` has to wait for.  done(event): whether
    // everything recorded has run.
    template <class Done>
    std::vector<Event> admit(const void* owner, Event event, int weight, int room, Done&& done) {
        std::vector<Event> waits;
        int mine = 0, others = 0;
        for (size_t k = 0; k < entries_.size();) {
            Entry& E = entries_[k];
            // a lone problem's launches need no look
            if ((entries_.size() > 1 || E.owner != owner) && done(E.event)) {
                entries_.erase(entries_.begin() + std::ptrdiff_t(k));
                continue;
            }
            (E.owner == owner ? mine : others) += E.weight;
            ++k;
        }
        int waited = 0;
        for (size_t k = 0; k < entries_.size() && (others - waited) + std::max(weight, mine + waited) > room;) {
            if (entries_[k].owner == owner) {
                ++k;
                continue;
            }
            waits.push_back(entries_[k].event);
            waited += entries_[k].weight;
            entries_.erase(entries_.begin() + std::ptrdiff_t(k));
        }
        forget(owner);
        entries_.push_back(Entry{owner, event, std::max(weight, mine + waited)});
        return waits;
    }
    // The owner's launches have run.
    void forget(const void* owner) {
        for (size_t k = 0; k < entries_.size(); ++k)
            if (entries_[k].owner == owner) {
                entries_.erase(entries_.begin() + std::ptrdiff_t(k));
                return;
            }
    }
    size_t size() const { return entries_.size(); }

private:
    struct Entry {
        const void* owner;
        Event event;
        int weight;
    };
    std::vector<Entry> entries_;  // oldest first
};

}  // namespace chysx_amd
