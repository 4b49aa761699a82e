// Work distribution of a launch: its queue's entries, 64 at a time.
#pragma once

#include "ljx_device.h"

namespace ljx {

// Hands a launch's n queue entries to its waves, 64 at a time, so that waves
// that drew short work take more and the launch's tail stays short.  Each
// wave's first chunk is its own by its number; after that it takes tickets.
// A ticket is one atomic by the whole wave, and those on one cache line run
// one every 11.3 ns on the whole chip (2,048 blocks took 12 ms of tickets for
// 67M rays from a single counter), so blocks draw from kFeeds counters on
// lines of their own, by block number modulo kFeeds, which is the XCD that
// dispatch in turn places them on.  Feed f owns every kFeeds-th run of
// kFeedRun chunks: an XCD's waves work on neighbouring entries, and every feed
// sees all parts of a queue of many runs.  (A queue of under kFeeds runs, 8,192
// entries, has work for as many feeds as it has runs.)
constexpr int kFeeds = 8, kFeedLine = 32, kFeedSet = kFeeds * kFeedLine;  // counters are kFeedLine apart: 128 bytes
constexpr int kFeedRun = 16;
constexpr int kMaxQueue = 1 << 26;
// A ticket's round trip takes over a microsecond, which two or three waves per
// SIMD do not hide.  For kernels of such occupancy a ticket covers several
// chunks of a long queue, as many as leave every wave `tickets` of them (media
// render's shadow walks 14.9 -> 7.5 ms); at eight waves per SIMD single chunks
// are better (terrain's closest hits 56.4 against 58.8 ms).
constexpr int kFeedTickets = 8;
// One wave's place in the queue, apart from the counters (host code too).
struct FeedPlace {
    int feeds, feed, waves, ticket, sub, span;
    bool more;  // tickets remain after every wave's first
    LJX_HD int chunk(int t) const {
        return ((t * span / kFeedRun) * feeds + feed) * kFeedRun + t * span % kFeedRun;
    }
    // Wave `wave` of `wpb` in block `block` of `blocks`; n <= kMaxQueue.  Grids
    // of fewer than kFeeds blocks use one feed.
    LJX_HD void place(int block, int blocks, int wave, int wpb, int n, int tickets) {
        const int chunks = (n + 63) / 64;
        feeds = blocks < kFeeds ? 1 : kFeeds;
        feed = block % feeds;
        waves = (blocks + feeds - 1 - feed) / feeds * wpb;
        span = 1;
        while (tickets > 0 && span < kFeedRun && chunks >= 2 * span * tickets * blocks * wpb) span *= 2;
        ticket = block / feeds * wpb + wave;
        sub = 0;
        more = chunk(waves) < chunks;
    }
    // First entry of the wave's current chunk; at or past n: none is left.
    LJX_HD int base() const { return (chunk(ticket) + sub) * 64; }
    // The next chunk: of this ticket, or of the feed's next, numbered by draw().
    template <class Draw>
    LJX_HD void advance(Draw &&draw) {
        if (++sub < span) return;
        sub = 0;
        ticket = more ? waves + draw() : kMaxQueue / 64 / span;  // the latter past every queue
    }
};
struct Feed : FeedPlace {
    int *counter;
    // counters: a set of kFeeds zeroed counters.
    __device__ __forceinline__ void start(int *counters, int n, int tickets = 0) {
        place(int(blockIdx.x), int(gridDim.x), int(threadIdx.x >> 6), int(blockDim.x >> 6), n, tickets);
        ticket = __builtin_amdgcn_readfirstlane(ticket);
        counter = counters + feed * kFeedLine;
    }
    __device__ __forceinline__ void next() {
        int *c = counter;
        advance([c] __device__() {
            int t = 0;
            if (__lane_id() == 0) t = atomicAdd(c, 1);
            return __builtin_amdgcn_readfirstlane(t);
        });
    }
};

}  // namespace ljx
