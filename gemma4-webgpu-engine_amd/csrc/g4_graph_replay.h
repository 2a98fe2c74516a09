// One replay of a captured graph as its kernel launches: what is enqueued, marked and waited for.
// Host code only; the runtime calls are passed in, so a CPU test can drive the order with fakes.
#ifndef G4_GRAPH_REPLAY_H
#define G4_GRAPH_REPLAY_H

#include <cstddef>

namespace g4 {

// launch(0) .. launch(n - 1) in order up to the first that fails, then mark() (the event that the
// graph's destroy waits for), also when a later launch failed: the earlier ones are on the stream
// and their buffers may be freed once destroy returns. drain() waits for the stream when the mark
// cannot be recorded. Each returns 0 on success; so does replay_chain, else the first failure.
// *pending: a mark has been recorded that destroy has to wait for.
template <typename Launch, typename Mark, typename Drain>
int replay_chain(size_t n, Launch launch, Mark mark, Drain drain, bool *pending) {
    int rc = 0;
    size_t enqueued = 0;
    while (enqueued < n && (rc = launch(enqueued)) == 0) ++enqueued;
    if (enqueued == 0) return rc;
    const int marked = mark();
    if (marked == 0) *pending = true;
    else (void)drain();
    return rc ? rc : marked;
}

}  // namespace g4

#endif  // G4_GRAPH_REPLAY_H
