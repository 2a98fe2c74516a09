// CPU driver for the replay of a graph as its kernel launches (gemma4-webgpu-engine_amd/csrc/
// g4_graph_replay.h), with fake runtime calls that record their order. Built and run by
// tests/test_graph_replay.py; prints "ok" and exits 0 when every rule holds.
#include <cstdio>
#include <cstdlib>
#include <string>

#include "g4_graph_replay.h"

namespace {

struct Run {
    int rc;
    bool pending;
    std::string calls;  // one letter per call: L launch, M mark, D drain
};

// A replay of n launches of which launch `fail_at` fails with 7 (-1: none) and whose mark returns `mark`.
Run replay(size_t n, long fail_at, int mark) {
    Run r{0, false, ""};
    r.rc = g4::replay_chain(
        n,
        [&](size_t i) {
            r.calls += 'L';
            return (long)i == fail_at ? 7 : 0;
        },
        [&] {
            r.calls += 'M';
            return mark;
        },
        [&] {
            r.calls += 'D';
            return 0;
        },
        &r.pending);
    return r;
}

void expect(const Run &r, int rc, bool pending, const char *calls, const char *what) {
    if (r.rc != rc || r.pending != pending || r.calls != calls) {
        std::printf("FAIL: %s: rc %d pending %d calls %s\n", what, r.rc, (int)r.pending, r.calls.c_str());
        std::exit(1);
    }
}

}  // namespace

int main() {
    expect(replay(1, -1, 0), 0, true, "LM", "one kernel");
    expect(replay(3, -1, 0), 0, true, "LLLM", "three kernels");
    // a launch that fails behind others: what is on the stream is marked, the failure is returned
    expect(replay(3, 1, 0), 7, true, "LLM", "the second launch fails");
    expect(replay(12, 11, 0), 7, true, "LLLLLLLLLLLLM", "the last launch fails");
    // nothing enqueued: nothing to wait for
    expect(replay(3, 0, 0), 7, false, "L", "the first launch fails");
    // a mark that cannot be recorded: the stream is waited for instead
    expect(replay(2, -1, 5), 5, false, "LLMD", "the mark fails");
    expect(replay(2, 1, 5), 7, false, "LLMD", "a launch and the mark fail");
    // an earlier replay's mark stays pending
    bool pending = true;
    (void)g4::replay_chain(1, [](size_t) { return 7; }, [] { return 0; }, [] { return 0; }, &pending);
    if (!pending) {
        std::printf("FAIL: an earlier replay is forgotten\n");
        return 1;
    }
    std::printf("ok\n");
    return 0;
}
