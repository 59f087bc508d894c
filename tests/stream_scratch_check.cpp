// Checks of the launchers' scratch memory (loken_amd/csrc/stream_scratch.hip) on the host, over the runtime of
// hip_stub/: one case per run, named by the first argument. Exit status 0: the case holds.
#include "stream_scratch.hip"

#include <stdio.h>
#include <string.h>

#define CHECK(c)                                                                  \
    do {                                                                          \
        if (!(c)) { fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #c); exit(1); } \
    } while (0)

static void* take(hipStream_t s, LkScratchUse use, size_t bytes) { return LkScratch(s).get(use, bytes); }
struct Recording {   // `s` records into capture `id` while this lives
    hipStream_t s;
    Recording(hipStream_t stream, unsigned long long id) : s(stream) { s->capture = id; ++fake::captures; }
    ~Recording() { s->capture = 0; --fake::captures; }
};

static void a_stream_keeps_its_buffers() {
    ihipStream_t a, b;
    void* p = take(&a, LK_SCRATCH_LINEAR, 1000);
    CHECK(p && take(&a, LK_SCRATCH_LINEAR, 1000) == p && take(&a, LK_SCRATCH_LINEAR, 1) == p);
    CHECK(take(&b, LK_SCRATCH_LINEAR, 1000) != p && take(&a, LK_SCRATCH_ROUTER, 1000) != p);
    CHECK(take(hipStreamPerThread, LK_SCRATCH_LINEAR, 1000) != take(nullptr, LK_SCRATCH_LINEAR, 1000));
    void* q = take(&a, LK_SCRATCH_LINEAR, 1 << 20);
    CHECK(q && q != p && take(&a, LK_SCRATCH_LINEAR, 1000) == q);
    fake::device = 1;
    CHECK(take(&a, LK_SCRATCH_LINEAR, 1000) != q);
    fake::device = 0;
    fake::out_of_memory = true;
    CHECK(!take(&a, LK_SCRATCH_BLOCK, 1000));
}

static void nothing_is_shared_with_a_graph() {
    ihipStream_t a, b, c;
    void* eager_a = take(&a, LK_SCRATCH_BLOCK, 4096);
    void* eager_b = take(&b, LK_SCRATCH_BLOCK, 100);
    void *first, *second, *own;
    {
        Recording r(&b, 7);
        first = take(&b, LK_SCRATCH_BLOCK, 4096);
        CHECK(first && first != eager_a && first != eager_b);          // nobody's from before
        CHECK(take(&b, LK_SCRATCH_BLOCK, 4000) == first);              // one buffer through one recording of a stream
        Recording forked(&c, 7);                                       // a second stream of the same capture runs beside it
        CHECK(take(&c, LK_SCRATCH_BLOCK, 4096) != first);
        CHECK(take(&a, LK_SCRATCH_BLOCK, 4096) == eager_a);            // another thread's calls go on meanwhile
        CHECK(take(&a, LK_SCRATCH_LINEAR, 4096) != nullptr);           // and may grow
    }
    {
        Recording r(&b, 8);                                            // the next graph of the same stream
        second = take(&b, LK_SCRATCH_BLOCK, 4096);
        CHECK(second && second != first && second != eager_a);
    }
    {
        Recording r(&a, 9);                                            // recorded where the calls ran
        own = take(&a, LK_SCRATCH_BLOCK, 4096);
        CHECK(own && own != eager_a && own != first && own != second);
    }
    CHECK(take(&b, LK_SCRATCH_BLOCK, 4096) != first && take(&b, LK_SCRATCH_BLOCK, 4096) != second);
    CHECK(take(&a, LK_SCRATCH_BLOCK, 4096) == eager_a);
    for (void* p : {first, second, own}) CHECK(fake::live.count(p));   // theirs until the release
}

static void what_nothing_reserved_is_refused_while_recording() {
    ihipStream_t a, b;
    {
        Recording r(&a, 1);
        CHECK(!take(&a, LK_SCRATCH_LINEAR, 100));
    }
    CHECK(take(&b, LK_SCRATCH_LINEAR, 100));
    {
        Recording r(&a, 2);
        CHECK(take(&a, LK_SCRATCH_LINEAR, 100));
        CHECK(!take(&a, LK_SCRATCH_LINEAR, 1000) && !take(&a, LK_SCRATCH_ROUTER, 100));
    }
    lk_stream_scratch_release(-1, ~0u);
    CHECK(fake::held() == 0);
    Recording r(&a, 3);
    CHECK(!take(&a, LK_SCRATCH_LINEAR, 100));
}

static void graphs_together_stay_within_their_bound() {
    ihipStream_t a;
    const size_t big = LK_SCRATCH_GRAPH_BYTES / 4;   // a quarter more is reserved each time
    CHECK(take(&a, LK_SCRATCH_TOKENS, big));
    for (int i = 1; i <= 4; ++i) {
        Recording r(&a, (unsigned long long)i);
        CHECK((take(&a, LK_SCRATCH_TOKENS, big) != nullptr) == (i <= 3));
    }
    lk_stream_scratch_release(-1, ~0u);
    CHECK(take(&a, LK_SCRATCH_TOKENS, big));
    Recording r(&a, 9);
    CHECK(take(&a, LK_SCRATCH_TOKENS, big));
}

static void an_outgrown_buffer_goes_unless_a_graph_has_it() {
    ihipStream_t a;
    for (size_t bytes : {1000, 10000, 100000}) CHECK(take(&a, LK_SCRATCH_BLOCK, bytes));
    CHECK(fake::live.size() == 1 && fake::held() < 130000);
    void *first, *second;
    {
        Recording r(&a, 4);
        first = take(&a, LK_SCRATCH_BLOCK, 1000);
        second = take(&a, LK_SCRATCH_BLOCK, 50000);
        ihipStream_t b;
        CHECK(take(&b, LK_SCRATCH_BLOCK, 10) && take(&b, LK_SCRATCH_BLOCK, 1000));   // a call beside the recording frees and allocates
    }
    CHECK(first != second && fake::live.count(first) && fake::live.count(second) && fake::live.size() == 4);
    fake::out_of_memory = true;                       // the larger one cannot be had: the next call tries again
    CHECK(!take(&a, LK_SCRATCH_BLOCK, 1 << 20) && !take(&a, LK_SCRATCH_BLOCK, 10));
    fake::out_of_memory = false;
    CHECK(take(&a, LK_SCRATCH_BLOCK, 10));
    lk_stream_scratch_release(-1, ~0u);
    CHECK(fake::held() == 0);
}

static void a_release_frees_its_own_part() {
    ihipStream_t a;
    void* held[2][LK_SCRATCH_USES][2];   // device, use, by a call / by a graph
    for (int d = 0; d < 2; ++d) {
        fake::device = d;
        for (int u = 0; u < LK_SCRATCH_USES; ++u) held[d][u][0] = take(&a, (LkScratchUse)u, 1000);
        Recording r(&a, 5);
        for (int u = 0; u < LK_SCRATCH_USES; ++u) held[d][u][1] = take(&a, (LkScratchUse)u, 1000);
    }
    fake::device = 0;
    auto lives = [&](int d, int u) { return fake::live.count(held[d][u][0]) + fake::live.count(held[d][u][1]); };
    fake::sync_fails = true;             // a device that cannot be waited for keeps everything
    lk_stream_scratch_release(-1, ~0u);
    CHECK(fake::frees == 0);
    fake::sync_fails = false;
    lk_stream_scratch_release(1, LK_SCRATCH_OF_LAUNCHERS);
    for (int u = 0; u < LK_SCRATCH_USES; ++u) {
        const bool linears = u == LK_SCRATCH_LINEAR || u == LK_SCRATCH_FIXUP;
        CHECK(lives(0, u) == 2 && lives(1, u) == (linears ? 2u : 0u));
    }
    lk_stream_scratch_release(-1, LK_SCRATCH_OF_LINEARS);
    for (int u = 0; u < LK_SCRATCH_USES; ++u) {
        const bool linears = u == LK_SCRATCH_LINEAR || u == LK_SCRATCH_FIXUP;
        CHECK(lives(0, u) == (linears ? 0u : 2u) && lives(1, u) == 0);
    }
    CHECK(fake::device == 0);
    lk_stream_scratch_release(0, LK_SCRATCH_OF_LAUNCHERS);
    CHECK(fake::held() == 0 && take(&a, LK_SCRATCH_BLOCK, 10));
}

static void streams_past_the_bound_share_in_order() {
    static ihipStream_t many[LK_SCRATCH_STREAMS + 3];
    for (int round = 0; round < 3; ++round)
        for (auto& s : many) CHECK(take(&s, LK_SCRATCH_LINEAR, 1000));
    CHECK(fake::allocations == LK_SCRATCH_STREAMS + 1 && fake::frees == 0);   // round after round nothing is freed or allocated
    ihipStream_t *x = &many[LK_SCRATCH_STREAMS], *y = x + 1;
    CHECK(take(x, LK_SCRATCH_LINEAR, 1000) == take(y, LK_SCRATCH_LINEAR, 1000));
    fake::log.clear();
    CHECK(take(&many[0], LK_SCRATCH_LINEAR, 1000) != take(&many[1], LK_SCRATCH_LINEAR, 1000) && fake::log.empty());
    {   // a launcher that calls others: one wait before its first buffer, one record behind its last launch
        LkScratch outer(x);
        CHECK(fake::log.empty());
        CHECK(outer.get(LK_SCRATCH_BLOCK, 10) && LkScratch(x).get(LK_SCRATCH_LAUNCHER, 10) && outer.get(LK_SCRATCH_BLOCK, 10));
        CHECK(fake::log.size() == 1 && fake::log[0] == "wait " + std::to_string((size_t)x));
    }
    CHECK(fake::log.size() == 2 && fake::log[1] == "record " + std::to_string((size_t)x));
    CHECK(take(y, LK_SCRATCH_BLOCK, 10) && fake::log[2] == "wait " + std::to_string((size_t)y) && fake::log.size() == 4);
    { LkScratch none(y); }               // took nothing: nothing to order
    CHECK(fake::log.size() == 4);
    {
        Recording r(y, 3);               // a graph has its own, past the bound too
        void* p = take(y, LK_SCRATCH_BLOCK, 10);
        CHECK(p && fake::log.size() == 4);
    }
    lk_stream_scratch_release(-1, ~0u);  // and the streams that are still there get their own again
    CHECK(fake::held() == 0);
    CHECK(take(x, LK_SCRATCH_LINEAR, 1000) != take(y, LK_SCRATCH_LINEAR, 1000) && fake::log.size() == 4);
}

static void without_an_event_the_shared_buffers_wait_on_the_host() {
    static ihipStream_t many[LK_SCRATCH_STREAMS + 1];
    fake::no_events = true;
    for (auto& s : many) CHECK(take(&s, LK_SCRATCH_LINEAR, 1000));
    CHECK(fake::log.size() == 1 && fake::log[0] == "synchronize " + std::to_string((size_t)&many[LK_SCRATCH_STREAMS]));
}

static void threads_hold_what_they_use() {
    // every thread marks the buffer it got while it holds it; on one stream, on streams of their own and past the bound
    static ihipStream_t many[LK_SCRATCH_STREAMS + 2];
    static std::map<void*, int> user;
    static std::mutex mu;
    for (int i = 0; i < LK_SCRATCH_STREAMS; ++i) take(&many[i], LK_SCRATCH_LINEAR, 10);
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; ++t)
        threads.emplace_back([t] {
            for (int i = 0; i < 2000; ++i) {
                LkScratch s(&many[t % 4 == 3 ? 0 : LK_SCRATCH_STREAMS - 2 + t % 4]);
                void* p = s.get(LK_SCRATCH_LINEAR, 10 + (size_t)(i % 500) * 7);
                CHECK(p);
                { std::lock_guard<std::mutex> lock(mu); CHECK(user[p]++ == 0); }
                { std::lock_guard<std::mutex> lock(mu); --user[p]; }
                if (t == 0 && i % 97 == 0) {
                    LkScratch other(&many[1]);
                    (void)other;
                }
                if (t == 5 && i % 301 == 300) break;
            }
            if (t == 5)
                for (int i = 0; i < 50; ++i) lk_stream_scratch_release(-1, i % 2 ? LK_SCRATCH_OF_LINEARS : LK_SCRATCH_OF_LAUNCHERS);
        });
    for (auto& t : threads) t.join();
    lk_stream_scratch_release(-1, ~0u);
    CHECK(fake::held() == 0);
}

static void a_counter_belongs_to_one_stream() {
    static ihipStream_t many[LK_SCRATCH_STREAMS + 2];
    std::map<int, int> seen;
    for (int i = 0; i < LK_SCRATCH_STREAMS; ++i) {
        const int t = LkScratch(&many[i]).ticket();
        CHECK(t >= 0 && t < LK_SCRATCH_TICKETS && seen[t]++ == 0 && LkScratch(&many[i]).ticket() == t);
    }
    const int shared = LkScratch(&many[LK_SCRATCH_STREAMS]).ticket();   // one set of buffers, one counter, in order
    CHECK(shared >= 0 && !seen[shared] && LkScratch(&many[LK_SCRATCH_STREAMS + 1]).ticket() == shared);
    {
        Recording r(&many[0], 5);
        CHECK(LkScratch(&many[0]).ticket() == -1);
    }
    for (int i = 0; i < 2 * LK_SCRATCH_TICKETS; ++i) {                 // a release gives them back
        take(&many[i % LK_SCRATCH_STREAMS], LK_SCRATCH_ROUTER, 10);
        if (i % 7 == 6) lk_stream_scratch_release(-1, ~0u);
    }
    CHECK(LkScratch(&many[3]).ticket() >= 0);
}

int main(int argc, char** argv) {
    const struct { const char* name; void (*run)(); } cases[] = {
#define CASE(f) {#f, f}
        CASE(a_stream_keeps_its_buffers), CASE(nothing_is_shared_with_a_graph),
        CASE(what_nothing_reserved_is_refused_while_recording), CASE(graphs_together_stay_within_their_bound),
        CASE(an_outgrown_buffer_goes_unless_a_graph_has_it),
        CASE(a_release_frees_its_own_part), CASE(streams_past_the_bound_share_in_order),
        CASE(without_an_event_the_shared_buffers_wait_on_the_host), CASE(threads_hold_what_they_use),
        CASE(a_counter_belongs_to_one_stream),
    };
    for (auto& c : cases) {
        if (argc < 2) puts(c.name);
        else if (!strcmp(argv[1], c.name)) return c.run(), 0;
    }
    return argc < 2 ? 0 : 2;
}
