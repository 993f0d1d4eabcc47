// Host test of csrc/copy_back.hpp over a stub of the HIP calls (hip/ here).
// One scenario per run: copy_back_test NAME; exit code 0 if it holds.
#include <sys/mman.h>

#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <functional>

// every range a helper makes present goes through here
static std::function<void()> in_range;
static std::atomic<int> ranges_made{0};
static int test_madvise(void *p, size_t n, int advice) {
    ++ranges_made;
    if (in_range) in_range();
    return madvise(p, n, advice);
}
#define madvise test_madvise
#include "../../mpqpcudasolver_amd/csrc/copy_back.hpp"
#undef madvise

#include <dirent.h>
#include <sys/wait.h>

#include <chrono>

#define CHECK(x)                                                        \
    do {                                                                \
        if (!(x)) {                                                     \
            std::fprintf(stderr, "%d: %s does not hold\n", __LINE__, #x); \
            std::exit(1);                                               \
        }                                                               \
    } while (0)

static int threads() {
    int n = 0;
    DIR *d = opendir("/proc/self/task");
    while (dirent *e = readdir(d)) n += e->d_name[0] != '.';
    closedir(d);
    return n;
}

static void pause_ms(int ms) { std::this_thread::sleep_for(std::chrono::milliseconds(ms)); }

struct Call {
    std::vector<unsigned char> dev;
    std::vector<std::vector<unsigned char>> dst;
    std::vector<CopyBack::Seg> segs;
};
// `sizes` bytes for the arrays; every third one is not wanted
__attribute__((no_sanitize("thread"))) static Call make_call(const std::vector<size_t> &sizes, unsigned seed) {
    Call c;
    size_t total = 0;
    for (size_t n : sizes) total += n;
    c.dev.resize(total);
    for (size_t i = 0; i < total; ++i) c.dev[i] = (unsigned char)((i * 2654435761u + seed) >> 13);
    c.dst.resize(sizes.size());
    size_t off = 0;
    for (size_t k = 0; k < sizes.size(); ++k) {
        if (k % 3 != 2 && sizes[k]) {
            c.dst[k].assign(sizes[k] + 2, 0xa5);  // a guard at either end
            c.segs.push_back({off, sizes[k], c.dst[k].data() + 1});
        }
        off += sizes[k];
    }
    return c;
}
static void check_call(const Call &c) {
    for (const CopyBack::Seg &s : c.segs) {
        const unsigned char *d = static_cast<const unsigned char *>(s.dst);
        CHECK(std::memcmp(d, c.dev.data() + s.off, s.bytes) == 0);
        CHECK(d[-1] == 0xa5 && d[s.bytes] == 0xa5);
    }
}
static size_t bytes_of(const std::vector<CopyBack::Seg> &segs) {
    size_t n = 0;
    for (const CopyBack::Seg &s : segs) n += s.bytes;
    return n;
}

static const size_t B = Staging::SLOT;
static const std::vector<std::vector<size_t>> SHAPES = {
    {}, {1}, {0, 7, 9}, {B - 1}, {B}, {B + 1}, {2 * B - 1}, {2 * B}, {2 * B + 3, 5, 11, 17},
    {B / 3, B / 2, 3 * B, 4099, 7 * B + 13, 9, B, 31}, {20 * B + 5, 3 * B + 1, B}};

static void run_call(Staging &S, CopyThreads &T, Call &c, int chunks) {
    FakeStream st;
    auto back = std::make_shared<CopyBack>(S, T, &st, bytes_of(c.segs));
    const size_t per = (c.segs.size() + chunks - 1) / chunks;
    for (size_t i = 0; i < c.segs.size(); i += per)
        back->copy(c.dev.data(), {c.segs.begin() + i, c.segs.begin() + std::min(i + per, c.segs.size())});
    back->finish();
    back->stop();
}

static void copies() {
    for (int helpers : {0, 1, 4}) {
        Staging S;
        S.make();
        CHECK(S.ok);
        CopyThreads T;
        T.make(helpers);
        const int mallocs = fake().mallocs, events = fake().events;
        for (int chunks : {1, 2})
            for (size_t k = 0; k < SHAPES.size(); ++k) {
                Call c = make_call(SHAPES[k], (unsigned)k);
                run_call(S, T, c, chunks);
                check_call(c);
            }
        // nothing is made inside a call
        CHECK(fake().mallocs == mallocs && fake().events == events);
        std::free(S.p[0]);
    }
    CHECK(ranges_made > 0);
}

// without pinned memory, or without its events, the copies go directly
static void no_staging() {
    for (int what : {0, 1}) {
        fake().fail_malloc = what == 0;
        fake().fail_event_from = what == 1 ? fake().events + 5 : -1;
        Staging S;
        S.make();
        CHECK(!S.ok);
        CopyThreads T;
        for (size_t k = 0; k < SHAPES.size(); ++k) {
            Call c = make_call(SHAPES[k], (unsigned)k);
            run_call(S, T, c, 1);
            check_call(c);
        }
        fake().fail_malloc = 0;
        fake().fail_event_from = -1;
        S.make();
        CHECK(S.ok);
    }
}

// a helper that comes when the call has ended touches nothing
static void late_helper() {
    Staging S;
    S.make();
    CopyThreads T;  // no thread: help() is called below
    Call c = make_call({3 * B, 2 * B}, 1);
    FakeStream st;
    auto back = std::make_shared<CopyBack>(S, T, &st, bytes_of(c.segs));
    back->copy(c.dev.data(), c.segs);
    back->finish();
    check_call(c);
    const int made = ranges_made;
    for (auto &d : c.dst) std::fill(d.begin(), d.end(), 0x11);
    back->help();
    CHECK(ranges_made == made);
    for (auto &d : c.dst)
        for (unsigned char x : d) CHECK(x == 0x11);
}

// a helper that is held up inside a range is waited for, and the rest of the
// call goes on without it
static void held_up_helper() {
    Staging S;
    S.make();
    CopyThreads T;
    T.make(1);
    Call c = make_call({12 * B}, 2);
    std::atomic<bool> entered{false}, leave{false}, left{false}, ended{false};
    const long long copied = FakeStream::copies();
    in_range = [&] {
        if (entered.exchange(true)) return;
        while (!leave) pause_ms(1);
        left = true;
    };
    std::thread call([&] {
        run_call(S, T, c, 1);
        CHECK(left);
        ended = true;
    });
    while (!entered) pause_ms(1);
    // every block is used, the first ones again
    for (int i = 0; i < 5000 && FakeStream::copies() < copied + 12; ++i) pause_ms(1);
    CHECK(FakeStream::copies() == copied + 12);
    pause_ms(20);
    CHECK(!ended);
    leave = true;
    call.join();
    check_call(c);
    in_range = nullptr;
    // the threads serve the next call
    Call d = make_call({12 * B}, 3);
    run_call(S, T, d, 1);
    check_call(d);
}

// a failed copy ends the call with an error, and nothing is copied from its block on
static void failed_copy() {
    for (int helpers : {0, 4}) {
        Staging S;
        S.make();
        CopyThreads T;
        T.make(helpers);
        Call c = make_call({20 * B}, 4);
        fake().fail_copy = 3;
        bool threw = false;
        FakeStream st;
        auto back = std::make_shared<CopyBack>(S, T, &st, bytes_of(c.segs));
        try {
            back->copy(c.dev.data(), c.segs);
            back->finish();
        } catch (const HipError &) {
            threw = true;
        }
        back->stop();
        hipStreamSynchronize(&st);
        fake().fail_copy = -1;
        CHECK(threw);
        CHECK(c.dst[0].back() == 0xa5);
        Call d = make_call({20 * B}, 5);
        run_call(S, T, d, 1);
        check_call(d);
    }
}

// no thread is made by a call, and none outlives the context
static void joined() {
    std::thread([] {}).join();  // (a sanitizer makes a thread of its own with the first)
    const int before = threads();
    {
        Staging S;
        S.make();
        CopyThreads T;
        T.make(4);
        T.make(4);
        CHECK(threads() == before + 4);
        for (int i = 0; i < 50; ++i) {
            Call c = make_call({2 * B + i}, i);
            run_call(S, T, c, 1);
            check_call(c);
            CHECK(threads() == before + 4);
        }
    }
    CHECK(threads() == before);
}

// a process that forks after warm_up() ends as any other
static void forked() {
    static CopyThreads T;
    T.make(4);
    const pid_t child = fork();
    if (child == 0) std::exit(0);
    for (int i = 0; i < 2000; ++i) {
        int status = 0;
        if (waitpid(child, &status, WNOHANG) == child) {
            CHECK(WIFEXITED(status) && WEXITSTATUS(status) == 0);
            return;
        }
        pause_ms(5);
    }
    kill(child, SIGKILL);
    CHECK(!"the child ended");
}

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "copies") copies();
    else if (what == "no_staging") no_staging();
    else if (what == "late_helper") late_helper();
    else if (what == "held_up_helper") held_up_helper();
    else if (what == "failed_copy") failed_copy();
    else if (what == "joined") joined();
    else if (what == "forked") forked();
    else return 2;
    return 0;
}
