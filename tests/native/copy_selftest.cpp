// copy_selftest.cpp -- the staged host copies (pmp_copy.hip) on the CPU against
// a simulated HIP runtime (hip_sim), under the sanitizers.  Exits non-zero on
// the first failed check (or a sanitizer report).
//
//   copy_selftest [part ...]     the parts by name; all of them by default
#include <dirent.h>
#include <signal.h>
#include <stdio.h>
#include <stdlib.h>

#include <set>
#include <string>
#include <thread>
#include <vector>

#include "pmp_copy.h"

using namespace pmp;
using Bytes = std::vector<uint8_t>;

#define CHECK(c)                                                                  \
    do {                                                                          \
        if (!(c)) {                                                               \
            fprintf(stderr, "copy_selftest: check failed at line %d: %s\n", __LINE__, #c); \
            exit(1);                                                              \
        }                                                                         \
    } while (0)

static hip_sim::Stats& st = hip_sim::stats();
constexpr size_t KiB = 1024, MiB = 1024 * KiB;

static Bytes noise(size_t n, unsigned seed) {
    Bytes b(n + 8);
    uint64_t x = 0x9E3779B97F4A7C15ull * (seed + 1);
    for (size_t k = 0; k < n; k += 8) {
        x = x * 6364136223846793005ull + 1442695040888963407ull;
        memcpy(&b[k], &x, 8);
    }
    b.resize(n);
    return b;
}

// Rows of `row` bytes, `pitch` apart, up and back down again: the same bytes.
// Returns the 2D copies that the runtime was asked for.
static int round_trip(Copier& c, hipStream_t s, size_t row, size_t rows, size_t pitch) {
    const Bytes host = noise(pitch * rows, (unsigned)(row + rows));
    Bytes dev(row * rows), back(row * rows, 0xAA);
    const int before = st.copies_2d;
    const HostCopy up{const_cast<uint8_t*>(host.data()), dev.data(), row, rows, pitch};
    CHECK(c.to_device(s, &up, 1) == hipSuccess);
    CHECK(s->idle());
    for (size_t r = 0; r < rows; ++r) CHECK(memcmp(&dev[r * row], &host[r * pitch], row) == 0);
    const HostCopy down = flat_copy(back.data(), dev.data(), row * rows);
    CHECK(c.to_host(s, &down, 1) == hipSuccess);
    CHECK(back == dev);
    return st.copies_2d - before;
}

// A pitched copy from pageable memory is never the runtime's own, which moves
// it row by row, whatever its size.
static void pitched() {
    hip_sim::Stream s;
    Copier c;
    for (size_t row : {700, 1920, 4099})
        for (size_t rows : {1, 3, 400, 960, 1100, 2300})
            for (size_t pad : {0, 5, 128}) CHECK(round_trip(c, &s, row, rows, row + pad) == 0);
    // nor without pinned memory
    st.fail_pinned = true;
    Copier d;
    for (size_t rows : {1, 400, 960, 2300}) CHECK(round_trip(d, &s, 1920, rows, 2048) == 0);
    st.fail_pinned = false;
}

// What an upload has done on return: everything by default, also in the sizes
// that the runtime copies itself; read the host memory (kRead); and after a
// failed copy nothing touches either side any more.
static void until() {
    hip_sim::Stream s;
    Copier c;
    for (size_t n : {1 * KiB, 700 * KiB, 2 * MiB, 7 * MiB, 13 * MiB, 30 * MiB}) {
        st.delay_us = 1000;
        const Bytes host = noise(n, (unsigned)n);
        for (Until u : {Until::kDone, Until::kRead, Until::kQueued}) {
            Bytes src = host, dev(n);
            const HostCopy up = flat_copy(src.data(), dev.data(), n);
            CHECK(c.to_device(&s, &up, 1, u) == hipSuccess);
            if (u == Until::kDone) CHECK(s.idle());
            if (u == Until::kQueued) s.sync();
            std::fill(src.begin(), src.end(), uint8_t(0));   // the caller's own again
            s.sync();
            CHECK(dev == host);
        }
        for (int at = 0; at < 8; ++at)
            for (bool out : {false, true}) {
                if (n < 6 * MiB && at > 1) continue;   // one copy
                st.delay_us = 200;
                Bytes src = host, dev(n);
                const HostCopy k = flat_copy(src.data(), dev.data(), n);
                st.fail_copy_in = at;
                const hipError_t e = out ? c.to_host(&s, &k, 1) : c.to_device(&s, &k, 1);
                const bool hit = st.fail_copy_in < 0;
                st.fail_copy_in = -1;
                CHECK((e == hipSuccess) == !hit);
                CHECK(s.idle());
                // the next transfer is whole
                st.delay_us = 0;
                Bytes to(n);
                src = host;
                const HostCopy up = flat_copy(src.data(), to.data(), n);
                CHECK(c.to_device(&s, &up, 1) == hipSuccess && to == host);
            }
    }
    st.delay_us = 0;
}

// The process's threads and, of those beside them, the ones that take no signal.
static void threads(size_t* all, size_t* deaf) {
    *all = *deaf = 0;
    DIR* d = opendir("/proc/self/task");
    CHECK(d);
    while (dirent* e = readdir(d)) {
        if (e->d_name[0] == '.') continue;
        FILE* f = fopen(("/proc/self/task/" + std::string(e->d_name) + "/status").c_str(), "r");
        if (!f) continue;   // gone meanwhile
        ++*all;
        char line[256];
        unsigned long long blocked = 0;
        while (fgets(line, sizeof(line), f)) sscanf(line, "SigBlk: %llx", &blocked);
        fclose(f);
        if ((blocked >> (SIGINT - 1)) & (blocked >> (SIGTERM - 1)) & (blocked >> (SIGUSR1 - 1)) & 1) ++*deaf;
    }
    closedir(d);
}

// Contexts share rings and threads: the second one's transfers allocate
// nothing and start no thread, many at once stay within bounds, and the last
// context gives everything back.
static void shared() {
    hip_sim::Stream s[12];
    size_t all0, deaf0, all, deaf;
    threads(&all0, &deaf0);
    CHECK(st.pinned_held == 0);
    {
        Copier a;
        CHECK(round_trip(a, &s[0], 20 * MiB, 1, 20 * MiB) == 0);
        const int pins = st.pinned_allocs;
        CHECK(pins > 0);
        threads(&all, &deaf);
        const size_t started = all - all0;
        CHECK(started <= 8 && deaf - deaf0 == started);
        CHECK(round_trip(a, &s[0], 20 * MiB, 1, 20 * MiB) == 0);
        {
            Copier b;
            for (size_t n : {8 * KiB, 600 * KiB, 9 * MiB, 20 * MiB}) CHECK(round_trip(b, &s[1], n, 1, n) == 0);
            CHECK(st.pinned_allocs == pins);
            threads(&all, &deaf);
            CHECK(all - all0 == started);
        }
        std::vector<std::thread> ts;
        std::atomic<int> busy{0};
        for (int k = 0; k < 12; ++k)
            ts.emplace_back([&, k] {
                Copier c;
                busy++;
                for (int r = 0; r < 4; ++r) {
                    const size_t n = 8 * MiB + 4099 * k;
                    round_trip(c, &s[k], n, 1, n);
                }
            });
        for (auto& t : ts) t.join();
        CHECK(st.pinned_held <= 4);
        threads(&all, &deaf);
        CHECK(all - all0 <= 8);
    }
    CHECK(st.pinned_held == 0 && st.events == 0);
    threads(&all, &deaf);
    CHECK(all == all0);
}

// A transfer does not wait for the DMAs that another stream's left behind.
static void streams() {
    hip_sim::Stream slow, s;
    Copier a, b;
    const size_t n = 8 * MiB;
    const Bytes x = noise(n, 1);
    Bytes dx(n), dy(n), y = x;
    const HostCopy up = flat_copy(y.data(), dx.data(), n);
    std::atomic<bool> go{false};
    slow.push([&] { while (!go) std::this_thread::yield(); });   // work before the upload
    CHECK(a.to_device(&slow, &up, 1, Until::kRead) == hipSuccess);
    std::fill(y.begin(), y.end(), uint8_t(0));
    const HostCopy up2 = flat_copy(x.data(), dy.data(), n);
    CHECK(b.to_device(&s, &up2, 1) == hipSuccess && dy == x);    // would hang
    go = true;
    slow.sync();
    CHECK(dx == x);
}

// Small downloads of several maps are the caller's alone, larger ones the
// threads' too; whole either way.
static void maps() {
    hip_sim::Stream s;
    Copier c;
    size_t all0, all, deaf;
    threads(&all0, &deaf);
    for (size_t px : {size_t(240 * 120), size_t(640 * 320)}) {
        const Bytes plane = noise(16 * px, 1), depth = noise(4 * px, 2), score = noise(4 * px, 3);
        Bytes p(16 * px), d(4 * px), sc(4 * px);
        const HostCopy down[3] = {flat_copy(p.data(), plane.data(), 16 * px), flat_copy(d.data(), depth.data(), 4 * px),
                                  flat_copy(sc.data(), score.data(), 4 * px)};
        CHECK(c.to_host(&s, down, 3) == hipSuccess);
        CHECK(p == plane && d == depth && sc == score);
        threads(&all, &deaf);
        CHECK((all > all0) == (24 * px > 1 * MiB));
    }
}

// Several threads on one context: host copies with more pieces than the ring
// has tasks, uploads and downloads of every path beside them, lists that mix
// pinned and pageable memory, downloads to fresh memory on both sides of their
// line.
static void together() {
    Copier c;
    std::vector<std::thread> ts;
    for (int k = 0; k < 2; ++k)
        ts.emplace_back([&, k] {
            const Bytes src = noise(70 * MiB + 12345, (unsigned)k);   // 281 pieces of 256 tasks
            for (int r = 0; r < 2; ++r) {
                Bytes dst(src.size());
                c.copy(dst.data(), src.data(), src.size());
                CHECK(dst == src);
                for (size_t n : {1 * KiB, 700 * KiB, 900 * KiB}) {
                    Bytes d(n);
                    c.copy(d.data(), src.data(), n);
                    CHECK(memcmp(d.data(), src.data(), n) == 0);
                }
            }
        });
    for (int k = 0; k < 2; ++k)
        ts.emplace_back([&] {
            hip_sim::Stream s;
            for (size_t n : {40 * KiB, 1 * MiB, 5 * MiB, 11 * MiB, 13 * MiB, 21 * MiB}) {
                const Bytes src = noise(n, (unsigned)n);
                Bytes dev(n), back(n);
                const HostCopy up = flat_copy(src.data(), dev.data(), n), down = flat_copy(back.data(), dev.data(), n);
                CHECK(c.to_device(&s, &up, 1) == hipSuccess && dev == src);
                CHECK(c.to_host(&s, &down, 1, true) == hipSuccess && back == src);
            }
        });
    ts.emplace_back([&] {
        hip_sim::Stream s;
        for (size_t n : {300 * KiB, 7 * MiB}) {
            void* pin = nullptr;
            CHECK(hipHostMalloc(&pin, n, hipHostMallocDefault) == hipSuccess);
            const Bytes a = noise(n, 3), b = noise(n, 4);
            memcpy(pin, b.data(), n);
            Bytes da(n), db(n), ra(n);
            const HostCopy up[2] = {flat_copy(a.data(), da.data(), n), flat_copy(pin, db.data(), n)};
            CHECK(c.to_device(&s, up, 2) == hipSuccess && da == a && db == b);
            const HostCopy down[2] = {flat_copy(ra.data(), db.data(), n), flat_copy(pin, da.data(), n)};
            CHECK(c.to_host(&s, down, 2) == hipSuccess && ra == b && memcmp(pin, a.data(), n) == 0);
            hipHostFree(pin);
        }
    });
    for (auto& t : ts) t.join();
}

int main(int argc, char** argv) {
    std::set<std::string> want(argv + 1, argv + argc);
    struct {
        const char* name;
        void (*f)();
    } parts[] = {{"pitched", pitched}, {"until", until}, {"shared", shared}, {"streams", streams}, {"maps", maps}, {"together", together}};
    for (auto& p : parts)
        if (want.empty() || want.count(p.name)) {
            p.f();
            CHECK(st.events == 0);
            printf("copy_selftest: %s ok\n", p.name);
        }
    return 0;
}
