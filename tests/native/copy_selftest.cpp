// copy_selftest.cpp -- the staged host copies (pmp_copy.hip) on the CPU against
// a simulated HIP runtime (hip_sim), under the sanitizers.  Exits non-zero on
// the first failed check (or a sanitizer report).
//
//   copy_selftest [part ...]     the parts by name; all of them by default
#include <stdio.h>
#include <stdlib.h>

#include <random>
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
    std::mt19937 g(seed);
    Bytes b(n);
    for (size_t k = 0; k < n; ++k) b[k] = (uint8_t)(g() >> 11);
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
    s->sync();
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
}

int main(int argc, char** argv) {
    std::set<std::string> want(argv + 1, argv + argc);
    struct {
        const char* name;
        void (*f)();
    } parts[] = {{"pitched", pitched}};
    for (auto& p : parts)
        if (want.empty() || want.count(p.name)) {
            p.f();
            CHECK(st.events == 0);
            printf("copy_selftest: %s ok\n", p.name);
        }
    return 0;
}
