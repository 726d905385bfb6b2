// CPU check of the workspace registry (sneppx-alg_amd/csrc/ws_registry.h) while
// a stream is being captured: nothing is allocated, filled or freed on that
// stream, and what a recorded call was given stays at its address.  Built and
// run by tests/test_ws_capture.py; exit status 0 when every check holds.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>
#include <thread>

#include "ws_registry.h"

static std::set<void*> g_held;
static long g_on_stream = 0, g_apart = 0;
static bool g_capturing = false, g_bad = false;

static void* on_stream(size_t bytes, void*, bool zeroed) {
    if (g_capturing) g_bad = true;
    g_on_stream++;
    void* p = malloc(bytes);
    memset(p, zeroed ? 0 : 0xAA, bytes);
    g_held.insert(p);
    return p;
}
static void* apart(size_t bytes, bool zeroed) {
    g_apart++;
    void* p = malloc(bytes);
    memset(p, zeroed ? 0 : 0xAA, bytes);
    g_held.insert(p);
    return p;
}
static void release(void* p, void*) {
    if (g_capturing || !g_held.erase(p)) g_bad = true;
    else free(p);
}
static void* get(void* stream, int slot, size_t bytes, bool zeroed = false) {
    return snx_ws::get(0, stream, slot, bytes, zeroed, g_capturing);
}

#define CHECK(c)                                                          \
    do {                                                                  \
        if (!(c)) {                                                       \
            fprintf(stderr, "check failed at line %d: %s\n", __LINE__, #c); \
            return 1;                                                     \
        }                                                                 \
    } while (0)

int main() {
    snx_ws::init(on_stream, release, apart);
    void* const S1 = (void*)0x1000;
    void* const S2 = (void*)0x2000;

    // a warmed stream: the recorded call takes the eager call's buffer
    void* a = get(S1, 0, 1000);
    g_capturing = true;
    CHECK(get(S1, 0, 900) == a && g_apart == 0);
    // a slot that no eager call used: taken apart, zeroed at once, and the
    // later eager call's too
    unsigned char* c = (unsigned char*)get(S1, 4, 64, true);
    CHECK(c && g_apart == 1);
    for (int i = 0; i < 64; i++) CHECK(c[i] == 0);
    // larger than the eager call's: another one, the old one neither freed nor moved
    void* b = get(S1, 0, 100000);
    CHECK(b && b != a && g_held.count(a) && g_apart == 2);
    g_capturing = false;
    CHECK(get(S1, 4, 64, true) == c && get(S1, 0, 100) == b && g_on_stream == 1);

    // a larger eager call later: both recorded buffers stay, the newest is handed out
    void* d = get(S1, 0, 1000000);
    CHECK(d != a && d != b && g_held.count(a) && g_held.count(b));
    CHECK(get(S1, 0, 10) == d);
    // which no graph has seen: the next one replaces it
    void* e = get(S1, 0, 10000000);
    CHECK(e != d && !g_held.count(d) && g_held.count(a) && g_held.count(b));
    CHECK(snx_ws::live() == 4 && (long)g_held.size() == 4);

    // bounded: recording ever larger calls keeps less than four times the largest
    size_t total = 0, last = 0;
    g_capturing = true;
    for (size_t n = 1; n < (64u << 20); n += n / 64 + 1) {
        void* p = get(S2, 0, n);
        const size_t want = (n + (n >> 2) + 4095) & ~(size_t)4095;
        static void* prev = nullptr;
        if (p != prev) {
            total += want;
            last = want;
            prev = p;
        }
    }
    g_capturing = false;
    CHECK(total < 5 * last + (1 << 20));

    // a thread that ends leaves all of them; the next one is given the newest
    void *x = nullptr, *y = nullptr, *z = nullptr;
    void* const S3 = (void*)0x3000;
    std::thread([&] {
        g_capturing = true;
        x = get(S3, 0, 64);
        g_capturing = false;
        y = get(S3, 0, 64000);
    }).join();
    std::thread([&] { z = get(S3, 0, 64); }).join();
    CHECK(x != y && z == y && g_held.count(x));

    for (void* s : {S1, S2, S3}) snx_ws::release_stream(s);
    CHECK(!g_bad && snx_ws::live() == 0 && g_held.empty());
    printf("ok: %ld on a stream, %ld apart\n", g_on_stream, g_apart);
    return 0;
}
