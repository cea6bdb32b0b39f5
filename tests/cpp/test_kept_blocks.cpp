// The device blocks the library keeps between uses (si_index.hip), on a device of this file's own
// with little memory: the HIP calls that allocate and free are defined here.  No GPU is used.
#include <map>

#include "si_index.hip"

static const size_t MB = 1 << 20;
static size_t g_total = 1000 * MB, g_used = 0;
static bool g_capture = false;
static std::map<void*, size_t> g_held;

static hipError_t fake_malloc(void** p, size_t bytes) {
    *p = (void*)8;   // (an allocation that failed may leave anything)
    if (g_used + bytes > g_total) return hipErrorOutOfMemory;
    static uintptr_t next = 4096;
    *p = (void*)next;
    next += bytes + 4096;
    g_held[*p] = bytes;
    g_used += bytes;
    return hipSuccess;
}
extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) { return fake_malloc(p, bytes); }
hipError_t hipMallocAsync(void** p, size_t bytes, hipStream_t) { return fake_malloc(p, bytes); }
hipError_t hipFree(void* p) {
    if (p) {
        g_used -= g_held.at(p);
        g_held.erase(p);
    }
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = g_capture ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
}
// (of the library's other files)
int64_t si_tune_long_len() { return -1; }
void si_learned_forget_index(siLearned*) {}

#define CHECK(x)                                        \
    do {                                                \
        if (!(x)) {                                     \
            printf("line %d: %s\n", __LINE__, #x);      \
            return 1;                                   \
        }                                               \
    } while (0)

// 600 MB of kept blocks, of 1000.
static bool keep_some() {
    size_t a = 0, b = 0;
    void *p = si_block_take(400 * MB, &a), *q = si_block_take(200 * MB, &b);
    if (!p || !q) return false;
    si_block_give(p, a, 0, true);
    si_block_give(q, b, 0, true);
    return g_used == 600 * MB;
}

int main() {
    si_block_users(1);
    // what the kept blocks leave no room for is allocated in their place, by every form
    void* p = nullptr;
    CHECK(keep_some());
    CHECK(si_malloc(&p, 900 * MB) == hipSuccess && g_used == 900 * MB);
    CHECK(hipFree(p) == hipSuccess && keep_some());
    CHECK(si_malloc_async(&p, 900 * MB, nullptr) == hipSuccess && g_used == 900 * MB);
    size_t got = 0;
    CHECK(hipFree(p) == hipSuccess && keep_some());
    CHECK((p = si_block_take(900 * MB, &got)) && g_used == 900 * MB);
    si_block_give(p, got, 0, false);
    CHECK(g_used == 0);
    // more than there is: an error, a null pointer, nothing held
    CHECK(keep_some());
    CHECK(si_malloc(&p, 1001 * MB) != hipSuccess && !p && g_used == 0);
    CHECK(keep_some());
    CHECK(!si_block_take(1001 * MB, &got) && g_used == 0);
    // a captured stream: an error, and the kept blocks stay
    CHECK(keep_some());
    g_capture = true;
    CHECK(si_malloc_async(&p, 900 * MB, nullptr) != hipSuccess && !p && g_used == 600 * MB);
    g_capture = false;
    // memory that lasts does not sit in a block much larger than itself; a call's may
    const size_t was = g_used;
    size_t lasting = 0, passing = 0;
    void *l = si_block_take(180 * MB, &lasting, true), *t = si_block_take(105 * MB, &passing);
    CHECK(l && lasting == 200 * MB && t && passing == 105 * MB);
    si_block_give(l, lasting, 0, true);
    si_block_give(t, passing, 0, true);
    CHECK((l = si_block_take(170 * MB, &lasting, true)) && lasting == 170 * MB && g_used == was + 275 * MB);
    CHECK((t = si_block_take(110 * MB, &passing)) && passing == 200 * MB && g_used == was + 275 * MB);
    si_block_give(l, lasting, 0, true);
    si_block_give(t, passing, 0, true);
    si_block_users(-1);   // the last user takes them along
    CHECK(g_used == 0);
    printf("ok\n");
    return 0;
}
