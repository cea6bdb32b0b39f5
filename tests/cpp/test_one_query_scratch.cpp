// The single-query scratch (si_internal.h OneQuery) when a step of its making fails: the HIP calls
// it makes are this file's own, told which of them to fail.  No GPU is used.
#include <cstdio>
#include <cstdlib>

#include "si_internal.h"

static int g_fail = 0, g_memory = 0, g_streams = 0;   // the step that fails (1..3), and what is held
static char g_buf[4096];

int si_set_error(int code, const char*, ...) { return code; }
extern "C" {
hipError_t hipHostMalloc(void** p, size_t, unsigned) {
    if (g_fail == 1) {
        *p = (void*)8;   // (an allocation that failed may leave anything)
        return hipErrorOutOfMemory;
    }
    ++g_memory;
    *p = g_buf;
    return hipSuccess;
}
hipError_t hipHostGetDevicePointer(void** d, void* h, unsigned) {
    if (g_fail == 2) return hipErrorInvalidValue;
    *d = h;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    if (g_fail == 3) return hipErrorOutOfMemory;
    ++g_streams;
    *s = (hipStream_t)16;
    return hipSuccess;
}
hipError_t hipHostFree(void* p) {
    if (p == g_buf) --g_memory;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) {
    --g_streams;
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "failed"; }
}

#define CHECK(x)                                                             \
    do {                                                                     \
        if (!(x)) {                                                          \
            printf("step %d, line %d: %s\n", g_fail, __LINE__, #x);          \
            return 1;                                                        \
        }                                                                    \
    } while (0)

int main() {
    for (int step = 1; step <= 3; ++step) {
        OneQuery o;
        g_fail = step;
        for (int turn = 0; turn < 2; ++turn) {   // a second call must not take half a scratch for a whole one
            CHECK(o.make(100) != SI_OK);
            CHECK(!o.h && !o.d && !o.st && !o.cap && g_memory == 0 && g_streams == 0);
        }
        g_fail = 0;
        CHECK(o.make(100) == SI_OK && o.h && o.d && o.st && o.cap == 100);
        CHECK(o.make(100) == SI_OK && g_memory == 1 && g_streams == 1);
        o.release();
        CHECK(g_memory == 0 && g_streams == 0 && !o.cap);
    }
    printf("ok\n");
    return 0;
}
