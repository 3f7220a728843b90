/* Stands before the HIP runtime's own hipMalloc, hipFree, hipHostMalloc and
 * hipEventElapsedTime in a process that loads it first (RTLD_GLOBAL): device
 * memory up to a limit or all but one piece of it, pinned memory up to a size per
 * piece, and one event time that comes out fifty times too long.  For the tests
 * of what the library does then. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <stddef.h>

static struct { void* p; size_t n; } g_piece[65536];
static int g_pieces;
static long g_used, g_limit = -1, g_calls, g_fail = -1, g_pinned = -1, g_times, g_slow = -1;

long shim_used(void) { return g_used; }
long shim_times(void) { return g_times; }
long shim_calls(void) { return g_calls; }
void shim_fail(long call) { g_calls = 0; g_fail = call; }
void shim_limit(long bytes) { g_limit = bytes; }
void shim_pinned(long bytes) { g_pinned = bytes; }
void shim_slow(long call) { g_times = 0; g_slow = call; }

/* the runtime that the library under test has loaded */
static void* runtime(const char* name) {
    static const char* const names[] = {"libamdhip64.so.7", "libamdhip64.so.6", "libamdhip64.so"};
    void* h = NULL;
    for (int i = 0; i < 3 && !h; ++i) h = dlopen(names[i], RTLD_NOW | RTLD_NOLOAD);
    return h ? dlsym(h, name) : NULL;
}

int hipMalloc(void** p, size_t n) {
    static int (*real)(void**, size_t);
    if (!real) real = (int (*)(void**, size_t))runtime("hipMalloc");
    if (++g_calls == g_fail) return 2;
    if (g_limit >= 0 && g_used + (long)n > g_limit) return 2;
    int rc = real(p, n);
    if (rc == 0 && g_pieces < 65536) {
        g_piece[g_pieces].p = *p;
        g_piece[g_pieces++].n = n;
        g_used += (long)n;
    }
    return rc;
}

int hipFree(void* p) {
    static int (*real)(void*);
    if (!real) real = (int (*)(void*))runtime("hipFree");
    for (int i = 0; i < g_pieces; ++i)
        if (g_piece[i].p == p) {
            g_used -= (long)g_piece[i].n;
            g_piece[i] = g_piece[--g_pieces];
            break;
        }
    return real(p);
}

int hipHostMalloc(void** p, size_t n, unsigned flags) {
    static int (*real)(void**, size_t, unsigned);
    if (!real) real = (int (*)(void**, size_t, unsigned))runtime("hipHostMalloc");
    if (g_pinned >= 0 && (long)n > g_pinned) return 2;
    return real(p, n, flags);
}

int hipEventElapsedTime(float* ms, void* a, void* b) {
    static int (*real)(float*, void*, void*);
    if (!real) real = (int (*)(float*, void*, void*))runtime("hipEventElapsedTime");
    int rc = real(ms, a, b);
    if (++g_times == g_slow) *ms *= 50.0f;
    return rc;
}
