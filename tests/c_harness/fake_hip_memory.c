/* Stand-ins for the HIP calls behind the library's workspace, for a process
 * without a GPU: loaded before the library with RTLD_GLOBAL, they take the
 * place of the runtime's own.  Streams are numbers, their own ids (0 is the null
 * stream, and HIP gives 1 and 2 a meaning of their own); an allocation is an
 * address that nobody reads.  Work is under way from each allocation until the
 * next hipDeviceSynchronize, and freeing memory out of its stream's order then
 * is wrong.  The program sets fake_limit, the memory of the device, and
 * fake_refuse, which makes frees fail; the counters say which calls were made. */
#include <stddef.h>
#include <stdint.h>

enum { MOST = 4096 };
static struct { char *p; size_t size; uintptr_t stream; } live[MOST];
static uintptr_t next_address = 4096;
size_t fake_limit = (size_t)-1, fake_bytes;
int fake_refuse, fake_working, fake_mallocs, fake_frees_async, fake_frees, fake_wrong;

static int find(void *p) {
    for (int i = 0; i < MOST; ++i)
        if (live[i].p == p) return i;
    return -1;
}
static int drop(void *p) {
    const int i = find(p);
    if (i < 0) return ++fake_wrong, 1;
    fake_bytes -= live[i].size;
    live[i].p = NULL;
    return 0;
}
int hipGetDevice(int *device) { return *device = 0; }
int hipStreamIsCapturing(void *s, int *status) { return (void)s, *status = 0; }
int hipStreamGetId(void *s, unsigned long long *id) { return *id = (uintptr_t)s, 0; }
int hipMallocAsync(void **p, size_t size, void *s) {
    ++fake_mallocs;
    if (fake_bytes + size > fake_limit) return 2;   /* hipErrorOutOfMemory */
    const int i = find(NULL);
    live[i].p = *p = (void *)next_address;
    live[i].size = size;
    live[i].stream = (uintptr_t)s;
    next_address += 4096;
    fake_bytes += size;
    fake_working = 1;
    return 0;
}
int hipFreeAsync(void *p, void *s) {
    ++fake_frees_async;
    if (fake_refuse) return 900;   /* hipErrorStreamCaptureUnsupported */
    const int i = find(p);
    if (i >= 0 && live[i].stream != (uintptr_t)s) ++fake_wrong;   /* its stream may still use it */
    return drop(p);
}
int hipFree(void *p) {
    ++fake_frees;
    if (fake_working) ++fake_wrong;
    return fake_refuse ? 900 : drop(p);
}
int hipDeviceSynchronize(void) { return fake_working = 0; }
int hipSetDevice(int device) { return device; }
int hipGetLastError(void) { return 0; }
int hipDeviceGetDefaultMemPool(void **pool, int device) { return *pool = NULL, device; }
int hipMemPoolTrimTo(void *pool, size_t keep) { return pool || keep; }
