/* Stand-ins for a few HIP and rocFFT functions, loaded before the engine: they call the real ones and count the waits for
 * a stream, and the one that is armed reports a failure at its k-th call from then on, after having done its work. */
#define _GNU_SOURCE
#include <dlfcn.h>
#include <string.h>

static char target[64];
static int before, failed, waits;

void arm(const char *name, int k)
{
    strncpy(target, name, sizeof(target) - 1);
    before = k;
    failed = waits = 0;
}
int failures(void) { return failed; }
int waits_since_failure(void) { return waits; }

static void *real(const char *lib, const char *name)
{
    void *h = dlopen(lib, RTLD_NOW | RTLD_NOLOAD);
    return h ? dlsym(h, name) : 0;
}
static int fails(const char *name)
{
    if (failed || strcmp(target, name) || before-- > 0) return 0;
    return failed = 1;
}
#define HIP "libamdhip64.so.7"
int hipGetLastError(void)
{
    const int r = ((int (*)(void))real(HIP, "hipGetLastError"))();
    return fails("hipGetLastError") ? 999 : r;
}
int hipEventRecord(void *event, void *stream)
{
    const int r = ((int (*)(void *, void *))real(HIP, "hipEventRecord"))(event, stream);
    return fails("hipEventRecord") ? 999 : r;
}
int hipStreamSynchronize(void *stream)
{
    waits += failed;
    return ((int (*)(void *))real(HIP, "hipStreamSynchronize"))(stream);
}
int rocfft_execute(void *plan, void **in, void **out, void *info)
{
    const int r = ((int (*)(void *, void **, void **, void *))real("librocfft.so.0", "rocfft_execute"))(plan, in, out, info);
    return fails("rocfft_execute") ? 1 : r;
}
