/* Stands in for the runtime's page-locked allocation, which it refuses (tests only). */
#include <stddef.h>

static int refused;

int hipHostMalloc(void **ptr, size_t bytes, unsigned flags) {
    (void)bytes;
    (void)flags;
    *ptr = NULL;
    ++refused;
    return 2; /* hipErrorOutOfMemory */
}

int no_pinned_refused(void) { return refused; }
