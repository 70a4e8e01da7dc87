/* Test infrastructure: BNN_BufferAlloc in front of the backend's own, for callers that resolve
 * the symbol while this library is in the global scope (the engine library).  The countdown-th
 * call from alloc_fail_arm on finds no memory; every other one is the backend's. */
#include <stddef.h>

#include "bnn-accelerator.h"

typedef BNN_Status (*alloc_fn)(BNN_Device, size_t, BNN_Buffer*);

static alloc_fn real_alloc;
static int calls_left;

void alloc_fail_arm(alloc_fn real, int countdown) {
    real_alloc = real;
    calls_left = countdown;
}

int alloc_fail_left(void) { return calls_left; }

BNN_Status BNN_BufferAlloc(BNN_Device device, size_t bytes, BNN_Buffer* out_buffer) {
    if (calls_left > 0 && --calls_left == 0) {
        *out_buffer = NULL;
        return BNN_ENOMEM;
    }
    return real_alloc(device, bytes, out_buffer);
}
