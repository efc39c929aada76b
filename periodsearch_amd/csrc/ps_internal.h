// ps_internal.h -- declarations shared by the host (ps_host.cpp) and device (ps_device.hip) halves of
// libpsamd.so.  Not part of the public ABI.
#pragma once

#include <cstddef>

struct ps_handle;
struct ps_batch;

// Records a message for ps_last_error() and returns code.
int ps_fail(int code, const char *fmt, ...);

// For the tests, which pin the route that a call took and what it does at the limits of memory.
extern "C" {
// The fits (ps_fit_batch, ps_scan, ps_batch_run) or vectors (ps_eval) of the last call that took the spread form.
int ps_test_spread(const ps_handle *h);
int ps_test_batch_spread(const ps_batch *b);
// Caps what later calls can have: bytes of device memory for the spread form's buffers, of pinned memory for
// the outputs of ps_eval.
void ps_test_limits(ps_handle *h, size_t arena, size_t pinned);
void ps_test_batch_limits(ps_batch *b, size_t arena);
// The bytes of a device's idle arenas (the spread form's memory) and its open handles.
size_t ps_test_arenas(int device, int *handles);
}
