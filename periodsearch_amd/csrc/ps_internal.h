// ps_internal.h -- declarations shared by the host (ps_host.cpp) and device (ps_device.hip) halves of
// libpsamd.so.  Not part of the public ABI.
#pragma once

struct ps_handle;

// Records a message for ps_last_error() and returns code.
int ps_fail(int code, const char *fmt, ...);

// For the tests, which pin the route that a call took.
extern "C" {
// The fits (ps_fit_batch, ps_scan) or vectors (ps_eval) of the handle's last call that took the spread form.
int ps_test_spread(const ps_handle *h);
}
