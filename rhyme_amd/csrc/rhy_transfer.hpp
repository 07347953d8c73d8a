// rhy_transfer.hpp -- copies between device state and the caller's host
// arrays (state mirrors, snapshot payloads).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace rhy {

// count values at dev (device) and host.
struct HostSpan {
  void* dev;
  void* host;
  size_t count;
};

// Copies every span on `stream` and waits for it.  Device values take esz
// bytes; host values the same, or, with as_double, are doubles of device
// floats.  to_host gives the direction.  wait = false: the caller waits for the
// stream itself before it returns, so that a copy that needs nothing from the
// host once queued does not (4 us of a snapshot's way in).
hipError_t copy_spans(hipStream_t stream, const HostSpan* spans, int nspans, size_t esz,
                      bool as_double, bool to_host, bool wait = true);

// Objects that may copy (boxes, batches): the staging memory is given back
// when the last one goes.
void transfer_user_add();
void transfer_user_drop();

}  // namespace rhy
