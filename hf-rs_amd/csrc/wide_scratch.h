// wide_scratch.h -- one queue for the kernels with the largest private segments.
//
// The runtime backs a kernel's private segment on the hardware queue it runs on,
// for every wave the chip could hold: 16,132 bytes a lane ((fd|dd)) x 64 lanes x 32
// waves x 256 CUs = 8.5 GB, kept by that queue.  A process has four hardware queues
// and about 32 GiB of address space for all their segments; the streams of several
// contexts are dealt over all four, and once each holds what (dd|dd) asks for
// (10,200 bytes, 5.3 GB), growing them one after another to 8.5 GB finds no room
// in the end: the launch fails with HSA_STATUS_ERROR_OUT_OF_RESOURCES.  Kernels
// beyond 10,240 bytes therefore run on one stream of the device, kept until the
// process ends, between events of the caller's: 3 x 5.4 + 8.5 GB.  They are chosen
// by class where they are launched; tests/test_private_segments.py checks the built
// kernels against the limit.
#pragma once
#include <hip/hip_runtime.h>

#include <functional>

namespace hfg {

// Runs launch(w) on the device's stream w for such kernels, after what stream s
// holds and before what it gets next.  Any thread.
void launch_wide(hipStream_t s, const std::function<void(hipStream_t)>& launch);

}  // namespace hfg
