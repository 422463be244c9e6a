// Host arrays to and from the device through pinned memory (host_stage.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <memory>

namespace fdmgpu {

class HostStage;

// Smallest copy the stage takes: below it the runtime's own copy of pageable
// memory is as fast or faster (a FP64 host solve, us, by the runtime / through the
// stage: 1.9 MiB 206-220 / 220-229, 3.8 MiB 390 / 335, 7.8 MiB 740 / 550).
constexpr size_t kStageMin = (size_t)3 << 20;

// The device's stage, shared by every plan that holds it and freed with the
// last of them; `create` false: only if there is one.  Null when it cannot be
// set up (the caller then copies as before).
std::shared_ptr<HostStage> host_stage(int device, bool create);

// Copies between host memory and the device on stream s, which belongs to the
// stage's device.  in: returns once every byte is read from src and enqueued.
// out: runs after what is enqueued on s; returns when dst is complete.
// hipErrorNotReady: another thread is using the stage (or no memory for the
// job's description); the copy is still to be made.
hipError_t stage_in(HostStage& st, void* dst, const void* src, size_t bytes, hipStream_t s);
hipError_t stage_out(HostStage& st, void* dst, const void* src, size_t bytes, hipStream_t s);

}  // namespace fdmgpu
