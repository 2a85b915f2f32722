// fake_hip.h -- controls of the host stand-in for the HIP runtime (fake_hip.cpp). Test infrastructure only.
#pragma once

#include <functional>

// Number of devices hipGetDevice / hipSetDevice believe in (default 1; 0 makes hipGetDevice fail).
void fake_hip_set_device_count(int n);
// hipMalloc / hipHostMalloc / stream / event objects that exist right now: 0 after everything has been given back.
long fake_hip_live_allocations();
// Called at the top of every hipGetDevice (the first runtime call of a file-store transfer that meets a device iov):
// lets a test know that a put or get is inside the library. Empty function = no hook.
void fake_hip_on_get_device(std::function<void()> fn);
// Queues `job` on a stream of the stand-in, behind whatever was queued before: how the stand-ins of the library's
// kernel entry points (sanitize_host.cpp) do their work "on the device", in stream order.
void fake_hip_enqueue(void *stream, std::function<void()> job);
// What hipStreamQuery says of a stream that has something queued (default hipErrorNotReady), as an int; and whether
// hipStreamIsCapturing says that a stream is being captured. hipStreamQuery on such a stream ends the process: on the real
// runtime the question invalidates the capture.
void fake_hip_set_query_result(int error);
void fake_hip_set_capturing(bool on);
// The timer slack (ns) of the thread that called hipStreamQuery last.
int fake_hip_timer_slack_of_last_query();
