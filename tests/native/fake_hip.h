// Controls of the device-less HIP runtime (fake_hip.cpp).
#pragma once
#include <cstddef>

// Closed: every stream synchronisation waits until the gate opens.
void fake_hip_gate(bool closed);
// Returns once some thread waits in a stream synchronisation.
void fake_hip_wait_for_waiter();
// Device memory, in all and free, that the runtime states (256 GiB at first).
void fake_hip_memory(std::size_t bytes);
// Kernels launched so far.
std::size_t fake_hip_launches();
