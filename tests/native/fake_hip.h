// Controls of the device-less HIP runtime (fake_hip.cpp).
#pragma once
#include <cstddef>

// Closed: every stream synchronisation waits until the gate opens.
void fake_hip_gate(bool closed);
// Returns once some thread waits in a stream synchronisation.
void fake_hip_wait_for_waiter();
// Kernels launched so far.
std::size_t fake_hip_launches();
