// Turns of the calls on one workspace (host only, no HIP dependency).
//
// A call of several kernels hands partials from one to the next in its workspace, and a
// workspace serves every call of its stream. The stream runs kernels in order, but threads
// that launch on it at the same time could put another call's kernel between two of one
// call. A call therefore holds its workspace's turn from its first launch to its last.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include <mutex>

namespace fdllm {

constexpr size_t kTurns = 61;  // workspaces that share one only wait for each other

inline std::mutex& turn_of(const void* workspace) {
  static std::mutex turns[kTurns];
  return turns[(reinterpret_cast<uintptr_t>(workspace) >> 8) % kTurns];
}

// Held until the end of the scope; none for a call without a workspace.
class WorkspaceTurn {
 public:
  explicit WorkspaceTurn(const void* workspace) {
    if (workspace != nullptr) lock_ = std::unique_lock<std::mutex>(turn_of(workspace));
  }

 private:
  std::unique_lock<std::mutex> lock_;
};

}  // namespace fdllm
