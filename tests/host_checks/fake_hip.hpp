// fake_hip.hpp -- a HIP runtime without a device, for checks of the library's
// host code on the CPU: the runtime sources link against fake_hip.cpp instead
// of libamdhip64.  Device memory is host memory.  Kernels are recorded and not
// run; copies are carried out in order when the stream is waited for, so a copy
// whose host memory is freed before that is seen.  Each kind of call can be
// made to fail.
#pragma once
#include <stddef.h>

#include <string>
#include <vector>

namespace fake {
struct Launch {
  std::string name;
  unsigned grid[3], block, lds;
};
extern std::vector<Launch> launches;
extern size_t pending_host_copies();  // queued copies that name pageable host memory
extern size_t freed_under_copy;       // frees of host memory that a queued copy names

// The nth call of the kind from now fails, once (0: none): an allocation by
// operator new, a kernel launch, a copy.
enum Kind { kNew, kLaunch, kCopy, kKinds };
void fail_nth(Kind kind, long n);
bool failed(Kind kind);  // whether that call has been reached
}  // namespace fake
