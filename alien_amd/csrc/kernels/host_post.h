// Words a kernel hands to a host thread that polls for them (alien_hip_ctx::fetch).
#pragma once

namespace alien_hip {

// pinned, coherent host memory: each 32-bit word is stored as tag << 32 | word, so that a word is
// known to be there, whole, when its tag is (tag 0: never used)
struct HostPost {
  unsigned long long* to = nullptr;
  unsigned tag = 0;
};

} // namespace alien_hip
