// Up to where an upload is a kernel of one workgroup (runtime.hip has the times of both sides).  The graph brings token ids with their values up to there.
#pragma once
#include <cstddef>

constexpr size_t kCopyKernelBytes = size_t(96) << 10;
