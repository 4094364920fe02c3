// -*- C++ -*-
/// @file kernels_batch.hip
/// @brief Batch sets: persistent kernels that mix several built-in kernels.
#include "registry.hpp"

#include "../kernels/catalog.hpp"

namespace P = loom_amd::programs;
namespace S = loom_amd::smallpt;

// The path tracer's sweeping batch kernel fits five waves per SIMD by itself;
// held to six, 16 jobs of frames, fib and Collatz take 2.21 ms instead of 2.29 (a pass
// kernel of the path tracer alone is the same at both).
LOOM_HIP_BATCH_WAVES_HINT(6, S::smallpt9<float>);

// the mixed benchmark batch: path-trace frames with fib and Collatz jobs
LOOM_HIP_REGISTER_BATCH("pt_int_mix", S::smallpt9<float>, P::fib<std::uint64_t>,
                        P::collatz<std::uint64_t>);
// integer-only batch (a smaller register file, higher occupancy)
LOOM_HIP_REGISTER_BATCH("int_mix", P::fib<std::uint64_t>, P::collatz<std::uint64_t>,
                        P::factorial<std::uint64_t>);
// two kernels whose START is pooled
LOOM_HIP_REGISTER_BATCH("start_mix", P::started<std::uint64_t>, P::started<std::uint32_t>);
