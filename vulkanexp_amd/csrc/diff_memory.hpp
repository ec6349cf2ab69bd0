// The device memory that a prepared differentiable context can do without.  Host code, no HIP.
#pragma once

#include <cstddef>
#include <cstdint>

namespace ddgi {

constexpr uint32_t kDiffRecRows = 5;            // float4s of a texel's sampling record
constexpr uint64_t kDiffRecords = 12u << 20;    // most texels whose records are kept (1 GiB; a 4K view has 8.3 M)
constexpr uint64_t kDiffTapProbes = 1u << 18;   // most probes whose texels are ordered by colour tap

struct DiffSpare {
	void* keys;      // three arrays of probes * taps counters, null: not even one counter per probe fits
	uint32_t taps;   // texels of a cell ordered by their first colour tap (64), or not (1)
	void* records;   // texels * kDiffRecRows float4s, null: the sampling weights are recomputed
};

// alloc(bytes): device memory, or null when it does not fit.  Called for everything the context cannot do
// without before this: what is left over decides.
template <class Alloc>
DiffSpare diff_spare_memory(uint64_t texels, uint64_t probes, const Alloc& alloc) {
	DiffSpare m{nullptr, 64u, nullptr};
	if(probes <= kDiffTapProbes) m.keys = alloc(size_t(probes) * m.taps * 3 * sizeof(uint32_t));
	if(!m.keys) {
		m.taps = 1u;
		m.keys = alloc(size_t(probes) * 3 * sizeof(uint32_t));
	}
	if(m.keys && texels <= kDiffRecords) m.records = alloc(size_t(texels) * kDiffRecRows * 4 * sizeof(float));
	return m;
}

}  // namespace ddgi
