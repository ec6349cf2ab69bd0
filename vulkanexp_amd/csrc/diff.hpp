// Arguments and launchers of the differentiable probe update (diff.hip).
#pragma once

#include "diff_memory.hpp"
#include "kernels.hpp"

namespace ddgi {

constexpr uint32_t kDiffChunk = 1024;  // G-buffer texels per backward work item (one cell)
constexpr uint32_t kDiffSumBlocks = 64;  // workgroups that add up the material partial sums

struct DiffArgs {
	GridConst grid;
	// fixed by prepare
	const float4* factors;          // [rays][4], thread (ray_order) order within a slot
	const uint16_t* perm;           // ray order
	const float4* dirs;             // world directions of the prepared frame (ray index order)
	const float* inv_sum;           // blend normalisation per texel (first 36: irradiance)
	const uint32_t* states;         // probe states after the prepared update
	const float2* dep;              // depth atlas after the prepared update
	const uint32_t* indices;        // probe per slot
	uint32_t slots;
	uint64_t rays;                  // slots * n
	const float* pos;               // G-buffer [N][3]
	const float* nrm;
	const float* tocam;
	const uint32_t* gmat;
	uint64_t N;
	uint32_t M;                     // material slots
	const uint32_t* sorted;         // texels sorted by cell
	const uint32_t* cell_item_start;  // [cells + 1]
	const uint32_t* item_begin;
	const uint32_t* item_count;
	const uint32_t* n_items;
	uint32_t max_items;
	// per call
	const float* albedo;            // [M][3]
	const float* sun;               // [3]
	const float* target;            // [N][3]
	float4* rad;                    // [rays]
	const float4* irr;              // differentiated irradiance atlas (tiled)
	const float4* rec;              // [N][kDiffRecRows] sampling records, nullptr: recomputed
	float* shade;                   // [N][3]
	float* loss_part;
	float* loss;
	long long* part_tile;           // [max_items][8][64][3]
	long long* part_mat_pix;        // [max_items][M][3]
	float* g_T;                     // [P][36][3]
	long long* part_mat_ray;        // [slots][M * 3 + 3]
	long long* part_rows;           // [kDiffSumBlocks][M * 3 + 3]
	const float* grad_loss;         // [1]
	float* g_albedo;                // [M][3]
	float* g_sun;                   // [3]
};

// Buffers of the texel binning; keys = cell * taps + first colour tap (taps = 64), or cells (taps = 1).
struct DiffBins {
	uint32_t taps;
	uint32_t *key_of;                // [N]
	uint32_t *key_count, *key_start, *cursor;  // [cells * taps]
	uint32_t *cell_item_start;       // [cells + 1]
	uint32_t *item_begin, *item_count, *n_items;
	uint32_t* sorted;                // [N]
};
hipError_t diff_bin(const DiffArgs& d, const DiffBins& b, hipStream_t s);
// The texels' sampling records (d.rec is set to them afterwards).
hipError_t diff_records(const DiffArgs& d, float4* rec, hipStream_t s);
hipError_t diff_radiance(const DiffArgs& d, hipStream_t s);
hipError_t diff_gather_forward(const DiffArgs& d, hipStream_t s);
hipError_t diff_backward(const DiffArgs& d, hipStream_t s);

}  // namespace ddgi
