// Kernel-argument structs and launcher declarations shared by the HIP translation units and the
// C-ABI implementation.  Everything a kernel reads is passed by value or as raw device pointers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/ddgi.h"
#include "bvh.hpp"

namespace ddgi {

constexpr float kPiF = 3.1415926538f;  // src/shaders/common.glsl:4
constexpr uint32_t kMaxRays = 512;
constexpr uint32_t kIrrTexels = 36;    // 6x6 interior of the 8x8 tile
constexpr uint32_t kDepTexels = 196;   // 14x14 interior of the 16x16 tile
constexpr uint32_t kBlendTexels = kIrrTexels + kDepTexels;
constexpr uint32_t kWeightRows = 256;  // blend weight rows: 36 irradiance + 12 zero + 196 depth + 12 zero
constexpr uint32_t kTraceBlock = 128;  // threads per traversal block
constexpr uint32_t kPrimaryBlock = 256;  // threads per block of the probe update's primary traversal
constexpr uint32_t kShadeBlock = 64;     // threads per block of the shading kernels (k_shade, k_reflection_shade, k_batch_shade)

// Grid constants derived on the host (FP32, same operations as the oracle's ray generation).
struct GridConst {
	float emin[3];
	float cell[3];        // (max - min) / (res - 1)
	float cell_len;       // length(cell)
	float hysteresis;
	float sharpness;
	float shadow_bias;
	float tmax_primary;   // length(max - min)
	int32_t res[3];
	uint32_t n;           // rays per probe
	uint32_t probe_count;
};

struct Rot {
	float r[9];  // row-major, rows X, Y, Z
};

struct LightConst {
	float dir[3];    // toward the light
	float color[3];  // radiance
	float sky[3];    // constant miss radiance
	float sky_brightness;  // the light colour's 4th component: sun scale of the atmospheric sky
	uint32_t sky_model;    // DDGI_SKY_CONSTANT or DDGI_SKY_ATMOSPHERE
};

// Per-instance shading record: normal matrix transpose(inverse(M)) row-major, custom index
// (offset-table entry) and the global id of the instance's first triangle.
struct InstanceDev {
	float nm[9];
	uint32_t custom_index;
	uint32_t prim_base;
	uint32_t mask;
};

struct SceneDev {
	const float4* nodes;       // the traversal's packed nodes (kPackedNodeBytes each)
	const float4* tris;
	const InstanceDev* inst;
	const uint32_t* offsets;   // 3 per entry (material, vertex offset, index offset)
	const uint32_t* indices;
	const float4* vertices;    // 4 float4 per vertex (64-byte record)
	const float* materials;    // 12 floats per material
	uint32_t tri_count;
	uint32_t node_count;
	uint32_t instance_count;
};

// One moved instance: its transform, its motion since the BVH was built (both row-major 3x4), the triangle
// records' meta word (mask | flip << 8) and its shading record.
struct InstanceMove {
	float xf[12];
	float rel[12];
	InstanceDev inst;
	uint32_t meta;
};

// Boxes (6 floats: lo, hi) of the triangle slots (level 0) and of 8, 64, 512, ... consecutive ones: level
// l has count[l] boxes from box first[l] on.
constexpr uint32_t kBoxLevels = 12;
struct BoxTree {
	float* boxes;
	uint32_t levels;
	uint32_t first[kBoxLevels], count[kBoxLevels];
};

struct SlotBoxArgs {
	float4* tris;
	const float* obj;        // object-space vertices per slot (9 floats)
	const float* slot_box;   // the builder's piece bounds per slot
	const float* rel_xf;     // per instance its motion since the build (3x4)
	const InstanceMove* moves;  // of instances first .. first + count - 1
	uint32_t first, count, tri_count;
	BoxTree tree;
};

// Internal hit record: (t, slot | back << 31, u, v); slot = triangle position in the BVH array,
// 0xFFFFFFFF = miss (t = -1).
// List counters, each on its own 128-byte line (device-scope atomics on one line serialise): the
// primary pass appends its front-face hits to kShadeSegments segments of the shade list, segment s
// counted at [kCounterStride * s] (workgroup b of an update appends to segment b % kShadeSegments, so each
// XCD has its own counter; item i of a batched volume to segment i % kShadeSegments); the miss list is counted at [kMissCountSlot]; the key sort stores the
// ordered list's length at [kShadeTotalSlot], which the shading reads.
constexpr uint32_t kShadeSegments = 8;
constexpr uint32_t kCounterStride = 32;
constexpr uint32_t kMissCountSlot = kCounterStride * kShadeSegments;
constexpr uint32_t kShadeTotalSlot = kMissCountSlot + kCounterStride;
constexpr uint32_t kBlendDoneSlot = kShadeTotalSlot + kCounterStride;  // PhaseStamps::done
constexpr uint32_t kListCounterBytes = (kBlendDoneSlot + kCounterStride) * 4;
// An update orders its shade list from this many rays (slots x rays per probe) up.  The ordering's four
// launches cost 25 to 60 us; it shortens the shading by less than that while the hits' probe tiles and BVH
// nodes fit the caches anyway.  Whole update without / with the ordering, us, instances of the scene 24, 80, 256:
//   rays   32768                        524288                       1048576                      2097152
//          122 / 145 144 / 170 168 / 192  186 / 213 228 / 245 266 / 285  245 / 250 324 / 300 385 / 372  391 / 358 550 / 477 689 / 591
constexpr uint64_t kShadeSortRays = 640u * 1024u;

// Phase times of an update, in ticks of the device's wall clock, in pinned host memory: [0] the start, then
// the starts of [1] tracing, [2] ordering or shading, [3] the blend, and [4] the end, written by the blend's
// last workgroup (`done`: device counter, 0 between launches).  Each kernel's first workgroup stores its
// own start: an event record between two kernels holds the second back for 4 us, and there were four.
struct PhaseStamps {
	unsigned long long* host;  // null: no stamps
	uint32_t* done;
};

struct TraceFrameArgs {
	SceneDev scene;
	GridConst grid;
	LightConst light;
	const uint32_t* indices;   // probe linear index per slot
	const uint32_t* count;     // device count of slots
	const float4* dirs;        // world ray directions of the frame
	const uint16_t* perm;      // thread order -> ray index (directionally coherent)
	const uint32_t* states;    // probe states (read by sampleProbes)
	const float4* irr;         // exposed irradiance atlas (tiled)
	const float2* dep;         // exposed depth atlas (tiled)
	float4* hits;
	float4* rays;              // (rgb, depth)
	uint32_t* shade_list;      // ray positions (slot * n + k) of the front-face hits, filled by the primary pass
	uint32_t* shade_count;     // list counters (kShadeSegments segments, miss list, ordered total)
	uint32_t* miss_list;       // atmospheric sky only: ray positions of the misses
	uint32_t max_slots;        // grid sized for this many slots
	// optional (statistics runs only): [0]/[1] primary node / triangle fetches, [2]/[3] shadow
	// node / triangle fetches, [4] shadow rays
	unsigned long long* visit_counters;
	// optional (differentiable prepare): 4 float4 per ray, rad = c0 + A a + (B a + C) L:
	// (c0, material bits), (A, lit bits), (B, 0), (C, 0); material 0xFFFFFFFF for misses/back faces
	float4* factors;
	// optional (shade-list ordering): the primary pass stores the cell key of each shade-list entry
	// (cell coordinates shifted right by key_shift, so that they stay below 64 and keys below 2^18);
	// null: the segments are shaded as they were appended
	uint32_t* shade_keys;
	uint32_t key_shift;
	// the shade list is kShadeSegments segments of seg_cap entries
	uint32_t seg_cap;
	// optional (launch_shade): arrays copied by workgroups that follow the shading ones, counted in float4
	const float4* copy_src[2];
	float4* copy_dst[2];
	uint32_t copy_n[2];
	uint32_t shade_blocks;  // set by launch_shade
	unsigned long long* stamps;  // optional: PhaseStamps::host
};
constexpr uint32_t kShadeSortCounts = 1024 * 128 + 1024;  // (list tile, coarse digit) counters + digit totals

struct SelectState {
	uint32_t last_offset;
	uint32_t loop_index;
	uint32_t count;
	uint32_t pad;
};

struct BlendArgs {
	GridConst grid;
	const uint32_t* indices;
	const uint32_t* count;
	const float4* rays;         // slot-major (rgb, depth)
	const float* wt;            // FP32 weights [kWeightRows][n_pad]: irradiance rows 0..35, depth rows 48..243
	const float* inv_sum;       // [232]
	const void* w_lo16;         // MFMA paths: weights split hi/lo in 16-bit types
	const void* w_hi16;
	uint32_t* states;
	const float4* irr_prev;
	const float2* dep_prev;
	float4* irr_out;
	float2* dep_out;
	uint32_t max_slots;
	uint32_t flags;             // kBlendIrradianceOnly: no depth stores, no state update
	PhaseStamps stamps;         // optional
};
constexpr uint32_t kBlendIrradianceOnly = 0x1;

// Final gather over a G-buffer (FinalGather.frag:38-77).
struct GatherArgs {
	SceneDev scene;
	GridConst grid;
	LightConst light;
	const uint32_t* states;
	const float4* irr;
	const float2* dep;
	const ddgi_gbuffer_texel* gbuffer;
	const float* direct;      // optional, one value per texel
	const float* reflection;  // optional, rgb per texel
	float* out;               // rgb per texel
	uint64_t count;
	float origin[3];          // camera position (the view vectors' origin)
	float sdir[3];            // normalize(light direction), computed on the host
};

// Ray-traced shadow pass (directLight.rgen) over G-buffer texels.
struct DirectLightArgs {
	SceneDev scene;
	const ddgi_gbuffer_texel* gbuffer;
	const float2* noise;     // optional: the blue-noise sample per texel
	const float4* previous;  // optional: the previous frame's output (its g, b pass through)
	float4* out;
	uint64_t count;
	float sdir[3];           // normalize(light direction), computed on the host
};

// Reflection pass (reflection.rgen) over G-buffer texels.
struct ReflectionArgs {
	SceneDev scene;
	GridConst grid;
	LightConst light;
	const uint32_t* states;
	const float4* irr;
	const float2* dep;
	const ddgi_gbuffer_texel* gbuffer;
	const float2* noise;  // optional: the blue-noise sample per texel
	float4* out;
	uint64_t count;
	float origin[3];      // camera position
	// the chunk of texels [first, first + chunk) being traced; front-face hits of the chunk are
	// queued (chunk-local texel index, cell key) and shaded in key order
	uint64_t first;
	uint32_t chunk;
	float4* hits;         // [chunk] hit records of the queued texels
	uint32_t* list;       // [chunk]
	uint32_t* keys;       // [chunk]
	uint32_t* list_count;
	uint32_t key_shift;
};

// A list to order by key (launch_key_sort): keys, entries and the device length; scratch: counts
// (kShadeSortCounts) and bucket_keys / bucket_list (the list's capacity each).
struct SortJob {
	const uint32_t* keys;
	uint32_t* list;
	const uint32_t* count;  // segment s's length at count[kCounterStride * s]
	uint32_t* counts;
	uint32_t* bucket_keys;
	uint32_t* bucket_list;
	uint32_t* total;        // optional: receives the list's length
	uint32_t fine_bits;     // key bits below the 10-bit coarse digit
	uint32_t segments;      // the input list: `segments` segments of seg_cap entries (1: contiguous)
	uint32_t seg_cap;
	uint32_t pad;
};
// The sort kernels' argument: one job, or (many != nullptr) job y of workgroup (x, y) at
// many + y * stride.
struct BatchItem;
constexpr uint32_t kFineChunk = 4096;  // list entries per workgroup of the sort's last pass
struct SortJobs {
	SortJob one;
	const char* many;
	uint32_t stride;
	unsigned long long* stamp;  // optional: receives the start (PhaseStamps)
	const BatchItem* chunks;  // (job, chunk of kFineChunk entries) per workgroup of a batch's last pass
};
uint32_t sort_fine_bits(uint32_t key_bits);

// ---- launchers (return hipGetLastError of the launch) ----
hipError_t launch_frame_dirs(const Rot& R, const float4* fib, float4* dirs, uint32_t count, hipStream_t s);
// Orders job.list (keys job.keys of key_bits <= 18 bits; input in job.segments segments, output
// contiguous, at most `capacity` entries) in place: by the keys' high 10 bits over the whole list,
// and by the whole key inside each fixed chunk of 4096 entries (a bucket of equal high bits longer
// than a chunk is ordered chunk by chunk); entries with equal keys come in any order.  Scratch:
// job.counts (kShadeSortCounts), job.bucket_keys and job.bucket_list (capacity each).  The
// caller's job.fine_bits is ignored (set from key_bits).
hipError_t launch_key_sort(SortJob job, uint64_t capacity, uint32_t key_bits, hipStream_t s, unsigned long long* stamp = nullptr);
// Cell-key layout of the shade ordering for a grid: coordinate shift and bits per axis.
void shade_key_layout(const GridConst& g, uint32_t* shift, uint32_t* bits_per_axis);
hipError_t launch_clear(uint32_t* words, uint32_t n, hipStream_t s);
hipError_t launch_trace_primary(const TraceFrameArgs& a, hipStream_t s);
hipError_t launch_shade(const TraceFrameArgs& a, hipStream_t s);
// Atmospheric-sky radiance of the frame's misses (the miss list).
hipError_t launch_sky(const TraceFrameArgs& a, hipStream_t s);
hipError_t launch_trace_rays(const SceneDev& sc, const ddgi_ray* rays, ddgi_hit* hits, uint64_t count, uint32_t mask,
							 bool any_hit, bool cull, hipStream_t s);
// Traversal nodes (kPackedNodeBytes each) of `node_count` wide nodes whose children cover the slot ranges
// `range` (4 per node, first >= second: empty), after re-transforming the triangles of moved instances.
hipError_t launch_make_nodes(const SlotBoxArgs& a, const uint2* range, const uint4* codes, float4* packed,
							 uint32_t node_count, hipStream_t s);
// Copies `count` staged moves (host memory the device can read) to `moves`, and their records to the
// instances' shading records and motions.
hipError_t launch_apply_moves(const InstanceMove* staged, InstanceMove* moves, InstanceDev* inst, float* rel_xf,
							  uint32_t first, uint32_t count, hipStream_t s);
hipError_t launch_gbuffer(const SceneDev& sc, const ddgi_ray* rays, uint64_t count, ddgi_gbuffer_texel* out, hipStream_t s);
hipError_t launch_gather(const GatherArgs& a, hipStream_t s);
hipError_t launch_direct_light(const DirectLightArgs& a, hipStream_t s);
hipError_t launch_reflection_trace(const ReflectionArgs& a, hipStream_t s);
hipError_t launch_reflection_shade(const ReflectionArgs& a, hipStream_t s);
hipError_t launch_init_probes(const SceneDev& sc, const GridConst& g, const float4* dirs512, uint32_t* states,
							  uint32_t* backface_counts, hipStream_t s);
hipError_t launch_iota(uint32_t* indices, uint32_t P, SelectState* st, hipStream_t s);
hipError_t launch_sample(const GridConst& g, const uint32_t* states, const float4* irr, const float2* dep,
						 const float* pos, const float* nrm, const float* tocam, uint64_t count, float* out,
						 hipStream_t s);
// The start of an update or a blend: the frame's directions fib * R, the thread -> ray order (the first n
// entries: rays sorted by the elevation of their world direction, ties by ray index), the weight rows of the
// blend (column k: ray order[k], so that the blend can consume ray records stored in that order) and the list of probes.
enum : uint32_t {
	kListKeep,    // the list stays; sel->count = count
	kListIota,    // 0 .. count - 1
	kListCopy,    // `count` entries of `listed`
	kListSelect,  // the due probes of probe_count by their states, at most `count` (0: no bound)
};
struct FrameBegin {
	Rot R;
	GridConst grid;
	const float4* fib;
	float4* dirs;
	uint16_t* order;         // null: natural order
	uint32_t* counters;      // optional: the shade-list counters, cleared
	float* wt;
	float* inv_sum;
	void* w_hi;
	void* w_lo;
	SelectState* sel;        // optional with kListKeep
	uint32_t* indices;
	const uint32_t* listed;
	const uint32_t* states;
	uint32_t mode;           // blend mode
	uint32_t list;           // kList...
	uint32_t count;
	uint32_t probe_count;
	uint32_t n_pad;          // set by the launcher
	unsigned long long* stamp;  // optional: receives the start (PhaseStamps)
	uint32_t* host_count;    // optional with kListSelect: pinned host memory that receives the count
};
hipError_t launch_frame_begin(FrameBegin a, hipStream_t s);
// Picks the workgroup shape by the number of slots and of the device's compute units (0: unknown); every
// shape gives the same sums (the same MFMAs per output element, in the same order).
hipError_t launch_blend(const BlendArgs& a, uint32_t mode, uint32_t cus, hipStream_t s);

// blend modes
constexpr uint32_t kBlendFP32 = 0;
constexpr uint32_t kBlendBF16 = 1;
constexpr uint32_t kBlendFP16 = 2;


// ---- batched update of many probe volumes (one graph launch per update) ----
constexpr uint32_t kMaxBatchVolumes = 256;
constexpr uint32_t kMaxItemThreads = 256 * 64;  // most traversal threads of a batch's work item
constexpr uint32_t kMfmaProbes = 64;   // probes per MFMA blend workgroup (BF16 / FP16)

// Everything the kernels of one volume read during a batched update.
struct BatchVolume {
	TraceFrameArgs trace;  // trace.dirs == dirs
	BlendArgs blend;       // blend.wt / inv_sum / w_hi16 / w_lo16 == the buffers below
	Rot R;                 // orientation of this update
	const float4* fib;     // fib(i, n)
	float4* dirs;          // world directions, written by k_batch_begin
	uint16_t* perm;        // ray order of the traversal threads, written by k_batch_begin
	float* wt;
	float* inv_sum;
	void* w_hi;
	void* w_lo;
	uint32_t threads;      // traversal threads: slots * rays
	uint32_t n_pad;        // rays rounded up to the MFMA chunk
	SortJob sort;          // ordering of the shade list (trace.shade_keys) before shading
};

struct BatchItem {
	uint32_t volume;
	uint32_t first;  // first traversal thread (trace items), slot (blend items), or the chunk (sort items)
};

struct BatchControl {
	uint32_t next[4];        // work-queue heads: [0] primary traversal
	unsigned long long t0;   // wall clock when the update started on the device
	unsigned long long pad;
	unsigned long long done[kMaxBatchVolumes];  // wall clock when a volume's last blend tile ended
};

struct BatchLaunch {
	const BatchVolume* vols;
	const BatchItem* trace_items;
	const BatchItem* blend_items;
	BatchControl* ctl;
	uint32_t volume_count;
	uint32_t trace_item_count;
	uint32_t trace_item_threads;  // traversal threads per item
	uint32_t blend_item_count;
	uint32_t blend_probes;        // slots per blend item
	uint32_t blend_mode;
	const BatchItem* shade_items;  // one workgroup of kShadeBlock shade-list entries each
	uint32_t shade_item_count;
	const BatchItem* sort_items;   // every kFineChunk entries that the volumes' shade lists can hold
	uint32_t sort_item_count;
};

hipError_t launch_batch_begin(const BatchLaunch& b, hipStream_t s);
hipError_t launch_batch_weights(const BatchLaunch& b, hipStream_t s);
hipError_t launch_batch_trace(const BatchLaunch& b, uint32_t block, uint32_t grid, hipStream_t s);
// Orders the shade list of every volume (BatchVolume::sort) in one set of launches.
hipError_t launch_batch_sort(const BatchLaunch& b, hipStream_t s);
// Shades every volume's ordered shade list: one workgroup per shade item, one thread per entry.
hipError_t launch_batch_shade(const BatchLaunch& b, hipStream_t s);
hipError_t launch_batch_blend(const BatchLaunch& b, hipStream_t s);
// Resident workgroups per CU of the persistent kernels (for sizing their grids).
hipError_t batch_trace_resident(uint32_t block, int* per_cu);

}  // namespace ddgi
