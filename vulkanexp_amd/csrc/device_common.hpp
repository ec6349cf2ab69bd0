// Device-side building blocks shared by the probe kernels (gfx950).
//
// Compiled with -ffp-contract=off in the trace translation unit: the intersection arithmetic
// must be exactly the FP32 operations listed here, in this order, with no fused multiply-add,
// so that hit ids, t and barycentrics are reproducible bit for bit on the host.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.hpp"
#include "packed_node.hpp"

namespace ddgi {

// ---------------------------------------------------------------------------------------------
// Ray precomputation for the watertight test (Woop, Benthin, Wald, JCGT 2(1) 2013): kz is the
// dominant axis of the direction (ties resolved x < y < z as written below), (kx, ky) the other
// two in cyclic order, swapped when d[kz] < 0 to keep the winding; shear constants Sx, Sy, Sz.
struct RayPrep {
	float o[3];
	int kx, ky, kz;
	float sx, sy, sz;
	float inv[3];  // 1/d
	float okx, oky, okz;
};

__device__ __forceinline__ float sel3(float a, float b, float c, int k) { return k == 0 ? a : (k == 1 ? b : c); }

// Workgroups are dealt round-robin to the 8 XCDs of an MI355X (workgroup i -> XCD i % 8), and each
// XCD has its own L2.  Remap so that XCD x processes one contiguous range of logical blocks (a
// slab of neighbouring probes whose rays touch overlapping BVH nodes and atlas tiles).  A
// bijection on [0, nblocks) for any nblocks.
constexpr uint32_t kNumXcd = 8;
__device__ __forceinline__ uint32_t xcd_remap(uint32_t block, uint32_t nblocks) {
	const uint32_t q = nblocks / kNumXcd, r = nblocks % kNumXcd;
	const uint32_t x = block % kNumXcd, k = block / kNumXcd;
	return x * q + min(x, r) + k;
}

// List append from a wavefront: every active lane with `pred` gets a distinct position in the list
// whose length is *counter, with one atomic per wave (issued by the lowest such lane).  Explicit, so
// that it does not depend on the compiler proving `counter` uniform.
__device__ __forceinline__ uint32_t wave_append(uint32_t* counter, bool pred) {
	const uint64_t mask = __ballot(pred);
	const uint32_t lane = __lane_id();
	const uint32_t before = uint32_t(__popcll(mask & ((uint64_t(1) << lane) - 1u)));
	uint32_t base = 0;
	if(mask != 0u) {
		const int leader = __ffsll((unsigned long long)mask) - 1;
		if(int(lane) == leader) base = atomicAdd(counter, uint32_t(__popcll(mask)));
		base = __shfl(base, leader);
	}
	return base + before;
}

__device__ __forceinline__ void ray_prepare(float ox, float oy, float oz, float dx, float dy, float dz, RayPrep& r) {
	const float ax = fabsf(dx), ay = fabsf(dy), az = fabsf(dz);
	const int kz = (ax > ay) ? ((ax > az) ? 0 : 2) : ((ay > az) ? 1 : 2);
	int kx = kz + 1;
	if(kx == 3) kx = 0;
	int ky = kx + 1;
	if(ky == 3) ky = 0;
	const float dkz = sel3(dx, dy, dz, kz);
	if(dkz < 0.0f) {
		const int t = kx;
		kx = ky;
		ky = t;
	}
	r.kx = kx;
	r.ky = ky;
	r.kz = kz;
	r.sx = sel3(dx, dy, dz, kx) / dkz;
	r.sy = sel3(dx, dy, dz, ky) / dkz;
	r.sz = 1.0f / dkz;
	r.o[0] = ox;
	r.o[1] = oy;
	r.o[2] = oz;
	r.inv[0] = 1.0f / dx;
	r.inv[1] = 1.0f / dy;
	r.inv[2] = 1.0f / dz;
	r.okx = sel3(ox, oy, oz, kx);
	r.oky = sel3(ox, oy, oz, ky);
	r.okz = sel3(ox, oy, oz, kz);
}

// Returns true when the triangle is hit with tmin <= t <= tmax; U,V,W,det are the edge functions.
__device__ __forceinline__ bool tri_intersect(const RayPrep& r, float4 a, float4 b, float4 c, float tmin, float tmax,
											  float& t, float& V, float& W, float& det) {
	const float Akx = sel3(a.x, a.y, a.z, r.kx) - r.okx, Aky = sel3(a.x, a.y, a.z, r.ky) - r.oky,
				Akz = sel3(a.x, a.y, a.z, r.kz) - r.okz;
	const float Bkx = sel3(b.x, b.y, b.z, r.kx) - r.okx, Bky = sel3(b.x, b.y, b.z, r.ky) - r.oky,
				Bkz = sel3(b.x, b.y, b.z, r.kz) - r.okz;
	const float Ckx = sel3(c.x, c.y, c.z, r.kx) - r.okx, Cky = sel3(c.x, c.y, c.z, r.ky) - r.oky,
				Ckz = sel3(c.x, c.y, c.z, r.kz) - r.okz;
	const float Ax = Akx - r.sx * Akz, Ay = Aky - r.sy * Akz;
	const float Bx = Bkx - r.sx * Bkz, By = Bky - r.sy * Bkz;
	const float Cx = Ckx - r.sx * Ckz, Cy = Cky - r.sy * Ckz;
	float U = Cx * By - Cy * Bx;
	V = Ax * Cy - Ay * Cx;
	W = Bx * Ay - By * Ax;
	if(U == 0.0f || V == 0.0f || W == 0.0f) {
		U = float(double(Cx) * double(By) - double(Cy) * double(Bx));
		V = float(double(Ax) * double(Cy) - double(Ay) * double(Cx));
		W = float(double(Bx) * double(Ay) - double(By) * double(Ax));
	}
	if((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
	det = U + V + W;
	if(det == 0.0f) return false;
	const float Az = r.sz * Akz, Bz = r.sz * Bkz, Cz = r.sz * Ckz;
	const float T = U * Az + V * Bz + W * Cz;
	t = T / det;
	return t >= tmin && t <= tmax;
}

struct HitResult {
	float t;
	uint32_t slot;  // triangle position in the BVH triangle array, 0xFFFFFFFF = miss
	uint32_t gid;   // global triangle id (ties go to the lower one)
	uint32_t meta;  // mask | flip_facing << 8 of the hit triangle
	float V, W, det;
};

// Closest-hit (ANY = false; ties -> lowest global id) or any-hit traversal of the BVH.
//
// Nodes are 4-wide, in the packed form of k_make_nodes: five 16-byte loads test four child boxes.  A
// wavefront runs until its longest ray ends with about a third of its lanes active, so what bounds the
// traversal is what a visit costs per wavefront: vector instructions (79 % of the SIMDs' issue cycles
// with FP32 boxes) and vector loads, whose data return costs about 22 cycles per load of the CU however
// few lanes are active (75 % of its cycles with the seven loads of an FP32 node).  Cutting one of them
// alone moved nothing; the packed node cuts both: a plane's distance is one v_fma_mix_f32 on the FP16
// plane (distance = q * (scale / d) + (origin - o) / d), and two loads fewer are returned.  The near and
// far plane rows are chosen by the sign of 1/d (which is the smaller distance, since the distance is
// monotonic in the plane), so no min / max pair is needed, and the far end is widened by a few ulps
// (robust traversal, Ize 2013).  A plane's two terms must be finite for that: the reciprocals of zero and
// very small direction components are bounded per ray (slab_reciprocals), which the triangle tests are not.
//
// For the closest hit the children the ray enters are sorted by entry distance (a five-comparator network on registers;
// sorting only the nearest, or leaving the middle pair, visits more and took 0.64 / 0.66 ms against
// 0.58 in the large workload's primary pass); the nearest is visited next and the others are pushed
// farthest first, so the next pop is the nearest remaining.  The result does not depend on the visiting
// order: closest hit is the minimum of (t, global id) over every triangle the conservative box tests
// let through.
//
// Stack: entries 0 .. STACK - 1 live in LDS laid out [entry][thread] (conflict-free; `stack` points at
// this thread's column, STRIDE is the block size), later ones in a private array.  Entry 0 is a
// sentinel, so that a pop needs no test for an empty stack; with three entries free in the LDS part
// the three pushes of a visit are unconditional stores with a conditional advance.  At most kWide - 1
// entries per level of the wide tree are pending.  12 LDS entries measured fastest (8 / 12 / 16 / 22:
// 0.605 / 0.574 / 0.580 / 0.629 ms): more LDS per workgroup keeps fewer of them on a CU.
//
// Large workload (4.2 M rays), primary pass: FP32 nodes with a ring stack 0.674 ms; packed nodes and
// this stack 0.575 ms at 7 waves per SIMD, 0.555 ms at 8, which its 64 registers now allow.
//
// Leaves are tested two triangles at a time, each triangle's 48 bytes loaded in one go, so that
// two loads are in flight and the mask word costs no extra round trip.
//
// With COUNT, n_nodes / n_tris receive the number of node (kPackedNodeBytes) and 48-byte triangle
// fetches (the algorithmic bytes of the traversal).
constexpr int kLdsStack = 12;  // LDS entries per thread
// entries beyond them, in a private array; one entry is the bottom's sentinel
constexpr int kStackMax = (int(kWide) - 1) * int(kMaxWideDepth) + 1;

// CULL: back-facing triangles are ignored (rasterizer back-face culling).
template <bool ANY, bool CULL>
__device__ __forceinline__ bool test_triangle(const RayPrep& r, float tmin, uint32_t mask, uint32_t slot, float4 ta,
											  float4 tb, float4 tc, HitResult& best) {
	if((__float_as_uint(tc.w) & mask) == 0u) return false;
	float t, V, W, det;
	if(!tri_intersect(r, ta, tb, tc, tmin, best.t, t, V, W, det)) return false;
	if(CULL && ((det < 0.0f) != ((__float_as_uint(tc.w) & 0x100u) != 0u))) return false;
	const uint32_t gid = __float_as_uint(ta.w);
	if(best.slot != 0xFFFFFFFFu && !(t < best.t || gid < best.gid)) return false;
	best.t = t;
	best.slot = slot;
	best.gid = gid;
	best.meta = __float_as_uint(tc.w);
	best.V = V;
	best.W = W;
	best.det = det;
	return true;
}

template <bool ANY, int STACK, int STRIDE, bool COUNT = false, bool CULL = false>
__device__ __forceinline__ HitResult traverse(const float4* __restrict__ nodes, const float4* __restrict__ tris,
											  const RayPrep& r, float tmin, float tmax, uint32_t mask,
											  uint32_t* stack, uint32_t& n_nodes_out, uint32_t& n_tris_out) {
	HitResult best;
	best.t = tmax;
	best.slot = 0xFFFFFFFFu;
	best.gid = 0xFFFFFFFFu;
	best.meta = 0u;
	best.V = best.W = best.det = 0.0f;
	uint32_t spill[kStackMax - STACK];
	constexpr uint32_t kNone = 0xFFFFFFFFu;  // no node (the stack's bottom) / no postponed leaf
	stack[0] = kNone;
	int sp = 1;  // stack entries
#define DDGI_STACK_POP(v)                                                        \
	{                                                                            \
		--sp;                                                                    \
		if(sp < STACK) v = stack[sp * STRIDE];                                   \
		else v = spill[sp - STACK];                                              \
	}
// order (key, code) pairs i, j by key
#define DDGI_CSWAP(i, j)                               \
	{                                                  \
		const bool sw_ = key[j] < key[i];              \
		const float ki_ = key[i], kj_ = key[j];        \
		const uint32_t ci_ = code[i], cj_ = code[j];   \
		key[i] = sw_ ? kj_ : ki_;                      \
		key[j] = sw_ ? ki_ : kj_;                      \
		code[i] = sw_ ? cj_ : ci_;                     \
		code[j] = sw_ ? ci_ : cj_;                     \
	}
	// Leaves are postponed (Aila and Laine's speculative traversal): a lane that reaches a leaf keeps
	// it in `leaf` and goes on descending from its stack until at least half of the active lanes of
	// the wavefront hold a leaf (or it has run out of nodes); the wavefront then tests leaves
	// together.  Waiting for every lane idles the lanes that hold one; testing at once idles the
	// others; half measured fastest (three, five and six eighths: 0.587 / 0.590 / 0.597 ms against
	// 0.580).
	uint32_t node = 0;  // root (always an inner node)
	uint32_t leaf = kNone;
	uint32_t n_nodes = 0, n_tris = 0;
	const float kInf = __int_as_float(0x7f800000);
	const float4 root = nodes[0];
	const float header[4] = {root.x, root.y, root.z, root.w};
	float inv[3] = {r.inv[0], r.inv[1], r.inv[2]};
	slab_reciprocals(r.o, header, inv);
	const bool neg[3] = {(__float_as_uint(inv[0]) >> 31) != 0u, (__float_as_uint(inv[1]) >> 31) != 0u,
						 (__float_as_uint(inv[2]) >> 31) != 0u};
	const char* __restrict__ node_bytes = reinterpret_cast<const char*>(nodes);
	typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
	for(;;) {
		// descend through inner nodes
		while(!(node & kLeafFlag)) {
			// 32-bit offsets from the array's base (the node array stays far below 4 GiB)
			const float4* nd = reinterpret_cast<const float4*>(node_bytes + node * kPackedNodeBytes);
			const float4 h = nd[0], px = nd[1], py = nd[2], pz = nd[3], cd = nd[4];
			++n_nodes;
			uint32_t code[4] = {__float_as_uint(cd.x), __float_as_uint(cd.y), __float_as_uint(cd.z), __float_as_uint(cd.w)};
			float tn[4], tf[4];
#pragma unroll
			for(int ax = 0; ax < 3; ++ax) {
				const float4 pl = ax == 0 ? px : (ax == 1 ? py : pz);
				const float org = ax == 0 ? h.x : (ax == 1 ? h.y : h.z);
				const float A = h.w * inv[ax], B = (org - r.o[ax]) * inv[ax];
				const uint32_t n01 = __float_as_uint(neg[ax] ? pl.z : pl.x), n23 = __float_as_uint(neg[ax] ? pl.w : pl.y);
				const uint32_t f01 = __float_as_uint(neg[ax] ? pl.x : pl.z), f23 = __float_as_uint(neg[ax] ? pl.y : pl.w);
				const half2_t qn[2] = {__builtin_bit_cast(half2_t, n01), __builtin_bit_cast(half2_t, n23)};
				const half2_t qf[2] = {__builtin_bit_cast(half2_t, f01), __builtin_bit_cast(half2_t, f23)};
#pragma unroll
				for(int k = 0; k < 4; ++k) {
					const float en = __builtin_fmaf(float(qn[k >> 1][k & 1]), A, B), ef = __builtin_fmaf(float(qf[k >> 1][k & 1]), A, B);
					tn[k] = ax == 0 ? en : fmaxf(tn[k], en);
					tf[k] = ax == 0 ? ef : fminf(tf[k], ef);
				}
			}
			// entry distance of each child the ray enters, infinity for the others
			float key[4];
#pragma unroll
			for(int k = 0; k < 4; ++k) {
				const float n = fmaxf(tn[k], tmin), f = fminf(tf[k], best.t);
				key[k] = n <= f * 1.000001f ? n : kInf;
			}
			if constexpr(ANY) {
				// any hit ends the ray, and finding it nearest first saves 1.5 % of the visits for 25 of
				// their 130 vector instructions: the first entered child goes on (0.5 M scattered rays
				// 125 -> 112 us; shadow pass of a full-HD view 134 -> 129 us).  The nearest first without
				// sorting the others: 1 M rays from inside a scene of 256 instances 166 us against 152, of a
				// camera in one of 24 78 against 66.  It is better where rays meet a closed room from outside,
				// whose walls the stored order tries late: 1 M rays 51 us against 67 (58 with FP32 boxes and
				// sorted), 40,000 rays 15 against 21 (14).
#pragma unroll
				for(int k = 1; k < 4; ++k) {
					const bool take = key[0] == kInf;
					key[0] = take ? key[k] : key[0];
					code[0] = take ? code[k] : code[0];
					key[k] = take ? kInf : key[k];
				}
			} else {  // sorted by key, the entered children come first
				DDGI_CSWAP(0, 1)
				DDGI_CSWAP(2, 3)
				DDGI_CSWAP(0, 2)
				DDGI_CSWAP(1, 3)
				DDGI_CSWAP(1, 2)
			}
			// push the others, farthest first; within the LDS part every slot is written and the stack
			// grows by those that were entered
			if(sp <= STACK - 3) {
#pragma unroll
				for(int k = 3; k >= 1; --k) {
					stack[sp * STRIDE] = code[k];
					sp += key[k] != kInf ? 1 : 0;
				}
			} else {
#pragma unroll
				for(int k = 3; k >= 1; --k) {
					if(key[k] == kInf) continue;
					if(sp < STACK) stack[sp * STRIDE] = code[k];
					else spill[sp - STACK] = code[k];
					++sp;
				}
			}
			node = code[0];
			if(key[0] == kInf) DDGI_STACK_POP(node)
			if(leaf == kNone && node != kNone && (node & kLeafFlag)) {  // postpone the leaf
				leaf = node;
				DDGI_STACK_POP(node)
			}
			// at least half of the active lanes hold a leaf
			if(uint32_t(__popcll(__ballot(leaf != kNone))) * 2u >= uint32_t(__popcll(__ballot(true)))) break;
		}
		// leaves: the postponed one, then any leaves next on the stack
		while(leaf != kNone) {
			const uint32_t first = (leaf & ~kLeafFlag) >> 3, cnt = (leaf & 7u) + 1u;
			for(uint32_t k = 0; k < cnt; k += 2) {
				const float4* tr = tris + size_t(first + k) * 3;
				const float4 ta = tr[0], tb = tr[1], tc = tr[2];
				const bool two = k + 1 < cnt;
				float4 ua = ta, ub = tb, uc = tc;
				if(two) {
					ua = tr[3];
					ub = tr[4];
					uc = tr[5];
				}
				n_tris += two ? 2u : 1u;
				// in index order, so that equal-t hits resolve exactly as a sequential scan would
				if(test_triangle<ANY, CULL>(r, tmin, mask, first + k, ta, tb, tc, best) && ANY) goto done;
				if(two && test_triangle<ANY, CULL>(r, tmin, mask, first + k + 1, ua, ub, uc, best) && ANY) goto done;
			}
			leaf = kNone;
			if(node != kNone && (node & kLeafFlag)) {
				leaf = node;
				DDGI_STACK_POP(node)
			}
		}
		if(node == kNone) break;
	}
done:
#undef DDGI_STACK_POP
#undef DDGI_CSWAP
	if(COUNT) {
		n_nodes_out = n_nodes;
		n_tris_out = n_tris;
	}
	return best;
}

// ---------------------------------------------------------------------------------------------
// Octahedral maps
__device__ __forceinline__ float gsign(float v) { return v > 0.0f ? 1.0f : (v < 0.0f ? -1.0f : 0.0f); }

// Direction of blend texel t: octDecode(specializedNormalizeLocalTexelCoord(c)) in FP32
// (irradiance.glsl:107-112, probesUpdate.glsl:33-42, with the reference's constants 0.33333 and
// 0.142857); t < 36: irradiance texel (x, y) = (t % 6, t / 6), else depth texel t - 36 of 14x14.
__device__ __forceinline__ void texel_direction(uint32_t t, float& x, float& y, float& z) {
	float u, v;
	if(t < kIrrTexels) {
		const int cx = int(t % 6u), cy = int(t / 6u);
		u = 0.33333f * (float(cx) - 2.5f);
		v = 0.33333f * (float(cy) - 2.5f);
	} else {
		const uint32_t d = t - kIrrTexels;
		const int cx = int(d % 14u), cy = int(d / 14u);
		u = 0.142857f * (float(cx) - 6.5f);
		v = 0.142857f * (float(cy) - 6.5f);
	}
	x = u;
	y = v;
	z = 1.0f - fabsf(u) - fabsf(v);
	if(z < 0.0f) {
		const float nx = (1.0f - fabsf(y)) * (x >= 0.0f ? 1.0f : -1.0f);
		const float ny = (1.0f - fabsf(x)) * (y >= 0.0f ? 1.0f : -1.0f);
		x = nx;
		y = ny;
	}
	const float l = sqrtf(x * x + y * y + z * z);
	x /= l;
	y /= l;
	z /= l;
}

// ---------------------------------------------------------------------------------------------
// Bilinear fetch inside one probe tile (texel coords 1 + (res-2)*uv, centres at k + 0.5): the first of the
// four texels (the others are the next ones in x, y and both) and the fractions.  u and v are octahedral
// coordinates in [0, 1], so the first texel lies in [0, RES - 2] on both axes; the minimum keeps whatever
// a NaN converts to inside the tile.
template <int RES>
__device__ __forceinline__ uint32_t tile_coords(float u, float v, float& wx, float& wy) {
	const float sx = 1.0f + float(RES - 2) * u - 0.5f;
	const float sy = 1.0f + float(RES - 2) * v - 0.5f;
	const float fx = floorf(sx), fy = floorf(sy);
	wx = sx - fx;
	wy = sy - fy;
	return min(uint32_t(int(fy) * RES + int(fx)), uint32_t((RES - 2) * RES + RES - 2));
}

// Correctly rounded division and square root for the shading's ranges.  The compiler's divisions take
// 12 instructions each (scaling for extreme exponents, a reciprocal with one Newton step, two corrections
// of the quotient); these are the same steps without the scaling, and the divisions by one denominator
// share its reciprocal.  The same bits as `/` and sqrtf() while no intermediate leaves the normal range
// (magnitudes between about 1e-29 and 1e29); zeros, infinities and NaNs come out as there.
struct Rcp {
	float d, r;
};
__device__ __forceinline__ Rcp rcp_rn(float d) {
	const float r = __builtin_amdgcn_rcpf(d);
	return {d, __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r)};
}
__device__ __forceinline__ float div_rn(float n, Rcp c) {
	float q = n * c.r;
	q = __builtin_fmaf(__builtin_fmaf(-c.d, q, n), c.r, q);
	q = __builtin_fmaf(__builtin_fmaf(-c.d, q, n), c.r, q);
	return __builtin_amdgcn_div_fixupf(q, c.d, n);
}
__device__ __forceinline__ float div_rn(float n, float d) { return div_rn(n, rcp_rn(d)); }
// The hardware's square root is within one ulp: the neighbour below when its product with the root is not
// below x, the neighbour above when that product still is.
__device__ __forceinline__ float sqrt_rn(float x) {
	const float s = __builtin_amdgcn_sqrtf(x);
	const float dn = __uint_as_float(__float_as_uint(s) - 1u), up = __uint_as_float(__float_as_uint(s) + 1u);
	float r = __builtin_fmaf(-dn, s, x) <= 0.0f ? dn : s;
	r = __builtin_fmaf(-up, s, x) > 0.0f ? up : r;
	return r;
}

struct Vec3 {
	float x, y, z;
};
__device__ __forceinline__ Vec3 v3(float x, float y, float z) { return {x, y, z}; }
__device__ __forceinline__ Vec3 operator+(Vec3 a, Vec3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ Vec3 operator-(Vec3 a, Vec3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ Vec3 operator*(Vec3 a, float s) { return {a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ Vec3 operator*(Vec3 a, Vec3 b) { return {a.x * b.x, a.y * b.y, a.z * b.z}; }
__device__ __forceinline__ float dot3(Vec3 a, Vec3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ Vec3 normalize3(Vec3 a) {
	const float l = sqrtf(dot3(a, a));
	return {a.x / l, a.y / l, a.z / l};
}

// normalize3 with the shared division (unit-scale and scene-scale vectors).
__device__ __forceinline__ Vec3 normalize_rn(Vec3 a) {
	const Rcp l = rcp_rn(sqrt_rn(dot3(a, a)));
	return {div_rn(a.x, l), div_rn(a.y, l), div_rn(a.z, l)};
}

__device__ __forceinline__ Vec3 cross3(Vec3 a, Vec3 b) {
	return {a.y * b.z - a.z * b.y, a.z * b.x - a.x * b.z, a.x * b.y - a.y * b.x};
}

// sin and cos of an FP32 angle by a fixed sequence of FP32 operations, so that a host replica gives
// the same bits: Cody-Waite reduction by the nearest multiple of pi/2 (pi/2 split into a float
// and its remainder), then the Taylor series of sin (to r^11) and cos (to r^12) on |r| <= pi/4,
// whose truncation error is below 1e-10, and the quadrant's sign/swap.
__device__ __forceinline__ void sincos_series(float x, float& s, float& c) {
	const float q = rintf(x * 0.636619772f);
	const float r = (x - q * 1.57079637f) - q * -4.37113883e-08f;
	const float r2 = r * r;
	const float sr = r + r * r2 * (-1.0f / 6.0f + r2 * (1.0f / 120.0f + r2 * (-1.0f / 5040.0f + r2 * (1.0f / 362880.0f +
																									r2 * (-1.0f / 39916800.0f)))));
	const float cr = 1.0f + r2 * (-0.5f + r2 * (1.0f / 24.0f + r2 * (-1.0f / 720.0f + r2 * (1.0f / 40320.0f +
															r2 * (-1.0f / 3628800.0f + r2 * (1.0f / 479001600.0f))))));
	switch(int(q) & 3) {
		case 0: s = sr; c = cr; break;
		case 1: s = cr; c = -sr; break;
		case 2: s = -sr; c = -cr; break;
		default: s = -cr; c = sr; break;
	}
}

// rotateAxis (common.glsl:6-8): mix(dot(axis, p) axis, p, cos a) + cross(axis, p) sin a.
__device__ __forceinline__ Vec3 rotate_axis(Vec3 p, Vec3 axis, float angle) {
	float s, c;
	sincos_series(angle, s, c);
	const Vec3 along = axis * dot3(axis, p);
	return (along * (1.0f - c) + p * c) + cross3(axis, p) * s;
}

// ---- atmospheric sky (src/shaders/sky.glsl:60-127, after O'Neil, GPU Gems 2 ch. 16) ----
// Planet of radius 100 km whose surface lies at y = -100, atmosphere 2.5 km thick, scale height a
// quarter of it; Rayleigh (Kr 0.0025, 1/lambda^4 for lambda = 650/570/475 nm) and Mie (Km 0.001,
// g = -0.99) single scattering integrated with 64 midpoint samples.  The reference's own choices
// are kept: the exit distance of a ray leaving the atmosphere adds the closest-approach offset
// where it should subtract it (and the reverse), a sample whose attenuation overflows is skipped
// without advancing the sample point, and a colour with an infinite channel gives black.
// Sample points are formed as position + (k + 1/2) * step instead of by repeated addition (the
// same point, without the FP32 drift of 64 additions at 1e5 m).  Exponentials use the hardware
// exp2 (__expf: relative error about 6e-8 |x| for the arguments here, |x| < 90).
namespace sky {
constexpr float kInner = 100000.0f;
constexpr float kOuter = 102500.0f;
constexpr float kScale = 1.0f / (kOuter - kInner);
constexpr float kScaleDepth = 0.25f;
constexpr float kPi = 3.1415926538f;  // common.glsl:4
constexpr float kKr = 0.0025f, kKm = 0.0010f, kG = -0.990f;
constexpr int kSamples = 64;

__device__ __forceinline__ float scale_fn(float c) {
	const float x = 1.0f - c;
	return kScaleDepth * __expf(fmaf(x, fmaf(x, fmaf(x, fmaf(x, 5.25f, -6.80f), 3.83f), 0.459f), -0.00287f));
}
// First crossing ahead of the sphere (radius r, centred at the origin) by a ray from outside, -1 if none.
__device__ __forceinline__ float enter_sphere(Vec3 o, Vec3 d, float r) {
	const float a = dot3(d, d), b = dot3(d, o), c = dot3(o, o) - r * r;
	const float g = b * b - a * c;
	if(g > 0.0f) {
		const float dis = (-sqrtf(g) - b) / a;
		if(dis > 0.0f) return dis;
	}
	return -1.0f;
}
// Exit distance from the sphere of a ray inside it, as sky.glsl:33-42 computes it.
__device__ __forceinline__ float leave_sphere(Vec3 o, Vec3 d, float r) {
	const float along = -dot3(o, d);
	const Vec3 pc = o + d * along;
	const float lpc = sqrtf(dot3(pc, pc));
	const float dist = sqrtf(r * r - lpc * lpc);
	const Vec3 off = pc - o;
	const float loff = sqrtf(dot3(off, off));
	return along > 0.0f ? dist - loff : dist + loff;
}
}  // namespace sky

__device__ __forceinline__ Vec3 sky_atmosphere(Vec3 origin, Vec3 dir, Vec3 sun_dir, Vec3 sun_color, float brightness,
											   bool show_sun) {
	using namespace sky;
	sun_color = sun_color * brightness;
	Vec3 pos = v3(origin.x, origin.y + (kInner + 100.0f), origin.z);
	float height = sqrtf(dot3(pos, pos));
	const Vec3 L = normalize3(sun_dir);
	if(fabsf(height - kInner) < 1e-3f) {
		pos = pos + normalize3(pos) * 1e-2f;
		height = sqrtf(dot3(pos, pos));
	}
	const Vec3 zero = v3(0.0f, 0.0f, 0.0f);
	if(height < kOuter) {
		if(height > kInner) {
			const float pd = enter_sphere(pos, dir, kInner);
			if(pd >= 0.0f) {
				const float c = fmaxf(0.1f, dot3(L, normalize3(pos + dir * pd)));
				return v3(c * 0.05f, c * 0.05f, c * 0.05f);
			}
		} else {
			return zero;
		}
		const float ray_depth = leave_sphere(pos, dir, kOuter);
		if(isinf(ray_depth) || isnan(ray_depth)) return zero;
		const float start_depth = __expf(kScale / kScaleDepth * (kInner - height));
		const float start_offset = start_depth * scale_fn(dot3(dir, pos) / height);
		const float seg = ray_depth / float(kSamples);
		const float scaled = seg * kScale;
		const Vec3 step = dir * seg;
		// 1 / lambda^4 per channel, times 4 pi Kr, plus 4 pi Km
		const Vec3 inv_wl = v3(1.0f / (0.650f * 0.650f * 0.650f * 0.650f), 1.0f / (0.570f * 0.570f * 0.570f * 0.570f),
							   1.0f / (0.475f * 0.475f * 0.475f * 0.475f));
		const Vec3 ext = v3(inv_wl.x * (kKr * 4.0f * kPi) + kKm * 4.0f * kPi, inv_wl.y * (kKr * 4.0f * kPi) + kKm * 4.0f * kPi,
							inv_wl.z * (kKr * 4.0f * kPi) + kKm * 4.0f * kPi);
		Vec3 color = zero;
		int k = 0;  // samples advanced so far
		for(int i = 0; i < kSamples; ++i) {
			const Vec3 sp = pos + step * (float(k) + 0.5f);
			// one reciprocal square root instead of a square root and two divisions (the loop is
			// VALU-bound; the sky's accuracy is set by the hardware exponentials, not by these)
			const float h2 = dot3(sp, sp), inv_h = rsqrtf(h2), h = h2 * inv_h;
			const float depth = __expf(kScale / kScaleDepth * (kInner - h));
			const float scatter = start_offset + depth * (scale_fn(dot3(L, sp) * inv_h) - scale_fn(dot3(dir, sp) * inv_h));
			const Vec3 att = v3(__expf(-scatter * ext.x), __expf(-scatter * ext.y), __expf(-scatter * ext.z));
			if(!isfinite(att.x) || !isfinite(att.y) || !isfinite(att.z)) continue;
			color = color + att * (depth * scaled);
			++k;
		}
		const Vec3 secondary = color * sun_color * kKm;
		color = color * inv_wl * sun_color * kKr;
		if(show_sun) {
			const float mc = -dot3(L, dir);
			const float m = fmaxf(1e-3f, 1.0f + kG * kG - 2.0f * kG * mc);
			const float phase = 1.5f * ((1.0f - kG * kG) / (2.0f + kG * kG)) * (1.0f + mc * mc) / (m * sqrtf(m));
			color = color + secondary * phase;
		}
		if(!isinf(color.x) && !isinf(color.y) && !isinf(color.z)) return color;
	} else {
		const float d = enter_sphere(pos, dir, kOuter);
		if(d > 0.0f) {
			const float c = dot3(L, normalize3(pos + dir * d)) * 0.5f;
			return v3(c * 0.5294117647f, c * 0.80784313725f, c * 0.92156862745f);
		}
	}
	return zero;
}

// spherePointToOctohedralUV (src/shaders/irradiance.glsl:119-138), GLSL sign() semantics.  The third
// component's quotient is only compared with 0, where the component itself serves.
__device__ __forceinline__ void oct_uv(float dx, float dy, float dz, float& u, float& v) {
	const float sx = gsign(dx), sy = gsign(dy), sz = gsign(dz);
	const Rcp sum = rcp_rn(dx * sx + dy * sy + dz * sz);
	float ox = div_rn(dx, sum), oy = div_rn(dy, sum);
	if(dz < 0.0f) {
		const float ax = fabsf(ox), ay = fabsf(oy);
		ox = sx * (1.0f - ay);
		oy = sy * (1.0f - ax);
	}
	u = ox * 0.5f + 0.5f;
	v = oy * 0.5f + 0.5f;
}

// The cage of a sampleProbes call (irradiance.glsl:145-163): the probe at its lower corner, the position's
// fractions inside it, and what the eight probes share.
struct Cage {
	int f[3];
	float alpha[3];
};

__device__ __forceinline__ bool make_cage(const GridConst& g, Vec3 position, Cage& c) {
	const float p[3] = {position.x, position.y, position.z};
	float gc[3];
#pragma unroll
	for(int a = 0; a < 3; ++a) gc[a] = (p[a] - g.emin[a]) / fabsf(g.cell[a]);
	if(gc[0] < 0.0f || gc[1] < 0.0f || gc[2] < 0.0f) return false;
#pragma unroll
	for(int a = 0; a < 3; ++a) {
		c.f[a] = int(gc[a]);
		const float p0 = float(c.f[a]) * g.cell[a] + g.emin[a];
		c.alpha[a] = fminf(fmaxf((p[a] - p0) / fabsf(g.cell[a]), 0.0f), 1.0f);
	}
	return true;
}

// Cage probe i: its linear index, position, direction from the shaded point and trilinear factor; false
// when it is off-grid or disabled.
__device__ __forceinline__ bool cage_corner(const GridConst& g, const uint32_t* __restrict__ states, const Cage& c,
											Vec3 position, int i, uint32_t& lin, Vec3& pp, Vec3& dtp, float& trw) {
	const int o0 = i & 1, o1 = (i >> 1) & 1, o2 = (i >> 2) & 1;
	// unsigned: a position 2^31 cells away has the largest int as its cell, whose upper corner would wrap to a
	// negative one and pass for on-grid
	const uint32_t p0i = uint32_t(c.f[0]) + o0, p1i = uint32_t(c.f[1]) + o1, p2i = uint32_t(c.f[2]) + o2;
	if(p0i >= uint32_t(g.res[0]) || p1i >= uint32_t(g.res[1]) || p2i >= uint32_t(g.res[2])) return false;
	lin = p0i + uint32_t(g.res[0]) * (p1i + uint32_t(g.res[1]) * p2i);
	if(states[lin] == 0u) return false;
	pp = v3(float(p0i) * g.cell[0] + g.emin[0], float(p1i) * g.cell[1] + g.emin[1], float(p2i) * g.cell[2] + g.emin[2]);
	dtp = normalize_rn(pp - position);
	const float trx = o0 ? c.alpha[0] : 1.0f - c.alpha[0];
	const float try_ = o1 ? c.alpha[1] : 1.0f - c.alpha[1];
	const float trz = o2 ? c.alpha[2] : 1.0f - c.alpha[2];
	trw = trx * try_ * trz + 0.001f;
	return true;
}

// Weight (visibility x backface x trilinear) and fallback weight of a cage probe for a normal, whose
// biased position is `biased` (irradiance.glsl:164-206).
__device__ __forceinline__ void cage_weight(const float2* __restrict__ dep, uint32_t lin, Vec3 pp, Vec3 dtp, float trw,
											Vec3 normal, Vec3 biased, float& weight, float& fbw) {
	const Vec3 bdir = pp - biased;
	const float bdist = sqrt_rn(dot3(bdir, bdir));
	const Rcp rb = rcp_rn(bdist);
	const Vec3 nb = v3(div_rn(bdir.x, rb), div_rn(bdir.y, rb), div_rn(bdir.z, rb));
	float du, dv, dwx, dwy;
	oct_uv(-nb.x, -nb.y, -nb.z, du, dv);
	const float bfw = fmaxf(0.0001f, (dot3(dtp, normal) + 1.0f) * 0.5f);
	weight = bfw * bfw + 0.2f;
	fbw = weight;
	// Chebyshev visibility from the bilinear depth moments; two texels of a row in one 16-byte load
	const float2* dt = dep + size_t(lin) * 256 + tile_coords<16>(du, dv, dwx, dwy);
	typedef float pair_t __attribute__((ext_vector_type(4), aligned(8)));
	const pair_t m0 = *reinterpret_cast<const pair_t*>(dt), m1 = *reinterpret_cast<const pair_t*>(dt + 16);
	const float mean = (m0[0] * (1.0f - dwx) + m0[2] * dwx) * (1.0f - dwy) + (m1[0] * (1.0f - dwx) + m1[2] * dwx) * dwy;
	const float m2 = (m0[1] * (1.0f - dwx) + m0[3] * dwx) * (1.0f - dwy) + (m1[1] * (1.0f - dwx) + m1[3] * dwx) * dwy;
	const float variance = fabsf(mean * mean - m2);
	const float dm = fmaxf(bdist - mean, 0.0001f);
	float cheb = div_rn(variance, variance + dm * dm);
	cheb = fmaxf(cheb * cheb * cheb, 0.0f);
	weight *= (bdist <= mean) ? 1.0f : cheb;
	weight = fmaxf(0.000001f, weight);
	if(weight < 0.2f) weight *= weight * weight * (1.0f / (0.2f * 0.2f));
	weight *= trw;
	fbw *= trw;
}

// What probe `lin` of a cage adds for one normal: its irradiance (square root space) times the weight, the
// weight, and the same with the fallback weight.
__device__ __forceinline__ void sample_corner(const float4* __restrict__ irr, const float2* __restrict__ dep, uint32_t lin,
											  Vec3 pp, Vec3 dtp, float trw, Vec3 normal, Vec3 biased, uint32_t tap, float wx,
											  float wy, float (&v)[8]) {
	float weight, fbw;
	cage_weight(dep, lin, pp, dtp, trw, normal, biased, weight, fbw);
	const float4* ct = irr + size_t(lin) * 64 + tap;
	const float4 c00 = ct[0], c10 = ct[1], c01 = ct[8], c11 = ct[9];
	const float cr = (c00.x * (1.0f - wx) + c10.x * wx) * (1.0f - wy) + (c01.x * (1.0f - wx) + c11.x * wx) * wy;
	const float cg = (c00.y * (1.0f - wx) + c10.y * wx) * (1.0f - wy) + (c01.y * (1.0f - wx) + c11.y * wx) * wy;
	const float cb = (c00.z * (1.0f - wx) + c10.z * wx) * (1.0f - wy) + (c01.z * (1.0f - wx) + c11.z * wx) * wy;
	Vec3 col;
	if(fminf(fminf(cr, cg), cb) >= 1.26217745e-29f) col = v3(sqrt_rn(cr), sqrt_rn(cg), sqrt_rn(cb));
	else col = v3(sqrtf(cr), sqrtf(cg), sqrtf(cb));  // 0, or too small for sqrt_rn's residuals (2^-96)
	v[0] = col.x * weight;
	v[1] = col.y * weight;
	v[2] = col.z * weight;
	v[3] = weight;
	v[4] = col.x * fbw;
	v[5] = col.y * fbw;
	v[6] = col.z * fbw;
	v[7] = fbw;
}

// sampleProbes (src/shaders/irradiance.glsl:145-237) on the tiled FP32 atlases, at one position for N
// normals, which share each probe's index, state, direction and trilinear factor.  Bound by vector
// instructions: 395 per probe and normal as separate calls with the compiler's divisions and square roots
// (63 % of the probe shading's), 240 so; the results are the same bits.  Large workload's shading 0.403 ->
// 0.374 ms, full-HD reflection shading 215 -> 190 us, final gather 175 -> 146 us.
template <int N>
__device__ __forceinline__ void sample_probes(const GridConst& g, const uint32_t* __restrict__ states,
											  const float4* __restrict__ irr, const float2* __restrict__ dep, Vec3 position,
											  const Vec3 (&normal)[N], Vec3 to_camera, Vec3 (&out)[N]) {
	Cage cage;
	if(!make_cage(g, position, cage)) {
#pragma unroll
		for(int k = 0; k < N; ++k) out[k] = v3(0.0f, 0.0f, 0.0f);
		return;
	}
	Vec3 biased[N], fin[N], fb[N];
	float tw[N], tfb[N], cwx[N], cwy[N];
	uint32_t tap[N];
#pragma unroll
	for(int k = 0; k < N; ++k) {
		biased[k] = position + (normal[k] + to_camera) * g.shadow_bias;
		float cu, cv;
		oct_uv(normal[k].x, normal[k].y, normal[k].z, cu, cv);
		tap[k] = tile_coords<8>(cu, cv, cwx[k], cwy[k]);
		fin[k] = fb[k] = v3(0.0f, 0.0f, 0.0f);
		tw[k] = tfb[k] = 0.0f;
	}
	for(int i = 0; i < 8; ++i) {
		uint32_t lin;
		Vec3 pp, dtp;
		float trw;
		if(!cage_corner(g, states, cage, position, i, lin, pp, dtp, trw)) continue;
#pragma unroll
		for(int k = 0; k < N; ++k) {
			float v[8];
			sample_corner(irr, dep, lin, pp, dtp, trw, normal[k], biased[k], tap[k], cwx[k], cwy[k], v);
			fin[k] = fin[k] + v3(v[0], v[1], v[2]);
			tw[k] += v[3];
			fb[k] = fb[k] + v3(v[4], v[5], v[6]);
			tfb[k] += v[7];
		}
	}
#pragma unroll
	for(int k = 0; k < N; ++k) {
		if(tw[k] > 1e-3f) fin[k] = fin[k] * (1.0f / tw[k]);
		if(tfb[k] > 1e-3f) fb[k] = fb[k] * (1.0f / tfb[k]);
		fin[k] = fin[k] * fin[k];
		fb[k] = fb[k] * fb[k];
		const float f = 8.0f * fminf(fmaxf(tw[k], 0.0f), 1.0f / 8.0f);
		out[k] = v3(fb[k].x * (1.0f - f) + fin[k].x * f, fb[k].y * (1.0f - f) + fin[k].y * f, fb[k].z * (1.0f - f) + fin[k].z * f);
	}
}

__device__ __forceinline__ Vec3 sample_probes(const GridConst& g, const uint32_t* __restrict__ states,
											  const float4* __restrict__ irr, const float2* __restrict__ dep, Vec3 position,
											  Vec3 normal, Vec3 to_camera) {
	const Vec3 n[1] = {normal};
	Vec3 out[1];
	sample_probes<1>(g, states, irr, dep, position, n, to_camera, out);
	return out[0];
}

// Order-independent (hence deterministic) accumulation: contributions are added as 64-bit
// fixed-point integers with 2^-50 resolution.
constexpr double kFixScale = 1125899906842624.0;  // 2^50
__device__ __forceinline__ long long to_fixed(float x) {
	const float s = x * 1125899906842624.0f;
	const float lim = 9.0e18f;
	return __float2ll_rn(fminf(fmaxf(s, -lim), lim));
}

// pbrMetallicRoughness (src/shaders/pbrMetallicRoughness.glsl:43-84)
__device__ __forceinline__ Vec3 pbr_metallic_roughness(Vec3 n, Vec3 v, Vec3 light_color, Vec3 light_dir, Vec3 albedo,
													   float metal, float rough) {
	const float f0 = 0.04f;
	const Vec3 diffuse = albedo * ((1.0f - f0) * (1.0f - metal));
	const float alpha = rough * rough;
	const Vec3 spec = v3(f0 * (1.0f - metal) + albedo.x * metal, f0 * (1.0f - metal) + albedo.y * metal,
						 f0 * (1.0f - metal) + albedo.z * metal);
	const float reflectance = fmaxf(fmaxf(spec.x, spec.y), spec.z);
	const float r90 = fminf(fmaxf(reflectance * 25.0f, 0.0f), 1.0f);
	const Vec3 l = normalize3(light_dir);
	const Vec3 h = normalize3(l + v);
	const float NdotL = fminf(fmaxf(dot3(n, l), 0.001f), 1.0f);
	const float NdotV = fminf(fmaxf(fabsf(dot3(n, v)), 0.001f), 1.0f);
	const float NdotH = fminf(fmaxf(dot3(n, h), 0.0f), 1.0f);
	const float VdotH = fminf(fmaxf(dot3(v, h), 0.0f), 1.0f);
	const float om = fminf(fmaxf(1.0f - VdotH, 0.0f), 1.0f);
	const float fw = om * om * om * om * om;
	const Vec3 F = v3(spec.x + (r90 - spec.x) * fw, spec.y + (r90 - spec.y) * fw, spec.z + (r90 - spec.z) * fw);
	const float a2 = alpha * alpha;
	const float attL = 2.0f * NdotL / (NdotL + sqrtf(a2 + (1.0f - a2) * (NdotL * NdotL)));
	const float attV = 2.0f * NdotV / (NdotV + sqrtf(a2 + (1.0f - a2) * (NdotV * NdotV)));
	const float G = attL * attV;
	const float ah = NdotH * alpha;
	const float k = alpha / ((1.0f - NdotH * NdotH) + ah * ah);
	const float D = fminf(fmaxf(k * k * (1.0f / kPiF), 0.0f), 4.0f);
	const float sp = G * D / (4.0f * NdotL * NdotV);
	const float inv_pi = 1.0f / kPiF;
	return v3(NdotL * light_color.x * ((1.0f - F.x) * diffuse.x * inv_pi + F.x * sp),
			  NdotL * light_color.y * ((1.0f - F.y) * diffuse.y * inv_pi + F.y * sp),
			  NdotL * light_color.z * ((1.0f - F.z) * diffuse.z * inv_pi + F.z * sp));
}

}  // namespace ddgi
