// The arithmetic of the traversal's packed nodes that decides whether a box test is conservative: the grid
// of a node, the planes on it and a ray's reciprocals.  Shared by the kernels (k_make_nodes, traverse) and
// by host programs, with the same FP32 and FP64 operations (no contraction) on both.
#pragma once

#include <cmath>
#include <cstdint>
#include <cstring>

#include "bvh.hpp"

#ifdef __HIPCC__
#define DDGI_HD __host__ __device__ __forceinline__
#else
#define DDGI_HD inline
#endif

namespace ddgi {

constexpr float kPlaneSteps = 2047.0f;  // grid steps over a node's extent: 11 bits, exact in FP16
constexpr uint32_t kPlaneInf = 0x7C00u, kPlaneNegInf = 0xFC00u;  // FP16 infinities

// The grid of a node whose children's (padded) boxes span mn .. mx, `size` along the longest axis: origin,
// scale (a power of two) and the growth of the boxes in position.  Not `fits`: the extent is too large for
// it (or infinite), and the children's planes are infinite.  The scale then only states how large the
// node's coordinates are, as slab_reciprocals wants it.
struct NodeGrid {
	float org[3], scale;
	double slack;
	bool fits;
};
DDGI_HD float next_power_of_two(float v) {  // v >= 0; v itself where it is one
	uint32_t b;
	std::memcpy(&b, &v, 4);
	b = (b + 0x007FFFFFu) & 0x7F800000u;
	std::memcpy(&v, &b, 4);
	return v;
}
DDGI_HD NodeGrid node_grid(const double mn[3], const double mx[3], double size) {
	NodeGrid g;
	g.slack = size * 1e-6;
	double ext = 0.0, reach = 0.0;
	for(int a = 0; a < 3; ++a) {
		const double lo = mn[a] - g.slack;
		g.org[a] = float(lo);
		if(double(g.org[a]) > lo) g.org[a] = nextafterf(g.org[a], -INFINITY);
		ext = fmax(ext, mx[a] + g.slack - double(g.org[a]));
		reach = fmax(reach, fmax(fabs(mn[a]), fabs(mx[a])));
	}
	g.fits = ext < 1e37;  // false for infinite extents too
	// the smallest power of two with kPlaneSteps steps over the extent
	g.scale = next_power_of_two(float((g.fits ? ext : reach) * (1.000001 / double(kPlaneSteps))));
	if(!g.fits) g.org[0] = g.org[1] = g.org[2] = 0.0f;
	return g;
}

DDGI_HD uint32_t plane_bits(int q) {  // an integer 0 .. 2047 as FP16
	if(q == 0) return 0u;
	const float f = float(q);
	uint32_t b;
	std::memcpy(&b, &f, 4);
	return ((b >> 23) - 112u) << 10 | ((b >> 13) & 0x3FFu);
}
// FP16 bits of the planes of a child's box [lo, hi] along one axis, low half lo: integers 0 .. kPlaneSteps,
// rounded outward; infinite ones for a node beyond the grid; inverted infinite ones for an empty child: its
// entry distance is infinity and its exit distance minus infinity from any finite distance, where an
// inversion of finite size is lost in the widening of the exit (1e-6 of the distance) far from the node.
DDGI_HD uint32_t child_planes(const NodeGrid& g, int axis, float lo, float hi, bool empty) {
	if(empty) return kPlaneInf | kPlaneNegInf << 16;
	if(!g.fits) return kPlaneNegInf | kPlaneInf << 16;
	const double inv = 1.0 / double(g.scale);
	const double l = floor((double(lo) - g.slack - double(g.org[axis])) * inv);
	const double h = ceil((double(hi) + g.slack - double(g.org[axis])) * inv);
	const double top = double(kPlaneSteps);
	return plane_bits(int(fmin(fmax(l, 0.0), top))) | plane_bits(int(fmin(fmax(h, 0.0), top))) << 16;
}

// The code of a child in a packed node.  An empty child's is that of a leaf of triangle slot 0: should its
// box be entered all the same (a ray whose distances are no numbers), a triangle of the scene is tested once
// more, which changes no hit.
inline uint32_t packed_code(uint32_t code) { return code == kEmptyChild ? kLeafFlag : code; }

// A ray's reciprocals for the box test (inv: 1 / direction on entry; `root`: the root node's header, origin
// and scale).  A plane's distance is fma(q, scale * inv, (org - o) * inv): while |org - o| and |plane - o|
// are at most `reach`, reciprocals up to 3e38 / reach keep both terms finite.  Larger ones (a direction
// component of zero, or so small that the terms would overflow: to a miss, or to infinity minus infinity)
// are replaced by that bound, which moves the ray by less than 1e-38 reach^2 / |direction|: far less than
// the boxes' padding of 1e-6, unless the coordinates are astronomical (from about 1e16 on, for directions of
// length one).  There the reciprocal becomes a NaN, and the axis excludes no box: the maxima and minima of
// the box test drop its distances.  A ray without a direction (all reciprocals infinite) hits nothing; it
// keeps the bound, and so only the boxes around its origin.  A ray from infinity enters no box with any
// finite reciprocal.
DDGI_HD void slab_reciprocals(const float o[3], const float root[4], float inv[3]) {
	const float from = fmaxf(fmaxf(fabsf(o[0]), fabsf(o[1])), fabsf(o[2]));
	const float reach = (from < INFINITY ? from : 0.0f) +
						fmaxf(fmaxf(fabsf(root[0]), fabsf(root[1])), fabsf(root[2])) + kPlaneSteps * root[3];
	const float at_least = fmaxf(reach, 1.0f);
	if(fmaxf(fmaxf(fabsf(inv[0]), fabsf(inv[1])), fabsf(inv[2])) * at_least <= 3e38f) return;  // nearly every ray
	const float least = fminf(fminf(fabsf(inv[0]), fabsf(inv[1])), fabsf(inv[2]));  // of the longest component
	const float bound = 3e38f / at_least;
	const float cap = reach * at_least * least <= 1e32f || least == INFINITY ? bound : NAN;
	for(int a = 0; a < 3; ++a)
		if(!(fabsf(inv[a]) <= bound)) inv[a] = copysignf(cap, inv[a]);
}

}  // namespace ddgi
