// Host-side check of the traversal's packed box test (vulkanexp_amd/csrc/packed_node.hpp), compiled and run
// by tests/test_packed_host.py:   packed_check SCENE MODE RAYS SEED REACH
// Builds the tree of a .scene file, packs its nodes as k_make_nodes does, and traces RAYS rays through the
// packed nodes and through the builder's FP32 boxes, with the kernels' FP32 box tests and one
// double-precision triangle test.  MODE says how the rays run:
//   generic  uniform directions
//   axis     along a coordinate axis, the other components +-0
//   plane    one component +-0
//   tiny     along a coordinate axis, the others of magnitude 1e-44 .. 1e-25
//   none     without a direction: all components +-0
//   infinite from a point with one infinite coordinate, every other one along another axis
//   far      from REACH away (and above) toward the scene's triangles
// from origins inside the scene's bounds (not farther than REACH from 0) unless far.
// Prints: rays hits mismatches-to-every-triangle packed-visits fp32-visits most-packed-visits
// (visits: node visits per ray).
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <string>
#include <vector>

#include "../vulkanexp_amd/csrc/bvh.hpp"
#include "../vulkanexp_amd/csrc/packed_node.hpp"

namespace ddgi {
namespace host {
void record_error(const std::string&) {}  // the library's error slot (api.hip), not linked here
}  // namespace host
}  // namespace ddgi

using namespace ddgi;

namespace {

struct Ray {
	float o[3], d[3];
};

// Moller-Trumbore in double; t in (1e-6, tmax)
bool hit(const float* v0, const float* v1, const float* v2, const Ray& r, double tmax, double& t) {
	double e1[3], e2[3], s[3], p[3], q[3];
	for(int k = 0; k < 3; ++k) {
		e1[k] = double(v1[k]) - v0[k];
		e2[k] = double(v2[k]) - v0[k];
		s[k] = double(r.o[k]) - v0[k];
	}
	p[0] = r.d[1] * e2[2] - r.d[2] * e2[1];
	p[1] = r.d[2] * e2[0] - r.d[0] * e2[2];
	p[2] = r.d[0] * e2[1] - r.d[1] * e2[0];
	const double det = e1[0] * p[0] + e1[1] * p[1] + e1[2] * p[2];
	if(det == 0.0) return false;
	const double u = (s[0] * p[0] + s[1] * p[1] + s[2] * p[2]) / det;
	if(!(u >= 0.0 && u <= 1.0)) return false;
	q[0] = s[1] * e1[2] - s[2] * e1[1];
	q[1] = s[2] * e1[0] - s[0] * e1[2];
	q[2] = s[0] * e1[1] - s[1] * e1[0];
	const double v = (r.d[0] * q[0] + r.d[1] * q[1] + r.d[2] * q[2]) / det;
	if(!(v >= 0.0 && u + v <= 1.0)) return false;
	t = (e2[0] * q[0] + e2[1] * q[1] + e2[2] * q[2]) / det;
	return t > 1e-6 && t < tmax;
}

float half(uint32_t h) {  // 0, infinities and normal numbers
	const uint32_t e = (h >> 10) & 31u, m = h & 0x3FFu;
	const float v = e == 31u ? INFINITY : (e == 0u ? 0.0f : std::ldexp(float(m | 0x400u), int(e) - 25));
	return (h & 0x8000u) ? -v : v;
}

struct Packed {
	float header[4];
	uint32_t planes[4][3];  // per child and axis, lo in the low half
	uint32_t code[4];
};

// the boxes of a subtree's slots, and the packed nodes over them
struct Box {
	float lo[3] = {3.402823466e+38f, 3.402823466e+38f, 3.402823466e+38f};
	float hi[3] = {-3.402823466e+38f, -3.402823466e+38f, -3.402823466e+38f};
	void grow(const Box& b) {
		for(int a = 0; a < 3; ++a) {
			lo[a] = std::min(lo[a], b.lo[a]);
			hi[a] = std::max(hi[a], b.hi[a]);
		}
	}
};

uint32_t code_of(const BvhHost& b, uint32_t node, uint32_t k) {
	uint32_t c;
	std::memcpy(&c, &b.nodes[size_t(node) * kNodeFloats + kCodeRow + k], 4);
	return c;
}

Box pack(const BvhHost& b, uint32_t node, std::vector<Packed>& out) {
	Box all, kid[4];
	Packed& p = out[node];
	double mn[3], mx[3], size = 0.0;
	for(uint32_t k = 0; k < 4; ++k) {
		const uint32_t c = code_of(b, node, k);
		p.code[k] = packed_code(c);
		if(c == kEmptyChild) continue;
		if(c & kLeafFlag) {
			const uint32_t first = (c & ~kLeafFlag) >> 3, cnt = (c & 7u) + 1u;
			for(uint32_t i = first; i < first + cnt; ++i) {
				Box s;
				std::memcpy(s.lo, &b.slot_box[size_t(i) * 6], 12);
				std::memcpy(s.hi, &b.slot_box[size_t(i) * 6 + 3], 12);
				kid[k].grow(s);
			}
		} else {
			kid[k] = pack(b, c, out);
		}
		all.grow(kid[k]);
		for(int a = 0; a < 3; ++a) {
			kid[k].lo[a] = pad_down(kid[k].lo[a]);
			kid[k].hi[a] = pad_up(kid[k].hi[a]);
		}
	}
	for(int a = 0; a < 3; ++a) {
		float l = kid[0].lo[a], h = kid[0].hi[a];
		for(int k = 1; k < 4; ++k) {
			l = std::min(l, kid[k].lo[a]);
			h = std::max(h, kid[k].hi[a]);
		}
		mn[a] = l;
		mx[a] = h;
		size = std::max(size, mx[a] - mn[a]);
	}
	const NodeGrid g = node_grid(mn, mx, size);
	for(int a = 0; a < 3; ++a) p.header[a] = g.org[a];
	p.header[3] = g.scale;
	for(uint32_t k = 0; k < 4; ++k)
		for(int a = 0; a < 3; ++a)
			p.planes[k][a] = child_planes(g, a, kid[k].lo[a], kid[k].hi[a], code_of(b, node, k) == kEmptyChild);
	return all;
}

// Entry distances of a node's children (infinity: not entered), by either form.
void keys_packed(const Packed& p, const float o[3], const float inv[3], float tmin, float best, float key[4]) {
	for(int k = 0; k < 4; ++k) {
		float tn = 0, tf = 0;
		for(int a = 0; a < 3; ++a) {
			const float A = p.header[3] * inv[a], B = (p.header[a] - o[a]) * inv[a];
			const bool neg = std::signbit(inv[a]);
			const float lo = half(p.planes[k][a] & 0xFFFFu), hi = half(p.planes[k][a] >> 16);
			const float en = std::fma(neg ? hi : lo, A, B), ef = std::fma(neg ? lo : hi, A, B);
			tn = a == 0 ? en : std::fmax(tn, en);
			tf = a == 0 ? ef : std::fmin(tf, ef);
		}
		const float n = std::fmax(tn, tmin), f = std::fmin(tf, best);
		key[k] = n <= f * 1.000001f ? n : INFINITY;
	}
}
void keys_fp32(const BvhHost& b, uint32_t node, const float o[3], const float inv[3], float tmin, float best, float key[4]) {
	const float* r = &b.nodes[size_t(node) * kNodeFloats];
	for(uint32_t k = 0; k < 4; ++k) {
		float n = tmin, f = best;
		for(int a = 0; a < 3; ++a) {
			const bool neg = std::signbit(inv[a]);
			const float lo = (r[(2 * a) * 4 + k] - o[a]) * inv[a], hi = (r[(2 * a + 1) * 4 + k] - o[a]) * inv[a];
			n = std::fmax(n, neg ? hi : lo);
			f = std::fmin(f, neg ? lo : hi);
		}
		key[k] = n <= f * 1.000001f && code_of(b, node, k) != kEmptyChild ? n : INFINITY;
	}
}

// Nearest hit through the tree: the children entered, nearest first; a popped kNone ends the ray, as in the
// kernels, whose stack ends with it.
double trace(const BvhHost& b, const std::vector<Packed>* packed, const Ray& r, uint64_t& visits) {
	constexpr uint32_t kNone = 0xFFFFFFFFu;
	float inv[3];
	for(int a = 0; a < 3; ++a) inv[a] = 1.0f / r.d[a];
	if(packed) slab_reciprocals(r.o, (*packed)[0].header, inv);
	std::vector<uint32_t> stack{kNone, 0u};
	double best = 1e30;
	for(;;) {
		const uint32_t c = stack.back();
		stack.pop_back();
		if(c == kNone) return best;
		if(c & kLeafFlag) {
			const uint32_t first = (c & ~kLeafFlag) >> 3, cnt = (c & 7u) + 1u;
			for(uint32_t i = first; i < first + cnt; ++i) {
				const float* t = &b.tris[size_t(i) * 12];
				double at;
				if(hit(t, t + 4, t + 8, r, best, at)) best = at;
			}
			continue;
		}
		++visits;
		float key[4];
		uint32_t order[4] = {0, 1, 2, 3};
		const float upper = std::nextafter(float(best), INFINITY);
		if(packed) keys_packed((*packed)[c], r.o, inv, 1e-6f, upper, key);
		else keys_fp32(b, c, r.o, inv, 1e-6f, upper, key);
		std::sort(order, order + 4, [&](uint32_t x, uint32_t y) { return key[x] > key[y]; });
		for(uint32_t k : order)
			if(key[k] != INFINITY) stack.push_back(packed ? (*packed)[c].code[k] : code_of(b, c, k));
	}
}

}  // namespace

int main(int argc, char** argv) {
	if(argc != 6) {
		std::fprintf(stderr, "usage: %s SCENE MODE RAYS SEED REACH\n", argv[0]);
		return 2;
	}
	void* sc = nullptr;
	if(ddgi_scene_load(argv[1], &sc) != DDGI_OK) {
		std::fprintf(stderr, "cannot load %s\n", argv[1]);
		return 2;
	}
	ddgi_scene_tables T;
	ddgi_scene_get_tables(sc, &T);
	BvhHost b;
	const char* err = nullptr;
	if(!build_bvh(T.vertices, T.vertex_count, T.indices, T.index_count, T.offsets, T.offset_count, T.instances,
				  T.instance_count, b, &err)) {
		std::fprintf(stderr, "build failed: %s\n", err ? err : "?");
		return 1;
	}
	std::vector<Packed> packed(b.node_count);
	pack(b, 0, packed);
	const std::string mode = argv[2];
	const double reach = std::atof(argv[5]);
	const long rays = std::atol(argv[3]);
	std::mt19937_64 rng(std::strtoull(argv[4], nullptr, 10));
	std::uniform_real_distribution<double> U(0.0, 1.0);
	long bad = 0, hits = 0;
	uint64_t vp = 0, vf = 0, most = 0;
	for(long q = 0; q < rays; ++q) {
		Ray r;
		for(int a = 0; a < 3; ++a) {
			const double lo = std::max<double>(T.bounds_min[a], -reach), hi = std::min<double>(T.bounds_max[a], reach);
			r.o[a] = float(lo + (hi - lo) * U(rng));
		}
		const int axis = int(U(rng) * 3.0);
		const double z = 2.0 * U(rng) - 1.0, ph = 2.0 * M_PI * U(rng), s = std::sqrt(1.0 - z * z);
		const double d[3] = {std::cos(ph) * s, std::sin(ph) * s, z};
		const float* at = &b.tris[size_t(U(rng) * b.tri_count) * 12];
		for(int a = 0; a < 3; ++a) {
			const double sign = U(rng) < 0.5 ? -1.0 : 1.0, e = U(rng);
			r.d[a] = float(d[a]);
			if(mode == "axis") r.d[a] = float(sign * (a == axis ? 1.0 : 0.0));
			if(mode == "plane" && a == axis) r.d[a] = float(sign * 0.0);
			if(mode == "tiny") r.d[a] = float(sign * (a == axis ? 1.0 : std::pow(10.0, -44.0 + 19.0 * e)));
			if(mode == "none") r.d[a] = float(sign * 0.0);
			if(mode == "infinite" && a == axis) r.o[a] = float(sign) * INFINITY;
			if(mode == "infinite" && q % 2) r.d[a] = float(sign * (a == (axis + 1) % 3 ? 1.0 : 0.0));
			// toward the triangle, within a tenth of the distance by which the box test widens a box's exit
			if(mode == "far") {
				const double to = at[a] + 1e-7 * reach * (2.0 * e - 1.0);
				r.o[a] = float(to + reach * (a == 1 ? std::abs(d[a]) + 0.1 : d[a]));
				r.d[a] = float((to - r.o[a]) / reach);
			}
		}
		double brute = 1e30, t;
		for(uint32_t i = 0; i < b.tri_count; ++i) {
			const float* v = &b.tris[size_t(i) * 12];
			if(hit(v, v + 4, v + 8, r, brute, t)) brute = t;
		}
		const uint64_t before = vp;
		bad += trace(b, &packed, r, vp) != brute;
		most = std::max(most, vp - before);
		trace(b, nullptr, r, vf);
		hits += brute < 1e30;
	}
	std::printf("%ld %ld %ld %.3f %.3f %llu\n", rays, hits, bad, double(vp) / double(rays), double(vf) / double(rays),
				(unsigned long long)most);
	return 0;
}
