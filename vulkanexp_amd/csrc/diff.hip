// Differentiable probe update: gradients of a shaded-G-buffer loss with respect to per-material
// albedo and the sun radiance, through probe sampling (src/shaders/irradiance.glsl:145-237), the
// border copy and the ray-to-texel irradiance blend (src/shaders/probesUpdate.glsl:70-103).
//
// Per-ray radiance is affine in the parameters (factors from the shading kernel):
//   rad = c0 + A (.) a[m] + (B (.) a[m] + C) (.) sun
// Forward:  rad -> irradiance blend (FP32 kernel, irradiance only) -> sampleProbes at every
//           G-buffer texel -> shade = out (.) a[g] * 0.996 (FinalGather.frag:62-72) -> MSE.
// Backward: hand-written adjoint.  All reductions are deterministic: the contributions are fixed-point
//           integers and their sums exact (order-independent).  The sampling weights (visibility,
//           trilinear) of a texel are kept in a record by the preparation where memory allows it, and
//           recomputed elsewhere; the blend weights are recomputed.
// G-buffer texels are binned by probe cell at prepare time, so a work item (a chunk of one cell's
// texels) scatters into only the 8 probe tiles of that cell's cage, accumulated in LDS.
#include "device_common.hpp"
#include "diff.hpp"

namespace ddgi {

namespace {

constexpr int kBlock = 256;

__device__ __forceinline__ bool cell_of(const GridConst& g, const float* pos, uint64_t x, uint32_t& cell) {
	const float ax = fabsf(g.cell[0]), ay = fabsf(g.cell[1]), az = fabsf(g.cell[2]);
	const float gx = (pos[x * 3] - g.emin[0]) / ax, gy = (pos[x * 3 + 1] - g.emin[1]) / ay, gz = (pos[x * 3 + 2] - g.emin[2]) / az;
	if(gx < 0.0f || gy < 0.0f || gz < 0.0f) return false;
	const int f0 = int(gx), f1 = int(gy), f2 = int(gz);
	if(f0 > g.res[0] - 1 || f1 > g.res[1] - 1 || f2 > g.res[2] - 1) return false;
	cell = uint32_t(f0) + uint32_t(g.res[0]) * (uint32_t(f1) + uint32_t(g.res[1]) * uint32_t(f2));
	return true;
}

__device__ __forceinline__ Vec3 load3(const float* p, uint64_t i) { return v3(p[i * 3], p[i * 3 + 1], p[i * 3 + 2]); }

// ---- the sampling of a texel ----
// The irradiance-independent part of a sampleProbes call: per cage slot i (0..7) the weight and fallback
// weight (0 when the probe does not contribute, bit i of mask), their totals, the probe of slot 0, and the
// first colour tap (texel cy0 * 8 + cx0 of the tile) with the bilinear fractions, the same for the 8
// probes (they depend on the normal only).
struct TexelWeights {
	float w[8], fw[8], cwx, cwy, tw, tfb;
	uint32_t base, t00, mask;
};

__device__ __forceinline__ TexelWeights make_weights(const DiffArgs& d, uint64_t x) {
	const GridConst& g = d.grid;
	TexelWeights c;
	c.mask = c.base = c.t00 = 0u;
	c.cwx = c.cwy = c.tw = c.tfb = 0.0f;
#pragma unroll
	for(int i = 0; i < 8; ++i) c.w[i] = c.fw[i] = 0.0f;
	const Vec3 position = load3(d.pos, x), normal = load3(d.nrm, x), to_camera = load3(d.tocam, x);
	Cage cage;
	if(!make_cage(g, position, cage)) return c;
	const Vec3 biased = position + (normal + to_camera) * g.shadow_bias;
	float cu, cv;
	oct_uv(normal.x, normal.y, normal.z, cu, cv);
	c.t00 = tile_coords<8>(cu, cv, c.cwx, c.cwy);
	c.base = uint32_t(cage.f[0]) + uint32_t(g.res[0]) * (uint32_t(cage.f[1]) + uint32_t(g.res[1]) * uint32_t(cage.f[2]));
#pragma unroll
	for(int i = 0; i < 8; ++i) {
		uint32_t lin;
		Vec3 pp, dtp;
		float trw, w, fw;
		if(!cage_corner(g, d.states, cage, position, i, lin, pp, dtp, trw)) continue;
		cage_weight(d.dep, lin, pp, dtp, trw, normal, biased, w, fw);
		c.mask |= 1u << i;
		c.w[i] = w;
		c.fw[i] = fw;
		c.tw += w;
		c.tfb += fw;
	}
	return c;
}

// The weights of texel x from its record (w[8], fw[8], cwx, cwy, base, t00 | mask << 8), or recomputed.
__device__ __forceinline__ TexelWeights texel_weights(const DiffArgs& d, uint64_t x) {
	if(!d.rec) return make_weights(d, x);
	const float4* r = d.rec + x * kDiffRecRows;
	const float4 q[5] = {r[0], r[1], r[2], r[3], r[4]};
	TexelWeights c;
#pragma unroll
	for(int i = 0; i < 2; ++i) {
		c.w[4 * i] = q[i].x, c.w[4 * i + 1] = q[i].y, c.w[4 * i + 2] = q[i].z, c.w[4 * i + 3] = q[i].w;
		c.fw[4 * i] = q[2 + i].x, c.fw[4 * i + 1] = q[2 + i].y, c.fw[4 * i + 2] = q[2 + i].z, c.fw[4 * i + 3] = q[2 + i].w;
	}
	c.cwx = q[4].x;
	c.cwy = q[4].y;
	c.base = __float_as_uint(q[4].z);
	const uint32_t meta = __float_as_uint(q[4].w);
	c.t00 = meta & 63u;
	c.mask = meta >> 8;
	c.tw = c.tfb = 0.0f;
#pragma unroll
	for(int i = 0; i < 8; ++i) {
		c.tw += c.w[i];
		c.tfb += c.fw[i];
	}
	return c;
}

// What sampleProbes makes of the weights: per channel the probes' square roots s and the normalised sums;
// the irradiance is fb^2 (1 - k) + fin^2 k.
struct TexelEval {
	float s[8][3], fin[3], fb[3], k, inv_w, inv_fb;
};

__device__ __forceinline__ TexelEval texel_eval(const DiffArgs& d, const TexelWeights& c) {
	TexelEval e;
	const uint32_t rx = uint32_t(d.grid.res[0]), ry = uint32_t(d.grid.res[1]);
	e.inv_w = c.tw > 1e-3f ? 1.0f / c.tw : 1.0f;
	e.inv_fb = c.tfb > 1e-3f ? 1.0f / c.tfb : 1.0f;
	e.k = 8.0f * fminf(fmaxf(c.tw, 0.0f), 1.0f / 8.0f);
#pragma unroll
	for(int ch = 0; ch < 3; ++ch) e.fin[ch] = e.fb[ch] = 0.0f;
#pragma unroll
	for(int i = 0; i < 8; ++i) {
		const bool on = (c.mask >> i) & 1u;
		// slots that do not contribute read some tile and drop what they read
		const uint32_t lin = on ? c.base + uint32_t(i & 1) + rx * (uint32_t((i >> 1) & 1) + ry * uint32_t(i >> 2)) : 0u;
		const float4* ct = d.irr + size_t(lin) * 64 + c.t00;
		const float4 c00 = ct[0], c10 = ct[1], c01 = ct[8], c11 = ct[9];
		const float a[3][4] = {{c00.x, c10.x, c01.x, c11.x}, {c00.y, c10.y, c01.y, c11.y}, {c00.z, c10.z, c01.z, c11.z}};
#pragma unroll
		for(int ch = 0; ch < 3; ++ch) {
			const float v = (a[ch][0] * (1.0f - c.cwx) + a[ch][1] * c.cwx) * (1.0f - c.cwy) +
							(a[ch][2] * (1.0f - c.cwx) + a[ch][3] * c.cwx) * c.cwy;
			e.s[i][ch] = on ? sqrtf(v) : 0.0f;
			e.fin[ch] += e.s[i][ch] * c.w[i];
			e.fb[ch] += e.s[i][ch] * c.fw[i];
		}
	}
#pragma unroll
	for(int ch = 0; ch < 3; ++ch) {
		e.fin[ch] *= e.inv_w;
		e.fb[ch] *= e.inv_fb;
	}
	return e;
}

// ---- prepare: sampling records, and texels binned by (cell, first colour tap) ----
__global__ __launch_bounds__(kBlock) void k_records(DiffArgs d, float4* __restrict__ rec) {
	const uint64_t x = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
	if(x >= d.N) return;
	const TexelWeights c = make_weights(d, x);
	float4* r = rec + x * kDiffRecRows;
	r[0] = make_float4(c.w[0], c.w[1], c.w[2], c.w[3]);
	r[1] = make_float4(c.w[4], c.w[5], c.w[6], c.w[7]);
	r[2] = make_float4(c.fw[0], c.fw[1], c.fw[2], c.fw[3]);
	r[3] = make_float4(c.fw[4], c.fw[5], c.fw[6], c.fw[7]);
	r[4] = make_float4(c.cwx, c.cwy, __uint_as_float(c.base), __uint_as_float(c.t00 | (c.mask << 8)));
}

// Adds 1 to counter[key] for every active lane and returns the lane's own position, with one atomic per
// distinct key of the wavefront (neighbouring texels mostly share theirs: one atomic per lane on a few
// hundred hot counters took 4 ms for a full-HD view).
__device__ __forceinline__ uint32_t wave_count(uint32_t* counter, uint32_t key) {
	const uint32_t lane = __lane_id();
	uint32_t pos = 0;
	for(uint64_t left = __ballot(true); left != 0u;) {
		const int leader = __ffsll((unsigned long long)left) - 1;
		const uint32_t k = uint32_t(__builtin_amdgcn_readlane(int(key), leader));
		const uint64_t same = __ballot(key == k) & left;
		if(key == k) {
			uint32_t base = 0;
			if(int(lane) == leader) base = atomicAdd(&counter[k], uint32_t(__popcll(same)));
			pos = uint32_t(__builtin_amdgcn_readlane(int(base), leader)) +
				  uint32_t(__popcll(same & ((uint64_t(1) << lane) - 1u)));
		}
		left &= ~same;
	}
	return pos;
}

__global__ void k_cells(DiffArgs d, uint32_t taps, uint32_t* __restrict__ key_of, uint32_t* __restrict__ key_count) {
	const uint64_t x = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if(x >= d.N) return;
	uint32_t c;
	if(!cell_of(d.grid, d.pos, x, c)) {
		key_of[x] = 0xFFFFFFFFu;
		return;
	}
	if(taps == 64u) {
		float cu, cv, wx, wy;
		oct_uv(d.nrm[x * 3], d.nrm[x * 3 + 1], d.nrm[x * 3 + 2], cu, cv);
		c = c * 64u + tile_coords<8>(cu, cv, wx, wy);
	}
	key_of[x] = c;
	wave_count(key_count, c);
}

// Sum over a workgroup of 1024 threads of (a, b), and this thread's exclusive prefix.
__device__ __forceinline__ void block_scan2(uint32_t a, uint32_t b, uint32_t* s_a, uint32_t* s_b, uint32_t& pa, uint32_t& pb,
											uint32_t& ta, uint32_t& tb) {
	const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6;
	uint32_t ia = a, ib = b;
	for(int o = 1; o < 64; o <<= 1) {
		const uint32_t xa = uint32_t(__shfl_up(int(ia), o)), xb = uint32_t(__shfl_up(int(ib), o));
		if(lane >= uint32_t(o)) {
			ia += xa;
			ib += xb;
		}
	}
	if(lane == 63u) {
		s_a[wave] = ia;
		s_b[wave] = ib;
	}
	__syncthreads();
	pa = ia - a;
	pb = ib - b;
	ta = tb = 0;
	for(uint32_t w = 0; w < 16u; ++w) {
		pa += w < wave ? s_a[w] : 0u;
		pb += w < wave ? s_b[w] : 0u;
		ta += s_a[w];
		tb += s_b[w];
	}
	__syncthreads();
}

// One workgroup: exclusive sums over the keys (texel offsets) and over the cells (work items of at most
// kDiffChunk texels of a cell).
__global__ __launch_bounds__(1024) void k_items(DiffArgs d, uint32_t taps, const uint32_t* __restrict__ key_count,
												uint32_t* __restrict__ key_start, uint32_t* __restrict__ cell_item_start,
												uint32_t* __restrict__ item_begin, uint32_t* __restrict__ item_count,
												uint32_t* __restrict__ n_items) {
	__shared__ uint32_t s_a[16], s_b[16];
	const uint32_t cells = d.grid.probe_count, t = threadIdx.x;
	uint32_t pix = 0, items = 0;
	for(uint32_t base = 0; base < cells; base += 1024u) {
		const uint32_t c = base + t;
		uint32_t cnt = 0;
		if(c < cells)
			for(uint32_t k = 0; k < taps; ++k) cnt += key_count[size_t(c) * taps + k];
		const uint32_t ni = (cnt + kDiffChunk - 1) / kDiffChunk;
		uint32_t pc, pi, tc, ti;
		block_scan2(cnt, ni, s_a, s_b, pc, pi, tc, ti);
		if(c < cells) {
			uint32_t at = pix + pc;
			cell_item_start[c] = items + pi;
			for(uint32_t k = 0; k < ni; ++k) {
				item_begin[items + pi + k] = at + k * kDiffChunk;
				item_count[items + pi + k] = min(kDiffChunk, cnt - k * kDiffChunk);
			}
			for(uint32_t k = 0; k < taps; ++k) {
				key_start[size_t(c) * taps + k] = at;
				at += key_count[size_t(c) * taps + k];
			}
		}
		pix += tc;
		items += ti;
	}
	if(t == 0) {
		cell_item_start[cells] = items;
		*n_items = items;
	}
}

__global__ void k_scatter(DiffArgs d, const uint32_t* __restrict__ key_of, const uint32_t* __restrict__ key_start,
						  uint32_t* __restrict__ cursor, uint32_t* __restrict__ sorted) {
	const uint64_t x = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if(x >= d.N) return;
	const uint32_t c = key_of[x];
	if(c == 0xFFFFFFFFu) return;
	const uint32_t pos = wave_count(cursor, c);
	sorted[key_start[c] + pos] = uint32_t(x);
}

// ---- forward ----
__global__ void k_radiance(DiffArgs d) {
	const uint64_t r = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if(r >= d.rays) return;
	const float4* f = d.factors + r * 4;
	const float4 c0 = f[0];
	const uint32_t m = __float_as_uint(c0.w);
	float4 out = make_float4(c0.x, c0.y, c0.z, 0.0f);
	if(m != 0xFFFFFFFFu) {
		const float4 A = f[1], B = f[2], C = f[3];
		const float* a = d.albedo + size_t(m) * 3;
		out.x += A.x * a[0] + (B.x * a[0] + C.x) * d.sun[0];
		out.y += A.y * a[1] + (B.y * a[1] + C.y) * d.sun[1];
		out.z += A.z * a[2] + (B.z * a[2] + C.z) * d.sun[2];
	}
	d.rad[r] = out;
}

// One thread per texel: 80 bytes of record, 16 of material and target in, 12 out, and 32 taps that
// neighbouring texels share.  Memory-bound: 63 us for a full-HD view (250 MB in 50 us at a copy's rate),
// against 128 us with the weights recomputed.
__global__ __launch_bounds__(kBlock) void k_gather_fwd(DiffArgs d) {
	__shared__ float red[kBlock / 64];
	const uint64_t x = uint64_t(blockIdx.x) * kBlock + threadIdx.x;
	float l = 0.0f;
	if(x < d.N) {
		const TexelWeights c = texel_weights(d, x);
		const TexelEval e = texel_eval(d, c);
		const float* a = d.albedo + size_t(d.gmat[x]) * 3;
#pragma unroll
		for(int ch = 0; ch < 3; ++ch) {
			const float o = e.fb[ch] * e.fb[ch] * (1.0f - e.k) + e.fin[ch] * e.fin[ch] * e.k;
			const float s = o * a[ch] * 0.996f;
			d.shade[x * 3 + ch] = s;
			const float err = s - d.target[x * 3 + ch];
			l += err * err;
		}
	}
	for(int o = 32; o > 0; o >>= 1) l += __shfl_xor(l, o);
	if(__lane_id() == 0) red[threadIdx.x >> 6] = l;
	__syncthreads();
	if(threadIdx.x == 0) d.loss_part[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// One workgroup; the partial sums added in double, in a fixed order (5 us; 329 us in one thread).
__global__ __launch_bounds__(1024) void k_loss(DiffArgs d, uint32_t parts) {
	__shared__ double red[1024];
	double s = 0.0;
	for(uint32_t i = threadIdx.x; i < parts; i += 1024u) s += double(d.loss_part[i]);
	red[threadIdx.x] = s;
	__syncthreads();
	for(uint32_t o = 512; o > 0; o >>= 1) {
		if(threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
		__syncthreads();
	}
	if(threadIdx.x == 0) d.loss[0] = float(red[0] / double(3ull * d.N));
}

// ---- backward ----
// Contributions are rounded to integers in units of 2^-50 and their sums are exact, hence independent of
// their order.  Those below kSmallUnits are summed in doubles (an addition there is one instruction, a
// conversion to 64-bit integers eight): kDiffChunk of them, the most that one sum takes, stay within the
// 2^53 to which doubles hold every integer.  Larger ones go to the 64-bit integers one by one.
constexpr float kUnits = 1125899906842624.0f;  // 2^50
constexpr float kSmallUnits = 8796093022208.0f;  // 2^43
static_assert(double(kSmallUnits) * kDiffChunk <= 9007199254740992.0 && kMaxRays <= kDiffChunk, "sums in doubles are exact");
__device__ __forceinline__ float to_units(float x) { return fminf(fmaxf(x * kUnits, -9.0e18f), 9.0e18f); }
__device__ __forceinline__ void add_units(unsigned long long* a, double v) { atomicAdd(a, (unsigned long long)(long long)v); }

// One workgroup per work item: its texels share one cage of 8 probes, whose gradient tiles it sums in
// LDS.  A wavefront evaluates 64 texels, one per lane, and then, for each channel, turns to eight texels at
// a time with one lane per cage probe (through LDS).  As the texels are ordered by their first tap, the
// eight nearly always share their four taps (and the 64 their material), so that a lane adds its
// contributions to registers and goes to the LDS tiles only when the taps change.  Full-HD view: 531 us
// with 96 LDS atomics per texel, most of them 64 lanes on one address; 233 us with eight lanes per texel
// throughout, where the evaluation is done eight times over; 112 us so (as multiples of it: 1.6 with the texels ordered
// by cell only, 1.13 with items of 2048 texels, 1.8 with 4096, 1.4 with 5 waves per SIMD, which spill; 109 us
// when contributions too large for a sum in doubles were not told apart).  Bound by vector
// instructions: the square roots, divisions and roundings of 96 contributions per texel.
// four waves per SIMD: 128 VGPRs
__global__ __launch_bounds__(kBlock, 4) void k_gather_bwd(DiffArgs d) {
	extern __shared__ unsigned long long lds[];
	unsigned long long* tile = lds;                  // [8][64][3]
	unsigned long long* mat = lds + 8 * 192;         // [M][3]
	__shared__ __attribute__((aligned(16))) float s_g[kBlock / 64][64 * 8];  // gradient per (texel, probe), one channel
	__shared__ __attribute__((aligned(16))) float s_b[kBlock / 64][64 * 4];  // tap weights per texel
	__shared__ uint32_t s_t[kBlock / 64][64];                                // first tap (| kLarge), kNo: no texel
	const uint32_t item = blockIdx.x;
	if(item >= *d.n_items) return;
	for(uint32_t k = threadIdx.x; k < 8 * 192 + d.M * 3; k += kBlock) lds[k] = 0ull;
	__syncthreads();
	const uint32_t begin = d.item_begin[item], cnt = d.item_count[item];
	const float inv3n = 2.0f / float(3ull * d.N);
	const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6, i = lane & 7u;
	unsigned long long* my_tile = tile + i * 192;
	constexpr uint32_t kNo = 0xFFFFFFFFu, kLarge = 64u;
	uint32_t cur_tap = kNo, cur_mat = kNo;  // wave-uniform: what the registers hold sums of
	double acc[4][3], macc[3];
#pragma unroll
	for(int q = 0; q < 4; ++q) acc[q][0] = acc[q][1] = acc[q][2] = 0.0;
	macc[0] = macc[1] = macc[2] = 0.0;
	const auto tap_of = [](uint32_t t00, int q) { return t00 + uint32_t(q & 1) + 8u * uint32_t(q >> 1); };
	const auto flush_taps = [&] {
#pragma unroll
		for(int q = 0; q < 4; ++q)
#pragma unroll
			for(int ch = 0; ch < 3; ++ch) {
				if(acc[q][ch] != 0.0) add_units(my_tile + tap_of(cur_tap, q) * 3 + ch, acc[q][ch]);
				acc[q][ch] = 0.0;
			}
	};
	const auto flush_mat = [&] {
#pragma unroll
		for(int ch = 0; ch < 3; ++ch) {
			double v = macc[ch];
			for(int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
			if(lane == 0 && v != 0.0) add_units(mat + size_t(cur_mat) * 3 + ch, v);
			macc[ch] = 0.0;
		}
	};
	for(uint32_t k0 = wave * 64u; k0 < cnt; k0 += kBlock) {  // wave-uniform; no barrier inside
		const bool on = k0 + lane < cnt;
		const uint64_t x = d.sorted[begin + (on ? k0 + lane : k0)];
		const TexelWeights c = texel_weights(d, x);
		const TexelEval e = texel_eval(d, c);
		const uint32_t m = d.gmat[x];
		const float* a = d.albedo + size_t(m) * 3;
		const uint32_t mat0 = uint32_t(__builtin_amdgcn_readfirstlane(int(m)));
		const bool one_mat = __ballot(on && m != mat0) == 0u;
		if(one_mat && mat0 != cur_mat) {
			flush_mat();
			cur_mat = mat0;
		}
		float go[3];
#pragma unroll
		for(int ch = 0; ch < 3; ++ch) {
			const float o = e.fb[ch] * e.fb[ch] * (1.0f - e.k) + e.fin[ch] * e.fin[ch] * e.k;
			const float gs = on ? (o * a[ch] * 0.996f - d.target[x * 3 + ch]) * inv3n : 0.0f;
			go[ch] = gs * a[ch] * 0.996f;
			const float gm = on ? rintf(to_units(gs * o * 0.996f)) : 0.0f;
			if(one_mat && fabsf(gm) < kSmallUnits) macc[ch] += double(gm);
			else if(gm != 0.0f) add_units(mat + size_t(m) * 3 + ch, double(gm));
		}
		*reinterpret_cast<float4*>(&s_b[wave][lane * 4]) = make_float4((1.0f - c.cwx) * (1.0f - c.cwy), c.cwx * (1.0f - c.cwy),
																	  (1.0f - c.cwx) * c.cwy, c.cwx * c.cwy);
#pragma unroll
		for(int ch = 0; ch < 3; ++ch) {
			// d loss / d (the probe's bilinear irradiance); sqrt'(v) taken at s >= 1e-6
			const float df = (1.0f - e.k) * 2.0f * e.fb[ch] * e.inv_fb, dw = e.k * 2.0f * e.fin[ch] * e.inv_w;
			float g[8], most = 0.0f;
#pragma unroll
			for(int p = 0; p < 8; ++p) {
				g[p] = to_units(go[ch] * (df * c.fw[p] + dw * c.w[p]) * 0.5f / fmaxf(e.s[p][ch], 1e-6f));
				most = fmaxf(most, fabsf(g[p]));
			}
			s_t[wave][lane] = on ? (most < kSmallUnits ? c.t00 : c.t00 | kLarge) : kNo;
			float4* dst = reinterpret_cast<float4*>(&s_g[wave][lane * 8]);
			dst[0] = make_float4(g[0], g[1], g[2], g[3]);
			dst[1] = make_float4(g[4], g[5], g[6], g[7]);
			// (the compiler orders these LDS accesses; a wavefront's LDS operations complete in order)
			__builtin_amdgcn_wave_barrier();
			for(uint32_t h = 0; h < 64u && k0 + h < cnt; h += 8u) {
				const uint32_t texel = h + (lane >> 3);
				const uint32_t t00 = s_t[wave][texel];
				const uint32_t tap0 = uint32_t(__builtin_amdgcn_readfirstlane(int(t00))) & ~kLarge;  // the first texel exists
				const float gv = s_g[wave][texel * 8 + i];
				const float4 b4 = *reinterpret_cast<const float4*>(&s_b[wave][texel * 4]);
				const float b[4] = {b4.x, b4.y, b4.z, b4.w};
				if(__ballot(t00 != kNo && t00 != tap0) == 0u) {  // one tap, none large
					if(tap0 != cur_tap) {
						flush_taps();
						cur_tap = tap0;
					}
#pragma unroll
					for(int q = 0; q < 4; ++q) acc[q][ch] += double(rintf(gv * b[q]));  // no texel: gv is 0
				} else if(t00 != kNo) {
#pragma unroll
					for(int q = 0; q < 4; ++q) {
						const float v = rintf(gv * b[q]);
						if(v != 0.0f) add_units(my_tile + tap_of(t00 & ~kLarge, q) * 3 + ch, double(v));
					}
				}
			}
			__builtin_amdgcn_wave_barrier();
		}
	}
	flush_taps();
	flush_mat();
	__syncthreads();
	long long* pt = d.part_tile + size_t(item) * 8 * 192;
	for(uint32_t k = threadIdx.x; k < 8 * 192; k += kBlock) pt[k] = (long long)tile[k];
	long long* pm = d.part_mat_pix + size_t(item) * d.M * 3;
	for(uint32_t k = threadIdx.x; k < d.M * 3; k += kBlock) pm[k] = (long long)mat[k];
}

// One block per probe: sum the partial tiles of the (up to 8) cells whose cage contains the
// probe, fold the border gradients onto the interior texels they copy, scale to float.  Four groups of
// 192 threads share the items (integer sums: any order gives the same; 18 us, 70 us with one group).
__global__ __launch_bounds__(768) void k_probe_grad(DiffArgs d) {
	__shared__ long long part[4][64 * 3];
	__shared__ long long g[64 * 3];
	const uint32_t p = blockIdx.x;
	const uint32_t rx = uint32_t(d.grid.res[0]), ry = uint32_t(d.grid.res[1]);
	const int px = int(p % rx), py = int((p % (rx * ry)) / rx), pz = int(p / (rx * ry));
	const uint32_t grp = threadIdx.x / 192u;
	uint32_t e = threadIdx.x - grp * 192u;  // texel * 3 + channel
	long long s = 0;
	for(int o = 0; o < 8; ++o) {
		const int cx = px - (o & 1), cy = py - ((o >> 1) & 1), cz = pz - ((o >> 2) & 1);
		if(cx < 0 || cy < 0 || cz < 0) continue;
		const uint32_t cell = uint32_t(cx) + rx * (uint32_t(cy) + ry * uint32_t(cz));
		const uint32_t first = d.cell_item_start[cell], last = d.cell_item_start[cell + 1];
#pragma unroll 4
		for(uint32_t it = first + grp; it < last; it += 4u) s += d.part_tile[(size_t(it) * 8 + o) * 192 + e];
	}
	part[grp][e] = s;
	__syncthreads();
	if(grp == 0) g[e] = part[0][e] + part[1][e] + part[2][e] + part[3][e];
	__syncthreads();
	if(grp != 0) e = 192u;  // the rest is one group's
	// border fold (adjoint of probesCopyBorders: dst <- src)
	if(e < 3) {
		const int R = 8;
		auto fold = [&](int dx, int dy, int sx, int sy) { g[(sy * R + sx) * 3 + e] += g[(dy * R + dx) * 3 + e]; };
		fold(0, 0, R - 2, R - 2);
		fold(0, R - 1, R - 2, 1);
		fold(R - 1, 0, 1, R - 2);
		fold(R - 1, R - 1, 1, 1);
		for(int j = 1; j + 1 < R; ++j) {
			fold(0, j, 1, R - 1 - j);
			fold(R - 1, j, R - 2, R - 1 - j);
			fold(j, 0, R - 1 - j, 1);
			fold(j, R - 1, R - 1 - j, R - 2);
		}
	}
	__syncthreads();
	if(e < 36 * 3) {
		const uint32_t t = e / 3, ch = e % 3;
		const int x = int(t % 6) + 1, y = int(t / 6) + 1;
		d.g_T[(size_t(p) * 36 + t) * 3 + ch] = float(double(g[(y * 8 + x) * 3 + ch]) / kFixScale);
	}
}

// One block per probe slot: d loss / d rad_i = (1 - h) sum_t w_ti inv_t dT_t with the weights
// recomputed from the ray directions, then the radiance adjoint into per-material / sun partials.
__global__ __launch_bounds__(kBlock) void k_blend_bwd(DiffArgs d) {
	extern __shared__ unsigned long long lds[];
	unsigned long long* mat = lds;                             // [M][3] then sun[3]
	__shared__ float s_g[36 * 3], s_dir[36 * 3];
	const uint32_t slot = blockIdx.x;
	const uint32_t probe = d.indices[slot];
	for(uint32_t k = threadIdx.x; k < d.M * 3 + 3; k += kBlock) lds[k] = 0ull;
	const float h = d.grid.hysteresis;
	if(threadIdx.x < 36) {
		float tx, ty, tz;
		texel_direction(threadIdx.x, tx, ty, tz);
		s_dir[threadIdx.x * 3] = tx;
		s_dir[threadIdx.x * 3 + 1] = ty;
		s_dir[threadIdx.x * 3 + 2] = tz;
	}
	if(threadIdx.x < 108) {
		const uint32_t t = threadIdx.x / 3;
		s_g[threadIdx.x] = d.g_T[size_t(probe) * 108 + threadIdx.x] * (1.0f - h) * d.inv_sum[t];
	}
	__syncthreads();
	const uint32_t n = d.grid.n;
	double sun[3] = {0.0, 0.0, 0.0};  // every ray adds to these: summed in registers first
	for(uint32_t j = threadIdx.x; j < n; j += kBlock) {
		const float4 dr = d.dirs[d.perm[j]];
		float gr[3] = {0.0f, 0.0f, 0.0f};
		for(int t = 0; t < 36; ++t) {
			const float w = fmaxf(0.0f, s_dir[t * 3] * dr.x + s_dir[t * 3 + 1] * dr.y + s_dir[t * 3 + 2] * dr.z);
			gr[0] += w * s_g[t * 3];
			gr[1] += w * s_g[t * 3 + 1];
			gr[2] += w * s_g[t * 3 + 2];
		}
		const float4* f = d.factors + (size_t(slot) * n + j) * 4;
		const uint32_t m = __float_as_uint(f[0].w);
		if(m == 0xFFFFFFFFu) continue;
		const float4 A = f[1], B = f[2], C = f[3];
		const float* a = d.albedo + size_t(m) * 3;
		const float Av[3] = {A.x, A.y, A.z}, Bv[3] = {B.x, B.y, B.z}, Cv[3] = {C.x, C.y, C.z};
		for(int ch = 0; ch < 3; ++ch) {
			atomicAdd(&mat[m * 3 + ch], (unsigned long long)to_fixed(gr[ch] * (Av[ch] + Bv[ch] * d.sun[ch])));
			const float gs = rintf(to_units(gr[ch] * (Bv[ch] * a[ch] + Cv[ch])));
			if(fabsf(gs) < kSmallUnits) sun[ch] += double(gs);
			else add_units(&mat[d.M * 3 + ch], double(gs));
		}
	}
#pragma unroll
	for(int ch = 0; ch < 3; ++ch) {
		for(int o = 32; o > 0; o >>= 1) sun[ch] += __shfl_xor(sun[ch], o);
		if(__lane_id() == 0) add_units(&mat[d.M * 3 + ch], sun[ch]);
	}
	__syncthreads();
	long long* pr = d.part_mat_ray + size_t(slot) * (d.M * 3 + 3);
	for(uint32_t k = threadIdx.x; k < d.M * 3 + 3; k += kBlock) pr[k] = (long long)mat[k];
}

// Columns (material channels, then the sun's) of the items' and slots' partial sums: workgroup b adds rows
// b, b + kDiffSumBlocks, ... (one row after another, coalesced), then one thread per column adds the
// workgroups' sums.  (One thread per column over every row: 214 us for a full-HD view.)
__global__ __launch_bounds__(kBlock) void k_grad_rows(DiffArgs d) {
	const uint32_t cols = d.M * 3 + 3, items = *d.n_items;
	for(uint32_t k = threadIdx.x; k < cols; k += kBlock) {
		long long s = 0;
		if(k < d.M * 3) {
#pragma unroll 8
			for(uint32_t it = blockIdx.x; it < items; it += kDiffSumBlocks) s += d.part_mat_pix[size_t(it) * d.M * 3 + k];
		}
#pragma unroll 8
		for(uint32_t sl = blockIdx.x; sl < d.slots; sl += kDiffSumBlocks) s += d.part_mat_ray[size_t(sl) * cols + k];
		d.part_rows[size_t(blockIdx.x) * cols + k] = s;
	}
}

__global__ void k_grad_final(DiffArgs d) {
	const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
	const uint32_t cols = d.M * 3 + 3;
	if(k >= cols) return;
	long long s = 0;
#pragma unroll 16
	for(uint32_t b = 0; b < kDiffSumBlocks; ++b) s += d.part_rows[size_t(b) * cols + k];
	const float v = float(double(s) / kFixScale) * d.grad_loss[0];
	if(k < d.M * 3) d.g_albedo[k] = v;
	else d.g_sun[k - d.M * 3] = v;
}

inline uint32_t nblocks(uint64_t n, uint32_t b) { return uint32_t((n + b - 1) / b); }

}  // namespace

hipError_t diff_bin(const DiffArgs& d, const DiffBins& b, hipStream_t s) {
	const size_t keys = size_t(d.grid.probe_count) * b.taps;
	hipError_t e;
	if((e = hipMemsetAsync(b.key_count, 0, keys * 4, s)) != hipSuccess) return e;
	if((e = hipMemsetAsync(b.cursor, 0, keys * 4, s)) != hipSuccess) return e;
	hipLaunchKernelGGL(k_cells, dim3(nblocks(d.N, 256)), dim3(256), 0, s, d, b.taps, b.key_of, b.key_count);
	hipLaunchKernelGGL(k_items, dim3(1), dim3(1024), 0, s, d, b.taps, b.key_count, b.key_start, b.cell_item_start,
					   b.item_begin, b.item_count, b.n_items);
	hipLaunchKernelGGL(k_scatter, dim3(nblocks(d.N, 256)), dim3(256), 0, s, d, b.key_of, b.key_start, b.cursor, b.sorted);
	return hipGetLastError();
}

hipError_t diff_records(const DiffArgs& d, float4* rec, hipStream_t s) {
	hipLaunchKernelGGL(k_records, dim3(nblocks(d.N, kBlock)), dim3(kBlock), 0, s, d, rec);
	return hipGetLastError();
}

hipError_t diff_radiance(const DiffArgs& d, hipStream_t s) {
	hipLaunchKernelGGL(k_radiance, dim3(nblocks(d.rays, 256)), dim3(256), 0, s, d);
	return hipGetLastError();
}

hipError_t diff_gather_forward(const DiffArgs& d, hipStream_t s) {
	const uint32_t parts = nblocks(d.N, kBlock);
	hipLaunchKernelGGL(k_gather_fwd, dim3(parts), dim3(kBlock), 0, s, d);
	hipLaunchKernelGGL(k_loss, dim3(1), dim3(1024), 0, s, d, parts);
	return hipGetLastError();
}

hipError_t diff_backward(const DiffArgs& d, hipStream_t s) {
	const size_t lds1 = (8 * 192 + size_t(d.M) * 3) * sizeof(unsigned long long);
	hipLaunchKernelGGL(k_gather_bwd, dim3(d.max_items), dim3(kBlock), lds1, s, d);
	hipLaunchKernelGGL(k_probe_grad, dim3(d.grid.probe_count), dim3(768), 0, s, d);
	const size_t lds2 = (size_t(d.M) * 3 + 3) * sizeof(unsigned long long);
	hipLaunchKernelGGL(k_blend_bwd, dim3(d.slots), dim3(kBlock), lds2, s, d);
	hipLaunchKernelGGL(k_grad_rows, dim3(kDiffSumBlocks), dim3(kBlock), 0, s, d);
	hipLaunchKernelGGL(k_grad_final, dim3(nblocks(d.M * 3 + 3, 64)), dim3(64), 0, s, d);
	return hipGetLastError();
}

}  // namespace ddgi
