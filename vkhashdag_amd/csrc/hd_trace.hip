// hd_trace.hip -- ESVO ray traversal of the device pool (shader/src/trace.frag:69-402 and
// include/hashdag/NodePoolTraversal.hpp:93-256).
//
// The march keeps trace.frag's fp32 operation order (the library is built with
// -ffp-contract=off and correctly rounded division / sqrt) so hits are bit-identical to the
// CPU transliteration. The ESVO march follows Laine & Karras, "Efficient Sparse Voxel Octrees"
// (I3D 2010), as restated in trace.frag, which carries the BSD-3 notice reproduced below; it
// applies to `march` in this file.
//
// Launch: one workgroup per pixel tile (8x8 or 16x16, from the tuning); the per-scale parent stack
// lives in LDS laid out [scale][thread] so a wavefront's stack accesses hit 64 consecutive banks.
// The march is bound by VALU issue (about 90 vector instructions per wave iteration, with the
// descend / advance / pop paths serialised under divergence), not by memory: fewer instructions
// per iteration and a shorter grid tail are what speed it up.
/*
 *  Copyright (c) 2009-2011, NVIDIA Corporation
 *  All rights reserved.
 *
 *  Redistribution and use in source and binary forms, with or without
 *  modification, are permitted provided that the following conditions are met:
 *      * Redistributions of source code must retain the above copyright
 *        notice, this list of conditions and the following disclaimer.
 *      * Redistributions in binary form must reproduce the above copyright
 *        notice, this list of conditions and the following disclaimer in the
 *        documentation and/or other materials provided with the distribution.
 *      * Neither the name of NVIDIA Corporation nor the
 *        names of its contributors may be used to endorse or promote products
 *        derived from this software without specific prior written permission.
 *
 *  THIS SOFTWARE IS PROVIDED BY THE COPYRIGHT HOLDERS AND CONTRIBUTORS "AS IS" AND
 *  ANY EXPRESS OR IMPLIED WARRANTIES, INCLUDING, BUT NOT LIMITED TO, THE IMPLIED
 *  WARRANTIES OF MERCHANTABILITY AND FITNESS FOR A PARTICULAR PURPOSE ARE
 *  DISCLAIMED. IN NO EVENT SHALL <COPYRIGHT HOLDER> BE LIABLE FOR ANY
 *  DIRECT, INDIRECT, INCIDENTAL, SPECIAL, EXEMPLARY, OR CONSEQUENTIAL DAMAGES
 *  (INCLUDING, BUT NOT LIMITED TO, PROCUREMENT OF SUBSTITUTE GOODS OR SERVICES;
 *  LOSS OF USE, DATA, OR PROFITS; OR BUSINESS INTERRUPTION) HOWEVER CAUSED AND
 *  ON ANY THEORY OF LIABILITY, WHETHER IN CONTRACT, STRICT LIABILITY, OR TORT
 *  (INCLUDING NEGLIGENCE OR OTHERWISE) ARISING IN ANY WAY OUT OF THE USE OF THIS
 *  SOFTWARE, EVEN IF ADVISED OF THE POSSIBILITY OF SUCH DAMAGE.
 */

#include "hd_internal.hpp"

#include <cmath>
#include <mutex>

namespace hd {

constexpr u32 kStack = 23;  // STACK_SIZE, fraction bits of float (trace.frag:52-54)
using u8 = unsigned char;
// Workgroup of the beam and traversal kernels: one wavefront, so that a few rays spread over the most CUs (and
// their L1s; 1M rays 404 -> 397 us, eight beam views 1093 -> 1086 us against 256 threads).
constexpr u32 kThreads = 64;
// The frame kernel's pixel tile (workgroup) is kT x kT, kT in {8, 16}, picked by the tuning.
constexpr u32 kMaxIter = 1u << 16;

__device__ inline float fmx(float a, float b) { return a < b ? b : a; } // std::max / GLSL max order
__device__ inline float fmn(float a, float b) { return b < a ? b : a; }
__device__ inline u32 f2u(float f) { return __float_as_uint(f); }
__device__ inline float u2f(u32 u) { return __uint_as_float(u); }
// DAG_GetLeafFirstChildBits (trace.frag:56-67): bit i of the result = (byte i of w0, w1 is not 0),
// i < 8. Bit 7 of each byte is set by the byte's top bit or by a carry out of its low 7 bits (no
// carry crosses bytes); two byte dot products with the weights 2^i add the eight flags, times 128.
__device__ inline u32 nonzero_bytes8(u32 w0, u32 w1) {
	const u32 t0 = (((w0 & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | w0) & 0x80808080u;
	const u32 t1 = (((w1 & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | w1) & 0x80808080u;
	return __builtin_amdgcn_udot4(t1, 0x80402010u, __builtin_amdgcn_udot4(t0, 0x08040201u, 0u, false), false) >> 7u;
}

struct MarchOut {
	bool hit;
	u32 vox[3], vox_size, iter;
	float hit_pos[3], norm[3];
	float t, scale; // t_min and scale_exp2 where the march stopped (beam.frag's outputs)
	// NodePoolTraversal result: clamp(o + t_min * d, cube) - 1 (valid when hit)
	float pick[3];
};

// A node as the march enters it at a scale: the pointer and the 8 child bits. Below the leaf scale
// the pointer is the leaf's byte, which is its child bits too. Inner nodes and leaves take one load
// path (word 1 exists for both: a leaf's second mask word, an inner node's first child).
template <bool kCount>
__device__ inline uint2 march_node(const u32 *__restrict__ W, u32 ptr, bool at_leaf, u32 &reads) {
	const u32 w0 = W[(u64)ptr], w1 = W[(u64)ptr + 1u];
	if (kCount)
		reads += at_leaf ? 2 : 1;
	return make_uint2(ptr, at_leaf ? nonzero_bytes8(w0, w1) : w0);
}

// DAG_RayMarch (trace.frag:69-270). stack: LDS base for this thread, stride = blockDim.
// kLod: the LOD cut-off is on (a finite proj_factor; without it scale_exp2 * inf is never below t).
// kCount: also count the pool words the march reads (reads += ...), for the algorithmic-bytes pass.
//
// The position is kept as the bits of its three floats: they stay multiples of the current cube size
// in [1, 2), so adding a cube is adding its bit, the child's index is that bit of each coordinate, and
// the bits that a step back changes say whether it leaves the parent (a bit above the cube's changed)
// and up to which scale (the highest one). A step out of the root borrows from the exponent: bit 23.
// A stack entry holds the node's child bits beside its pointer, so a pop reads no pool word: the
// chain of a ray that goes from empty cube to empty cube is LDS and registers.
// 1M incoherent rays on a 4096^3 terrain: 440 -> 397 us, a 1080p frame with shadows 439 -> 402 us (vector
// instructions 2.23e8 -> 1.85e8, LDS kept small enough for 32 waves a CU: the bits are bytes).
template <bool kCount, bool kLod>
__device__ inline MarchOut march(const u32 *__restrict__ W, u32 root, u32 leaf_level, float proj_factor,
                                 float proj_bias, float ox, float oy, float oz, float dx, float dy, float dz,
                                 u32 *stack, u8 *bits, u32 stride, u32 &reads) {
	MarchOut out;
	out.hit = false;
	out.iter = 0;
	out.vox_size = 0;
	out.t = 0.0f;
	out.scale = 0.0f;
	for (int i = 0; i < 3; ++i)
		out.vox[i] = 0, out.hit_pos[i] = 0.0f, out.norm[i] = 0.0f, out.pick[i] = 0.0f;
	if (root == kNull)
		return out;
	ox += 1.0f, oy += 1.0f, oz += 1.0f;
	const float eps = u2f((127u - kStack) << 23u);
	dx = fabsf(dx) > eps ? dx : (dx >= 0 ? eps : -eps);
	dy = fabsf(dy) > eps ? dy : (dy >= 0 ? eps : -eps);
	dz = fabsf(dz) > eps ? dz : (dz >= 0 ? eps : -eps);
	const float tcx = 1.0f / -fabsf(dx), tcy = 1.0f / -fabsf(dy), tcz = 1.0f / -fabsf(dz);
	float tbx = tcx * ox, tby = tcy * oy, tbz = tcz * oz;
	u32 oct = 0;
	if (dx > 0.0f)
		oct ^= 1u, tbx = 3.0f * tcx - tbx;
	if (dy > 0.0f)
		oct ^= 2u, tby = 3.0f * tcy - tby;
	if (dz > 0.0f)
		oct ^= 4u, tbz = 3.0f * tcz - tbz;
	// A NaN on the x axis makes t_min NaN: such a ray enters no node and ends without a result. A NaN
	// on another axis never wins a comparison below, and fminf passes over it as the comparisons do.
	if (tbx != tbx)
		return out;
	float t_min = fmx(fmx(2.0f * tcx - tbx, 2.0f * tcy - tby), 2.0f * tcz - tbz);
	float t_max = fmn(fmn(tcx - tbx, tcy - tby), tcz - tbz);
	float h = t_max;
	t_min = fmx(t_min, 0.0f);
	t_max = fmn(t_max, 1.0f);
	constexpr u32 kOne = 127u << 23u; // 1.0f
	u32 scale = kStack - 1, cube = 1u << (kStack - 1);
	u32 px = kOne, py = kOne, pz = kOne;
	if (1.5f * tcx - tbx > t_min)
		px |= cube;
	if (1.5f * tcy - tby > t_min)
		py |= cube;
	if (1.5f * tcz - tbz > t_min)
		pz |= cube;
	float scale_exp2 = 0.5f;
	const u32 leaf_scale = kStack - leaf_level;
	uint2 node = march_node<kCount>(W, root, scale == leaf_scale, reads);
	u32 iter = 1;
	// A valid ray takes at most a few thousand steps; the cap only guards the device against a
	// malformed pool (it is never reached by the parity cases).
	for (;; ++iter) {
		if (iter > kMaxIter)
			return out;
		const float tx = u2f(px) * tcx - tbx, ty = u2f(py) * tcy - tby, tz = u2f(pz) * tcz - tbz;
		const float tc_max = fminf(fminf(tx, ty), tz);
		const u32 child = (((px >> scale) & 1u) | (((py >> scale) & 1u) << 1u) | (((pz >> scale) & 1u) << 2u)) ^ oct;
		if (((node.y >> child) & 1u) != 0u && t_min <= t_max) {
			if (scale < leaf_scale || (kLod && scale_exp2 * proj_factor < tc_max + proj_bias))
				break;
			if (tc_max < h) {
				stack[(scale - leaf_scale) * stride] = node.x;
				bits[(scale - leaf_scale) * stride] = (u8)node.y;
			}
			h = tc_max;
			if (kCount)
				reads += 1;
			// one load for both node kinds: an inner node's child pointer, or the leaf word holding the
			// child's byte
			const bool inner = scale > leaf_scale;
			const u32 below = (u32)__builtin_popcount(node.y & ((1u << child) - 1u));
			const u32 w = W[(u64)node.x + (inner ? below + 1u : child >> 2u)];
			--scale;
			cube >>= 1u;
			scale_exp2 *= 0.5f;
			const float cx = scale_exp2 * tcx + tx, cy = scale_exp2 * tcy + ty, cz = scale_exp2 * tcz + tz;
			px |= cx > t_min ? cube : 0u;
			py |= cy > t_min ? cube : 0u;
			pz |= cz > t_min ? cube : 0u;
			if (inner)
				node = march_node<kCount>(W, w, scale == leaf_scale, reads);
			else
				node.x = node.y = (w >> ((child & 3u) << 3u)) & 0xFFu;
		} else {
			const u32 qx = px - (tx <= tc_max ? cube : 0u), qy = py - (ty <= tc_max ? cube : 0u),
			          qz = pz - (tz <= tc_max ? cube : 0u);
			const u32 diff = (px ^ qx) | (py ^ qy) | (pz ^ qz);
			px = qx, py = qy, pz = qz;
			t_min = tc_max;
			if (diff >= 2u * cube) {
				scale = 31u - (u32)__builtin_clz(diff);
				if (scale >= kStack)
					break;
				cube = 1u << scale;
				scale_exp2 = u2f((scale - kStack + 127u) << 23u);
				node.x = stack[(scale - leaf_scale) * stride];
				node.y = bits[(scale - leaf_scale) * stride];
				px &= 0u - cube, py &= 0u - cube, pz &= 0u - cube;
				h = 0.0f;
			}
		}
	}
	const float fx = u2f(px), fy = u2f(py), fz = u2f(pz);
	// normal / voxel / hit position (trace.frag:223-258)
	float ex = tcx * (fx + scale_exp2) - tbx, ey = tcy * (fy + scale_exp2) - tby, ez = tcz * (fz + scale_exp2) - tbz;
	float n[3];
	if (ex > ey && ex > ez)
		n[0] = -1, n[1] = 0, n[2] = 0;
	else if (ey > ez)
		n[0] = 0, n[1] = -1, n[2] = 0;
	else
		n[0] = 0, n[1] = 0, n[2] = -1;
	if ((oct & 1u) == 0u)
		n[0] = -n[0];
	if ((oct & 2u) == 0u)
		n[1] = -n[1];
	if ((oct & 4u) == 0u)
		n[2] = -n[2];
	const u32 voxel_level = leaf_level + 1u, voxel_scale = kStack - voxel_level;
	const bool ok = scale < kStack && t_min <= t_max;
	out.iter = iter;
	out.t = t_min;
	out.scale = scale_exp2;
	if (!ok) { // a miss reports zeros (trace.frag leaves them unused)
		for (int i = 0; i < 3; ++i)
			out.vox[i] = 0, out.hit_pos[i] = 0.0f, out.norm[i] = 0.0f, out.pick[i] = 0.0f;
		out.vox_size = 0;
		return out;
	}
	u32 vs = 1u << (scale - voxel_scale);
	float pp[3] = {fx, fy, fz}, oo[3] = {ox, oy, oz}, dd[3] = {dx, dy, dz};
	for (int i = 0; i < 3; ++i) {
		u32 v = (f2u(pp[i]) & 0x7FFFFFu) >> voxel_scale;
		if (oct & (1u << i))
			v = (1u << voxel_level) - vs - v;
		out.vox[i] = v;
		float vmin = u2f((v << voxel_scale) | (127u << 23u)), vmax = u2f(((v + vs) << voxel_scale) | (127u << 23u));
		float hp = fmn(fmx(oo[i] + t_min * dd[i], vmin), vmax);
		if (n[i] != 0)
			hp = n[i] > 0 ? vmax + eps * 2 : vmin - eps;
		out.hit_pos[i] = hp - 1.0f;
		out.norm[i] = n[i];
		// NodePoolTraversal: undo mirroring of pos, clamp(o + t d, pos, pos + scale) - 1
		float q = pp[i];
		if (oct & (1u << i))
			q = 3.0f - scale_exp2 - q;
		out.pick[i] = fmn(fmx(oo[i] + t_min * dd[i], q), q + scale_exp2) - 1.0f;
	}
	out.vox_size = vs;
	out.iter = iter;
	out.hit = ok;
	return out;
}

struct RGB {
	float r, g, b;
};
__device__ inline RGB unorm8(u32 c) {
	return {float(c & 0xFFu) / 255.0f, float((c >> 8) & 0xFFu) / 255.0f, float((c >> 16) & 0xFFu) / 255.0f};
}
__device__ inline RGB rgb565(u32 c) {
	return {float(c & 0x1Fu) / 31.0f, float((c >> 5) & 0x3Fu) / 63.0f, float((c >> 11) & 0x1Fu) / 31.0f};
}
// Color_GetLeafColor (trace.frag:304-349)
template <bool kCount>
__device__ inline RGB leaf_color(const u32 *__restrict__ L, u32 idx, u32 x, u32 y, u32 z, u32 &reads) {
	u32 macro_cnt = L[idx + 1u], block_cnt = L[idx + 2u];
	if (kCount)
		reads += 5; // counts, macro pair, next macro
	u32 macro_offset = idx + 4u, block_offset = macro_offset + (macro_cnt << 1u);
	u32 weight_offset = block_offset + (block_cnt << 1u);
	u32 vox_id = morton3(x, y, z);
	u32 macro_id = vox_id >> 14u;
	if (macro_id >= macro_cnt)
		return {0, 0, 0};
	u32 mx = L[macro_offset + (macro_id << 1u)], my = L[(macro_offset + (macro_id << 1u)) | 1u];
	block_offset += mx << 1u;
	block_cnt = macro_id + 1u < macro_cnt ? L[macro_offset + ((macro_id + 1u) << 1u)] - mx : block_cnt - mx;
	vox_id &= 0x3FFFu;
	if (block_cnt == 0u)
		return {0, 0, 0};
	for (u32 s = 0; s <= 14u && block_cnt != 0u; ++s) {
		u32 step = block_cnt >> 1u;
		if (kCount)
			reads += 1;
		if ((L[(block_offset + (step << 1u)) | 1u] >> 18u) <= vox_id) {
			block_cnt -= (step + 1u);
			block_offset += (step + 1u) << 1u;
		} else
			block_cnt = step;
	}
	block_offset -= 2u;
	u32 bx = L[block_offset], by = L[block_offset | 1u];
	u32 bpw = (by >> 16u) & 0x3u;
	if (kCount)
		reads += 2 + (bpw ? 2 : 0);
	if (bpw == 0u)
		return unorm8(bx);
	vox_id -= (by >> 18u);
	u32 bit_id = my + (by & 0xFFFFu) + vox_id * bpw;
	u32 bo = bit_id & 31u;
	u32 w = L[weight_offset + (bit_id >> 5u)] >> bo;
	if (bo + bpw <= 32u)
		w &= (1u << bpw) - 1u;
	else
		w = w | ((L[weight_offset + (bit_id >> 5u) + 1u] & ((1u << (bo + bpw - 32u)) - 1u)) << (32u - bo));
	float a = float(w) / float((1u << bpw) - 1u);
	RGB p = rgb565(bx), q = rgb565(bx >> 16u);
	return {p.r * (1.0f - a) + q.r * a, p.g * (1.0f - a) + q.g * a, p.b * (1.0f - a) + q.b * a};
}
// Color_Fetch (trace.frag:351-364)
template <bool kCount>
__device__ inline RGB color_fetch(const u32 *__restrict__ CN, const u32 *__restrict__ CL, u32 root, u32 voxel_level,
                                  u32 leaf_level, u32 x, u32 y, u32 z, u32 &reads) {
	u32 ptr = root;
	for (u32 l = 0; l < leaf_level; ++l) {
		u32 tag = ptr >> 30u, data = ptr & 0x3FFFFFFFu;
		if (tag != 0)
			return unorm8(data);
		u32 sh = voxel_level - 1u - l;
		if (kCount)
			reads += 1;
		ptr = CN[((u64)ptr << 3u) | ((x >> sh) & 1u) | (((y >> sh) & 1u) << 1u) | (((z >> sh) & 1u) << 2u)];
	}
	u32 tag = ptr >> 30u, data = ptr & 0x3FFFFFFFu;
	if (tag == 2u) {
		u32 m = (1u << (voxel_level - leaf_level)) - 1u;
		return leaf_color<kCount>(CL, data, x & m, y & m, z & m, reads);
	}
	return unorm8(data);
}

struct TraceArgs {
	const u32 *words, *cnodes, *cleaves;
	u32 root, color_root, leaf_level, color_leaf_level;
	const hd_view *views;
	const u32 *tile_start; // prefix of tiles per view (n_views + 1)
	u32 n_views;
	u32 *rgba, *records;
	unsigned long long *counters; // [primary rays, shadow rays, march iterations, words read] (may be null)
	const u32 *roots;             // if set: (root, color root) read from the device (graph replays)
	const float *beam;            // beam images of the HD_TRACE_BEAM views (may be null)
	const u32 *beam_start;        // prefix of beam texels per view (n_views + 1)
};

// Beam prepass (beam.frag:59-223, BeamPass.cpp:9-111): one coarse ray per 8x8-pixel block through
// the block's centre on the ceil(W/8) x ceil(H/8) beam image, LOD with a block's projection factor
// (the view's / 8); the block's value is max(t - cube size, 0) where the march stopped, +inf on a
// miss. The trace starts each pixel at the smallest of the 2x2 beam texels around it, times 0.98
// (a MIN-reduction bilinear fetch, trace.frag:384-390), with that distance as the LOD bias.
constexpr u32 kBeamBlock = 8;
__device__ inline u32 beam_dim(u32 n) { return (n + kBeamBlock - 1u) / kBeamBlock; }
__device__ inline float beam_sample(const float *__restrict__ B, u32 Wb, u32 Hb, float u, float v) {
	float x = u * float(Wb) - 0.5f, y = v * float(Hb) - 0.5f;
	int x0 = (int)floorf(x), y0 = (int)floorf(y);
	auto cl = [](int a, u32 n) { return (u32)min(max(a, 0), (int)n - 1); };
	u32 xa = cl(x0, Wb), xb = cl(x0 + 1, Wb), ya = cl(y0, Hb), yb = cl(y0 + 1, Hb);
	return fminf(fminf(B[ya * Wb + xa], B[ya * Wb + xb]), fminf(B[yb * Wb + xa], B[yb * Wb + xb])) * 0.98f;
}

__device__ inline u32 q8(float x) { return (u32)(fmn(fmx(x, 0.0f), 1.0f) * 255.0f + 0.5f); }

template <bool kCount, u32 kT> __global__ void __launch_bounds__(kT *kT) k_trace(TraceArgs A) {
	constexpr u32 kTT = kT * kT;
	extern __shared__ u32 stack_lds[]; // node levels x kTT words, then as many bytes (trace_lds_bytes)
	// view of this tile (binary search over the tile prefix); a fixed grid may run past the last tile
	u32 tile = blockIdx.x, lo = 0, hi = A.n_views;
	if (tile >= A.tile_start[A.n_views])
		return;
	const u32 root = A.roots ? A.roots[0] : A.root, color_root = A.roots ? A.roots[1] : A.color_root;
	while (hi - lo > 1) {
		u32 mid = (lo + hi) >> 1;
		if (A.tile_start[mid] <= tile)
			lo = mid;
		else
			hi = mid;
	}
	const hd_view V = A.views[lo];
	// Tiles go out in reverse raster order, bottom row first: a view's lower rows usually see the
	// near ground, whose marches are the longest, so they start first and the short sky tiles fill
	// the end of the grid (longest-first order shortens its tail).
	u32 t = A.tile_start[lo + 1] - 1u - tile;
	u32 tiles_x = (V.width + kT - 1) / kT;
	u32 px = (t % tiles_x) * kT + (threadIdx.x % kT), py = (t / tiles_x) * kT + (threadIdx.x / kT);
	if (px >= V.width || py >= V.height)
		return;
	u32 *stack = stack_lds + threadIdx.x;
	u8 *bits = (u8 *)(stack_lds + A.leaf_level * kTT) + threadIdx.x;
	// Camera_GenRay (trace.frag:366-370), gl_FragCoord at pixel centres, origin top-left
	const float u = (float(px) + 0.5f) / float(V.width), w = (float(py) + 0.5f) / float(V.height);
	const float cx = u * 2.0f - 1.0f, cy = w * 2.0f - 1.0f;
	float dx = V.look[0] - V.side[0] * cx - V.up[0] * cy, dy = V.look[1] - V.side[1] * cx - V.up[1] * cy,
	      dz = V.look[2] - V.side[2] * cx - V.up[2] * cy;
	float len = sqrtf(dx * dx + dy * dy + dz * dz);
	dx = dx / len, dy = dy / len, dz = dz / len;
	u32 reads = 0;
	MarchOut h;
	if ((V.flags & HD_TRACE_BEAM) && A.beam) {
		const float t0 = beam_sample(A.beam + A.beam_start[lo], beam_dim(V.width), beam_dim(V.height), u, w);
		if (isinf(t0)) { // the block's coarse ray missed: so does this pixel
			h.hit = false;
			h.iter = 0, h.vox_size = 0, h.t = 0.0f, h.scale = 0.0f;
			for (int i = 0; i < 3; ++i)
				h.vox[i] = 0, h.hit_pos[i] = 0.0f, h.norm[i] = 0.0f, h.pick[i] = 0.0f;
		} else
			h = march<kCount, true>(A.words, root, A.leaf_level, V.proj_factor, t0, V.pos[0] + t0 * dx, V.pos[1] + t0 * dy,
			                  V.pos[2] + t0 * dz, dx, dy, dz, stack, bits, kTT, reads);
	} else
		h = march<kCount, true>(A.words, root, A.leaf_level, V.proj_factor, 0.0f, V.pos[0], V.pos[1], V.pos[2], dx, dy,
		                  dz, stack, bits, kTT, reads);
	u32 iters = h.iter;
	float lx = 4.0f, ly = 5.0f, lz = 3.0f;
	float ll = sqrtf(lx * lx + ly * ly + lz * lz);
	lx = lx / ll, ly = ly / ll, lz = lz / ll;
	bool shadow = false;
	if (h.hit && (V.flags & HD_TRACE_SHADOW)) {
		MarchOut s = march<kCount, false>(A.words, root, A.leaf_level, __builtin_inff(), 0.0f, h.hit_pos[0], h.hit_pos[1],
		                           h.hit_pos[2], lx, ly, lz, stack, bits, kTT, reads);
		shadow = s.hit;
		iters += s.iter;
	}
	float r = 0, g = 0, b = 0;
	if (h.hit) {
		float nd = h.norm[0] * lx + h.norm[1] * ly + h.norm[2] * lz;
		float diffuse = shadow ? 0.5f : fmx(nd, 0.0f) * 0.5f + 0.5f;
		RGB c = color_fetch<kCount>(A.cnodes, A.cleaves, color_root, A.leaf_level + 1u, A.color_leaf_level,
		                            h.vox[0], h.vox[1], h.vox[2], reads);
		r = diffuse * c.r, g = diffuse * c.g, b = diffuse * c.b;
	}
	u64 o = V.out_offset + (u64)py * V.width + px;
	A.rgba[o] = q8(r) | (q8(g) << 8) | (q8(b) << 16) | (255u << 24);
	if (A.records && (V.flags & HD_TRACE_RECORDS)) {
		u32 *rec = A.records + o * 12u;
		rec[0] = h.vox[0], rec[1] = h.vox[1], rec[2] = h.vox[2];
		rec[3] = h.vox_size | (h.hit ? 0x80000000u : 0u);
		rec[4] = f2u(h.hit_pos[0]), rec[5] = f2u(h.hit_pos[1]), rec[6] = f2u(h.hit_pos[2]);
		rec[7] = f2u(h.norm[0]), rec[8] = f2u(h.norm[1]), rec[9] = f2u(h.norm[2]);
		rec[10] = h.iter;
		rec[11] = shadow ? 1u : 0u;
	}
	if (kCount && A.counters) {
		atomicAdd(&A.counters[0], 1ull);
		atomicAdd(&A.counters[1], h.hit && (V.flags & HD_TRACE_SHADOW) ? 1ull : 0ull);
		atomicAdd(&A.counters[2], (unsigned long long)iters);
		atomicAdd(&A.counters[3], (unsigned long long)reads);
	}
}

// One thread per beam texel of every HD_TRACE_BEAM view (views without the flag have no texels).
__global__ void __launch_bounds__(kThreads) k_beam(TraceArgs A, float *__restrict__ beam) {
	extern __shared__ u32 stack_lds[];
	const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= A.beam_start[A.n_views])
		return;
	const u32 root = A.roots ? A.roots[0] : A.root;
	u32 lo = 0, hi = A.n_views;
	while (hi - lo > 1) {
		u32 mid = (lo + hi) >> 1;
		if (A.beam_start[mid] <= i)
			lo = mid;
		else
			hi = mid;
	}
	const hd_view V = A.views[lo];
	const u32 Wb = beam_dim(V.width), Hb = beam_dim(V.height), t = i - A.beam_start[lo];
	const u32 bx = t % Wb, by = t / Wb;
	float cx = (float(bx) + 0.5f) / float(Wb), cy = (float(by) + 0.5f) / float(Hb);
	cx = cx * 2.0f - 1.0f;
	cy = cy * 2.0f - 1.0f;
	float dx = V.look[0] - V.side[0] * cx - V.up[0] * cy, dy = V.look[1] - V.side[1] * cx - V.up[1] * cy,
	      dz = V.look[2] - V.side[2] * cx - V.up[2] * cy;
	float len = sqrtf(dx * dx + dy * dy + dz * dz);
	dx = dx / len, dy = dy / len, dz = dz / len;
	u32 reads = 0;
	u32 *stack = stack_lds + threadIdx.x;
	u8 *bits = (u8 *)(stack_lds + A.leaf_level * kThreads) + threadIdx.x;
	MarchOut h = march<false, true>(A.words, root, A.leaf_level, V.proj_factor * (1.0f / float(kBeamBlock)), 0.0f, V.pos[0],
	                          V.pos[1], V.pos[2], dx, dy, dz, stack, bits, kThreads, reads);
	beam[i] = h.hit ? fmaxf(h.t - h.scale, 0.0f) : __builtin_inff();
}

__global__ void __launch_bounds__(kThreads) k_traversal(const u32 *__restrict__ W, u32 root, u32 leaf_level,
                                                         const float *__restrict__ o, const float *__restrict__ d,
                                                         u64 n, float *__restrict__ out) {
	extern __shared__ u32 stack_lds[];
	u64 i = (u64)blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	u32 reads = 0;
	u32 *stack = stack_lds + threadIdx.x;
	u8 *bits = (u8 *)(stack_lds + leaf_level * kThreads) + threadIdx.x;
	MarchOut h = march<false, false>(W, root, leaf_level, __builtin_inff(), 0.0f, o[3 * i], o[3 * i + 1], o[3 * i + 2],
	                          d[3 * i], d[3 * i + 1], d[3 * i + 2], stack, bits, kThreads, reads);
	out[4 * i] = h.hit ? h.pick[0] : 0.0f;
	out[4 * i + 1] = h.hit ? h.pick[1] : 0.0f;
	out[4 * i + 2] = h.hit ? h.pick[2] : 0.0f;
	out[4 * i + 3] = h.hit ? 1.0f : 0.0f;
}

// A call's views, tile prefix and beam prefix for the trace kernels: up to kPutViews views go to the device as
// the arguments of a one-workgroup kernel; more take a copy each. (A small copy from pageable memory holds the
// host for about 10 us: a 255 x 201 frame 107 -> 102 us.)
constexpr u32 kPutViews = 16;
struct PutViews {
	u32 views[kPutViews * sizeof(hd_view) / 4], tiles[kPutViews + 1], beams[kPutViews + 1];
};
__global__ void __launch_bounds__(64) k_put_views(PutViews a, u32 n, u32 *__restrict__ views, u32 *__restrict__ tiles,
                                                  u32 *__restrict__ beams) {
	for (u32 i = threadIdx.x; i < n * (u32)(sizeof(hd_view) / 4); i += 64)
		views[i] = a.views[i];
	for (u32 i = threadIdx.x; i <= n; i += 64) {
		tiles[i] = a.tiles[i];
		if (beams)
			beams[i] = a.beams[i];
	}
}
static int put_views(hipStream_t s, const hd_view *views, const u32 *tiles, const u32 *beams, u32 n, hd_view *dv, u32 *dt,
                     u32 *db) {
	if (n <= kPutViews) {
		PutViews a;
		std::memcpy(a.views, views, n * sizeof(hd_view));
		std::memcpy(a.tiles, tiles, (n + 1) * 4);
		std::memcpy(a.beams, beams, (n + 1) * 4);
		k_put_views<<<1, 64, 0, s>>>(a, n, (u32 *)dv, dt, db);
		HD_TRY(hipGetLastError());
		return HD_OK;
	}
	HD_TRY(hipMemcpyAsync(dv, views, n * sizeof(hd_view), hipMemcpyHostToDevice, s));
	HD_TRY(hipMemcpyAsync(dt, tiles, (n + 1) * 4, hipMemcpyHostToDevice, s));
	if (db)
		HD_TRY(hipMemcpyAsync(db, beams, (n + 1) * 4, hipMemcpyHostToDevice, s));
	return HD_OK;
}

// The frame kernel at the tuned tile (tiles counted with the same tile by trace_tile_count).
// The march keeps one stack word per node level and thread in LDS (pushes and pops stay at scales
// >= the leaf scale, so the slots are scale - leaf_scale in [0, levels)); sizing the stack to the
// pool's levels rather than the 23 float scales leaves room for more resident waves.
static u32 trace_lds_bytes(u32 levels, u32 threads) { return levels * threads * 5u; }
static void launch_trace(bool count, u32 n_tiles, hipStream_t s, const TraceArgs &A) {
	if (g_tuning.trace_tile == 8) {
		const u32 lds = trace_lds_bytes(A.leaf_level, 64);
		if (count)
			k_trace<true, 8><<<n_tiles, 64, lds, s>>>(A);
		else
			k_trace<false, 8><<<n_tiles, 64, lds, s>>>(A);
	} else {
		const u32 lds = trace_lds_bytes(A.leaf_level, 256);
		if (count)
			k_trace<true, 16><<<n_tiles, 256, lds, s>>>(A);
		else
			k_trace<false, 16><<<n_tiles, 256, lds, s>>>(A);
	}
}
static u32 trace_tile_count(const hd_view &v) {
	const u32 t = g_tuning.trace_tile;
	return div_up(v.width, t) * div_up(v.height, t);
}

int trace_on_stream(Pool &p, hipStream_t s, u32 root, u32 color_root, const hd_view *d_views, const u32 *d_tiles,
                    u32 n_views, u32 n_tiles, u32 *rgba, const u32 *d_roots) {
	TraceArgs A{p.words, p.cnodes, p.cleaves, root,    color_root, p.dc.L, p.dc.color_leaf,
	            d_views, d_tiles,  n_views,   rgba,    nullptr,    nullptr, d_roots, nullptr, nullptr};
	launch_trace(false, n_tiles, s, A);
	HD_TRY(hipGetLastError());
	return HD_OK;
}

} // namespace hd

using namespace hd;

extern "C" int hd_trace(hd_pool *h, uint32_t root, uint32_t color_root, const hd_view *views, uint32_t n_views,
                        uint32_t *rgba, uint32_t *records) {
	if (!h || !views || !n_views || !rgba)
		return set_error("hd_trace: null argument"), HD_ERR_ARG;
	Pool &p = h->p;
	std::vector<u32> tiles(n_views + 1, 0), beams(n_views + 1, 0);
	for (u32 v = 0; v < n_views; ++v) {
		if (!views[v].width || !views[v].height)
			return set_error("hd_trace: empty view"), HD_ERR_ARG;
		if ((views[v].flags & HD_TRACE_RECORDS) && !records)
			return set_error("hd_trace: records requested without a buffer"), HD_ERR_ARG;
		if ((views[v].flags & HD_TRACE_BEAM) && !std::isfinite(views[v].proj_factor))
			return set_error("hd_trace: the beam prepass needs a finite proj_factor (LOD on)"), HD_ERR_ARG;
		tiles[v + 1] = tiles[v] + trace_tile_count(views[v]);
	}
	HD_RET(hd_trace_beam_sizes(views, n_views, beams.data()));
	hd_view *dv;
	u32 *dt, *db = nullptr;
	float *beam = nullptr;
	HD_RET(p.scratch.get<hd_view>("trace_views", n_views, &dv));
	HD_RET(p.scratch.get<u32>("trace_tiles", n_views + 1, &dt));
	if (beams[n_views]) {
		HD_RET(p.scratch.get<u32>("trace_beam_start", n_views + 1, &db));
		HD_RET(p.scratch.get<float>("trace_beam", beams[n_views], &beam));
	}
	HD_RET(put_views(p.stream, views, tiles.data(), beams.data(), n_views, dv, dt, db));
	TraceArgs A{p.words, p.cnodes, p.cleaves, root,   color_root, p.dc.L, p.dc.color_leaf,
	            dv,      dt,       n_views,   rgba, records, nullptr, nullptr, beam, db};
	if (beams[n_views])
		k_beam<<<div_up(beams[n_views], kThreads), kThreads, trace_lds_bytes(p.dc.L, kThreads), p.stream>>>(A, beam);
	launch_trace(false, tiles[n_views], p.stream, A);
	HD_TRY(hipGetLastError());
	HD_TRY(hipStreamSynchronize(p.stream));
	return HD_OK;
}

// Asynchronous variant for timing loops and graph capture: views and the tile prefix already on the
// device (hd_trace_prepare), nothing copied, no synchronisation.
// counters (device u64[4], zeroed by the caller) selects the instrumented variant that also counts
// rays, march iterations and the pool words read (the algorithmic bytes of the frame).
extern "C" int hd_trace_async(hd_pool *h, uint32_t root, uint32_t color_root, const hd_view *d_views,
                              const uint32_t *d_tile_start, uint32_t n_views, uint32_t n_tiles, uint32_t *rgba,
                              uint32_t *records, uint64_t *counters) {
	Pool &p = h->p;
	TraceArgs A{p.words,      p.cnodes, p.cleaves, root, color_root, p.dc.L, p.dc.color_leaf, d_views, d_tile_start,
	            n_views,      rgba,     records,   (unsigned long long *)counters, nullptr, nullptr, nullptr};
	launch_trace(counters != nullptr, n_tiles, p.stream, A);
	HD_TRY(hipGetLastError());
	return HD_OK;
}

extern "C" int hd_trace_beam_sizes(const hd_view *views, uint32_t n_views, uint32_t *beam_start) {
	beam_start[0] = 0;
	for (u32 v = 0; v < n_views; ++v)
		beam_start[v + 1] = beam_start[v] + ((views[v].flags & HD_TRACE_BEAM)
		                                         ? div_up(views[v].width, kBeamBlock) * div_up(views[v].height, kBeamBlock)
		                                         : 0u);
	return HD_OK;
}

// Asynchronous beam prepass + trace: views, tile and beam-texel prefixes already on the device.
extern "C" int hd_trace_beam_async(hd_pool *h, uint32_t root, uint32_t color_root, const hd_view *d_views,
                                   const uint32_t *d_tile_start, const uint32_t *d_beam_start, uint32_t n_views,
                                   uint32_t n_tiles, uint32_t n_beam, float *d_beam, uint32_t *rgba) {
	Pool &p = h->p;
	TraceArgs A{p.words, p.cnodes, p.cleaves, root, color_root, p.dc.L, p.dc.color_leaf, d_views, d_tile_start,
	            n_views, rgba,     nullptr,   nullptr, nullptr, d_beam, d_beam_start};
	if (n_beam)
		k_beam<<<div_up(n_beam, kThreads), kThreads, trace_lds_bytes(p.dc.L, kThreads), p.stream>>>(A, d_beam);
	launch_trace(false, n_tiles, p.stream, A);
	HD_TRY(hipGetLastError());
	return HD_OK;
}

extern "C" int hd_trace_tiles(const hd_view *views, uint32_t n_views, uint32_t *tile_start) {
	tile_start[0] = 0;
	for (u32 v = 0; v < n_views; ++v)
		tile_start[v + 1] = tile_start[v] + trace_tile_count(views[v]);
	return HD_OK;
}

extern "C" int hd_traversal(hd_pool *h, uint32_t root, const float *o, const float *d, uint64_t n, float *out) {
	Pool &p = h->p;
	if (!n)
		return HD_OK;
	k_traversal<<<div_up(n, kThreads), kThreads, trace_lds_bytes(p.dc.L, kThreads), p.stream>>>(p.words, root, p.dc.L, o,
	                                                                                         d, n, out);
	HD_TRY(hipGetLastError());
	HD_TRY(hipStreamSynchronize(p.stream));
	return HD_OK;
}

// A pick: the kernel reads the rays from pinned host memory and writes the hits there. (Three device
// allocations, two copies in and one out took 56 of a one-ray call's 82 us: 26 us without them. Each ray
// crosses the bus once either way.)
extern "C" int hd_traversal_host(hd_pool *h, uint32_t root, const float *o, const float *d, uint64_t n, float *out) {
	if (!h || (n && (!o || !d || !out)))
		return set_error("hd_traversal_host: null argument"), HD_ERR_ARG;
	if (n > kHostRays)
		return set_error("hd_traversal_host: %llu rays, at most %llu", (unsigned long long)n,
		                 (unsigned long long)kHostRays), HD_ERR_CAPACITY;
	Pool &p = h->p;
	std::lock_guard<std::mutex> lock(p.rays_mu);
	float *po = p.h_rays, *pd = po + 3 * kHostRays, *hits = pd + 3 * kHostRays;
	std::memcpy(po, o, n * 12);
	std::memcpy(pd, d, n * 12);
	HD_RET(hd_traversal(h, root, po, pd, n, hits));
	std::memcpy(out, hits, n * 16);
	return HD_OK;
}

// ---------------------------------------------------------------- trace without allocation
// hd_trace for callers that cannot allocate device memory: the staged views, the tile and beam
// prefixes and the beam prepass image live in one file-scope device array instead of the pool's
// scratch. Layout (u32 words): views [0, 64 x 18), tile prefix [1152, 1217), beam prefix
// [1217, 1282), beam image from word 1536 (2^20 floats, 256-byte aligned). Every call on a GPU
// shares that GPU's copy: overlapping calls on one GPU race.
namespace {
constexpr u32 kNoAllocViews = 64;
constexpr u32 kNoAllocBeam = 1u << 20;
constexpr u32 kNoAllocViewWords = kNoAllocViews * (u32)(sizeof(hd_view) / 4);
constexpr u32 kNoAllocBeamOff = 1536;
constexpr u64 kNoAllocWords = kNoAllocBeamOff + (u64)kNoAllocBeam;
static_assert(sizeof(hd_view) % 8 == 0 && kNoAllocViewWords + 2 * (kNoAllocViews + 1) <= kNoAllocBeamOff &&
              kNoAllocBeamOff % 64 == 0);
} // namespace

static __device__ __align__(256) u32 scratch[kNoAllocWords];

namespace {
constexpr int kNoAllocDevices = 64;
std::mutex g_scratch_mu;
u32 *g_scratch_ptr[kNoAllocDevices] = {};

// The device address of `scratch` on the current device, looked up once per device (each GPU holds
// its own copy at its own address; the host-side name is not a device address).
int scratch_address(u32 **out) {
	int dev = 0;
	HD_TRY(hipGetDevice(&dev));
	if (dev < 0 || dev >= kNoAllocDevices)
		return set_error("hd_trace_noalloc: device %d beyond the %d supported", dev, kNoAllocDevices), HD_ERR_DEVICE;
	std::lock_guard<std::mutex> lock(g_scratch_mu);
	if (!g_scratch_ptr[dev]) {
		void *ptr = nullptr;
		HD_TRY(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
		if (!ptr)
			return set_error("hd_trace_noalloc: no device address for the scratch array"), HD_ERR_DEVICE;
		g_scratch_ptr[dev] = static_cast<u32 *>(ptr);
	}
	*out = g_scratch_ptr[dev];
	return HD_OK;
}
} // namespace

extern "C" int hd_trace_noalloc(hd_pool *h, uint32_t root, uint32_t color_root, const hd_view *views,
                                uint32_t n_views, uint32_t *rgba, uint32_t *records) {
	if (!h || !views || !n_views || !rgba)
		return set_error("hd_trace_noalloc: null argument"), HD_ERR_ARG;
	if (n_views > kNoAllocViews)
		return set_error("hd_trace_noalloc: %u views, at most %u", n_views, kNoAllocViews), HD_ERR_CAPACITY;
	Pool &p = h->p;
	u32 tiles[kNoAllocViews + 1], beams[kNoAllocViews + 1];
	tiles[0] = 0;
	u64 n_beam = 0;
	for (u32 v = 0; v < n_views; ++v) {
		if (!views[v].width || !views[v].height)
			return set_error("hd_trace_noalloc: empty view"), HD_ERR_ARG;
		if ((views[v].flags & HD_TRACE_RECORDS) && !records)
			return set_error("hd_trace_noalloc: records requested without a buffer"), HD_ERR_ARG;
		if ((views[v].flags & HD_TRACE_BEAM) && !std::isfinite(views[v].proj_factor))
			return set_error("hd_trace_noalloc: the beam prepass needs a finite proj_factor (LOD on)"), HD_ERR_ARG;
		tiles[v + 1] = tiles[v] + trace_tile_count(views[v]);
		if (views[v].flags & HD_TRACE_BEAM)
			n_beam += (u64)div_up(views[v].width, kBeamBlock) * div_up(views[v].height, kBeamBlock);
	}
	if (n_beam > kNoAllocBeam)
		return set_error("hd_trace_noalloc: %llu beam texels, at most %u", (unsigned long long)n_beam, kNoAllocBeam),
		       HD_ERR_CAPACITY;
	HD_RET(hd_trace_beam_sizes(views, n_views, beams));
	u32 *base = nullptr;
	HD_RET(scratch_address(&base));
	hd_view *dv = reinterpret_cast<hd_view *>(base);
	u32 *dt = base + kNoAllocViewWords, *db = dt + kNoAllocViews + 1;
	float *beam = reinterpret_cast<float *>(base + kNoAllocBeamOff);
	HD_RET(put_views(p.stream, views, tiles, beams, n_views, dv, dt, n_beam ? db : nullptr));
	TraceArgs A{p.words, p.cnodes, p.cleaves, root,   color_root,          p.dc.L,         p.dc.color_leaf,
	            dv,      dt,       n_views,   rgba,   records,             nullptr,        nullptr,
	            n_beam ? beam : nullptr,     n_beam ? db : nullptr};
	if (n_beam)
		k_beam<<<div_up((u32)n_beam, kThreads), kThreads, trace_lds_bytes(p.dc.L, kThreads), p.stream>>>(A, beam);
	launch_trace(false, tiles[n_views], p.stream, A);
	HD_TRY(hipGetLastError());
	// the host arrays above are read by the copies: wait before they go out of scope
	HD_TRY(hipStreamSynchronize(p.stream));
	return HD_OK;
}

// Event timing on the pool stream: hd_timer_begin records a start event, hd_timer_end records an
// end event, waits for it and returns the elapsed milliseconds between the two.
namespace {
hipEvent_t g_ev0 = nullptr, g_ev1 = nullptr;
}
extern "C" int hd_timer_begin(hd_pool *h) {
	if (!g_ev0) {
		HD_TRY(hipEventCreate(&g_ev0));
		HD_TRY(hipEventCreate(&g_ev1));
	}
	HD_TRY(hipEventRecord(g_ev0, h->p.stream));
	return HD_OK;
}
extern "C" int hd_timer_end(hd_pool *h, float *ms) {
	HD_TRY(hipEventRecord(g_ev1, h->p.stream));
	HD_TRY(hipEventSynchronize(g_ev1));
	HD_TRY(hipEventElapsedTime(ms, g_ev0, g_ev1));
	return HD_OK;
}
