// hd_gc.hip -- device garbage collection of the node pool (NodePoolThreadedGC, NodePoolThreadedGC.hpp:29-403).
//
// forward  (top-down, :72-103): level by level the live set is the set of node pointers reachable from
//          the roots and the filled chain's root, held as a bitmap over the level's words (bit o: a
//          live node starts at word o); the live nodes of a level mark their children in the next one.
// backward (bottom-up, :105-348): leaves stay in their bucket and are packed in pointer order (bitmap
//          order); inner nodes get their children remapped, are re-hashed into a possibly new bucket and
//          appended there in pointer order, with the page-tail padding of the reference's bucket caches;
//          every bucket counter of the level is rewritten. A node's new pointer is kept at half its old
//          offset (nodes are two words or more, so no two share a place). Roots are remapped at level
//          0, the filled chain at each level (:378-381).
// Processing order equals the reference run on one worker, so the compacted pool words are
// identical to its output.
//
// Every launch has a size fixed by the pool's configuration (counts live in device memory), so the
// whole collection needs no host round trip: hd_gc queues it and waits once, and a frame graph
// captures it between its edit passes and its trace (hd_edit.hip).
//
// What bounds it: launches (a level's kernels are a few dependent reads each) on small worlds, then the
// child marks and the scattered reads of the children's new pointers. Work follows the used words and
// the live nodes, never the level's capacity: a 4096^3 terrain's levels hold 2^27 words each, of which
// under 3 % are used. The collection of a 4096^3 terrain after 256 edits: 3257 -> 975 us with a
// 640x360 frame (0.25 ms of it), 120 launches fewer.
#include "hd_internal.hpp"

#include <algorithm>
#include <string>

namespace hd {
namespace {

constexpr u32 kGcThreads = 256;
constexpr u32 kGcGrid = 2048;    // workgroups of the grid-stride kernels (bounded dispatch)
constexpr u32 kGcSortCap = 1024; // nodes that a wavefront sorts in LDS

__device__ inline u32 low_mask(u32 k) { return k >= 32u ? ~0u : ((1u << k) - 1u); }

// Clears what the collection starts from: the bitmap words over each bucket's used words and the new
// buckets' node counts. One thread per bucket of the pool. (Bits past a bucket's used words may be left
// from an earlier collection: nothing reads them.)
struct GcLevels {
	u32 *bits[HD_MAX_LEVELS];
};
__global__ void k_gc_clear(const u32 *__restrict__ bucket_words, DevConfig c, u64 total_buckets, GcLevels G,
                           u32 *__restrict__ cnt, u64 n_cnt) {
	const u64 t0 = (u64)blockIdx.x * blockDim.x + threadIdx.x, stride = (u64)gridDim.x * blockDim.x;
	for (u64 i = t0; i < n_cnt; i += stride)
		cnt[i] = 0u;
	for (u64 gb = t0; gb < total_buckets; gb += stride) {
		u32 l = 0;
		while (l + 1u < c.L && gb >= c.level_base[l + 1u])
			++l;
		const u64 lo = (gb - c.level_base[l]) << c.wbpb(), n = min(bucket_words[gb], c.words_per_bucket());
		if (n)
			for (u64 w = lo >> 5; w <= (lo + n - 1u) >> 5; ++w)
				G.bits[l][w] = 0u;
	}
}

// The live bits of word g of a level's bitmap that belong to the bucket whose used words are [lo, hi).
__device__ inline u32 live_word(const u32 *__restrict__ bits, u64 g, u64 lo, u64 hi) {
	u32 m = bits[g];
	if ((g << 5) < lo)
		m &= ~low_mask((u32)(lo - (g << 5)));
	if (((g + 1) << 5) > hi)
		m &= low_mask((u32)(hi - (g << 5)));
	return m;
}
// Calls f(o) for the start o of every live node of the level, one node per lane: a wavefront takes
// kWaveBuckets buckets at a time, four bitmap words of each per round (a bucket of an ordinary world has
// one or two used ones), and hands the words' set bits out to its lanes in pointer order, so a wave's
// nodes are neighbours in memory and no lane waits for another's fuller word. (One thread per bitmap
// word of the whole level, as before, walked up to 16 nodes in turn and read 2^22 words a level.)
constexpr u32 kWaveBuckets = 16, kBucketLanes = 64 / kWaveBuckets;
template <typename F>
__device__ inline void for_live(const u32 *__restrict__ bits, const u32 *__restrict__ bucket_words, const DevConfig &c,
                                u32 level, F f) {
	const u32 lane = threadIdx.x & 63u, nb = 1u << c.bucket_bits[level];
	const u64 wave = ((u64)blockIdx.x * blockDim.x + threadIdx.x) >> 6, waves = ((u64)gridDim.x * blockDim.x) >> 6;
	for (u64 b0 = wave * kWaveBuckets; b0 < nb; b0 += waves * kWaveBuckets) {
		const u64 b = b0 + lane / kBucketLanes, lo = b << c.wbpb();
		const u64 hi = lo + (b < nb ? min(bucket_words[c.level_base[level] + b], c.words_per_bucket()) : 0u);
		for (u64 g = (lo >> 5) + lane % kBucketLanes; __ballot((g << 5) < hi && hi > lo); g += kBucketLanes) {
			const u32 m = (g << 5) < hi && hi > lo ? live_word(bits, g, lo, hi) : 0u;
			const u32 cnt = (u32)__builtin_popcount(m);
			u32 x = cnt; // inclusive prefix over the lanes
#pragma unroll
			for (u32 d = 1; d < 64; d <<= 1) {
				const u32 y = __shfl_up(x, d);
				if (lane >= d)
					x += y;
			}
			const u32 total = (u32)__builtin_amdgcn_readlane((int)x, 63);
			for (u32 t0 = 0; t0 < total; t0 += 64u) {
				const u32 t = t0 + lane;
				u32 s = 0; // the first lane whose prefix exceeds t
#pragma unroll
				for (u32 d = 32; d > 0; d >>= 1)
					if ((u32)__shfl((int)x, (int)(s + d - 1u)) <= t)
						s += d;
				s = min(s, 63u);
				u32 ms = (u32)__shfl((int)m, (int)s);
				const u32 r = t - ((u32)__shfl((int)x, (int)s) - (u32)__shfl((int)cnt, (int)s));
				const u64 gs = ((u64)(u32)__shfl((int)(g >> 32), (int)s) << 32) | (u32)__shfl((int)(u32)g, (int)s);
				if (t < total) {
					for (u32 k = 0; k < r; ++k)
						ms &= ms - 1u;
					f((u32)((gs << 5) + (u32)__builtin_ctz(ms)));
				}
			}
		}
	}
}

// ---- forward
// the roots mark level 0, and the filled chain every level (its nodes have the most parents of all: with
// their bits set first no parent's atomic queues on them), as far down as it hangs together: what is below a
// missing node nobody holds
__global__ void k_gc_mark_roots(const u32 *__restrict__ roots, u32 n, const u32 *__restrict__ filled, DevConfig c,
                                GcLevels G) {
	const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
	const u32 l = i < n ? 0u : i - n;
	if (l >= c.L || (i >= n && !filled))
		return;
	u32 r = i < n ? roots[i] : filled[l];
	for (u32 k = 0; i >= n && k < l; ++k)
		r = filled[k] == kNull ? kNull : r;
	const u64 base = (u64)c.level_base[l] << c.wbpb(), words = 1ull << (c.bucket_bits[l] + c.wbpb());
	if (r == kNull || (u64)r < base || (u64)r - base >= words)
		return;
	const u64 o = (u64)r - base;
	atomicOr(&G.bits[l][o >> 5], 1u << (o & 31u));
}
// Every live node of level l marks its children in level l + 1. A hash-consed child can have millions
// of parents (the filled and uniform subtrees above all), whose atomics would queue on one address
// (about 10 ns each): the bit is read first, and of the workgroup's threads that still see it clear, the
// first to write the child into its slot of a small LDS table goes on. Stale reads and lost slots only
// cost a redundant atomic: bits go from 0 to 1 only. The widest workgroup shares one table among the most
// threads: with 256 threads and half the slots a 4096^3 terrain's marks take 271 instead of 197 us.
constexpr u32 kMarkThreads = 1024, kMarkSlots = 8192;
__global__ void __launch_bounds__(kMarkThreads) k_gc_expand(const u32 *__restrict__ words, const u32 *__restrict__ bits,
                                                            const u32 *__restrict__ bucket_words, DevConfig c,
                                                            u32 level, u64 base, u64 cbase, u64 cwords, u32 *cbits) {
	__shared__ u32 seen[kMarkSlots];
	for (u32 i = threadIdx.x; i < kMarkSlots; i += kMarkThreads)
		seen[i] = kNull;
	__syncthreads();
	for_live(bits, bucket_words, c, level, [&](u32 o) {
		u32 nw[9], co[8], bw[8], need = 0;
#pragma unroll
		for (u32 k = 0; k < 9; ++k) // the pool is padded past its end
			nw[k] = words[base + o + k];
		const u32 cnt = (u32)__builtin_popcount(nw[0] & 0xFFu);
#pragma unroll
		for (u32 k = 0; k < 8; ++k) {
			const u64 at = (u64)nw[k + 1] - cbase;
			const bool in = k < cnt && at < cwords;
			co[k] = in ? (u32)at : 0u;
			bw[k] = in ? cbits[co[k] >> 5] : ~0u;
		}
#pragma unroll
		for (u32 k = 0; k < 8; ++k)
			if (!((bw[k] >> (co[k] & 31u)) & 1u) &&
			    atomicExch(&seen[(co[k] * 0x9E3779B1u) >> (32 - 13)], co[k]) != co[k])
				need |= 1u << k;
#pragma unroll
		for (u32 k = 0; k < 8; ++k)
			if ((need >> k) & 1u)
				atomicOr(&cbits[co[k] >> 5], 1u << (co[k] & 31u));
	});
}
static_assert(kMarkSlots == 1u << 13, "the table's hash takes 13 bits");

// ---- backward
// leaves keep their bucket (:229-274): each bucket's live leaves, in pointer order, are packed in
// place from its start (a node never moves up, so reads stay ahead of writes); one thread per bucket
__global__ void k_gc_pack_leaves(u32 *__restrict__ words, u32 *__restrict__ bucket_words, DevConfig c, u32 level,
                                 const u32 *__restrict__ bits, u32 *__restrict__ newp, u32 *__restrict__ meta) {
	const u32 b = blockIdx.x * blockDim.x + threadIdx.x;
	if (b >= (1u << c.bucket_bits[level]))
		return;
	const u32 gb = c.level_base[level] + b;
	const u64 wbase = (u64)gb << c.wbpb(), lo = (u64)b << c.wbpb(), hi = lo + min(bucket_words[gb], c.words_per_bucket());
	if (hi == lo)
		return;
	u32 bw = 0;
	for (u64 w = lo >> 5; w <= (hi - 1) >> 5; ++w) {
		u32 m = live_word(bits, w, lo, hi);
		for (; m; m &= m - 1u) {
			const u64 o = (w << 5) + (u32)__builtin_ctz(m), off = o - lo;
			const u32 leaf[2] = {words[wbase + off], words[wbase + off + 1]};
			const u32 np = append_to_bucket(words, c, gb, bw, leaf, 2);
			if (np == kNull)
				atomicOr(&meta[kMetaOverflow], 4u);
			newp[o >> 1] = np;
		}
	}
	bucket_words[gb] = bw;
}
// The nodes that a new bucket of a level receives, in the order of arrival: the first cap in a list of the
// bucket's own, the others in a chain (head: the latest one's old offset + 1; next, at half its old offset: the
// one before it). cap is what a bucket of 2-word nodes holds, so only a bucket that overflows has a chain.
struct GcLists {
	u32 cap, *cnt, *head, *list, *next;
};
// The live nodes of an inner level: each one's children remapped (cnewp: the new pointers of the level
// below), the node written to the stage at its old offset (the pack rewrites the pool's words in place),
// re-hashed (:147-148) and listed in its new bucket, unordered. Thread 0 moves the filled chain's entry of
// the level below.
__global__ void __launch_bounds__(kGcThreads) k_gc_key(const u32 *__restrict__ words, const u32 *__restrict__ bits,
                                                       const u32 *__restrict__ bucket_words, DevConfig c, u32 level,
                                                       u64 base, u64 cbase, u64 cwords, const u32 *__restrict__ cnewp,
                                                       u32 *__restrict__ stage, GcLists B, u32 *__restrict__ newp,
                                                       u32 *__restrict__ filled) {
	if ((threadIdx.x | blockIdx.x) == 0 && filled) {
		const u32 f = filled[level + 1u];
		const u64 o = (u64)f - cbase; // (of a node that was dropped: launch_refill finds the chain again)
		if (f != kNull && o < cwords)
			filled[level + 1u] = cnewp[o >> 1];
	}
	for_live(bits, bucket_words, c, level, [&](u32 o) {
		u32 buf[9];
#pragma unroll
		for (u32 k = 0; k < 9; ++k)
			buf[k] = words[base + o + k];
		u32 k = (u32)__builtin_popcount(buf[0] & 0xFFu), lost = 0;
		u32 np[8];
#pragma unroll
		for (u32 j = 0; j < 8; ++j) {
			const u64 co = (u64)buf[j + 1] - cbase;
			np[j] = j < k && co < cwords ? cnewp[co >> 1] : kNull;
			lost |= (j < k && np[j] == kNull ? 1u : 0u) << j;
		}
		if (lost) { // children that a full bucket dropped leave the node (a trace would follow a null pointer)
			u32 mask = buf[0] & 0xFFu, r = 0;
			for (u32 m = mask; m; m &= m - 1u, ++r)
				if ((lost >> r) & 1u)
					mask &= ~(m & (0u - m));
#pragma unroll 1
			for (u32 p = 0; p < 7; ++p) // the others move up, in order
#pragma unroll
				for (u32 j = 0; j < 7; ++j) {
					const bool up = np[j] == kNull;
					const u32 x = np[j];
					np[j] = up ? np[j + 1] : x;
					np[j + 1] = up ? x : np[j + 1];
				}
			buf[0] = (buf[0] & ~0xFFu) | mask;
			k = (u32)__builtin_popcount(mask);
			if (k == 0u) {
				newp[o >> 1] = kNull;
				return;
			}
		}
#pragma unroll
		for (u32 j = 0; j < 8; ++j)
			buf[j + 1] = np[j];
		const u32 kb = murmur_regs(buf, k + 1u) & ((1u << c.bucket_bits[level]) - 1u);
		const u32 lp = atomicAdd(&B.cnt[kb], 1u);
#pragma unroll
		for (u32 j = 0; j < 9; ++j)
			if (j <= k)
				stage[(u64)o + j] = buf[j];
		if (lp < B.cap)
			B.list[(u64)kb * B.cap + lp] = o;
		else
			B.next[o >> 1] = atomicExch(&B.head[kb], o + 1u);
	});
}
// One node of a new bucket written at word `at` of the bucket (kNull: the bucket was full).
__device__ inline void gc_place(u32 *__restrict__ words, const u32 *__restrict__ stage, u64 wbase, u32 o, u32 n, u32 at,
                                u32 *__restrict__ newp) {
	if (at == kNull) {
		newp[o >> 1] = kNull;
		return;
	}
	u32 buf[9];
#pragma unroll
	for (u32 j = 0; j < 9; ++j)
		buf[j] = j < n ? stage[(u64)o + j] : 0u;
#pragma unroll
	for (u32 j = 0; j < 9; ++j)
		if (j < n)
			words[wbase + at + j] = buf[j];
	newp[o >> 1] = (u32)(wbase + at);
}
// The next node's place in a bucket filled to bw: past the page's tail when it would straddle it
// (the caller clears [bw, at)), kNull when the bucket is full (later, smaller nodes may still fit).
__device__ inline u32 gc_next(const DevConfig &c, u32 bw, u32 sz) {
	const u32 wpp = c.words_per_page();
	u32 at = bw;
	if ((at & (wpp - 1u)) + sz > wpp)
		at = (at / wpp + 1u) * wpp;
	return at + sz > c.words_per_bucket() ? kNull : at;
}
// A bucket of at most 64 nodes (one wavefront, a node per lane): ranked by old offset across the
// lanes, sizes in rank order, places by a wave scan while they fit the first page (else one by one).
__device__ inline u32 gc_pack_small(u32 *__restrict__ words, const DevConfig &c, const u32 *__restrict__ stage, u64 wbase,
                                    u32 m, const u32 *__restrict__ list, u32 *__restrict__ newp, u32 *__restrict__ meta,
                                    u32 lane) {
	const u32 o0 = lane < m ? list[lane] : kNull;
	u32 rk = lane;
	if (lane < m)
		rk = 0;
	for (u32 y = 0; y < m; ++y)
		rk += lane < m && (u32)__builtin_amdgcn_readlane((int)o0, (int)y) < o0 ? 1u : 0u;
	const u32 o = (u32)__builtin_amdgcn_ds_permute((int)(rk << 2), (int)o0); // lane r: the node ranked r
	const u32 sz = lane < m ? (u32)__builtin_popcount(stage[o] & 0xFFu) + 1u : 0u;
	u32 x = sz;
#pragma unroll
	for (u32 d = 1; d < 64; d <<= 1) {
		const u32 y = __shfl_up(x, d);
		if (lane >= d)
			x += y;
	}
	u32 bw = (u32)__builtin_amdgcn_readlane((int)x, 63), at = x - sz;
	if (bw > c.words_per_page()) { // uniform
		bw = 0;
		for (u32 r = 0; r < m; ++r) {
			const u32 s = (u32)__builtin_amdgcn_readlane((int)sz, (int)r), a = gc_next(c, bw, s);
			if (lane == r)
				at = a;
			if (a == kNull) {
				if (lane == 0)
					atomicOr(&meta[kMetaOverflow], 4u);
				continue;
			}
			for (u32 z = bw + lane; z < a; z += 64u)
				words[wbase + z] = 0u;
			bw = a + s;
		}
	}
	if (lane < m)
		gc_place(words, stage, wbase, o, sz, at, newp);
	return bw;
}
__device__ inline void gc_wave_sync() {
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// The m nodes in so (LDS, at most kGcSortCap; one wavefront) into a bucket filled to bw: bitonic sort,
// places one by one (sp). Returns what the bucket is filled to.
__device__ inline u32 gc_pack_sorted(u32 *__restrict__ words, const DevConfig &c, const u32 *__restrict__ stage, u64 wbase,
                                     u32 m, u32 bw, u32 *__restrict__ newp, u32 *__restrict__ meta, u32 lane, u32 *so,
                                     u32 *sp) {
	u32 P = 1;
	while (P < m)
		P <<= 1;
	for (u32 k = m + lane; k < P; k += 64)
		so[k] = ~0u;
	gc_wave_sync();
	for (u32 size = 2; size <= P; size <<= 1) // bitonic sort, ascending
		for (u32 stride = size >> 1; stride > 0; stride >>= 1) {
			for (u32 k = lane; k < P; k += 64) {
				const u32 q = k ^ stride;
				if (q > k) {
					const bool up = (k & size) == 0;
					const u32 a = so[k], d = so[q];
					if ((a > d) == up) {
						so[k] = d;
						so[q] = a;
					}
				}
			}
			gc_wave_sync();
		}
	for (u32 k = lane; k < m; k += 64)
		sp[k] = (u32)__builtin_popcount(stage[so[k]] & 0xFFu) + 1u; // node sizes
	gc_wave_sync();
	if (lane == 0) { // positions in pointer order; a page tail a node skips is zero (the cache's resize)
		for (u32 k = 0; k < m; ++k) {
			const u32 sz = sp[k], at = gc_next(c, bw, sz);
			sp[k] = at;
			if (at == kNull) {
				atomicOr(&meta[kMetaOverflow], 4u);
				continue;
			}
			for (u32 z = bw; z < at; ++z)
				words[wbase + z] = 0u;
			bw = at + sz;
		}
	}
	gc_wave_sync();
	for (u32 k = lane; k < m; k += 64)
		gc_place(words, stage, wbase, so[k], (u32)__builtin_popcount(stage[so[k]] & 0xFFu) + 1u, sp[k], newp);
	return __builtin_amdgcn_readfirstlane(bw);
}
// A bucket of 65 to kGcSortCap listed nodes (one wavefront).
__device__ inline u32 gc_pack_large(u32 *__restrict__ words, const DevConfig &c, const u32 *__restrict__ stage, u64 wbase,
                                    u32 m, const u32 *__restrict__ list, u32 *__restrict__ newp, u32 *__restrict__ meta,
                                    u32 lane, u32 *so, u32 *sp) {
	gc_wave_sync(); // the previous bucket's readers of so / sp are done
	for (u32 k = lane; k < m; k += 64)
		so[k] = list[k];
	return gc_pack_sorted(words, c, stage, wbase, m, 0u, newp, meta, lane, so, sp);
}
// Any number of nodes, listed and chained (one wavefront): range after range of old offsets, each narrow
// enough for the LDS sort. level_words: the offsets lie below it.
__device__ inline u32 gc_pack_ranges(u32 *__restrict__ words, const DevConfig &c, const u32 *__restrict__ stage, u64 wbase,
                                     u32 m, const u32 *__restrict__ list, const GcLists &B, u32 head, u64 level_words,
                                     u32 *__restrict__ newp, u32 *__restrict__ meta, u32 lane, u32 *so, u32 *sp) {
	u64 width = level_words;
	for (u32 k = m; k > kGcSortCap / 2u; k >>= 1)
		width >>= 1;
	u32 bw = 0, left = m;
	for (u64 lo = 0; left && lo < level_words;) {
		// (nodes are two words or more, so a range of 2 kGcSortCap offsets always fits)
		width = max(width, (u64)kGcSortCap);
		u32 n = 0;
		gc_wave_sync();
		for (u32 k0 = 0; k0 < min(m, B.cap); k0 += 64u) {
			const u32 k = k0 + lane, o = k < min(m, B.cap) ? list[k] : 0u;
			const bool in = k < min(m, B.cap) && o >= lo && o < lo + width;
			const u64 b = __ballot(in);
			const u32 at = n + (u32)__popcll(b & ((1ull << lane) - 1ull));
			if (in && at < kGcSortCap)
				so[at] = o;
			n += (u32)__popcll(b);
		}
		for (u32 q = head; q; q = B.next[(q - 1u) >> 1]) { // (the same on every lane)
			const u32 o = q - 1u;
			if (o >= lo && o < lo + width) {
				if (lane == 0 && n < kGcSortCap)
					so[n] = o;
				++n;
			}
		}
		if (n > kGcSortCap) {
			width >>= 1;
			continue;
		}
		if (n)
			bw = gc_pack_sorted(words, c, stage, wbase, n, bw, newp, meta, lane, so, sp);
		left -= n;
		lo += width;
		width = min(2u * width, level_words);
	}
	return bw;
}
// The new buckets of an inner level, kPackBuckets per wavefront: their nodes sorted by old pointer,
// placed one after another with page-tail padding (lf_gc_shrink_inner_bucket's cache, :105-182, and
// the flush, :198-227) and written in parallel; every bucket's counter is rewritten and its node
// count cleared for the next level. The wave reads its buckets' counts at once and skips the empty ones.
constexpr u32 kPackBuckets = 4;
__global__ void __launch_bounds__(kGcThreads) k_gc_pack_inner(u32 *__restrict__ words, u32 *__restrict__ bucket_words,
                                                              DevConfig c, u32 level, const u32 *__restrict__ stage,
                                                              GcLists B, u32 *__restrict__ newp, u32 *__restrict__ meta) {
	__shared__ u32 s_off[kGcThreads / 64][kGcSortCap];
	__shared__ u32 s_pos[kGcThreads / 64][kGcSortCap];
	const u32 lane = threadIdx.x & 63u, w = threadIdx.x >> 6, nb = 1u << c.bucket_bits[level];
	for (u64 b0 = ((u64)blockIdx.x * (kGcThreads / 64) + w) * kPackBuckets; b0 < nb;
	     b0 += (u64)gridDim.x * (kGcThreads / 64) * kPackBuckets) {
		const bool in = lane < kPackBuckets && b0 + lane < nb;
		const u32 mm = in ? B.cnt[b0 + lane] : 0u;
		u32 bw = 0;
		for (u64 todo = __ballot(mm != 0u); todo; todo &= todo - 1ull) {
			const int k = __builtin_ctzll(todo);
			const u32 m = (u32)__builtin_amdgcn_readlane((int)mm, k), b = (u32)b0 + (u32)k;
			const u64 wbase = (u64)(c.level_base[level] + b) << c.wbpb();
			const u32 *ls = B.list + (u64)b * B.cap;
			u32 r;
			if (m <= min(64u, B.cap))
				r = gc_pack_small(words, c, stage, wbase, m, ls, newp, meta, lane);
			else if (m <= min(kGcSortCap, B.cap))
				r = gc_pack_large(words, c, stage, wbase, m, ls, newp, meta, lane, s_off[w], s_pos[w]);
			else {
				r = gc_pack_ranges(words, c, stage, wbase, m, ls, B, m > B.cap ? B.head[b] : 0u,
				                   1ull << (c.bucket_bits[level] + c.wbpb()), newp, meta, lane, s_off[w], s_pos[w]);
				if (lane == 0)
					B.head[b] = 0u;
			}
			bw = (int)lane == k ? r : bw;
		}
		if (in) {
			bucket_words[c.level_base[level] + b0 + lane] = bw;
			if (mm)
				B.cnt[b0 + lane] = 0u;
		}
	}
}
// roots and the filled chain's root remapped through level 0's new pointers
__global__ void k_gc_roots(u32 *__restrict__ roots, u32 n, u32 *__restrict__ filled, const u32 *__restrict__ newp,
                           u64 base, u64 words) {
	const u32 i = blockIdx.x * blockDim.x + threadIdx.x;
	u32 *r = i < n ? roots + i : (i == n && filled ? filled : nullptr);
	if (!r || *r == kNull || (u64)*r < base || (u64)*r - base >= words)
		return;
	*r = newp[((u64)*r - base) >> 1];
}

inline u32 grid(u64 n, u32 t = kGcThreads) { return (u32)std::max<u64>(1, (n + t - 1) / t); }

} // namespace

// Device buffers of a collection, sized by the pool's configuration (reused across calls).
int GcPlan::prepare(Pool &p, const char *prefix) {
	const u32 L = p.dc.L, wpb = p.dc.words_per_bucket();
	lv.assign(L, Level{});
	u64 max_words = 0, max_buckets = 0;
	std::string pre(prefix);
	for (u32 l = 0; l < L; ++l) {
		Level &V = lv[l];
		V.buckets = 1ull << p.dc.bucket_bits[l];
		V.words = V.buckets * wpb;
		V.base = (u64)p.dc.level_base[l] << p.dc.wbpb();
		HD_RET(p.scratch.get<u32>(pre + "gc_bits" + std::to_string(l), (V.words + 31) / 32 + 1, &V.bits));
		max_words = std::max(max_words, V.words);
		max_buckets = std::max(max_buckets, V.buckets);
	}
	cap = wpb / 2; // (of 2-word nodes)
	HD_RET(p.scratch.get<u32>(pre + "gc_newp0", max_words / 2 + 1, &newp[0]));
	HD_RET(p.scratch.get<u32>(pre + "gc_newp1", max_words / 2 + 1, &newp[1]));
	HD_RET(p.scratch.get<u32>(pre + "gc_stage", max_words + 16, &stage));
	HD_RET(p.scratch.get<u32>(pre + "gc_list", max_buckets * cap + max_words / 2 + 1, &list));
	next = list + max_buckets * cap;
	HD_RET(p.scratch.get<u32>(pre + "gc_cnt", 2 * max_buckets, &cnt)); // and the chains' heads
	return HD_OK;
}

// Queues a whole collection on stream s: roots (device, n_roots) are remapped in place; the filled
// chain (when the pool has one) is a root and moves with its nodes in d_filled. No host
// synchronisation and no allocation (capture-safe once the plan is prepared).
int gc_queue(Pool &p, const GcPlan &G, hipStream_t s, u32 *d_roots, u32 n_roots, bool has_filled) {
	const u32 L = p.dc.L;
	u64 max_buckets = 0;
	GcLevels B{};
	for (u32 l = 0; l < L; ++l) {
		B.bits[l] = G.lv[l].bits;
		max_buckets = std::max(max_buckets, G.lv[l].buckets);
	}
	k_gc_clear<<<std::min(grid(p.total_buckets), kGcGrid), kGcThreads, 0, s>>>(p.bucket_words, p.dc, p.total_buckets, B,
	                                                                          G.cnt, 2 * max_buckets);
	k_gc_mark_roots<<<grid(n_roots + L), kGcThreads, 0, s>>>(d_roots, n_roots, has_filled ? p.d_filled : nullptr, p.dc, B);
	auto waves = [&](u32 l) { return std::min(grid(G.lv[l].buckets / kWaveBuckets * 64), kGcGrid); };
	for (u32 l = 0; l + 1 < L; ++l) {
		const GcPlan::Level &V = G.lv[l], &C = G.lv[l + 1];
		k_gc_expand<<<std::min(grid(V.buckets / kWaveBuckets * 64, kMarkThreads), 512u), kMarkThreads, 0, s>>>(
		    p.words, V.bits, p.bucket_words, p.dc, l, V.base, C.base, C.words, C.bits);
	}
	k_gc_pack_leaves<<<grid(G.lv[L - 1].buckets), kGcThreads, 0, s>>>(p.words, p.bucket_words, p.dc, L - 1,
	                                                                 G.lv[L - 1].bits, G.newp[(L - 1) & 1], p.meta);
	const GcLists lists{G.cap, G.cnt, G.cnt + max_buckets, G.list, G.next};
	for (int l = (int)L - 2; l >= 0; --l) {
		const GcPlan::Level &V = G.lv[l], &C = G.lv[l + 1];
		u32 *newp = G.newp[l & 1];
		k_gc_key<<<waves((u32)l), kGcThreads, 0, s>>>(p.words, V.bits, p.bucket_words, p.dc, (u32)l, V.base, C.base,
		                                              C.words, G.newp[(l + 1) & 1], G.stage, lists, newp,
		                                              has_filled ? p.d_filled : nullptr);
		k_gc_pack_inner<<<grid((V.buckets + kPackBuckets - 1) / kPackBuckets * 64), kGcThreads, 0, s>>>(
		    p.words, p.bucket_words, p.dc, (u32)l, G.stage, lists, newp, p.meta);
	}
	k_gc_roots<<<grid(n_roots + 1), kGcThreads, 0, s>>>(d_roots, n_roots, has_filled ? p.d_filled : nullptr, G.newp[0],
	                                                    G.lv[0].base, G.lv[0].words);
	if (has_filled) // a chain node that a full bucket dropped is appended again
		launch_refill(p, s);
	HD_TRY(hipGetLastError());
	return HD_OK;
}

} // namespace hd

using namespace hd;

extern "C" int hd_gc(hd_pool *h, uint32_t *roots, uint32_t n) {
	if (!h || (!roots && n))
		return set_error("hd_gc: null argument"), HD_ERR_ARG;
	Pool &p = h->p;
	HD_RET(p.gc_plan.prepare(p, ""));
	u32 *droots;
	HD_RET(p.scratch.get<u32>("gc_roots", n ? n : 1, &droots));
	if (n)
		HD_TRY(hipMemcpyAsync(droots, roots, n * 4, hipMemcpyHostToDevice, p.stream));
	const bool has_filled = !p.filled.empty();
	HD_RET(gc_queue(p, p.gc_plan, p.stream, droots, n, has_filled));
	if (n)
		HD_TRY(hipMemcpyAsync(roots, droots, n * 4, hipMemcpyDeviceToHost, p.stream));
	if (has_filled)
		HD_TRY(hipMemcpyAsync(p.filled.data(), p.d_filled, p.dc.L * 4, hipMemcpyDeviceToHost, p.stream));
	HD_TRY(hipStreamSynchronize(p.stream));
	return HD_OK;
}
