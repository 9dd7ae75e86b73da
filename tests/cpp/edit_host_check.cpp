// The host side of plain edits (hd_edit.hip: planning, buffers, the order of passes) on a stand-in for the HIP
// runtime: nothing runs, launches are reported by name, device memory is addresses only, and what the host
// reads back is what a test says. Compiled for the host alone; no device is needed.
//     edit_host_check NAME   runs one test (exit status 0: passed)
#include "../../vkhashdag_amd/csrc/hd_edit.hip"

#include <cstdarg>
#include <cstdio>
#include <functional>
#include <map>
#include <set>
#include <string>

using namespace hd;

struct Fake {
	u64 free_bytes = 256ull << 30, next = 1ull << 40, allocs = 0;
	bool same_address = false; // an allocation gets the address that was freed last, whatever its size
	u64 freed = 0;
	std::map<u64, u64> held; // address, bytes
	std::map<const void *, std::string> names;
	std::function<bool(size_t)> refuse; // an allocation that fails
	std::function<void(const std::string &, void **)> launch;
	std::function<bool(void *, const void *, size_t)> read; // device to host: true if it filled the destination
} fake;

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
	if (n > fake.free_bytes || (fake.refuse && fake.refuse(n)))
		return hipErrorOutOfMemory;
	const u64 at = fake.same_address && fake.freed ? fake.freed : fake.next;
	fake.freed = 0;
	fake.next += (n + (1u << 21)) & ~((1ull << 21) - 1u);
	fake.free_bytes -= n;
	fake.held[at] = n;
	++fake.allocs;
	*p = (void *)at;
	return hipSuccess;
}
hipError_t hipFree(void *p) {
	if (!p)
		return hipSuccess;
	const auto it = fake.held.find((u64)p);
	if (it == fake.held.end())
		printf("hipFree of %p, which is not held\n", p), exit(1);
	fake.free_bytes += it->second;
	fake.freed = it->first;
	fake.held.erase(it);
	return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *free_b, size_t *total) { return *free_b = fake.free_bytes, *total = 288ull << 30, hipSuccess; }
hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind kind, hipStream_t) {
	if (kind == hipMemcpyDeviceToHost && !(fake.read && fake.read(dst, src, n)))
		memset(dst, 0, n);
	return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **args, size_t, hipStream_t) {
	if (fake.launch)
		fake.launch(fake.names[f], args);
	return hipSuccess;
}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) {
	fake.names[f] = name;
}
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s) {
	return *g = *b = dim3(1), *n = 0, *s = nullptr, hipSuccess;
}
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "an error"; }
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *, hipDeviceAttribute_t, int) { return hipErrorInvalidValue; }
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *, int) { return hipErrorInvalidValue; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *, hipGraph_t, hipGraphNode_t *, char *, size_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *) { return hipSuccess; }
hipError_t hipHostFree(void *p) { return free(p), hipSuccess; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return *p = calloc(1, n), hipSuccess; }
}

namespace hd {
Tuning g_tuning;
void set_error(const char *fmt, ...) {
	va_list ap;
	va_start(ap, fmt);
	vprintf(fmt, ap);
	va_end(ap);
	printf("\n");
}
int set_config(Pool &, const hd_config &) { return HD_ERR_ARG; }
int make_filled(Pool &) { return HD_OK; }
int GcPlan::prepare(Pool &, const char *) { return HD_ERR_ARG; }
int gc_queue(Pool &, const GcPlan &, hipStream_t, u32 *, u32, bool) { return HD_ERR_ARG; }
int trace_on_stream(Pool &, hipStream_t, u32, u32, const hd_view *, const u32 *, u32, u32, u32 *, const u32 *) {
	return HD_ERR_ARG;
}
} // namespace hd

#define CHECK(x)                                                                                                   \
	do {                                                                                                           \
		if (!(x))                                                                                                  \
			printf("%s:%d: %s does not hold\n", __FILE__, __LINE__, #x), exit(1);                                   \
	} while (0)

static void make_pool(Pool &p, u32 voxel_level, u32 color_leaf) {
	p.dc = DevConfig{};
	p.dc.wbpp = 9, p.dc.pbpb = 2, p.dc.L = voxel_level - 1, p.dc.voxel_level = voxel_level, p.dc.color_leaf = color_leaf;
	for (u32 l = 0; l < p.dc.L; ++l)
		p.dc.bucket_bits[l] = 10, p.dc.level_base[l] = l << 10;
	p.total_buckets = (u64)p.dc.L << 10;
	p.total_words = p.total_buckets << 11;
	p.cnode_cap = 1u << 24, p.cleaf_cap = 1u << 28;
	p.h_pass = (u32 *)calloc(16, 4);
}
static hd_edit_desc ball(u32 x, u32 y, u32 z, u32 r, bool colored) {
	hd_edit_desc d{};
	d.kind = HD_EDIT_SPHERE_FILL, d.p0[0] = x, d.p0[1] = y, d.p0[2] = z, d.r2 = (u64)r * r;
	d.colored = colored, d.color.colors = 0x010203u * (x + y + z) & 0xFFFFFFu, d.color.has_value = colored;
	return d;
}
// The pass whose top-down was launched last.
struct Pass {
	u32 first = 0, count = 0;
	bool chained = false;
};
static Pass top_down(const std::string &kernel, void **args, const hd_edit_desc *base) {
	const EditParams &P = *(const EditParams *)args[0];
	(void)kernel;
	return Pass{(u32)(P.edits - base), P.n_edits, kernel.find("a_topILj2E") != std::string::npos};
}

// ---- a piece of a pass that did not hold stays sync-free when the device's memory is gone meanwhile
static void test_piece() {
	setenv("HD_EDIT_STAGING_WORDS", "1", 1); // (the buffers held are then much smaller than the plan counts)
	Pool p;
	make_pool(p, 12, 8);
	std::vector<hd_edit_desc> e;
	for (u32 k = 0; k < 64; ++k)
		e.push_back(ball(256 + 512 * (k % 8), 256 + 512 * (k / 8), 2048, 160 + k % 3, true));
	const hd_edit_desc *base = nullptr;
	Pass now;
	bool cut = false;
	std::vector<Pass> seen;
	fake.launch = [&](const std::string &k, void **args) {
		CHECK(k.find("k_root") == std::string::npos); // (a kernel of the synchronized pipeline)
		if (k.find("a_top") == std::string::npos)
			return;
		if (!base)
			base = ((const EditParams *)args[0])->edits;
		now = top_down(k, args, base);
		seen.push_back(now);
	};
	fake.read = [&](void *dst, const void *, size_t n) {
		if (dst != p.h_pass || n != 4 * kPmHdr)
			return false;
		memset(dst, 0, n);
		if (!cut) // the first pass is cut at its second edit
			p.h_pass[kPmCut] = ~1u, fake.free_bytes = 64u << 20;
		cut = true;
		return true;
	};
	u32 r = 0, c = 0;
	CHECK(edit_plain(p, 1u, kColorNull, e.data(), (u32)e.size(), &r, &c) == HD_OK);
	u32 next = 0; // the edits once each, in order, the cut pass aside
	for (size_t k = 1; k < seen.size(); ++k) {
		CHECK(seen[k].first == next);
		next += seen[k].count;
	}
	printf("first pass %u edits, %llu MB held\n", seen[0].count, (unsigned long long)(p.scratch.held() >> 20));
	CHECK(seen[0].count == 64 && next == 64);
}

// ---- a dedup table that grows is cleared, also where the new one lies at the old one's address
static void test_table() {
	Pool p;
	make_pool(p, 12, 8);
	fake.same_address = true;
	std::map<u64, u64> cleared; // address, words
	fake.launch = [&](const std::string &k, void **args) {
		if (k.find("a_fill_u32") != std::string::npos && *(u32 *)args[2] == 0u)
			cleared[*(u64 *)args[0]] = *(u64 *)args[1];
	};
	u32 r = 0, c = 0;
	u64 before = 0;
	for (u32 n : {1u, 8u, 64u}) {
		std::vector<hd_edit_desc> e;
		for (u32 k = 0; k < n; ++k)
			e.push_back(ball(256 + 512 * (k % 8), 256 + 512 * (k / 8), 2048, 100, true));
		cleared.clear();
		CHECK(edit_plain(p, 1u, kColorNull, e.data(), n, &r, &c) == HD_OK);
		const DevBuf &tab = p.scratch.bufs["a_tab"];
		CHECK(tab.bytes > before); // (the calls are larger each time)
		before = tab.bytes;
		CHECK(cleared.count((u64)tab.p) && cleared[(u64)tab.p] >= tab.bytes / 8 * 2);
	}
}

// ---- the per-bucket lists start empty also when an allocation after theirs failed
static void test_lists() {
	Pool p;
	make_pool(p, 12, 8);
	std::set<u64> filled;
	fake.launch = [&](const std::string &k, void **args) {
		if (k.find("a_fill_u32") != std::string::npos)
			filled.insert(*(u64 *)args[0]);
	};
	const hd_edit_desc e = ball(256, 256, 2048, 100, true);
	u32 r = 0, c = 0;
	const size_t list = p.total_buckets * kWalkList * 4;
	fake.refuse = [&](size_t n) { return n == list + list / 4; };
	CHECK(edit_plain(p, 1u, kColorNull, &e, 1, &r, &c) == HD_ERR_DEVICE);
	CHECK(p.scratch.bufs["a_head"].p && !p.scratch.bufs["a_blist"].p); // (that one was refused)
	fake.refuse = nullptr;
	CHECK(edit_plain(p, 1u, kColorNull, &e, 1, &r, &c) == HD_OK);
	CHECK(filled.count((u64)p.scratch.bufs["a_bcnt"].p) && filled.count((u64)p.scratch.bufs["a_head"].p));
}

// ---- calls that fit the device's memory one edit at a time are not refused
static std::vector<hd_edit_desc> apart(u32 n, u32 r) {
	std::vector<hd_edit_desc> e;
	for (u32 k = 0; k < n; ++k)
		e.push_back(ball(256 + 512 * (k % 8), 256 + 512 * (k / 8), 2048, r, true));
	return e;
}
// The passes of a plain call: in order, each edit once.
static std::vector<Pass> passes(Pool &p, const std::vector<hd_edit_desc> &e) {
	std::vector<Pass> seen;
	const hd_edit_desc *base = nullptr;
	fake.launch = [&](const std::string &k, void **args) {
		CHECK(k.find("k_root") == std::string::npos); // (a kernel of the synchronized pipeline)
		if (k.find("a_top") == std::string::npos)
			return;
		if (!base)
			base = ((const EditParams *)args[0])->edits;
		seen.push_back(top_down(k, args, base));
	};
	u32 r = 0, c = 0, next = 0;
	CHECK(edit_plain(p, 1u, kColorNull, e.data(), (u32)e.size(), &r, &c) == HD_OK);
	for (const Pass &q : seen) {
		CHECK(q.first == next && q.chained == (q.count > 1));
		next += q.count;
	}
	CHECK(next == e.size());
	return seen;
}
static void test_memory() { // little is free: shorter passes, the rest of the memory left to others
	for (u64 mb : {16384u, 2048u, 768u, 256u, 96u}) {
		Pool p;
		make_pool(p, 12, 8);
		fake.held.clear();
		fake.free_bytes = mb << 20;
		const std::vector<Pass> seen = passes(p, apart(64, 160));
		printf("%llu MB free: %zu passes, %llu MB held\n", (unsigned long long)mb, seen.size(),
		       (unsigned long long)(p.scratch.held() >> 20));
		CHECK(mb < 16384u || seen.size() == 1);
		CHECK(p.scratch.held() < std::max<u64>(mb << 19, 80u << 20)); // (one such edit alone takes 70 MB)
	}
}
static void test_refused() { // the device says no all the same (its memory is in pieces, or somebody was faster)
	Pool p;
	make_pool(p, 12, 8);
	fake.refuse = [&](size_t n) { return n > (30u << 20); };
	CHECK(passes(p, apart(64, 160)).size() == 64);
	fake.refuse = nullptr;
	CHECK(passes(p, apart(64, 160)).size() == 1);
}
static void test_column() { // a column fill that cannot have its buffers: the synchronized pipeline
	Pool p;
	make_pool(p, 12, 8);
	p.hm_mn = (u32 *)8;
	fake.read = [&](void *dst, const void *, size_t n) {
		if (n != 8 * HD_MAX_LEVELS) // the nodes per level that column_count reads
			return false;
		for (u32 l = 0; l < HD_MAX_LEVELS; ++l)
			((u64 *)dst)[l] = 3ull << 2 * l;
		return true;
	};
	fake.launch = [&](const std::string &k, void **) {
		if (k.find("k_root") != std::string::npos)
			printf("column: the synchronized pipeline\n"), exit(0);
	};
	hd_edit_desc e{};
	e.kind = HD_EDIT_COLUMN_FILL, e.p1[0] = e.p1[1] = 4096;
	u32 r = 0, c = 0;
	CHECK(edit_plain(p, 1u, kColorNull, &e, 1, &r, &c) == HD_OK); // (all there: sync-free)
	p.scratch.release();
	fake.refuse = [&](size_t n) { return n > (100u << 20); };
	edit_plain(p, 1u, kColorNull, &e, 1, &r, &c);
	CHECK(!"the fill reached the synchronized pipeline");
}

// ---- passes that do not hold: what a call loses by them
// The device, as far as the host sees it: fills over a world whose nodes above level `full` are all there and
// below it none. A chained pass is cut at the first edit that enters a node which was null before the
// pass and which an earlier edit of it fills (early: its top-down knows), or, with late = k > 0, at its k-th edit
// whatever it does, or it reports a full bucket.
struct Device {
	Pool &p;
	const std::vector<hd_edit_desc> &e;
	u32 full, late = 0;
	bool early = true, full_bucket = false;
	std::set<u64> nodes;
	const hd_edit_desc *base = nullptr;
	Pass now;
	u32 cut = ~0u; // the pass's first edit that must not share it
	u32 singles = 0, chained = 0, left = 0, again = 0, next = 0, widest = 0;
	bool open = false;

	template <typename F> void entered(const hd_edit_desc &d, F f) const { // nodes of level full .. the color leaves
		const i64 r = (i64)std::sqrt((double)d.r2) + 1;
		for (u32 l = full; l <= p.dc.color_leaf; ++l) {
			const i64 S = (i64)1 << (p.dc.voxel_level - l);
			for (i64 z = (d.p0[2] - r) / S; z <= (d.p0[2] + r) / S; ++z)
				for (i64 y = (d.p0[1] - r) / S; y <= (d.p0[1] + r) / S; ++y)
					for (i64 x = (d.p0[0] - r) / S; x <= (d.p0[0] + r) / S; ++x)
						if (reaches(d, {x * S, y * S, z * S}, S))
							f((u64)l << 48 | (u64)z << 32 | (u64)y << 16 | (u64)x);
		}
	}
	void settle() { // the pass before went through
		if (!open)
			return;
		open = false;
		CHECK(now.first == next);
		for (u32 k = now.first; k < now.first + now.count; ++k)
			entered(e[k], [&](u64 n) { nodes.insert(n); });
		next += now.count;
		(now.count > 1 ? chained : singles) += 1;
		widest = std::max(widest, now.count);
	}
	void run() {
		fake.launch = [this](const std::string &k, void **args) {
			CHECK(k.find("k_root") == std::string::npos);
			if (k.find("a_chain_restore") != std::string::npos) {
				CHECK(cut != ~0u || full_bucket);
				++again;
				open = false;
			}
			if (k.find("a_top") == std::string::npos)
				return;
			if (!base)
				base = ((const EditParams *)args[0])->edits;
			const Pass q = top_down(k, args, base);
			if (open && (cut == ~0u || now.count == 1) && !(full_bucket && now.count > 1))
				settle(); // (else the host has still to learn that the pass before did not hold)
			else if (open)
				return;
			now = q;
			open = true;
			cut = ~0u;
			std::set<u64> mine;
			for (u32 j = 0; j < q.count && cut == ~0u; ++j) {
				const hd_edit_desc &d = e[q.first + j];
				bool meets = false;
				entered(d, [&](u64 n) { meets |= !nodes.count(n) && mine.count(n); });
				if (q.chained && (meets || (late && j == late)))
					cut = j;
				entered(d, [&](u64 n) { mine.insert(n); });
			}
		};
		fake.read = [this](void *dst, const void *, size_t n) {
			memset(dst, 0, n);
			if (dst == p.h_pass + kHostMeet && n == 4) {
				if (cut != ~0u && early)
					*(u32 *)dst = ~cut, ++left, open = false;
			} else if (dst == p.h_pass && n == 4 * kPmHdr) {
				p.h_pass[kPmCut] = full_bucket ? ~0u : cut == ~0u ? 0u : ~cut;
				p.h_pass[kPmFull] = full_bucket;
			}
			return true;
		};
		u32 r = 0, c = 0;
		CHECK(edit_plain(p, 1u, kColorNull, e.data(), (u32)e.size(), &r, &c) == HD_OK);
		settle();
		CHECK(next == e.size());
		CHECK(p.passes - p.passes_cut == singles + chained && p.passes_left == left && p.passes_cut == again);
	}
	// in passes of one edit: a chained pass takes up to three, its top-down one and a quarter
	double time() const { return singles + 3.0 * chained + 1.25 * left + 3.0 * again; }
};
static double air(const char *name, const std::vector<hd_edit_desc> &e, u32 full, bool wary, u32 late = 0,
                  bool early = true, bool full_bucket = false) {
	Pool p;
	make_pool(p, 12, 8);
	p.edit_wary = wary;
	fake.free_bytes = 256ull << 30;
	fake.held.clear();
	Device d{p, e, full};
	d.late = late, d.early = early, d.full_bucket = full_bucket;
	d.run();
	printf("%s%s: %zu edits, %u single, %u chained (up to %u), %u left, %u cut: %.2f of one by one\n", name,
	       wary ? ", wary" : "", e.size(), d.singles, d.chained, d.widest, d.left, d.again, d.time() / (double)e.size());
	return d.time();
}
static std::vector<hd_edit_desc> lattice(u32 nx, u32 ny, u32 nz, u32 step, u32 r) {
	std::vector<hd_edit_desc> e;
	for (u32 k = 0; k < nx * ny * nz; ++k)
		e.push_back(ball(100 + step * (k % nx), 100 + step * (k / nx % ny), 3200 + step * (k / nx / ny), r, true));
	return e;
}
// At most a sixteenth slower than one by one, and a pass and a half that did not hold (of a wary pool: its
// top-down).
static double bound(u32 n, bool wary) { return n * (1.0 + 1.0 / 16.0) + (wary ? 1.25 : 4.5); }
static void test_air() {
	for (bool wary : {false, true}) {
		for (u32 n : {2u, 3u, 4u, 8u, 16u, 120u})
			CHECK(air("row", lattice(n, 1, 1, 32, 6), 2, wary) <= bound(n, wary));
		CHECK(air("sheet", lattice(16, 16, 1, 48, 10), 2, wary) <= bound(256, wary));
		CHECK(air("lattice", lattice(8, 8, 8, 48, 10), 2, wary) <= bound(512, wary));
	}
}
static void test_ground() { // nothing is null above the color leaves: nearly everything shares passes
	for (bool wary : {false, true}) {
		CHECK(air("ground", lattice(16, 16, 1, 48, 10), 9, wary) <= 6.0);
		CHECK(air("ground", lattice(3, 1, 1, 48, 10), 9, wary) <= 3.0);
	}
}
static void test_cut() { // passes that are found out at their end only
	for (u32 late : {1u, 2u, 5u, 40u})
		CHECK(air("cut", lattice(16, 16, 2, 48, 10), 9, false, late) <= bound(512, false));
	CHECK(air("meets seen at the end", lattice(16, 16, 1, 48, 10), 2, false, 0, false) <= bound(256, false));
	CHECK(air("full buckets", lattice(16, 16, 2, 48, 10), 9, false, 0, true, true) <= bound(512, false));
}

int main(int argc, char **argv) {
	const std::map<std::string, void (*)()> tests{{"piece", test_piece}, {"table", test_table}, {"lists", test_lists}, {"memory", test_memory},
	                                                 {"refused", test_refused}, {"column", test_column},
	                                                 {"air", test_air}, {"ground", test_ground}, {"cut", test_cut}};
	if (argc != 2 || !tests.count(argv[1]))
		return printf("unknown test\n"), 2;
	setvbuf(stdout, nullptr, _IONBF, 0);
	tests.at(argv[1])();
	return printf("%s: passed\n", argv[1]), 0;
}
