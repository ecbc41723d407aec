/* bvh_build.hip - GPU binned-SAH BVH builder (16 bins) for gfx950.
 *
 * Replaces the BLAS/TLAS builds hidden in OptiX (rtpModelUpdate,
 * lib/RenderCore_PrimeRef/core_mesh.cpp:63-64; optixAccelBuild,
 * lib/rendercore_optix7/core_mesh.cpp:123). Breadth-first, the levels driven
 * from device memory (a level's kernels read its node range there, so the host
 * launches several levels before it looks). Two kinds of node:
 *   up to SMALL primitives: one wave per node does everything in one kernel per
 *     level (k_level): centroid bounds, bins in LDS, split, stable partition;
 *   above: chunks of CHUNK primitives, a block each, bin into LDS and merge into
 *     the node's global bins (k_big_bin); a wave per node picks the split
 *     (k_big_decide); the chunks partition and gather the children's centroid
 *     bounds on the way (k_big_part).
 * What bounds a build is atomics and launches: per-primitive global atomics of
 * blocks that straddle small nodes, one thread per split decision, and a host
 * round trip per level took most of it before. With the bins of small nodes in
 * their wave's LDS, 16 lanes scanning an axis's bins (one DPP row) and two
 * children slots reserved per split by one atomic per block, SetGeometry's build
 * (with the layout) takes, before -> now: 1,000 triangles 1.68 -> 0.36 ms, 20,000
 * 2.8 -> 0.75, 200,000 8.6 -> 1.5, 1 M 24.7 -> 4.2, 4 M 78 -> 16; the top level of
 * 1,000 instances 1.42 -> 0.29 ms. min/max are taken on order-preserving integer
 * keys (exact, so their order does not matter).
 *
 * Split rules (identical in every builder of this project): centroid
 * c = (lo + hi) * 0.5; axis valid when its centroid extent e > 0 and 16/e is
 * finite; bin = min(15, int((c - cmin) * (16 / e))); cost of the split after
 * bin i = nL * A(L) + nR * A(R) with A = dx*dy + dy*dz + dz*dx; first minimum
 * over axes 0..2 and i = 0..14; one primitive -> leaf; n <= maxLeaf -> leaf
 * unless A(node) + cost < n * A(node); no valid axis -> leaf up to
 * maxDegenerateLeaf primitives, else the range is halved.
 */
#include "bvh.h"
#include "lh_math.h"
#include <algorithm>

namespace lh {

static const int BINS = 16;
static const int SMALL = 512;          /* primitives a wave handles by itself */
static const int CHUNK = 2048;         /* primitives of a larger node per block */
static const int LEVEL_WAVES = 8;      /* nodes per block of k_level */
static const int MAX_LEVELS = 65536;
/* bins of a node (ints): counts [48], lo keys [48][3], hi keys [48][3]; a big
 * node's scratch holds its centroid bounds' keys in front */
static const int B_CNT = 0, B_LO = 3 * BINS, B_HI = B_LO + 9 * BINS, B_SIZE = B_HI + 9 * BINS; /* 336 */
static const int S_CMIN = 0, S_CMAX = 3, S_BINS = 6, S_STRIDE = 344;

struct BigRec
{
	int node, start, cnt, chunk0;      /* chunks chunk0 .. of the level */
	int mode, split, left, child;      /* axis 0..2 or 3 (halved); last left bin; left count; left child */
	int childBig[2];                   /* the children's records at the next level, -1: not big */
	int cursor[2];                     /* next position of the left / right child */
};

/* Level d: nodes [start[d], start[d] + cnt[d]), big nodes (low word) and their
 * chunks (high word) in head[d]. Lists and scratch alternate by level parity. */
struct BuildArgs
{
	BuildNode* nodes;
	uint32_t* out;                     /* leaves' primitives */
	uint32_t* buf[2];
	const float4* lo;
	const float4* hi;
	int* cnt;
	int* start;
	unsigned long long* head;
	BigRec* big[2];
	int* scr[2];
	int* table[2];                     /* chunk -> big record */
	int* keys;                         /* root box, root centroid bounds: 2 x (min 3, max 3) */
	int n, maxLeaf, maxDegen;
};

static __device__ __forceinline__ int KINF() { return fkey(__builtin_huge_valf()); }
static __device__ __forceinline__ int KNINF() { return fkey(-__builtin_huge_valf()); }

__device__ __forceinline__ float half_area(v3 lo, v3 hi)
{
	const v3 d = hi - lo;
	return d.x * d.y + d.y * d.z + d.z * d.x;
}

__device__ __forceinline__ v3 centroid(float4 a, float4 b) { return mk3((a.x + b.x) * 0.5f, (a.y + b.y) * 0.5f, (a.z + b.z) * 0.5f); }

/* DPP moves within the wave; lanes without a source get `none`. */
template <int CTRL, int ROWS = 0xf> __device__ __forceinline__ int dpp(int none, int v) { return __builtin_amdgcn_update_dpp(none, v, CTRL, ROWS, 0xf, false); }
enum { ROW_SHL = 0x100, ROW_SHR = 0x110, BCAST15 = 0x142, BCAST31 = 0x143 };
__device__ __forceinline__ int imin(int a, int b) { return a < b ? a : b; }
__device__ __forceinline__ int imax(int a, int b) { return a > b ? a : b; }
/* minimum / maximum over the wave, in every lane */
__device__ __forceinline__ int wave_min(int v)
{
	v = imin(v, dpp<ROW_SHR + 1>(0x7fffffff, v)), v = imin(v, dpp<ROW_SHR + 2>(0x7fffffff, v));
	v = imin(v, dpp<ROW_SHR + 4>(0x7fffffff, v)), v = imin(v, dpp<ROW_SHR + 8>(0x7fffffff, v));
	v = imin(v, dpp<BCAST15, 0xa>(0x7fffffff, v)), v = imin(v, dpp<BCAST31, 0xc>(0x7fffffff, v));
	return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_max(int v) { return ~wave_min(~v); }

__global__ void k_tri_bounds(const float4* __restrict__ v, int n, float4* __restrict__ lo, float4* __restrict__ hi)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	const v3 a = xyz(v[3 * i]), b = xyz(v[3 * i + 1]), c = xyz(v[3 * i + 2]);
	const v3 l = kmin3(a, kmin3(b, c)), h = kmax3(a, kmax3(b, c));
	lo[i] = make_float4(l.x, l.y, l.z, 0.0f);
	hi[i] = make_float4(h.x, h.y, h.z, 0.0f);
}

/* One word of each record; bound by the 64-byte lines those words lie in. One
 * atomic per wave, at most 1024 of them in a launch. */
__global__ void k_max_word(const uint32_t* __restrict__ v, int stride, int n, uint32_t* __restrict__ out)
{
	uint32_t m = 0;
	for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) m = max(m, v[(size_t)i * stride]);
	m = (uint32_t)(wave_max((int)(m ^ 0x80000000u))) ^ 0x80000000u;
	if ((threadIdx.x & 63) == 0) atomicMax(out, m);
}

__global__ void k_build_init(BuildArgs A)
{
	if (threadIdx.x < 12) A.keys[threadIdx.x] = threadIdx.x % 6 < 3 ? KINF() : KNINF();
	if (threadIdx.x < 3) A.cnt[threadIdx.x] = threadIdx.x == 0 ? 1 : 0, A.start[threadIdx.x] = 0, A.head[threadIdx.x] = 0;
}

/* Identity order, root box and root centroid bounds: per block 12 atomics. */
__global__ void __launch_bounds__(256) k_root_bounds(BuildArgs A)
{
	__shared__ int s[4][12];
	int m[6], x[6];
	for (int k = 0; k < 6; k++) m[k] = KINF(), x[k] = KNINF();
	for (int i = blockIdx.x * 256 + threadIdx.x; i < A.n; i += gridDim.x * 256)
	{
		A.buf[0][i] = (uint32_t)i;
		const float4 a = A.lo[i], b = A.hi[i];
		const v3 c = centroid(a, b);
		m[0] = imin(m[0], fkey(a.x)), m[1] = imin(m[1], fkey(a.y)), m[2] = imin(m[2], fkey(a.z));
		x[0] = imax(x[0], fkey(b.x)), x[1] = imax(x[1], fkey(b.y)), x[2] = imax(x[2], fkey(b.z));
		m[3] = imin(m[3], fkey(c.x)), m[4] = imin(m[4], fkey(c.y)), m[5] = imin(m[5], fkey(c.z));
		x[3] = imax(x[3], fkey(c.x)), x[4] = imax(x[4], fkey(c.y)), x[5] = imax(x[5], fkey(c.z));
	}
	const int wave = threadIdx.x >> 6;
	for (int k = 0; k < 6; k++)
	{
		const int a = wave_min(m[k]), b = wave_max(x[k]), at = (k / 3) * 6 + k % 3;
		if ((threadIdx.x & 63) == 0) s[wave][at] = a, s[wave][at + 3] = b;
	}
	__syncthreads();
	if (threadIdx.x >= 12) return;
	int v = s[0][threadIdx.x];
	const bool isMin = threadIdx.x % 6 < 3;
	for (int w = 1; w < 4; w++) v = isMin ? imin(v, s[w][threadIdx.x]) : imax(v, s[w][threadIdx.x]);
	if (isMin) atomicMin(&A.keys[threadIdx.x], v);
	else atomicMax(&A.keys[threadIdx.x], v);
}

__device__ __forceinline__ int chunks_of(int cnt) { return (cnt + CHUNK - 1) / CHUNK; }

/* A new record of the level's big list (called by a whole wave): its place, its
 * chunks in the table, its scratch emptied. Returns the record's index. */
__device__ __forceinline__ int push_big(const BuildArgs& A, int level, int node, int start, int cnt, int lane)
{
	const int par = level & 1, nch = chunks_of(cnt);
	unsigned long long at = 0;
	if (lane == 0) at = atomicAdd(A.head + level, 1ull | (unsigned long long)nch << 32);
	const int rec = __builtin_amdgcn_readfirstlane((int)(uint32_t)at), chunk0 = __builtin_amdgcn_readfirstlane((int)(uint32_t)(at >> 32));
	if (lane == 0)
	{
		BigRec r = {};
		r.node = node, r.start = start, r.cnt = cnt, r.chunk0 = chunk0, r.childBig[0] = r.childBig[1] = -1;
		A.big[par][rec] = r;
	}
	for (int i = lane; i < nch; i += 64) A.table[par][chunk0 + i] = rec;
	int* s = A.scr[par] + (size_t)rec * S_STRIDE;
	for (int i = lane; i < S_BINS + B_SIZE; i += 64)
		s[i] = i < S_CMAX ? KINF() : i < S_BINS ? KNINF() : i < S_BINS + B_LO ? 0 : i < S_BINS + B_HI ? KINF() : KNINF();
	return rec;
}

__global__ void __launch_bounds__(64) k_root_node(BuildArgs A)
{
	const int lane = threadIdx.x;
	if (lane == 0)
	{
		BuildNode r;
		for (int c = 0; c < 3; c++) r.lo[c] = keyf(A.keys[c]), r.hi[c] = keyf(A.keys[3 + c]);
		r.leftFirst = 0, r.count = A.n;
		A.nodes[0] = r;
	}
	if (A.n <= SMALL) return;
	push_big(A, 0, 0, 0, A.n, lane);
	if (lane < 6) A.scr[0][lane] = A.keys[6 + lane];
}

/* scale of a valid axis from its centroid bounds' keys */
__device__ __forceinline__ bool axis_scale(int kmin, int kmax, float& cmin, float& scale)
{
	cmin = keyf(kmin);
	const float ext = keyf(kmax) - cmin;
	if (!(ext > 0.0f)) return false;
	scale = 16.0f / ext;
	return scale < __builtin_huge_valf();
}

__device__ __forceinline__ int bin_of(float c, float cmin, float scale)
{
	const int b = (int)((c - cmin) * scale);
	return b > BINS - 1 ? BINS - 1 : b < 0 ? 0 : b;
}

/* Adds a primitive to bins (LDS). */
__device__ __forceinline__ void bin_add(int* bins, int a, int b, float4 lo, float4 hi)
{
	const int slot = a * BINS + b;
	atomicAdd(&bins[B_CNT + slot], 1);
	atomicMin(&bins[B_LO + slot * 3 + 0], fkey(lo.x)), atomicMin(&bins[B_LO + slot * 3 + 1], fkey(lo.y)), atomicMin(&bins[B_LO + slot * 3 + 2], fkey(lo.z));
	atomicMax(&bins[B_HI + slot * 3 + 0], fkey(hi.x)), atomicMax(&bins[B_HI + slot * 3 + 1], fkey(hi.y)), atomicMax(&bins[B_HI + slot * 3 + 2], fkey(hi.z));
}

struct Split
{
	int mode, split, left;       /* mode -1: none */
	float cost;
	v3 Llo, Lhi, Rlo, Rhi;
};

/* The best split of a node from its bins: lane 16 a + i holds bin i of axis a
 * (a DPP row per axis); inclusive scans from both ends give every split's two
 * sides at once. All 64 lanes call it. valid: bit a set when axis a is valid. */
__device__ __forceinline__ Split best_split(const int* bins, int valid, int lane)
{
	const int a = lane >> 4, i = lane & 15;
	const bool in = lane < 48;
	int c = in ? bins[B_CNT + lane] : 0, m[3], x[3];
	for (int k = 0; k < 3; k++) m[k] = in ? bins[B_LO + lane * 3 + k] : KINF(), x[k] = in ? bins[B_HI + lane * 3 + k] : KNINF();
	int lc = c, rc = c, lm[3], lx[3], rm[3], rx[3];
	for (int k = 0; k < 3; k++) lm[k] = rm[k] = m[k], lx[k] = rx[k] = x[k];
#define SCAN(S) \
	lc += dpp<ROW_SHR + S>(0, lc), rc += dpp<ROW_SHL + S>(0, rc); \
	for (int k = 0; k < 3; k++) \
	{ \
		lm[k] = imin(lm[k], dpp<ROW_SHR + S>(0x7fffffff, lm[k])), lx[k] = imax(lx[k], dpp<ROW_SHR + S>((int)0x80000000, lx[k])); \
		rm[k] = imin(rm[k], dpp<ROW_SHL + S>(0x7fffffff, rm[k])), rx[k] = imax(rx[k], dpp<ROW_SHL + S>((int)0x80000000, rx[k])); \
	}
	SCAN(1) SCAN(2) SCAN(4) SCAN(8)
#undef SCAN
	/* the right side of the split after bin i starts at bin i + 1 */
	rc = dpp<ROW_SHL + 1>(0, rc);
	for (int k = 0; k < 3; k++) rm[k] = dpp<ROW_SHL + 1>(KINF(), rm[k]), rx[k] = dpp<ROW_SHL + 1>(KNINF(), rx[k]);
	const v3 Llo = mk3(keyf(lm[0]), keyf(lm[1]), keyf(lm[2])), Lhi = mk3(keyf(lx[0]), keyf(lx[1]), keyf(lx[2]));
	const v3 Rlo = mk3(keyf(rm[0]), keyf(rm[1]), keyf(rm[2])), Rhi = mk3(keyf(rx[0]), keyf(rx[1]), keyf(rx[2]));
	const float la = half_area(Llo, Lhi), ra = half_area(Rlo, Rhi);
	const float cost = (lc == 0 || rc == 0) ? __builtin_huge_valf() : (float)lc * la + (float)rc * ra;
	const bool can = in && i < BINS - 1 && ((valid >> a) & 1) && cost < __builtin_huge_valf();
	const int best = wave_min(can ? fkey(cost) : 0x7fffffff);
	const uint64_t at = __ballot(can && fkey(cost) == best);
	Split s;
	s.mode = -1, s.split = 0, s.left = 0, s.cost = __builtin_huge_valf();
	if (at == 0) return s;
	const int w = __ffsll((unsigned long long)at) - 1;     /* the first axis and bin of the minimum */
	const auto rl = [&](float v) { return bitsf((uint32_t)__builtin_amdgcn_readlane((int)fbits(v), w)); };
	s.mode = w >> 4, s.split = w & 15, s.left = __builtin_amdgcn_readlane(lc, w), s.cost = rl(cost);
	s.Llo = mk3(rl(Llo.x), rl(Llo.y), rl(Llo.z)), s.Lhi = mk3(rl(Lhi.x), rl(Lhi.y), rl(Lhi.z));
	s.Rlo = mk3(rl(Rlo.x), rl(Rlo.y), rl(Rlo.z)), s.Rhi = mk3(rl(Rhi.x), rl(Rhi.y), rl(Rhi.z));
	return s;
}

/* No valid axis: the range halved by position, the halves' boxes. */
__device__ __forceinline__ Split half_split(const BuildArgs& A, const uint32_t* prims, int start, int cnt, int lane)
{
	Split s;
	s.mode = 3, s.split = 0, s.left = cnt / 2, s.cost = 0.0f;
	int m[6], x[6];
	for (int k = 0; k < 6; k++) m[k] = KINF(), x[k] = KNINF();
	for (int i = lane; i < cnt; i += 64)
	{
		const uint32_t p = prims[start + i];
		const float4 l = A.lo[p], h = A.hi[p];
		const int o = i < s.left ? 0 : 3;
		m[o] = imin(m[o], fkey(l.x)), m[o + 1] = imin(m[o + 1], fkey(l.y)), m[o + 2] = imin(m[o + 2], fkey(l.z));
		x[o] = imax(x[o], fkey(h.x)), x[o + 1] = imax(x[o + 1], fkey(h.y)), x[o + 2] = imax(x[o + 2], fkey(h.z));
	}
	float lo[6], hi[6];
	for (int k = 0; k < 6; k++) lo[k] = keyf(wave_min(m[k])), hi[k] = keyf(wave_max(x[k]));
	s.Llo = mk3(lo[0], lo[1], lo[2]), s.Lhi = mk3(hi[0], hi[1], hi[2]), s.Rlo = mk3(lo[3], lo[4], lo[5]), s.Rhi = mk3(hi[3], hi[4], hi[5]);
	return s;
}

/* Split or leaf (mode -1) by the rules above. */
__device__ __forceinline__ Split decide(const BuildArgs& A, const BuildNode& nd, const int* bins, int valid, const uint32_t* prims, int lane)
{
	Split s = best_split(bins, valid, lane);
	if (s.mode < 0) return nd.count <= A.maxDegen ? s : half_split(A, prims, nd.leftFirst, nd.count, lane);
	const float area = half_area(mk3(nd.lo[0], nd.lo[1], nd.lo[2]), mk3(nd.hi[0], nd.hi[1], nd.hi[2]));
	if (nd.count <= A.maxLeaf && !(area + s.cost < (float)nd.count * area)) s.mode = -1;
	return s;
}

__device__ __forceinline__ void write_children(const BuildArgs& A, int node, const BuildNode& nd, const Split& s, int child)
{
	BuildNode L, R;
	L.lo[0] = s.Llo.x, L.lo[1] = s.Llo.y, L.lo[2] = s.Llo.z, L.hi[0] = s.Lhi.x, L.hi[1] = s.Lhi.y, L.hi[2] = s.Lhi.z;
	R.lo[0] = s.Rlo.x, R.lo[1] = s.Rlo.y, R.lo[2] = s.Rlo.z, R.hi[0] = s.Rhi.x, R.hi[1] = s.Rhi.y, R.hi[2] = s.Rhi.z;
	L.leftFirst = nd.leftFirst, L.count = s.left;
	R.leftFirst = nd.leftFirst + s.left, R.count = nd.count - s.left;
	A.nodes[child] = L, A.nodes[child + 1] = R;
	A.nodes[node].leftFirst = child, A.nodes[node].count = 0;
}

/* Bins of the level's big nodes, a block per chunk. */
__global__ void __launch_bounds__(256) k_big_bin(BuildArgs A, int d)
{
	__shared__ int s[B_SIZE];
	const int par = d & 1, chunks = (int)(A.head[d] >> 32);
	for (int ch = blockIdx.x; ch < chunks; ch += gridDim.x)
	{
		const int rec = A.table[par][ch];
		const BigRec& r = A.big[par][rec];
		int* g = A.scr[par] + (size_t)rec * S_STRIDE;
		const int p0 = r.start + (ch - r.chunk0) * CHUNK, p1 = imin(p0 + CHUNK, r.start + r.cnt);
		float cmin[3], scale[3];
		bool ok[3];
		for (int a = 0; a < 3; a++) ok[a] = axis_scale(g[S_CMIN + a], g[S_CMAX + a], cmin[a], scale[a]);
		for (int i = threadIdx.x; i < B_SIZE; i += 256) s[i] = i < B_LO ? 0 : i < B_HI ? KINF() : KNINF();
		__syncthreads();
		for (int p = p0 + (int)threadIdx.x; p < p1; p += 256)
		{
			const uint32_t prim = A.buf[par][p];
			const float4 lo = A.lo[prim], hi = A.hi[prim];
			const v3 c = centroid(lo, hi);
			for (int a = 0; a < 3; a++)
				if (ok[a]) bin_add(s, a, bin_of(comp(c, a), cmin[a], scale[a]), lo, hi);
		}
		__syncthreads();
		for (int i = threadIdx.x; i < B_SIZE; i += 256)
		{
			const int v = s[i];
			if (s[B_CNT + (i < B_LO ? i : i < B_HI ? (i - B_LO) / 3 : (i - B_HI) / 3)] == 0) continue;   /* an empty bin */
			if (i < B_LO) atomicAdd(&g[S_BINS + i], v);
			else if (i < B_HI) atomicMin(&g[S_BINS + i], v);
			else atomicMax(&g[S_BINS + i], v);
		}
		__syncthreads();
	}
}

/* Splits of the level's big nodes, a wave each. */
__global__ void __launch_bounds__(256) k_big_decide(BuildArgs A, int d)
{
	const int lane = threadIdx.x & 63, par = d & 1, count = (int)(uint32_t)A.head[d];
	const int next = A.start[d] + A.cnt[d];
	for (int rec = blockIdx.x * 4 + (threadIdx.x >> 6); rec < count; rec += gridDim.x * 4)
	{
		BigRec& r = A.big[par][rec];
		const int* g = A.scr[par] + (size_t)rec * S_STRIDE;
		const int node = r.node;
		const BuildNode nd = A.nodes[node];
		int valid = 0;
		for (int a = 0; a < 3; a++)
		{
			float cmin, scale;
			if (axis_scale(g[S_CMIN + a], g[S_CMAX + a], cmin, scale)) valid |= 1 << a;
		}
		const Split s = decide(A, nd, g + S_BINS, valid, A.buf[par], lane);
		int child = 0;
		if (s.mode >= 0)
		{
			if (lane == 0) child = next + atomicAdd(A.cnt + d + 1, 2);
			child = __builtin_amdgcn_readfirstlane(child);
			const int cl = s.left, cr = nd.count - s.left;
			const int bl = cl > SMALL ? push_big(A, d + 1, child, nd.leftFirst, cl, lane) : -1;
			const int br = cr > SMALL ? push_big(A, d + 1, child + 1, nd.leftFirst + cl, cr, lane) : -1;
			if (lane == 0)
			{
				write_children(A, node, nd, s, child);
				r.childBig[0] = bl, r.childBig[1] = br;
				r.cursor[0] = nd.leftFirst, r.cursor[1] = nd.leftFirst + cl;
			}
		}
		if (lane == 0) r.mode = s.mode, r.split = s.split, r.left = s.left, r.child = child;
	}
}

/* Partition of the level's big nodes into the other buffer (a leaf's primitives
 * to the output), a block per chunk: one atomic per chunk and side reserves its places. Children that are big get
 * their centroid bounds here. */
__global__ void __launch_bounds__(256) k_big_part(BuildArgs A, int d)
{
	__shared__ int nl[4], nr[4], base[2], box[4][12];
	constexpr int PER = CHUNK / 256;
	const int par = d & 1, chunks = (int)(A.head[d] >> 32), wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
	for (int ch = blockIdx.x; ch < chunks; ch += gridDim.x)
	{
		const int rec = A.table[par][ch];
		BigRec& r = A.big[par][rec];
		const int* g = A.scr[par] + (size_t)rec * S_STRIDE;
		const int mode = r.mode, p0 = r.start + (ch - r.chunk0) * CHUNK, p1 = imin(p0 + CHUNK, r.start + r.cnt);
		float cmin = 0.0f, scale = 0.0f;
		if (mode >= 0 && mode < 3) (void)axis_scale(g[S_CMIN + mode], g[S_CMAX + mode], cmin, scale);
		uint32_t prim[PER], leftBits = 0;
		int m[6], x[6], wl = 0, wr = 0;
		for (int k = 0; k < 6; k++) m[k] = KINF(), x[k] = KNINF();
#pragma unroll
		for (int k = 0; k < PER; k++)
		{
			const int p = p0 + k * 256 + (int)threadIdx.x;
			bool left = false;
			if (p < p1)
			{
				prim[k] = A.buf[par][p];
				const v3 c = centroid(A.lo[prim[k]], A.hi[prim[k]]);
				left = mode == 3 ? p - r.start < r.left : bin_of(comp(c, mode), cmin, scale) <= r.split;
				if (left)
				{
					m[0] = imin(m[0], fkey(c.x)), m[1] = imin(m[1], fkey(c.y)), m[2] = imin(m[2], fkey(c.z));
					x[0] = imax(x[0], fkey(c.x)), x[1] = imax(x[1], fkey(c.y)), x[2] = imax(x[2], fkey(c.z));
				}
				else
				{
					m[3] = imin(m[3], fkey(c.x)), m[4] = imin(m[4], fkey(c.y)), m[5] = imin(m[5], fkey(c.z));
					x[3] = imax(x[3], fkey(c.x)), x[4] = imax(x[4], fkey(c.y)), x[5] = imax(x[5], fkey(c.z));
				}
			}
			if (left) leftBits |= 1u << k;
			wl += __popcll(__ballot(left)), wr += __popcll(__ballot(p < p1 && !left));
		}
		if (lane == 0) nl[wave] = wl, nr[wave] = wr;
		const int bl = r.childBig[0], br = r.childBig[1];
		if (bl >= 0 || br >= 0)
			for (int k = 0; k < 6; k++)
			{
				const int a = wave_min(m[k]), b = wave_max(x[k]), at = (k / 3) * 6 + k % 3;
				if (lane == 0) box[wave][at] = a, box[wave][at + 3] = b;
			}
		__syncthreads();
		if (threadIdx.x < 12 && (bl >= 0 || br >= 0))
		{
			const int t = threadIdx.x, side = t / 6, f = t % 6;
			int v = box[0][t];
			for (int w = 1; w < 4; w++) v = f < 3 ? imin(v, box[w][t]) : imax(v, box[w][t]);
			const int cb = side ? br : bl;
			if (cb >= 0)
			{
				int* s = A.scr[par ^ 1] + (size_t)cb * S_STRIDE;
				if (f < 3) atomicMin(&s[S_CMIN + f], v);
				else atomicMax(&s[S_CMAX + f - 3], v);
			}
		}
		if (threadIdx.x == 64)
		{
			const int l = nl[0] + nl[1] + nl[2] + nl[3], q = nr[0] + nr[1] + nr[2] + nr[3];
			base[0] = l ? atomicAdd(&r.cursor[0], l) : 0, base[1] = q ? atomicAdd(&r.cursor[1], q) : 0;
		}
		__syncthreads();
		int atL = base[0], atR = base[1];
		for (int w = 0; w < wave; w++) atL += nl[w], atR += nr[w];
#pragma unroll
		for (int k = 0; k < PER; k++)
		{
			const int p = p0 + k * 256 + (int)threadIdx.x;
			const bool in = p < p1, left = in && ((leftBits >> k) & 1u);
			const uint64_t bmL = __ballot(left), bmR = __ballot(in && !left), mine = left ? bmL : bmR;
			const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mine >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mine, 0u));
			if (in && mode >= 0) A.buf[par ^ 1][(mode == 3 ? p : (left ? atL : atR) + rank)] = prim[k];
			else if (in) A.out[p] = prim[k];
			atL += __popcll(bmL), atR += __popcll(bmR);
		}
		__syncthreads();
	}
}

/* All nodes of a level with at most SMALL primitives, a wave per node; the
 * block's splits take their children's ids with one atomic. */
__global__ void __launch_bounds__(64 * LEVEL_WAVES) k_level(BuildArgs A, int d)
{
	__shared__ int sbins[LEVEL_WAVES][B_SIZE];
	__shared__ int nSplit[2][LEVEL_WAVES], first[2];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, par = d & 1;
	const int begin = A.start[d], count = A.cnt[d], next = begin + count;
	if (blockIdx.x == 0 && threadIdx.x == 0) A.start[d + 1] = next, A.cnt[d + 2] = 0, A.head[d + 2] = 0;
	const uint32_t* prims = A.buf[par];
	int* bins = sbins[wave];
	int flip = 0;
	for (int i0 = blockIdx.x * LEVEL_WAVES; i0 < count; i0 += gridDim.x * LEVEL_WAVES, flip ^= 1)
	{
		const int node = begin + i0 + wave;
		BuildNode nd;
		nd.leftFirst = 0, nd.count = 0;
		if (i0 + wave < count) nd = A.nodes[node];
		const int start = nd.leftFirst, cnt = nd.count <= SMALL ? nd.count : 0;   /* 0: interior (a big node just split) or not ours */
		Split s;
		s.mode = -1;
		uint32_t prim = 0;
		float4 lo = make_float4(0, 0, 0, 0), hi = lo;
		float cmin[3] = { 0, 0, 0 }, scale[3] = { 0, 0, 0 };
		if (lane < cnt) prim = prims[start + lane];
		if (cnt > 1)
		{
			if (lane < cnt) lo = A.lo[prim], hi = A.hi[prim];
			/* centroid bounds; the first 64 primitives stay in registers */
			int m[3] = { KINF(), KINF(), KINF() }, x[3] = { KNINF(), KNINF(), KNINF() };
			const auto grow = [&](float4 l, float4 h) {
				const v3 c = centroid(l, h);
				m[0] = imin(m[0], fkey(c.x)), m[1] = imin(m[1], fkey(c.y)), m[2] = imin(m[2], fkey(c.z));
				x[0] = imax(x[0], fkey(c.x)), x[1] = imax(x[1], fkey(c.y)), x[2] = imax(x[2], fkey(c.z));
			};
			if (lane < cnt) grow(lo, hi);
			for (int i = lane + 64; i < cnt; i += 64)
			{
				const uint32_t p = prims[start + i];
				grow(A.lo[p], A.hi[p]);
			}
			int valid = 0;
			for (int a = 0; a < 3; a++)
				if (axis_scale(wave_min(m[a]), wave_max(x[a]), cmin[a], scale[a])) valid |= 1 << a;
			for (int i = lane; i < B_SIZE; i += 64) bins[i] = i < B_LO ? 0 : i < B_HI ? KINF() : KNINF();
			const auto add = [&](float4 l, float4 h) {
				const v3 c = centroid(l, h);
				for (int a = 0; a < 3; a++)
					if ((valid >> a) & 1) bin_add(bins, a, bin_of(comp(c, a), cmin[a], scale[a]), l, h);
			};
			if (lane < cnt) add(lo, hi);
			for (int i = lane + 64; i < cnt; i += 64)
			{
				const uint32_t p = prims[start + i];
				add(A.lo[p], A.hi[p]);
			}
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
			s = decide(A, nd, bins, valid, prims, lane);
		}
		if (lane == 0) nSplit[flip][wave] = s.mode >= 0 ? 1 : 0;
		__syncthreads();
		if (threadIdx.x == 0)
		{
			int t = 0;
			for (int w = 0; w < LEVEL_WAVES; w++) t += nSplit[flip][w];
			first[flip] = t ? atomicAdd(A.cnt + d + 1, 2 * t) : 0;
		}
		__syncthreads();
		if (cnt == 0) continue;
		if (s.mode < 0)
		{	/* leaf */
			if (lane < cnt) A.out[start + lane] = prim;
			for (int i = lane + 64; i < cnt; i += 64) A.out[start + i] = prims[start + i];
			continue;
		}
		int child = next + first[flip];
		for (int w = 0; w < wave; w++) child += 2 * nSplit[flip][w];
		if (lane == 0) write_children(A, node, nd, s, child);
		/* stable partition into the other buffer */
		int atL = start, atR = start + s.left;
		const float c0 = s.mode < 3 ? cmin[s.mode == 0 ? 0 : s.mode == 1 ? 1 : 2] : 0.0f, sc = s.mode < 3 ? scale[s.mode == 0 ? 0 : s.mode == 1 ? 1 : 2] : 0.0f;
		for (int i = lane; i - lane < cnt; i += 64)
		{
			const bool in = i < cnt;
			if (i >= 64 && in) prim = prims[start + i], lo = A.lo[prim], hi = A.hi[prim];
			const v3 c = centroid(lo, hi);
			const bool left = in && (s.mode == 3 ? i < s.left : bin_of(comp(c, s.mode), c0, sc) <= s.split);
			const uint64_t bmL = __ballot(left), bmR = __ballot(in && !left), mine = left ? bmL : bmR;
			const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mine >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mine, 0u));
			if (in) A.buf[par ^ 1][(left ? atL : atR) + rank] = prim;
			atL += __popcll(bmL), atR += __popcll(bmR);
		}
	}
}

#define CK(x) do { const hipError_t e_ = (x); if (e_ != hipSuccess) return e_; } while (0)

hipError_t tri_bounds(const float4* dVerts, int n, float4* dLo, float4* dHi, hipStream_t stream)
{
	if (n <= 0) return hipSuccess;
	k_tri_bounds<<<(n + 255) / 256, 256, 0, stream>>>(dVerts, n, dLo, dHi);
	return hipGetLastError();
}

hipError_t max_word(const uint32_t* dRecords, int stride, int n, uint32_t* dMax, hipStream_t stream)
{
	if (n <= 0) return hipSuccess;
	k_max_word<<<std::min((n + 255) / 256, 256), 256, 0, stream>>>(dRecords, stride, n, dMax);
	return hipGetLastError();
}

/* Workspace: two id buffers, level counters, big lists (at most n / (SMALL + 1)
 * big nodes per level and one chunk more than CHUNK-sized pieces per node). */
static int max_big(int n) { return n / (SMALL + 1) + 1; }
static int max_chunks(int n) { return n / CHUNK + max_big(n) + 1; }
static size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

static size_t carve(char* base, int n, BuildArgs& A)
{
	size_t at = 0;
	const auto take = [&](size_t bytes) { char* p = base ? base + at : nullptr; at += up256(bytes); return (void*)p; };
	for (int i = 0; i < 2; i++) A.buf[i] = (uint32_t*)take(sizeof(uint32_t) * (size_t)n);
	A.cnt = (int*)take(sizeof(int) * (MAX_LEVELS + 4)), A.start = (int*)take(sizeof(int) * (MAX_LEVELS + 4));
	A.head = (unsigned long long*)take(sizeof(unsigned long long) * (MAX_LEVELS + 4));
	A.keys = (int*)take(sizeof(int) * 16);
	const int big = n > SMALL ? max_big(n) : 0;
	for (int i = 0; i < 2; i++)
	{
		A.big[i] = (BigRec*)take(sizeof(BigRec) * (size_t)big);
		A.scr[i] = (int*)take(sizeof(int) * (size_t)big * S_STRIDE);
		A.table[i] = (int*)take(sizeof(int) * (size_t)(n > SMALL ? max_chunks(n) : 0));
	}
	return at;
}

size_t gpu_build_workspace_bytes(int n)
{
	BuildArgs A;
	return n > 0 ? carve(nullptr, n, A) : 0;
}

static int log2_ceil(int v) { int k = 0; while (((int64_t)1 << k) < v) k++; return k; }

hipError_t gpu_build(const float4* dLo, const float4* dHi, int n, int maxLeaf, int maxDegen, DeviceBuild& out, void* ws, size_t wsBytes, hipStream_t stream)
{
	out.primCount = n, out.nodeCount = 0, out.depth = 0;
	out.levelStart.clear();
	if (n <= 0) return hipSuccess;
	if (!ws || !out.nodes || !out.prims || wsBytes < gpu_build_workspace_bytes(n)) return hipErrorInvalidValue;
	BuildArgs A;
	(void)carve((char*)ws, n, A);
	A.nodes = out.nodes, A.out = out.prims, A.lo = dLo, A.hi = dHi, A.n = n, A.maxLeaf = maxLeaf, A.maxDegen = maxDegen;
	k_build_init<<<1, 64, 0, stream>>>(A);
	k_root_bounds<<<std::min((n + 1023) / 1024, 1024), 256, 0, stream>>>(A);
	k_root_node<<<1, 64, 0, stream>>>(A);
	int d = 0;                         /* levels launched */
	const auto levels = [&](int k, bool big) {
		for (; k > 0 && d < MAX_LEVELS; k--, d++)
		{
			/* a level has at most 2^d nodes and n / 2 splits; the kernels step over what the grid does not cover */
			const int nodes = d < 20 ? std::min(1 << d, n) : n;
			if (big)
			{
				const int chunks = std::min(max_chunks(n), n / CHUNK + (d < 20 ? 1 << d : n) + 1);
				k_big_bin<<<std::min(chunks, 4096), 256, 0, stream>>>(A, d);
				k_big_decide<<<std::min((std::min(max_big(n), nodes) + 3) / 4, 2048), 256, 0, stream>>>(A, d);
				k_big_part<<<std::min(chunks, 4096), 256, 0, stream>>>(A, d);
			}
			k_level<<<std::min((nodes + LEVEL_WAVES - 1) / LEVEL_WAVES, 2048), 64 * LEVEL_WAVES, 0, stream>>>(A, d);
		}
	};
	/* Levels with big nodes until none is left, then the others; each batch as
	 * deep as a balanced tree would be and a few levels more, so that the host
	 * looks two or three times. */
	if (n > SMALL)
		for (int batch = log2_ceil(n / SMALL + 1) + 1;; batch = 2)
		{
			levels(batch, true);
			unsigned long long left = 0;
			CK(hipGetLastError());
			CK(hipMemcpyAsync(&left, A.head + d, sizeof(left), hipMemcpyDeviceToHost, stream));
			CK(hipStreamSynchronize(stream));
			if ((uint32_t)left == 0) break;
			if (d >= MAX_LEVELS) return hipErrorInvalidValue;
		}
	std::vector<int> cnt;
	int total = 0;
	for (int batch = log2_ceil(std::min(n, SMALL)) + 4;; batch = 4)
	{
		levels(batch, false);
		const int from = (int)cnt.size();
		cnt.resize(d + 1);
		CK(hipGetLastError());
		CK(hipMemcpyAsync(cnt.data() + from, A.cnt + from, sizeof(int) * (size_t)(d + 1 - from), hipMemcpyDeviceToHost, stream));
		CK(hipStreamSynchronize(stream));
		if (cnt.back() == 0) break;
		if (d >= MAX_LEVELS) return hipErrorInvalidValue;
		cnt.pop_back();                /* level d's node count is final, but its level is still to run */
	}
	for (size_t k = 0; k < cnt.size() && cnt[k] > 0; k++) out.levelStart.push_back(total), total += cnt[k], out.depth++;
	out.levelStart.push_back(total);
	out.nodeCount = total;
	return hipSuccess;
}

/* min / max in std::min / std::max form, (b < a) ? b : a and (a < b) ? b : a:
 * a NaN operand resolves the same way as in the oracle's builder. */
__device__ __forceinline__ float smin(float a, float b) { return (b < a) ? b : a; }
__device__ __forceinline__ float smax(float a, float b) { return (a < b) ? b : a; }

__device__ __forceinline__ void refit_node(BuildNode* __restrict__ nodes, const uint32_t* __restrict__ prims, const float4* __restrict__ v, int x)
{
	const BuildNode b = nodes[x];
	float lo[3] = { INFINITY, INFINITY, INFINITY }, hi[3] = { -INFINITY, -INFINITY, -INFINITY };
	if (b.count > 0)
		for (int k = 0; k < b.count; k++)
		{
			const float4* t = v + 3 * (size_t)prims[b.leftFirst + k];
			const float4 p0 = t[0], p1 = t[1], p2 = t[2];
			const float a0[3] = { p0.x, p0.y, p0.z }, a1[3] = { p1.x, p1.y, p1.z }, a2[3] = { p2.x, p2.y, p2.z };
			for (int c = 0; c < 3; c++)
				lo[c] = smin(lo[c], smin(smin(a0[c], a1[c]), a2[c])), hi[c] = smax(hi[c], smax(smax(a0[c], a1[c]), a2[c]));
		}
	else
		for (int k = 0; k < 2; k++)
		{
			const BuildNode ch = nodes[b.leftFirst + k];
			for (int c = 0; c < 3; c++) lo[c] = smin(lo[c], ch.lo[c]), hi[c] = smax(hi[c], ch.hi[c]);
		}
	for (int c = 0; c < 3; c++) nodes[x].lo[c] = lo[c], nodes[x].hi[c] = hi[c];
}

__global__ void k_refit_level(BuildNode* nodes, const uint32_t* prims, const float4* v, int first, int count)
{
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < count) refit_node(nodes, prims, v, first + i);
}

/* Several levels in one block, deepest first. */
__global__ void __launch_bounds__(LEVELS_BLOCK) k_refit_levels(BuildNode* nodes, const uint32_t* prims, const float4* v, const LevelRange r)
{
	for (int d = r.n - 1; d >= 0; d--)
	{
		for (int x = r.s[d] + (int)threadIdx.x; x < r.s[d + 1]; x += LEVELS_BLOCK) refit_node(nodes, prims, v, x);
		__syncthreads();
	}
}

hipError_t refit_levels(BuildNode* dNodes, const uint32_t* dPrims, const float4* dVerts, const std::vector<int>& levelStart, hipStream_t stream)
{
	for (int d = (int)levelStart.size() - 1; d > 0;)
	{
		const LevelRange r = small_levels(levelStart, d, false);
		if (r.n > 1) k_refit_levels<<<1, LEVELS_BLOCK, 0, stream>>>(dNodes, dPrims, dVerts, r), d -= r.n;
		else
		{
			const int first = levelStart[d - 1], count = levelStart[d] - first;
			k_refit_level<<<(count + 255) / 256, 256, 0, stream>>>(dNodes, dPrims, dVerts, first, count), d--;
		}
	}
	return hipGetLastError();
}

} // namespace lh
