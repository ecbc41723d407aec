/* kernel_checks.hip - entry points for tests of what the C ABI does not reach:
 * the traversal's stacks (run on the host), the builder with leaves of any size and
 * the short forms of the math functions.
 * Built beside the library into tests/bin/libkernel_checks.so. */
#include "../lighthouse2_amd/csrc/trace_stack.h"
#include "../lighthouse2_amd/csrc/bvh.h"
#include "../lighthouse2_amd/csrc/lh_math.h"
#include <vector>

using namespace lh;

#define CHECK_API extern "C" __attribute__((visibility("default")))

/* ---- stacks ----------------------------------------------------------------
 * Random visits (up to three entries on top) and pops beside a plain array that
 * drops what goes beyond TRACE_MAX_STACK. The overflow area lies between words
 * that no pop may return. Returns the first step that differs, or -1. */
static uint32_t next(uint32_t& s) { s ^= s << 13; s ^= s >> 17; s ^= s << 5; return s; }

struct Model
{
	std::vector<uint32_t> v;
	void push(uint32_t x) { if ((int)v.size() < TRACE_MAX_STACK) v.push_back(x); }
	uint32_t pop() { const uint32_t x = v.back(); v.pop_back(); return x; }
};

template <typename STACK, typename VISIT>
static int run_stack(STACK& st, int ldsWords, int ovfWords, uint32_t seed, int grow, VISIT visit)
{
	const int PAD = 1024;
	std::vector<uint32_t> lds(ldsWords, 0xbad0bad0u), ovf(PAD + ovfWords + PAD, 0xbad0bad0u);
	st.lds = (lds_u32*)lds.data(), st.ovf = ovf.data() + PAD, st.sp = 0;
	Model m;
	for (int step = 0; step < 4000; step++)
	{
		const bool up = (int)(next(seed) % 100) < ((step / 500) % 2 ? 100 - grow : grow);   /* phases of growing and of shrinking */
		if (up)
		{
			uint32_t e[3];
			const int n = 1 + (int)(next(seed) % 3);
			for (int k = 0; k < n; k++) e[k] = (uint32_t)(step * 4 + k), m.push(e[k]);
			visit(st, e, n);
		}
		else if (!m.v.empty() && st.pop() != m.pop()) return step;
		if (st.sp != (int)m.v.size()) return step;
	}
	while (!m.v.empty())
		if (st.pop() != m.pop()) return 4000;
	for (int k = 0; k < PAD; k++)
		if (ovf[k] != 0xbad0bad0u || ovf[PAD + ovfWords + k] != 0xbad0bad0u) return 4001;
	return -1;
}

template <int DEPTH, int STRIDE>
static int run_quad(uint32_t seed, int grow)
{
	QuadStack<DEPTH, STRIDE> st;
	st.col = (int)(seed % STRIDE);
	return run_stack(st, DEPTH * STRIDE, TRACE_MAX_STACK - DEPTH, seed, grow, [](QuadStack<DEPTH, STRIDE>& s, const uint32_t* e, int n) {
		for (int k = 0; k < n; k++) s.put(s.sp + k, e[k]);
		s.grow(n);
	});
}

/* which: 0 a lane's stack, 1 a quad's of a small launch, 2 a quad's that goes on with a lane's */
CHECK_API int check_stack(int which, uint32_t seed, int grow)
{
	if (which == 1) return run_quad<32, 16>(seed, grow);
	if (which == 2) return run_quad<TRACE_LDS_STACK, TRACE_BLOCK>(seed, grow);
	Stack<TRACE_BLOCK> st;
	st.tid = (int)(seed % TRACE_BLOCK);
	return run_stack(st, TRACE_LDS_STACK * TRACE_BLOCK, TRACE_OVF_STACK, seed, grow, [](Stack<TRACE_BLOCK>& s, const uint32_t* e, int n) {
		s.push3(e[0], true, n > 1 ? e[1] : 0, n > 1, n > 2 ? e[2] : 0, n > 2);
	});
}

/* ---- builder ------------------------------------------------------------------
 * gpu_build over n device boxes; nodes (2 n) and prims (n) are device memory,
 * wsBytes of them at ws (0: how many it needs, returned). Returns the node count,
 * or minus the error. */
CHECK_API int64_t check_build(const float4* lo, const float4* hi, int n, int maxLeaf, int maxDegenerateLeaf, BuildNode* nodes, uint32_t* prims, void* ws,
	uint64_t wsBytes)
{
	if (wsBytes == 0) return (int64_t)gpu_build_workspace_bytes(n);
	DeviceBuild b;
	b.nodes = nodes, b.prims = prims;
	const hipError_t e = gpu_build(lo, hi, n, maxLeaf, maxDegenerateLeaf, b, ws, (size_t)wsBytes, nullptr);
	return e == hipSuccess ? b.nodeCount : -(int64_t)e;
}

/* ---- short math ---------------------------------------------------------------
 * out[i] of n device floats: 0 rcp_tame(a), 1 sqrt_tame(a), 2 div_core(a, b), 3 exp_neg(a), 4 cw_expf(a). */
__global__ void k_short(int which, const float* a, const float* b, float* out, int n)
{
	for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
		out[i] = which == 0 ? rcp_tame(a[i]) : which == 1 ? sqrt_tame(a[i]) : which == 2 ? div_core(a[i], b[i]) : which == 3 ? exp_neg(a[i]) : cw_expf(a[i]);
}

CHECK_API int check_short(int which, const float* a, const float* b, float* out, int n)
{
	if (n <= 0 || which < 0 || which > 4 || !a || !out || (which == 2 && !b)) return (int)hipErrorInvalidValue;
	k_short<<<4096, 256>>>(which, a, b, out, n);
	return (int)hipGetLastError();
}
