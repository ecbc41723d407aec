/* trace_stack.h - the traversal's stacks of node references: the first entries in
 * LDS, the others in an overflow area in memory. Plain enough to run on the host. */
#pragma once
#include "trace.h"

namespace lh {

/* An LDS pointer typed as such, so that loads through it stay LDS loads. */
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) uint32_t lds_u32;
#else
typedef uint32_t lds_u32;
#endif

template <int BLOCK>
struct Stack
{
	lds_u32* lds;       /* TRACE_LDS_STACK x BLOCK */
	uint32_t* ovf;      /* this thread's overflow area */
	int tid, sp;
	/* The host checks that the tree depth fits TRACE_MAX_STACK; a push beyond
	 * it is dropped (never written out of bounds). */
	__host__ __device__ __forceinline__ void push(uint32_t v)
	{
		if (sp < TRACE_LDS_STACK) lds[sp * BLOCK + tid] = v, sp++;
		else if (sp < TRACE_MAX_STACK) ovf[sp - TRACE_LDS_STACK] = v, sp++;
	}
	/* Pushes c (bottom) if hc, then b if hb, then a (top) if ha. With room
	 * for three entries in LDS, every lane writes all three slots and only
	 * moves its stack pointer for the pushed ones: no divergent branch. */
	__host__ __device__ __forceinline__ void push3(uint32_t c, bool hc, uint32_t b, bool hb, uint32_t a, bool ha)
	{
		if (sp + 3 <= TRACE_LDS_STACK)
		{
			lds[sp * BLOCK + tid] = c;
			sp += hc ? 1 : 0;
			lds[sp * BLOCK + tid] = b;
			sp += hb ? 1 : 0;
			lds[sp * BLOCK + tid] = a;
			sp += ha ? 1 : 0;
		}
		else
		{
			if (hc) push(c);
			if (hb) push(b);
			if (ha) push(a);
		}
	}
	/* LDS read for every lane (the row clamped into the LDS part), the
	 * overflow area read only by lanes below it. */
	__host__ __device__ __forceinline__ uint32_t pop()
	{
		sp--;
		uint32_t v = lds[min(sp, TRACE_LDS_STACK - 1) * BLOCK + tid];
		if (sp >= TRACE_LDS_STACK) v = ovf[sp - TRACE_LDS_STACK];
		return v;
	}
};

/* One stack per ray, entries written by the quad's lanes: DEPTH in LDS
 * (interleaved over STRIDE rays), the others in the ray's overflow area. */
template <int DEPTH, int STRIDE>
struct QuadStack
{
	lds_u32* lds;
	uint32_t* ovf;
	int col, sp;
	__host__ __device__ __forceinline__ void put(int at, uint32_t v)
	{
		if (at < DEPTH) lds[at * STRIDE + col] = v;
		else if (at < TRACE_MAX_STACK) ovf[at - DEPTH] = v;
	}
	/* n entries were put on top; those beyond TRACE_MAX_STACK were dropped, as by Stack */
	__host__ __device__ __forceinline__ void grow(int n) { sp = min(sp + n, TRACE_MAX_STACK); }
	__host__ __device__ __forceinline__ uint32_t pop()
	{
		sp--;
		uint32_t v = lds[min(sp, DEPTH - 1) * STRIDE + col];
		if (sp >= DEPTH) v = ovf[sp - DEPTH];
		return v;
	}
};

} // namespace lh
