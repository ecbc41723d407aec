/* denoise.hip - learned-denoiser kernels for gfx950 (see denoise.h).
 *
 * Convolutions are implicit GEMMs on the matrix cores,
 * v_mfma_f32_16x16x16_bf16 (bf16 operands, fp32 accumulation). Operand
 * layout of one 16x16x16 product in a wave of 64 lanes: A[m][k] with
 * m = lane % 16, k = 4 (lane / 16) + i; B[k][n] with n = lane % 16,
 * k = 4 (lane / 16) + i; D[m][n] with n = lane % 16, m = 4 (lane / 16) + i
 * (i = 0..3 the element of the lane's 4-vector).
 *
 * Forward / input gradient: M = 64 output pixels of one row per wave, N =
 * output channels, K = 9 taps x input channels; activations are NHWC, so the
 * 4 k-values a lane needs are 4 consecutive channels of one pixel (one 8-byte
 * load) and the weights [tap][n][k] give the same for B.
 * Weight gradient: M = output channels, N = input channels, K = pixels; a
 * wave walks down a 32-pixel column segment with its rows staged as they lie
 * in memory and read through the transposing LDS read, so that both operands
 * get consecutive pixels; a second kernel adds the blocks' partial sums in a
 * fixed order (deterministic).
 */
#include "denoise.h"

#include <mutex>

namespace lh {

typedef short s4v __attribute__((__vector_size__(4 * sizeof(short))));
typedef float f4v __attribute__((__vector_size__(4 * sizeof(float))));

__device__ __forceinline__ float bf2f(bf16_t b) { return __builtin_bit_cast(float, (uint32_t)b << 16); }
/* round to nearest even, NaN stays a quiet NaN: v_cvt_pk_bf16_f32, whose result equals the
 * integer formula's for all 2^32 inputs (six instructions per value before) */
__device__ __forceinline__ bf16_t f2bf(float f) { return __builtin_bit_cast(bf16_t, (__bf16)f); }
__device__ __forceinline__ uint32_t pack_bf(float lo, float hi)
{
	typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
	const bf2v v = { (__bf16)lo, (__bf16)hi };
	return __builtin_bit_cast(uint32_t, v);
}

static bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }
static bool aligned16_3(const void* a, const void* b, const void* c) { return (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c) & 15) == 0; }

static const int DW_BLOCKS = 512;

/* ---- 3x3 convolution, forward and input gradient ------------------------ */
template <int NB, bool RELU, bool F32OUT>
__global__ void __launch_bounds__(256) k_conv3x3(const bf16_t* __restrict__ x, int Cin, const bf16_t* __restrict__ w,
	const float* __restrict__ bias, void* __restrict__ y, int H, int W)
{
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int row = blockIdx.y * 4 + wave;
	const int x0 = blockIdx.x * 64;
	if (row >= H) return;
	const int Cout = NB * 16;
	const int ml = lane & 15, kq = (lane >> 4) * 4;
	f4v acc[4][NB];
#pragma unroll
	for (int mb = 0; mb < 4; mb++)
#pragma unroll
		for (int nb = 0; nb < NB; nb++) acc[mb][nb] = (f4v){ 0.0f, 0.0f, 0.0f, 0.0f };
	for (int tap = 0; tap < 9; tap++)
	{
		const int yy = row + tap / 3 - 1, dx = tap % 3 - 1;
		const bool rowOk = yy >= 0 && yy < H;
		const bf16_t* xrow = x + (size_t)(rowOk ? yy : 0) * W * Cin;
		for (int c = 0; c < Cin; c += 16)
		{
			s4v b[NB];
#pragma unroll
			for (int nb = 0; nb < NB; nb++) b[nb] = *(const s4v*)(w + ((size_t)(tap * Cout + nb * 16 + ml) * Cin + c + kq));
#pragma unroll
			for (int mb = 0; mb < 4; mb++)
			{
				const int xx = x0 + mb * 16 + ml + dx;
				s4v a = (s4v){ 0, 0, 0, 0 };
				if (rowOk && xx >= 0 && xx < W) a = *(const s4v*)(xrow + (size_t)xx * Cin + c + kq);
#pragma unroll
				for (int nb = 0; nb < NB; nb++) acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b[nb], acc[mb][nb], 0, 0, 0);
			}
		}
	}
#pragma unroll
	for (int nb = 0; nb < NB; nb++)
	{
		const int ch = nb * 16 + ml;
		const float bv = bias ? bias[ch] : 0.0f;
#pragma unroll
		for (int mb = 0; mb < 4; mb++)
#pragma unroll
			for (int i = 0; i < 4; i++)
			{
				const int px = x0 + mb * 16 + kq + i;
				if (px >= W) continue;
				float v = acc[mb][nb][i] + bv;
				if (RELU) v = v > 0.0f ? v : 0.0f;
				const size_t o = ((size_t)row * W + px) * Cout + ch;
				if (F32OUT) ((float*)y)[o] = v;
				else ((bf16_t*)y)[o] = f2bf(v);
			}
	}
}

/* Decoders of the SVGF feature words (tools_shared.h:130-136,169-176):
 * albedo HDRtoRGB32 (10:11:11), normal PackNormal2, depth as float bits. */
__device__ __forceinline__ float3 feat_albedo(uint32_t c)
{
	return make_float3((float)(c >> 22) * (1.0f / 1023.0f), (float)((c >> 11) & 2047u) * (1.0f / 2047.0f), (float)(c & 2047u) * (1.0f / 2047.0f));
}
__device__ __forceinline__ float3 feat_normal(uint32_t p)
{
	return make_float3((float)((p >> 2) & 1023u) * (1.0f / 511.0f) - 1.0f, (float)((p >> 12) & 1023u) * (1.0f / 511.0f) - 1.0f,
		(float)(p >> 22) * (1.0f / 511.0f) - 1.0f);
}

static const float DN_ALBEDO_FLOOR = 0.02f;

/* The frame the output convolution's display variant (dn_conv3x3_display)
 * writes: features of the frame and its display image, w x h inside the
 * network's padded image. */
struct FrameIO
{
	const uint4* feat;
	int w, h;
	float4* image;
};

/* The display value of one pixel from the network's first 3 output channels,
 * as k_frame_output computes it. */
__device__ __forceinline__ float4 frame_display(float o0, float o1, float o2, uint32_t featX)
{
	const float3 a = feat_albedo(featX);
	const float o[3] = { o0, o1, o2 }, al[3] = { a.x, a.y, a.z };
	float v[3];
	for (int k = 0; k < 3; k++) v[k] = sqrtf(sqrtf(expm1f(fmaxf(o[k], 0.0f)) * fmaxf(al[k], DN_ALBEDO_FLOOR)));
	return make_float4(v[0], v[1], v[2], 0.0f);
}

typedef __bf16 bf8v __attribute__((ext_vector_type(8)));
/* What the epilogue does besides the plain store: IO_DISPLAY writes the display
 * image of a frame; IO_MASK zeroes outputs whose activation (the tensor `act`,
 * shaped like y) is not positive, the ReLU gradient of the layer below; IO_SPLIT
 * (64 outputs) is the gradient of the decoder's concatenation: channels 32..63
 * to y (the skip tensor), 2 x 2 sums of channels 0..31, masked by `act` (coarse
 * size), to ypool. */
enum { IO_NONE = 0, IO_DISPLAY = 1, IO_MASK = 2, IO_SPLIT = 3 };

/* dword of two bf16 gradients, each kept where its activation is positive */
__device__ __forceinline__ uint32_t relu_mask2(uint32_t act, uint32_t g)
{
	return (bf2f((bf16_t)(act & 0xffffu)) > 0.0f ? g & 0xffffu : 0u) | (bf2f((bf16_t)(act >> 16)) > 0.0f ? g & 0xffff0000u : 0u);
}

/* Tiled variants for the network's shapes (k_conv3x3_t for small images, k_conv_rows
 * for large ones). A block's pixels and their halo are staged once in LDS with
 * 16-byte loads, a thread's loads in flight together, CP channels per pixel (8 of
 * padding against bank conflicts). The 9 taps run as v_mfma_f32_16x16x32_bf16
 * products with A = 16 output channels x 32 input channels of the [tap][Cout][Cin]
 * weights and B = 32 input channels x 16 pixels from LDS (lane: pixel lane % 16,
 * channels 8 (lane / 16) + 0..7); D then gives each lane 4 consecutive output
 * channels of one pixel; bf16 outputs pair channel blocks across lanes for 16-byte
 * writes (below). CIN = 16 is padded to K = 32 with zero channels. CAT: the input is
 * the 64-channel concatenation [nearest 2x upsample of coarse (32 channels),
 * x (32 channels)]; the coarse pixels under the tile (and their halo) are staged
 * separately and upsampled by the fragment addressing. */

/* Large images: a wave computes 4 rows x 16 MBW pixels, a block's four waves a
 * tile of 16 MBW x 16, staged as above (18 of 16 rows are read; 8 x 64 tiles, 10
 * of 8). All nine taps' weight fragments sit in registers before the products
 * start, and an input row's fragment, read from LDS once per horizontal shift,
 * serves the up to three output rows it touches: 36 LDS reads for 144 products at
 * 32 -> 32 channels. (With a wave per row 36 reads served 72 products, and every
 * wave fetched every weight through L1 as it went, more bytes than the tile's own,
 * waiting at each tap.) A row's sums run over the taps in the same order, so the
 * results are those of the 16-pixel tiles bit for bit.
 *   LOOP, for 64 channels: the weights are 147 KB a block and 144 registers a lane,
 * so two blocks a CU stay and walk their XCD's tiles with them, one block's loads
 * under the other's products (a block per tile: 121 us for the decoder's first
 * convolution at 1920 x 1088, 100 -> 151 us for its gradient). With fewer weights
 * three blocks a CU hide the loads better than a loop does.
 *   Measured within forward passes and training steps at 1920 x 1088 (kernel trace;
 * in brackets the bytes a layer must move at a copy's 5.06 TB/s): 16 -> 32 55 us (40),
 * 32 -> 32 66 (53), with pooling 70 (59), 64 -> 32 89 (59), 32 -> 16 float 54 (53), display
 * 52; gradients 32 -> 32 94 (79), 16 -> 32 89 (66), 32 -> 64 104 (66). With a wave per row
 * the whole forward pass took 715 us where it now takes 450 to 475. Memory bounds all
 * but the 64-channel ones, which wait for it between their tiles' products as well. */
template <int CIN, int NB, bool RELU, bool F32OUT, bool CAT, bool POOL, int IO, int MBW>
__global__ void __launch_bounds__(256, NB == 4 || CIN == 64 ? 2 : 3) k_conv_rows(const bf16_t* __restrict__ x, const bf16_t* __restrict__ coarse,
	const bf16_t* __restrict__ w, const float* __restrict__ bias, void* __restrict__ y, int H, int W, bf16_t* __restrict__ ypool,
	FrameIO io, const bf16_t* __restrict__ act, int across, int tiles)
{
	static_assert(IO != IO_SPLIT || (NB == 4 && !F32OUT && !RELU && !POOL), "the concatenation's gradient has 64 channels");
	static_assert(IO != IO_DISPLAY || (NB == 1 && F32OUT && !RELU), "the display epilogue reads the first output channels");
	constexpr int CX = CAT ? 32 : CIN, CKX = CX < 32 ? 32 : CX;   /* channels of x, padded to K */
	constexpr int CP = CKX + 8, CH8 = CX / 8, CHP = CKX / 8, KS = CAT ? 2 : CKX / 32, WCIN = CAT ? 64 : CIN;
	constexpr bool LOOP = CIN == 64 || NB == 4;
	constexpr int TX = 16 * MBW, TY = 16, TW = TX + 2, TR = TY + 2;
	constexpr int CPC = 40, TWC = TX / 2 + 2, TRC = TY / 2 + 2;   /* coarse tile */
	constexpr int Cout = NB * 16;
	__shared__ __attribute__((aligned(16))) bf16_t xs[TR * TW * CP];
	__shared__ __attribute__((aligned(16))) float bs[Cout];
	__shared__ __attribute__((aligned(16))) bf16_t cs[CAT ? TRC * TWC * CPC : IO == IO_SPLIT ? (TY / 2) * (TX / 2) * CPC : 8];   /* coarse pixels, or those of the coarse mask */
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ml = lane & 15, kg = lane >> 4;
	bf8v wt[9][KS][NB];
#pragma unroll
	for (int tap = 0; tap < 9; tap++)
#pragma unroll
		for (int ks = 0; ks < KS; ks++)
#pragma unroll
			for (int nb = 0; nb < NB; nb++)
			{
				const int k = ks * 32 + kg * 8;
				wt[tap][ks][nb] = k < WCIN ? *(const bf8v*)(w + ((size_t)(tap * Cout + nb * 16 + ml) * WCIN + k)) : (bf8v){ 0, 0, 0, 0, 0, 0, 0, 0 };
			}
	if (tid < Cout) bs[tid] = bias ? bias[tid] : 0.0f;
	const int wy = wave * 4;                                 /* the wave's first row in the tile */
	const int fine = (wy * TW + ml) * CP + kg * 8;   /* the lane's place in the tile, and in the coarse one for the middle tap and the left (+ 1: the right) */
	const int codd = ((wy >> 1) * TWC + (ml >> 1) + 1) * CPC + kg * 8, ceven = ((wy >> 1) * TWC + ((ml + 1) >> 1)) * CPC + kg * 8;
	constexpr bool PAIRED = !F32OUT && (NB % 2) == 0, PAIRS = POOL || IO == IO_SPLIT;
	constexpr int PNB = IO == IO_SPLIT ? 2 : NB;         /* channel blocks that are pooled */
	/* XCD blockIdx % 8 gets an eighth of the tiles, in one piece: halos are read from its own L2 */
	const int xcd = blockIdx.x & 7, end = (int)((long long)tiles * (xcd + 1) >> 3);
	for (int tile = (int)((long long)tiles * xcd >> 3) + (blockIdx.x >> 3); tile < end; tile += gridDim.x >> 3)
	{
		const int x0 = (tile % across) * TX, r0 = (tile / across) * TY;
		int lt = tid;
		if (LOOP) asm volatile("" : "+v"(lt));            /* the staging's addresses are worked out per tile: kept over the loop they spill */
		if (LOOP) __syncthreads();                       /* the waves have read the last tile */
		{	/* the tile's loads in flight together */
			constexpr int N = TR * TW * CHP, IT = (N + 255) / 256, BATCH = IT < 12 ? IT : (IT + 1) / 2;
#pragma unroll
			for (int it0 = 0; it0 < IT; it0 += BATCH)
			{
				uint4 v[BATCH];
#pragma unroll
				for (int j = 0; j < BATCH; j++)
				{
					const int i = lt + (it0 + j) * 256;
					const int c8 = i % CHP, p = (i / CHP) % TW, gy = r0 - 1 + i / (CHP * TW), gx = x0 - 1 + p;
					v[j] = it0 + j < IT && i < N && c8 < CH8 && gy >= 0 && gy < H && gx >= 0 && gx < W ?
						*(const uint4*)(x + ((size_t)gy * W + gx) * CX + c8 * 8) : make_uint4(0, 0, 0, 0);
				}
#pragma unroll
				for (int j = 0; j < BATCH; j++)
				{
					const int i = lt + (it0 + j) * 256;
					if (it0 + j < IT && i < N) *(uint4*)(xs + (i / CHP) * CP + (i % CHP) * 8) = v[j];
				}
			}
			if (IO == IO_SPLIT)
			{
				constexpr int NM = (TY / 2) * (TX / 2) * 4;
				static_assert(IO != IO_SPLIT || NM == 256, "a load each");
				const int cy = (r0 >> 1) + lt / (TX * 2), cx = (x0 >> 1) + (lt >> 2) % (TX / 2);
				*(uint4*)(cs + (lt >> 2) * CPC + (lt & 3) * 8) = cy < (H >> 1) && cx < (W >> 1) ?
					*(const uint4*)(act + ((size_t)cy * (W >> 1) + cx) * 32 + (lt & 3) * 8) : make_uint4(0, 0, 0, 0);
			}
			if (CAT)
			{
				constexpr int NC = TRC * TWC * 4, ITC = (NC + 255) / 256;
				const int Hc = H >> 1, Wc = W >> 1;
				uint4 v[ITC];
#pragma unroll
				for (int j = 0; j < ITC; j++)
				{
					const int i = lt + j * 256;
					const int c8 = i % 4, p = (i / 4) % TWC, cy = (r0 >> 1) - 1 + i / (4 * TWC), cx = (x0 >> 1) - 1 + p;
					v[j] = i < NC && cy >= 0 && cy < Hc && cx >= 0 && cx < Wc ? *(const uint4*)(coarse + ((size_t)cy * Wc + cx) * 32 + c8 * 8) : make_uint4(0, 0, 0, 0);
				}
#pragma unroll
				for (int j = 0; j < ITC; j++)
				{
					const int i = lt + j * 256;
					if (i < NC) *(uint4*)(cs + (i / 4) * CPC + (i % 4) * 8) = v[j];
				}
			}
		}
		f4v acc[4][MBW][NB];
#pragma unroll
		for (int o = 0; o < 4; o++)
#pragma unroll
			for (int mb = 0; mb < MBW; mb++)
#pragma unroll
				for (int nb = 0; nb < NB; nb++) acc[o][mb][nb] = (f4v){ 0.0f, 0.0f, 0.0f, 0.0f };
		__syncthreads();
#pragma unroll
		for (int ir = 0; ir < 6; ir++)                      /* input row of the tile wy + ir */
#pragma unroll
			for (int dx = 0; dx < 3; dx++)
#pragma unroll
				for (int ks = 0; ks < KS; ks++)
#pragma unroll
					for (int mb = 0; mb < MBW; mb++)
					{
						bf8v a;
						if (CAT && ks == 0) a = *(const bf8v*)(cs + (((ir + 1) >> 1) * TWC + mb * 8 + (dx == 2)) * CPC + (dx == 1 ? codd : ceven));
						else a = *(const bf8v*)(xs + (ir * TW + mb * 16 + dx) * CP + (CAT ? 0 : ks * 32) + fine);
#pragma unroll
						for (int o = 0; o < 4; o++)
						{
							const int dy = ir - o;
							if (dy < 0 || dy > 2) continue;
#pragma unroll
							for (int nb = 0; nb < NB; nb++) acc[o][mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wt[dy * 3 + dx][ks][nb], a, acc[o][mb][nb], 0, 0, 0);
						}
					}
#pragma unroll
		for (int mb = 0; mb < MBW; mb++)
		{
			const int px = x0 + mb * 16 + ml;
			if constexpr (IO == IO_DISPLAY)
			{	/* channels 0..3 of the four rows are with lanes 0..15; swaps hand row kg to the lanes of kg, and each lane
				 * writes one pixel of the frame */
				float v[4];
#pragma unroll
				for (int i = 0; i < 4; i++)
				{
					auto u = [&](int o) { const float f = acc[o][mb][0][i]; return __builtin_bit_cast(uint32_t, f); };   /* (the cast of a vector's element takes element 0) */
					const uint32_t r01 = __builtin_amdgcn_permlane16_swap(u(0), u(1), false, false)[0], r23 = __builtin_amdgcn_permlane16_swap(u(2), u(3), false, false)[0];
					v[i] = __builtin_bit_cast(float, (uint32_t)__builtin_amdgcn_permlane32_swap(r01, r23, false, false)[0]) + bs[i];
				}
				const int py = r0 + wy + kg;
				if (py < io.h && px < io.w)
				{
					const size_t q = (size_t)px + (size_t)py * io.w;
					io.image[q] = frame_display(v[0], v[1], v[2], io.feat[q].x);
				}
				continue;
			}
			float above[PAIRS ? PNB : 1][4];                 /* sums of the pixel pairs of the row above */
#pragma unroll
			for (int o = 0; o < 4; o++)
			{
				const int ry = r0 + wy + o;
				uint32_t pk[NB][2], pq[PAIRS ? PNB : 1][2];
#pragma unroll
				for (int nb = 0; nb < NB; nb++)
				{
					const f4v bv = *(const f4v*)(bs + nb * 16 + kg * 4);
					float v[4];
#pragma unroll
					for (int i = 0; i < 4; i++)
					{
						v[i] = acc[o][mb][nb][i] + bv[i];
						if (RELU) v[i] = v[i] > 0.0f ? v[i] : 0.0f;
					}
					if (F32OUT)
					{
						if (ry < H && px < W) *(float4*)((float*)y + ((size_t)ry * W + px) * Cout + nb * 16 + kg * 4) = make_float4(v[0], v[1], v[2], v[3]);
					}
					else
					{
						pk[nb][0] = pack_bf(v[0], v[1]), pk[nb][1] = pack_bf(v[2], v[3]);
						if (!PAIRED && ry < H && px < W) *(uint2*)((bf16_t*)y + ((size_t)ry * W + px) * Cout + nb * 16 + kg * 4) = make_uint2(pk[nb][0], pk[nb][1]);
					}
					if (PAIRS && nb < PNB)
					{	/* 2x2 sums of the stored (bf16) values: (left + right) of the top row + of the bottom row, as
						 * dn_pool2 (times 1/4) and dn_upcat_bwd on the stored tensor */
						float hs[4];
#pragma unroll
						for (int i = 0; i < 4; i++)
						{
							const float r = bf2f((bf16_t)(pk[nb][i >> 1] >> (16 * (i & 1))));
							hs[i] = r + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, r), 0xb1, 0xf, 0xf, true));   /* lane ^ 1 */
						}
						const int pb = nb < PNB ? nb : 0;
						if (o & 1)
						{
							float q[4];
#pragma unroll
							for (int i = 0; i < 4; i++) q[i] = (above[pb][i] + hs[i]) * (IO == IO_SPLIT ? 1.0f : 0.25f);
							pq[pb][0] = pack_bf(q[0], q[1]), pq[pb][1] = pack_bf(q[2], q[3]);
						}
						else
#pragma unroll
							for (int i = 0; i < 4; i++) above[pb][i] = hs[i];
					}
				}
				/* channel blocks in pairs: row swaps of 16 lanes leave each lane 8 consecutive channels of its pixel (kg even:
				 * block nb, channels 4 kg .. + 7; kg odd: block nb + 1, channels 4 (kg - 1) .. + 7), so one 16-byte store
				 * covers whole 64-byte pixels */
				const int ch8 = (kg & 1) ? 16 + (kg - 1) * 4 : kg * 4;
				auto octet = [](const uint32_t (&p)[2], const uint32_t (&q)[2])
				{
					const auto a = __builtin_amdgcn_permlane16_swap(p[0], q[0], false, false);
					const auto b = __builtin_amdgcn_permlane16_swap(p[1], q[1], false, false);
					return make_uint4(a[0], b[0], a[1], b[1]);
				};
				if (PAIRED)
				{
#pragma unroll
					for (int nb = IO == IO_SPLIT ? 2 : 0; nb < NB; nb += 2)
					{
						uint4 q = octet(pk[nb], pk[nb + 1]);
						constexpr int YC = IO == IO_SPLIT ? 32 : Cout;
						const size_t at = ((size_t)ry * W + px) * YC + nb * 16 + ch8 - (Cout - YC);
						if (ry < H && px < W)
						{
							if (IO == IO_MASK)
							{
								const uint4 m = *(const uint4*)(act + at);
								q = make_uint4(relu_mask2(m.x, q.x), relu_mask2(m.y, q.y), relu_mask2(m.z, q.z), relu_mask2(m.w, q.w));
							}
							*(uint4*)((bf16_t*)y + at) = q;
						}
					}
				}
				if constexpr (PAIRS)
					if (o & 1)
					{
						static_assert(PNB == 2, "one pair");
						uint4 q = octet(pq[0], pq[1]);
						if (IO == IO_SPLIT)
						{
							const uint4 m = *(const uint4*)(cs + (((wy + o) >> 1) * (TX / 2) + ((mb * 16 + ml) >> 1)) * CPC + ch8);
							q = make_uint4(relu_mask2(m.x, q.x), relu_mask2(m.y, q.y), relu_mask2(m.z, q.z), relu_mask2(m.w, q.w));
						}
						if (!(ml & 1) && ry < H && px < W) *(uint4*)(ypool + ((size_t)(ry >> 1) * (W >> 1) + (px >> 1)) * 32 + ch8) = q;
					}
			}
		}
		if (!LOOP) break;
	}
}

template <int CIN, int NB, bool RELU, bool F32OUT, bool CAT, bool POOL, int IO>
__global__ void __launch_bounds__(256) k_conv3x3_t(const bf16_t* __restrict__ x, const bf16_t* __restrict__ coarse,
	const bf16_t* __restrict__ w, const float* __restrict__ bias, void* __restrict__ y, int H, int W, bf16_t* __restrict__ ypool,
	FrameIO io, const bf16_t* __restrict__ act)
{
	constexpr int MBW = 1, ROWS = 4;
	static_assert(IO != IO_SPLIT || (NB == 4 && !F32OUT && !RELU && !POOL), "the concatenation's gradient has 64 channels");
	static_assert(IO != IO_DISPLAY || (NB == 1 && F32OUT && !RELU), "the display epilogue reads the first output channels");
	constexpr int CX = CAT ? 32 : CIN;                  /* channels of x */
	constexpr int CKX = CX < 32 ? 32 : CX;              /* channels per pixel of the x tile (K, padded) */
	constexpr int CP = CKX + 8, TW = 16 * MBW + 2, TR = ROWS + 2, CH8 = CX / 8, CHP = CKX / 8;
	constexpr int KS = CAT ? 2 : CKX / 32;              /* 32-channel steps of K per tap */
	constexpr int WCIN = CAT ? 64 : CIN;                /* weight row length */
	constexpr int CPC = 40, TWC = 8 * MBW + 2, TRC = ROWS / 2 + 2; /* coarse tile */
	constexpr int NT = 64 * ROWS;                       /* threads per block: a wave per output row */
	constexpr int Cout = NB * 16;
	__shared__ __attribute__((aligned(16))) bf16_t xs[TR * TW * CP];
	__shared__ __attribute__((aligned(16))) bf16_t cs[CAT ? TRC * TWC * CPC : 8];
	const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ml = lane & 15, kg = lane >> 4;
	const int tx = blockIdx.x, ty = blockIdx.y;
	const int x0 = tx * (16 * MBW), r0 = ty * ROWS;
	{
		constexpr int N = TR * TW * CHP, IT = (N + NT - 1) / NT, BATCH = 8;
#pragma unroll
		for (int it0 = 0; it0 < IT; it0 += BATCH)
		{
			uint4 v[BATCH];
#pragma unroll
			for (int j = 0; j < BATCH; j++)
			{
				const int i = tid + (it0 + j) * NT;
				const int c8 = i % CHP, p = (i / CHP) % TW, gy = r0 - 1 + i / (CHP * TW), gx = x0 - 1 + p;
				v[j] = it0 + j < IT && i < N && c8 < CH8 && gy >= 0 && gy < H && gx >= 0 && gx < W ?
					*(const uint4*)(x + ((size_t)gy * W + gx) * CX + c8 * 8) : make_uint4(0, 0, 0, 0);
			}
#pragma unroll
			for (int j = 0; j < BATCH; j++)
			{
				const int i = tid + (it0 + j) * NT;
				if (it0 + j < IT && i < N) *(uint4*)(xs + (i / CHP) * CP + (i % CHP) * 8) = v[j];
			}
		}
		if (CAT)
		{
			constexpr int NC = TRC * TWC * 4, ITC = (NC + NT - 1) / NT;
			const int Hc = H >> 1, Wc = W >> 1;
			uint4 v[ITC];
#pragma unroll
			for (int j = 0; j < ITC; j++)
			{
				const int i = tid + j * NT;
				const int c8 = i % 4, p = (i / 4) % TWC, cy = (r0 >> 1) - 1 + i / (4 * TWC), cx = (x0 >> 1) - 1 + p;
				v[j] = i < NC && cy >= 0 && cy < Hc && cx >= 0 && cx < Wc ? *(const uint4*)(coarse + ((size_t)cy * Wc + cx) * 32 + c8 * 8) : make_uint4(0, 0, 0, 0);
			}
#pragma unroll
			for (int j = 0; j < ITC; j++)
			{
				const int i = tid + j * NT;
				if (i < NC) *(uint4*)(cs + (i / 4) * CPC + (i % 4) * 8) = v[j];
			}
		}
	}
	auto wfrag = [&](int tap, int ks, int nb) -> bf8v {
		const int k = ks * 32 + kg * 8;
		return k < WCIN ? *(const bf8v*)(w + ((size_t)(tap * Cout + nb * 16 + ml) * WCIN + k)) : (bf8v){ 0, 0, 0, 0, 0, 0, 0, 0 };
	};
	/* bias now, beside the tile's loads, so that the epilogue waits on nothing;
	 * weight fragments a tap ahead of their products */
	float bv[NB][4];
#pragma unroll
	for (int nb = 0; nb < NB; nb++)
#pragma unroll
		for (int i = 0; i < 4; i++) bv[nb][i] = bias ? bias[nb * 16 + kg * 4 + i] : 0.0f;
	bf8v wc[KS][NB], w1[KS][NB];
#pragma unroll
	for (int ks = 0; ks < KS; ks++)
#pragma unroll
		for (int nb = 0; nb < NB; nb++) wc[ks][nb] = wfrag(0, ks, nb);
	f4v acc[MBW][NB];
#pragma unroll
	for (int mb = 0; mb < MBW; mb++)
#pragma unroll
		for (int nb = 0; nb < NB; nb++) acc[mb][nb] = (f4v){ 0.0f, 0.0f, 0.0f, 0.0f };
	__syncthreads();
	const auto products = [&](int tap) {
		const int dy = tap / 3, dx = tap % 3;
#pragma unroll
		for (int ks = 0; ks < KS; ks++)
#pragma unroll
			for (int mb = 0; mb < MBW; mb++)
			{
				const int m = mb * 16 + ml;
				bf8v a;
				if (CAT && ks == 0) a = *(const bf8v*)(cs + ((((wave + dy - 1) >> 1) + 1) * TWC + ((m + dx - 1) >> 1) + 1) * CPC + kg * 8);
				else a = *(const bf8v*)(xs + ((wave + dy) * TW + m + dx) * CP + (CAT ? 0 : ks * 32) + kg * 8);
#pragma unroll
				for (int nb = 0; nb < NB; nb++) acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wc[ks][nb], a, acc[mb][nb], 0, 0, 0);
			}
	};
#pragma unroll 1
	for (int tap = 0; tap < 9; tap++)
	{
		if (tap < 8)
#pragma unroll
			for (int ks = 0; ks < KS; ks++)
#pragma unroll
				for (int nb = 0; nb < NB; nb++) w1[ks][nb] = wfrag(tap + 1, ks, nb);
		products(tap);
#pragma unroll
		for (int ks = 0; ks < KS; ks++)
#pragma unroll
			for (int nb = 0; nb < NB; nb++) wc[ks][nb] = w1[ks][nb];
	}
	const int ry = r0 + wave;
	constexpr bool PAIRS = POOL || IO == IO_SPLIT;       /* 2 x 2 sums of the first PNB channel blocks */
	constexpr int PNB = IO == IO_SPLIT ? 2 : NB;
	float hs[PAIRS ? MBW : 1][PNB][4];                   /* sums of horizontal pixel pairs */
	/* bf16 output with channel blocks in pairs: lanes kg and kg ^ 1 swap half
	 * their fragments so that each lane writes 8 consecutive channels (16 B)
	 * and one store instruction covers whole 64 B pixel rows; kg even keeps
	 * block nb (channels 4 kg .. 4 kg + 7), kg odd block nb + 1 (channels
	 * 16 + 4 (kg - 1) .. + 7). */
	constexpr bool PAIRED = !F32OUT && (NB % 2) == 0;
	uint32_t pk[MBW][NB][2];
#pragma unroll
	for (int nb = 0; nb < NB; nb++)
	{
		const int ch = nb * 16 + kg * 4;
#pragma unroll
		for (int mb = 0; mb < MBW; mb++)
		{
			const int px = x0 + mb * 16 + ml;
			float v[4];
#pragma unroll
			for (int i = 0; i < 4; i++)
			{
				v[i] = acc[mb][nb][i] + bv[nb][i];
				if (RELU) v[i] = v[i] > 0.0f ? v[i] : 0.0f;
			}
			const size_t o = ((size_t)ry * W + px) * Cout + ch;
			if (PAIRED)
				pk[mb][nb][0] = pack_bf(v[0], v[1]), pk[mb][nb][1] = pack_bf(v[2], v[3]);
			else if (IO == IO_DISPLAY)
			{	/* lanes holding channels 0..3 write the display pixel of the frame */
				if (kg == 0 && ry < io.h && px < io.w)
				{
					const size_t q = (size_t)px + (size_t)ry * io.w;
					io.image[q] = frame_display(v[0], v[1], v[2], io.feat[q].x);
				}
			}
			else if (ry < H && px < W)
			{
				if (F32OUT) *(float4*)((float*)y + o) = make_float4(v[0], v[1], v[2], v[3]);
				else *(uint2*)((bf16_t*)y + o) = make_uint2(pack_bf(v[0], v[1]),
					pack_bf(v[2], v[3]));
			}
			if (PAIRS && nb < PNB)                        /* the stored (bf16) values, left + right */
#pragma unroll
				for (int i = 0; i < 4; i++)
				{
					const float r = bf2f(f2bf(v[i]));
					hs[PAIRS ? mb : 0][nb < PNB ? nb : 0][i] = r + __shfl_xor(r, 1);
				}
		}
	}
	if (PAIRED)
	{
		const bool even = !(kg & 1);
#pragma unroll
		for (int mb = 0; mb < MBW; mb++)
		{
			const int px = x0 + mb * 16 + ml;
#pragma unroll
			for (int nb = IO == IO_SPLIT ? 2 : 0; nb < NB; nb += 2)
			{
				const uint32_t s0 = even ? pk[mb][nb + 1][0] : pk[mb][nb][0], s1 = even ? pk[mb][nb + 1][1] : pk[mb][nb][1];
				const uint32_t r0 = (uint32_t)__shfl_xor((int)s0, 16), r1 = (uint32_t)__shfl_xor((int)s1, 16);
				uint4 q = even ? make_uint4(pk[mb][nb][0], pk[mb][nb][1], r0, r1) : make_uint4(r0, r1, pk[mb][nb + 1][0], pk[mb][nb + 1][1]);
				const int ch = even ? nb * 16 + kg * 4 : (nb + 1) * 16 + (kg - 1) * 4;
				constexpr int YC = IO == IO_SPLIT ? 32 : Cout;
				const size_t at = ((size_t)ry * W + px) * YC + ch - (Cout - YC);
				if (ry < H && px < W)
				{
					if (IO == IO_MASK)
					{
						const uint4 a = *(const uint4*)(act + at);
						q = make_uint4(relu_mask2(a.x, q.x), relu_mask2(a.y, q.y), relu_mask2(a.z, q.z), relu_mask2(a.w, q.w));
					}
					*(uint4*)((bf16_t*)y + at) = q;
				}
			}
		}
	}
	if (PAIRS)
	{
		/* 2x2 average, (top pair) + (bottom pair), as dn_pool2 on the stored tensor (IO_SPLIT: the sum, as
		 * dn_upcat_bwd). Odd rows pass their pair sums to the even rows through LDS. */
		float* ex = (float*)xs;
		__syncthreads();                                  /* every wave is done with the staged tile */
		if (wave & 1)
#pragma unroll
			for (int mb = 0; mb < MBW; mb++)
#pragma unroll
				for (int nb = 0; nb < PNB; nb++)
#pragma unroll
					for (int i = 0; i < 4; i++) ex[(((wave >> 1) * MBW + mb) * PNB * 4 + nb * 4 + i) * 64 + lane] = hs[PAIRS ? mb : 0][nb][i];
		__syncthreads();
		const int Wp = W >> 1, pr = (r0 >> 1) + (wave >> 1);
		if (!(wave & 1) && ry + 1 < H && !(ml & 1))
#pragma unroll
			for (int mb = 0; mb < MBW; mb++)
			{
				const int px = x0 + mb * 16 + ml;
				if (px >= W) continue;
#pragma unroll
				for (int nb = 0; nb < PNB; nb++)
				{
					bf16_t q[4];
#pragma unroll
					for (int i = 0; i < 4; i++)
						q[i] = f2bf((hs[PAIRS ? mb : 0][nb][i] + ex[(((wave >> 1) * MBW + mb) * PNB * 4 + nb * 4 + i) * 64 + lane]) *
							(IO == IO_SPLIT ? 1.0f : 0.25f));
					const size_t at = ((size_t)pr * Wp + (px >> 1)) * (PNB * 16) + nb * 16 + kg * 4;
					uint2 o = make_uint2((uint32_t)q[0] | (uint32_t)q[1] << 16, (uint32_t)q[2] | (uint32_t)q[3] << 16);
					if (IO == IO_SPLIT)
					{
						const uint2 a = *(const uint2*)(act + at);
						o = make_uint2(relu_mask2(a.x, o.x), relu_mask2(a.y, o.y));
					}
					*(uint2*)(ypool + at) = o;
				}
			}
	}
}

/* Images with few 64-pixel-wide tiles of 4 rows run 4 x 16 tiles, a wave per row:
 * four to eight times the blocks, so that a small layer spreads over more compute
 * units instead of running at the latency of a few blocks. The line is 128 such
 * tiles (128 x 128, 64 tiles: 4.6 against 6.3 us for 32 -> 32 with pooling, 6.7 against
 * 10.3 for the concatenation; 240 x 144, 144 tiles: 6.3 and 6.4, 14.7 and 11.1), and
 * 256 for layers of at most half of 32 -> 32's weights, which wait less for them at
 * each tap (16 -> 32 at 144, 192, 252 and 260 tiles: 4.5 against 5.5, 4.8 and 5.8, 5.4 and 5.9,
 * 5.4 and 5.9; 32 -> 16 3.9 and 4.6, 3.9 and 4.7, 4.6 and 4.7, 4.7 and 4.8). */
static bool small_image(int H, int W, int weights) { return ((W + 63) / 64) * ((H + 3) / 4) < (weights <= 512 ? 256 : 128); }


/* The tiled convolution with the tile that suits the image. Large ones: 32 x 16
 * pixels, 16 x 16 where the sums of 64 outputs or the plain 64-channel tile would
 * not leave two blocks a CU. */
template <int CIN, int NB, bool RELU, bool F32OUT, bool CAT, bool POOL, int IO>
static hipError_t conv_tile(const bf16_t* x, const bf16_t* coarse, const bf16_t* w, const float* bias, void* y, int H, int W, bf16_t* ypool,
	const FrameIO& io, const bf16_t* act, hipStream_t s)
{
	constexpr int MBW = NB == 4 || (CIN == 64 && !CAT) ? 1 : 2, TX = 16 * MBW;
	const int across = (W + TX - 1) / TX, tiles = across * ((H + 15) / 16);
	const int blocks = (NB == 4 || CIN == 64) && tiles > 512 ? 512 : (tiles + 7) & ~7;   /* two a CU walk the tiles; or one a tile, a multiple of the XCDs */
	if (small_image(H, W, CIN * NB * 16))
		k_conv3x3_t<CIN, NB, RELU, F32OUT, CAT, POOL, IO><<<dim3((W + 15) / 16, (H + 3) / 4), 256, 0, s>>>(x, coarse, w, bias, y, H, W, ypool, io, act);
	else
		k_conv_rows<CIN, NB, RELU, F32OUT, CAT, POOL, IO, MBW><<<blocks, 256, 0, s>>>(x, coarse, w, bias, y, H, W,
			ypool, io, act, across, tiles);
	return hipGetLastError();
}

template <int CIN, int NB, bool CAT>
static hipError_t conv_t(const bf16_t* x, const bf16_t* coarse, const bf16_t* w, const float* bias, void* y, int H, int W, int flags, hipStream_t s)
{
	const bool relu = flags & DN_RELU, f32 = flags & DN_OUT_F32;
	const FrameIO io{};
	if (relu && f32) return conv_tile<CIN, NB, true, true, CAT, false, IO_NONE>(x, coarse, w, bias, y, H, W, nullptr, io, nullptr, s);
	if (relu) return conv_tile<CIN, NB, true, false, CAT, false, IO_NONE>(x, coarse, w, bias, y, H, W, nullptr, io, nullptr, s);
	if (f32) return conv_tile<CIN, NB, false, true, CAT, false, IO_NONE>(x, coarse, w, bias, y, H, W, nullptr, io, nullptr, s);
	return conv_tile<CIN, NB, false, false, CAT, false, IO_NONE>(x, coarse, w, bias, y, H, W, nullptr, io, nullptr, s);
}

hipError_t dn_conv3x3_pool(const bf16_t* x, int Cin, const bf16_t* w, const float* bias, bf16_t* y, int Cout, int H, int W,
	bf16_t* ypool, hipStream_t s)
{
	if (Cout != 32 || (Cin != 16 && Cin != 32) || H <= 0 || W <= 0 || H % 2 || W % 2) return hipErrorInvalidValue;
	if (Cin == 16) return conv_tile<16, 2, true, false, false, true, IO_NONE>(x, nullptr, w, bias, y, H, W, ypool, FrameIO{}, nullptr, s);
	return conv_tile<32, 2, true, false, false, true, IO_NONE>(x, nullptr, w, bias, y, H, W, ypool, FrameIO{}, nullptr, s);
}

hipError_t dn_conv3x3_cat(const bf16_t* coarse, const bf16_t* skip, const bf16_t* w, const float* bias, void* y, int Cout, int H, int W,
	int flags, hipStream_t s)
{
	if (Cout != 32 || H <= 0 || W <= 0 || H % 2 || W % 2) return hipErrorInvalidValue;
	return conv_t<64, 2, true>(skip, coarse, w, bias, y, H, W, flags, s);
}

template <int NB>
static hipError_t conv_nb(const bf16_t* x, int Cin, const bf16_t* w, const float* bias, void* y, int H, int W, int flags, hipStream_t s)
{
	const dim3 grid((W + 63) / 64, (H + 3) / 4), block(256);
	const bool relu = flags & DN_RELU, f32 = flags & DN_OUT_F32;
	if (relu && f32) k_conv3x3<NB, true, true><<<grid, block, 0, s>>>(x, Cin, w, bias, y, H, W);
	else if (relu) k_conv3x3<NB, true, false><<<grid, block, 0, s>>>(x, Cin, w, bias, y, H, W);
	else if (f32) k_conv3x3<NB, false, true><<<grid, block, 0, s>>>(x, Cin, w, bias, y, H, W);
	else k_conv3x3<NB, false, false><<<grid, block, 0, s>>>(x, Cin, w, bias, y, H, W);
	return hipGetLastError();
}

hipError_t dn_conv3x3(const bf16_t* x, int Cin, const bf16_t* w, const float* bias, void* y, int Cout, int H, int W, int flags, hipStream_t s)
{
	if (Cin <= 0 || Cin % 16 || Cout <= 0 || Cout % 16 || Cout > 64 || H <= 0 || W <= 0) return hipErrorInvalidValue;
	if (Cin == 16 && Cout == 32) return conv_t<16, 2, false>(x, nullptr, w, bias, y, H, W, flags, s);
	if (Cin == 16 && Cout == 16) return conv_t<16, 1, false>(x, nullptr, w, bias, y, H, W, flags, s);
	if (Cin == 32)
	{
		if (Cout == 16) return conv_t<32, 1, false>(x, nullptr, w, bias, y, H, W, flags, s);
		if (Cout == 32) return conv_t<32, 2, false>(x, nullptr, w, bias, y, H, W, flags, s);
		if (Cout == 64) return conv_t<32, 4, false>(x, nullptr, w, bias, y, H, W, flags, s);
	}
	if (Cin == 64 && Cout == 32) return conv_t<64, 2, false>(x, nullptr, w, bias, y, H, W, flags, s);
	switch (Cout / 16)
	{
	case 1: return conv_nb<1>(x, Cin, w, bias, y, H, W, flags, s);
	case 2: return conv_nb<2>(x, Cin, w, bias, y, H, W, flags, s);
	case 3: return conv_nb<3>(x, Cin, w, bias, y, H, W, flags, s);
	default: return conv_nb<4>(x, Cin, w, bias, y, H, W, flags, s);
	}
}

/* The output convolution (32 -> 16) writing the display image of a
 * filter-core frame from its epilogue: equal to dn_conv3x3 (fp32 out) +
 * dn_frame_output bit for bit, without the fp32 output tensor. (Reading the
 * frame into the first convolution's tile the same way was measured slower
 * than dn_frame_input + dn_conv3x3: 181 against 99 µs at 1080p.) */
hipError_t dn_conv3x3_display(const bf16_t* x, const bf16_t* wts, const float* bias, const uint4* features, int w, int h, float4* image,
	int Hp, int Wp, hipStream_t s)
{
	if (w <= 0 || h <= 0 || Hp < h || Wp < w) return hipErrorInvalidValue;
	const FrameIO io{ features, w, h, image };
	return conv_tile<32, 1, false, true, false, false, IO_DISPLAY>(x, nullptr, wts, bias, nullptr, Hp, Wp, nullptr, io, nullptr, s);
}

/* Input gradients with what follows them in the backward pass done by the
 * epilogue: the ReLU gradient of the layer below (dn_conv3x3 + dn_relu_bwd), or
 * the concatenation's (dn_conv3x3 to 64 channels + dn_upcat_bwd + dn_relu_bwd
 * of the coarse half), bit for bit. Level 0 at 1088 x 1920: the ReLU pass alone
 * moved 402 MB (66 us) per layer, the 64-channel tensor 268 MB out and back. */
hipError_t dn_conv3x3_dx_relu(const bf16_t* gy, int Cin, const bf16_t* w, const bf16_t* act, bf16_t* gx, int Cout, int H, int W, hipStream_t s)
{
	if (Cout != 32 || (Cin != 16 && Cin != 32) || H <= 0 || W <= 0 || !aligned16_3(gy, act, gx)) return hipErrorInvalidValue;
	if (Cin == 16) return conv_tile<16, 2, false, false, false, false, IO_MASK>(gy, nullptr, w, nullptr, gx, H, W, nullptr, FrameIO{}, act, s);
	return conv_tile<32, 2, false, false, false, false, IO_MASK>(gy, nullptr, w, nullptr, gx, H, W, nullptr, FrameIO{}, act, s);
}

hipError_t dn_conv3x3_dx_cat(const bf16_t* gy, const bf16_t* w, const bf16_t* actCoarse, bf16_t* gcoarse, bf16_t* gskip, int H, int W, hipStream_t s)
{
	if (H <= 0 || W <= 0 || H % 2 || W % 2 || !aligned16_3(gy, actCoarse, gcoarse) || !aligned16(gskip)) return hipErrorInvalidValue;
	return conv_tile<32, 4, false, false, false, false, IO_SPLIT>(gy, nullptr, w, nullptr, gskip, H, W, gcoarse, FrameIO{}, actCoarse, s);
}

/* ---- weight gradient ---------------------------------------------------
 * dW[tap][co][ci] = sum_p dy[p][co] x[p + tap - (1,1)][ci] as a GEMM over
 * pixels on v_mfma_f32_16x16x32_bf16 (M = output channels, N = input channels,
 * K = 32 pixels of a row). Writing q = p + (dx - 1) for the input pixel, a tap
 * pairs input row ty + r - 1 at pixels q with the output-gradient row ty at
 * pixels q + 1 - dx.
 *
 * A wave owns a 32-pixel column segment of a few rows and all nine taps (36
 * accumulator tiles at 32 x 32 channels), so it needs no barrier while it walks
 * down: it copies the next input row and gradient row ([pixel][channel], as they
 * lie in memory) into LDS of its own, and reads fragments with the transposing
 * LDS read (ds_read_b64_tr_b16: 16 lanes get one channel each of 4 pixels). The
 * fragments of the last three input rows stay in registers, so every row is
 * read from memory and from LDS once for its nine uses; the gradient row is read
 * at its three shifts. Rows are loaded two steps ahead of their use. The block's
 * 8 waves add their sums in wave order through LDS, and k_dw_reduce adds the
 * blocks' in a fixed order (deterministic).
 *
 * All layers of a network go in one launch (their inputs and gradients are kept
 * by the backward pass): a layer of a small image fills a fraction of the chip
 * on its own. The 64 input channels of the decoder's concatenation run as two
 * halves, the coarse one read from the coarse tensor (row and pixel halved).
 * The 19 layers of the network at 1088 x 1920 (1.7 GB of inputs and gradients,
 * 340 us at a copy's rate): 1,034 us and 413 us for partial sums with 9-wave
 * blocks that transposed while staging and a launch per layer, 466 and 22 us
 * now; at 256 x 256 362 us in all, now 40. */
typedef __bf16 bf8v_dw __attribute__((ext_vector_type(8)));
typedef short s4x __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s4x lds_s4x;
typedef short s8x __attribute__((ext_vector_type(8)));

static constexpr int DWW = 8;                       /* waves per block */
static constexpr int DW_SEG = 32;                   /* pixels of a wave's segment */
static constexpr int DW_MAXJOBS = 32;
static constexpr int DW_ROWSTRIDE = 40;             /* bf16 per LDS pixel: 32 channels and padding */
static constexpr int DW_STAGE = (DW_SEG + DW_SEG + 2) * DW_ROWSTRIDE;

struct DwJob
{
	const bf16_t* x;
	const bf16_t* dy;
	float* dw;
	float* db;          /* null: no bias gradient from this job */
	uint32_t part;      /* its partial sums in the workspace: blocks x n floats from here */
	int H, W;
	int16_t cx, cy;     /* channels of x and dy: 16 or 32 */
	int16_t up;         /* 1: x is the coarse tensor [H/2][W/2][cx], upsampled */
	int16_t ldw, off;   /* dw row length and first column of this job's channels */
	int16_t sx;         /* channels per pixel of x in memory */
	int rows, tilesX, chunks, block0, blocks;
	int out0;           /* first output of the job in the reduction's grid, in groups of 32 */
};
struct DwBatch { DwJob j[DW_MAXJOBS]; int n; };
static_assert(sizeof(DwBatch) <= 4000, "kernel argument size");

__device__ __forceinline__ bf8v_dw tr_frag(const bf16_t* lds, int firstPixel, int ch, int lane)
{
	const bf16_t* p = lds + (firstPixel + 8 * (lane >> 4) + ((lane & 15) >> 2)) * DW_ROWSTRIDE + ch + (lane & 3) * 4;
	const s4x a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4x*)p);
	const s4x b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4x*)(p + 4 * DW_ROWSTRIDE));
	const s8x v = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
	return __builtin_bit_cast(bf8v_dw, v);
}

/* One chunk (a segment of J.rows rows) into acc[tap][mb][nb], accb[mb] (column 0.. of sum dy). */
template <int CX, int CY>
__device__ __forceinline__ void dw_chunk(const DwJob& J, int chunk, bf16_t* lx, f4v (&acc)[9][2][2], f4v (&accb)[2])
{
	constexpr int MB = CY / 16, NB = CX / 16, XG = CX / 8, DG = CY / 8;           /* 16-byte groups per pixel */
	constexpr int XI = DW_SEG * XG / 64, DI = ((DW_SEG + 2) * DG + 63) / 64;      /* loads per lane and row */
	bf16_t* ld = lx + DW_SEG * DW_ROWSTRIDE;
	const int lane = threadIdx.x & 63, H = J.H, W = J.W;
	const int x0 = (chunk % J.tilesX) * DW_SEG, y0 = (chunk / J.tilesX) * J.rows, y1 = min(y0 + J.rows, H);
	const auto loadX = [&](uint4 (&v)[XI], int row) {
#pragma unroll
		for (int j = 0; j < XI; j++)
		{
			const int i = lane + 64 * j, g = i % XG, px = x0 + i / XG;
			const size_t at = J.up ? (size_t)(row >> 1) * (W >> 1) + (px >> 1) : (size_t)row * W + px;
			v[j] = row >= 0 && row < H && row <= y1 && px < W ? *(const uint4*)(J.x + at * J.sx + g * 8) : make_uint4(0, 0, 0, 0);
		}
	};
	const auto loadD = [&](uint4 (&v)[DI], int row) {    /* pixels x0 - 1 .. x0 + 32 */
#pragma unroll
		for (int j = 0; j < DI; j++)
		{
			const int i = lane + 64 * j, g = i % DG, k = i / DG, px = x0 - 1 + k;
			v[j] = k < DW_SEG + 2 && row < y1 && px >= 0 && px < W ? *(const uint4*)(J.dy + ((size_t)row * W + px) * CY + g * 8) : make_uint4(0, 0, 0, 0);
		}
	};
	const auto storeX = [&](const uint4 (&v)[XI]) {
#pragma unroll
		for (int j = 0; j < XI; j++)
		{
			const int i = lane + 64 * j;
			*(uint4*)(lx + (i / XG) * DW_ROWSTRIDE + (i % XG) * 8) = v[j];
		}
	};
	const auto storeD = [&](const uint4 (&v)[DI]) {
#pragma unroll
		for (int j = 0; j < DI; j++)
		{
			const int i = lane + 64 * j;
			if (i < (DW_SEG + 2) * DG) *(uint4*)(ld + (i / DG) * DW_ROWSTRIDE + (i % DG) * 8) = v[j];
		}
	};
	bf8v_dw ring[3][NB];                                 /* input rows ty - 1, ty, ty + 1 */
	uint4 xv[2][XI], dv[2][DI];
	{
		uint4 a[XI], b[XI];
		loadX(a, y0 - 1), loadX(b, y0);
		loadX(xv[0], y0 + 1), loadD(dv[0], y0);
		loadX(xv[1], y0 + 2), loadD(dv[1], y0 + 1);
		storeX(a);
#pragma unroll
		for (int nb = 0; nb < NB; nb++) ring[0][nb] = tr_frag(lx, 0, nb * 16, lane);
		storeX(b);
#pragma unroll
		for (int nb = 0; nb < NB; nb++) ring[1][nb] = tr_frag(lx, 0, nb * 16, lane);
	}
	const bf8v_dw ones = { (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f, (__bf16)1.0f };
	const auto step = [&](uint4 (&xs)[XI], uint4 (&dsv)[DI], int ty) {
		storeX(xs), storeD(dsv);
		loadX(xs, ty + 3), loadD(dsv, ty + 2);
#pragma unroll
		for (int nb = 0; nb < NB; nb++) ring[2][nb] = tr_frag(lx, 0, nb * 16, lane);
#pragma unroll
		for (int dx = 0; dx < 3; dx++)
		{
			bf8v_dw A[MB];
#pragma unroll
			for (int mb = 0; mb < MB; mb++) A[mb] = tr_frag(ld, 2 - dx, mb * 16, lane);
#pragma unroll
			for (int r = 0; r < 3; r++)
#pragma unroll
				for (int mb = 0; mb < MB; mb++)
#pragma unroll
					for (int nb = 0; nb < NB; nb++)
						acc[3 * r + dx][mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[mb], ring[r][nb], acc[3 * r + dx][mb][nb], 0, 0, 0);
			if (dx == 1)
#pragma unroll
				for (int mb = 0; mb < MB; mb++) accb[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[mb], ones, accb[mb], 0, 0, 0);
		}
#pragma unroll
		for (int nb = 0; nb < NB; nb++) ring[0][nb] = ring[1][nb], ring[1][nb] = ring[2][nb];
	};
	for (int ty = y0; ty < y1; ty += 2)
	{
		step(xv[0], dv[0], ty);
		if (ty + 1 < y1) step(xv[1], dv[1], ty + 1);
	}
}

/* Sums of the block's waves, in wave order, to partial[9][CY][CX] and bias[CY]:
 * in four rounds, each wave laying a quarter of its tiles into LDS. */
template <int CX, int CY>
__device__ __forceinline__ void dw_store(float* lds, const f4v (&acc)[9][2][2], const f4v (&accb)[2], float* out)
{
	constexpr int MB = CY / 16, NB = CX / 16;
	constexpr int TILES = 9 * MB * NB;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	f4v t[TILES];
#pragma unroll
	for (int tap = 0; tap < 9; tap++)
#pragma unroll
		for (int mb = 0; mb < MB; mb++)
#pragma unroll
			for (int nb = 0; nb < NB; nb++) t[(tap * MB + mb) * NB + nb] = acc[tap][mb][nb];
	constexpr int PER = (TILES + 3) / 4;
#pragma unroll
	for (int round = 0; round < 4; round++)
	{
		__syncthreads();
#pragma unroll
		for (int k = 0; k < PER; k++)
			if (round * PER + k < TILES) *(f4v*)(lds + ((wave * PER + k) * 64 + lane) * 4) = t[round * PER + k < TILES ? round * PER + k : 0];
		__syncthreads();
		for (int e = threadIdx.x; e < PER * 64; e += 64 * DWW)
		{
			const int tile = round * PER + e / 64, l = e % 64;
			if (tile >= TILES) continue;
			f4v sum = *(const f4v*)(lds + e * 4);
#pragma unroll
			for (int w = 1; w < DWW; w++) sum += *(const f4v*)(lds + (w * PER * 64 + e) * 4);
			const int tap = tile / (MB * NB), mb = (tile / NB) % MB, nb = tile % NB;
			/* D layout: lane holds rows 4 (lane / 16) + i, column lane % 16 */
#pragma unroll
			for (int i = 0; i < 4; i++) out[(tap * CY + mb * 16 + (l >> 4) * 4 + i) * CX + nb * 16 + (l & 15)] = sum[i];
		}
	}
	__syncthreads();
	if ((lane & 15) == 0)
#pragma unroll
		for (int mb = 0; mb < MB; mb++) *(f4v*)(lds + (wave * 2 + mb) * 16 + (lane >> 4) * 4) = accb[mb];
	__syncthreads();
	if ((int)threadIdx.x < CY)
	{
		float sum = 0.0f;
		for (int w = 0; w < DWW; w++) sum += lds[(w * 2 + (int)threadIdx.x / 16) * 16 + (int)threadIdx.x % 16];
		out[9 * CY * CX + threadIdx.x] = sum;
	}
}

template <int CX, int CY>
__device__ __forceinline__ void dw_job(const DwJob& J, float* lds, float* ws)
{
	const int wave = threadIdx.x >> 6, b = (int)blockIdx.x - J.block0, chunk = b * DWW + wave;
	f4v acc[9][2][2], accb[2];
#pragma unroll
	for (int k = 0; k < 9; k++)
#pragma unroll
		for (int m = 0; m < 4; m++) acc[k][m >> 1][m & 1] = (f4v){ 0.0f, 0.0f, 0.0f, 0.0f };
	accb[0] = accb[1] = (f4v){ 0.0f, 0.0f, 0.0f, 0.0f };
	if (chunk < J.chunks) dw_chunk<CX, CY>(J, chunk, (bf16_t*)lds + wave * DW_STAGE, acc, accb);
	dw_store<CX, CY>(lds, acc, accb, ws + J.part + (size_t)b * (9 * CX * CY + CY));
}

__global__ void __launch_bounds__(64 * DWW, 2) k_conv3x3_dw(const DwBatch B, float* __restrict__ ws)
{
	constexpr int SUMS = DWW * 9 * 64 * 4 * 4, STAGE = DWW * DW_STAGE * 2;
	__shared__ __attribute__((aligned(16))) char lds[SUMS > STAGE ? SUMS : STAGE];
	int k = 0;
	while (k + 1 < B.n && B.j[k + 1].block0 <= (int)blockIdx.x) k++;
	const DwJob& J = B.j[k];
	if (J.cx == 32 && J.cy == 32) dw_job<32, 32>(J, (float*)lds, ws);
	else if (J.cx == 16 && J.cy == 32) dw_job<16, 32>(J, (float*)lds, ws);
	else if (J.cx == 32) dw_job<32, 16>(J, (float*)lds, ws);
	else dw_job<16, 16>(J, (float*)lds, ws);
}

/* Sums of every job's blocks in a fixed order: 8 lanes per output each add
 * every 8th block partial (32 consecutive outputs per block row, coalesced),
 * then the 8 sums are added in lane order. */
__global__ void __launch_bounds__(256) k_dw_reduce(const DwBatch B, const float* __restrict__ ws)
{
	__shared__ float red[8][33];
	int k = 0;
	while (k + 1 < B.n && B.j[k + 1].out0 <= (int)blockIdx.x) k++;
	const DwJob& J = B.j[k];
	const int lane = threadIdx.x & 31, part = threadIdx.x >> 5, nw = 9 * J.cx * J.cy, n = nw + J.cy;
	const int i = ((int)blockIdx.x - J.out0) * 32 + lane;
	float s = 0.0f;
	if (i < n)
		for (int b = part; b < J.blocks; b += 8) s += ws[J.part + (size_t)b * n + i];
	red[part][lane] = s;
	__syncthreads();
	if (part != 0 || i >= n) return;
	float t = 0.0f;
#pragma unroll
	for (int q = 0; q < 8; q++) t += red[q][lane];
	if (i < nw) J.dw[(size_t)(i / J.cx) * J.ldw + J.off + i % J.cx] = t;
	else if (J.db) J.db[i - nw] = t;
}

/* Jobs of a list of layers: chunk heights (the same for all layers: enough
 * chunks for 8,192 waves, each at least 8 rows: fewer waves leave compute units
 * idle at the end, shorter chunks re-read two rows of their neighbours' input;
 * lists of few segment rows, a single layer of a small image among them, take 2 or
 * 4, as a block's walk is then the whole time), block and workspace ranges; taller
 * chunks where the partial sums would exceed maxFloats. One layer 32 -> 32, us with
 * chunks of 8 / 4 / 2 rows: 64 x 64 (128 segment rows) 19.5 / 14.9 / 13.0, 128 x 192
 * (768) 19.7 / 15.5 / 14.8, 160 x 256 (1,280) 20.0 / 16.4 / 16.4, 256 x 256 (2,048) 20.4 /
 * 17.8 / 18.9, 272 x 480 (4,080) 22.9 / 22.1 / 25.7, 544 x 960 (16,320) 34.4 / 53.6. (Before
 * all layers shared a launch: 12.9, 15.8, 18.1, 22.6, 42.6 and 73.9.) false: a shape that is not supported. */
static bool dw_plan(const DwLayer* L, int layers, size_t maxFloats, DwBatch& B, size_t& floats, int& blocks, int& outs)
{
	B.n = 0;
	int64_t steps = 0;
	int tallest = 1;
	if (!L || layers <= 0) return false;
	for (int i = 0; i < layers; i++)
	{
		const DwLayer& l = L[i];
		const bool ok = (l.Cout == 32 && (l.Cin == 16 || l.Cin == 32 || l.Cin == 64)) || (l.Cout == 16 && (l.Cin == 16 || l.Cin == 32));
		if (!ok || !l.x || !l.dy || !l.dw || l.H <= 0 || l.W <= 0 || (l.W + 63) / 64 > DW_BLOCKS) return false;   /* W beyond DW_BLOCKS * 64 pixels */
		if (l.coarse && (l.Cin != 64 || l.H % 2 || l.W % 2)) return false;
		const int parts = l.Cin == 64 ? 2 : 1;
		if (B.n + parts > DW_MAXJOBS) return false;
		for (int p = 0; p < parts; p++)
		{
			DwJob& J = B.j[B.n++];
			J = DwJob{};
			J.dy = l.dy, J.dw = l.dw, J.db = p == 0 ? l.db : nullptr;
			J.H = l.H, J.W = l.W, J.cy = (int16_t)l.Cout, J.ldw = (int16_t)l.Cin, J.off = (int16_t)(32 * p);
			J.cx = (int16_t)(l.Cin == 64 ? 32 : l.Cin);
			J.sx = (int16_t)(l.Cin == 64 && !l.coarse ? 64 : J.cx);
			J.up = (int16_t)(l.coarse && p == 0 ? 1 : 0);
			J.x = l.coarse ? (p == 0 ? l.coarse : l.x) : l.x + 32 * p;
			J.tilesX = (l.W + DW_SEG - 1) / DW_SEG;
			steps += (int64_t)J.tilesX * l.H;
			tallest = tallest > l.H ? tallest : l.H;
		}
	}
	const int least = steps <= 1280 ? 2 : steps < 4096 ? 4 : 8;
	int rows = (int)(steps / 8192 < least ? least : steps / 8192 < tallest ? steps / 8192 : tallest);
	while (true)
	{
		blocks = outs = 0, floats = 0;
		for (int k = 0; k < B.n; k++)
		{
			DwJob& J = B.j[k];
			const int n = 9 * J.cx * J.cy + J.cy;
			J.rows = rows < J.H ? rows : J.H;
			J.chunks = J.tilesX * ((J.H + J.rows - 1) / J.rows), J.blocks = (J.chunks + DWW - 1) / DWW;
			J.block0 = blocks, J.out0 = outs, J.part = (uint32_t)floats;
			blocks += J.blocks, outs += (n + 31) / 32, floats += (size_t)J.blocks * n;
		}
		if (floats <= maxFloats) return true;
		if (rows >= tallest) return false;
		rows += (rows + 7) / 8;
	}
}

static hipError_t dw_launch(const DwBatch& B, int blocks, int outs, void* ws, hipStream_t s)
{
	k_conv3x3_dw<<<blocks, 64 * DWW, 0, s>>>(B, (float*)ws);
	k_dw_reduce<<<outs, 256, 0, s>>>(B, (const float*)ws);
	return hipGetLastError();
}

size_t dn_dw_workspace_bytes(int Cin, int Cout) { return (size_t)DW_BLOCKS * (9 * Cout * Cin + Cout) * sizeof(float); }

hipError_t dn_conv3x3_dw(const bf16_t* x, int Cin, const bf16_t* dy, int Cout, int H, int W, float* dw, float* db, void* ws, hipStream_t s)
{
	DwLayer l = { x, nullptr, dy, dw, db, Cin, Cout, H, W };
	DwBatch B;
	size_t floats;
	int blocks, outs;
	if (!ws || !dw_plan(&l, 1, dn_dw_workspace_bytes(Cin, Cout) / sizeof(float), B, floats, blocks, outs)) return hipErrorInvalidValue;
	return dw_launch(B, blocks, outs, ws, s);
}

static const size_t DW_BATCH_FLOATS = (size_t)1 << 30;

size_t dn_dw_batch_workspace_bytes(const DwLayer* layers, int n)
{
	DwBatch B;
	size_t floats;
	int blocks, outs;
	return dw_plan(layers, n, DW_BATCH_FLOATS, B, floats, blocks, outs) ? floats * sizeof(float) : 0;
}

hipError_t dn_conv3x3_dw_batch(const DwLayer* layers, int n, void* ws, size_t wsBytes, hipStream_t s)
{
	DwBatch B;
	size_t floats;
	int blocks, outs;
	if (!ws || !dw_plan(layers, n, DW_BATCH_FLOATS, B, floats, blocks, outs) || floats * sizeof(float) > wsBytes) return hipErrorInvalidValue;
	return dw_launch(B, blocks, outs, ws, s);
}

/* ---- weight gradient without allocation --------------------------------
 * The workspace of dn_conv3x3_dw_noalloc is a file-scope device array sized
 * for the largest supported shape (Cin 64, Cout 32: DW_BLOCKS x (9 x 32 x 64
 * + 32) floats, 37.8 MB); each device holds its own copy until the process
 * ends. Every block partial that the reduction reads is written by the same
 * call first, so nothing needs clearing between calls; calls that overlap
 * on one device share the array and race. */
static constexpr size_t DW_SCRATCH_FLOATS = (size_t)DW_BLOCKS * (9 * 32 * 64 + 32);
static __device__ __align__(256) float scratch[DW_SCRATCH_FLOATS];

static constexpr int MAX_DEVICES = 64;
static std::mutex g_scratchLock;
static void* g_scratchPtr[MAX_DEVICES];   /* device address of scratch per device, looked up once */

size_t dn_dw_scratch_bytes() { return DW_SCRATCH_FLOATS * sizeof(float); }

hipError_t dn_conv3x3_dw_noalloc(const bf16_t* x, int Cin, const bf16_t* dy, int Cout, int H, int W, float* dw, float* db, hipStream_t s)
{
	if (dn_dw_workspace_bytes(Cin, Cout) > dn_dw_scratch_bytes()) return hipErrorInvalidValue;
	int dev = 0;
	hipError_t e = hipGetDevice(&dev);
	if (e != hipSuccess) return e;
	if (dev < 0 || dev >= MAX_DEVICES) return hipErrorInvalidDevice;
	void* ptr = nullptr;
	{
		std::lock_guard<std::mutex> g(g_scratchLock);
		if (!g_scratchPtr[dev])
		{	/* the host-side name is not a device address: ask the runtime for this device's copy */
			e = hipGetSymbolAddress(&g_scratchPtr[dev], HIP_SYMBOL(scratch));
			if (e != hipSuccess)
			{
				g_scratchPtr[dev] = nullptr;
				return e;
			}
		}
		ptr = g_scratchPtr[dev];
	}
	return dn_conv3x3_dw(x, Cin, dy, Cout, H, W, dw, db, ptr, s);
}

/* ---- elementwise and layout kernels ------------------------------------ */
/* 16-byte versions of the elementwise kernels below: a thread handles 8
 * channels of one pixel (C a multiple of 8, 16-byte aligned tensors), a grid
 * row (blockIdx.y) one image row, so no per-element index division; the
 * per-element arithmetic is the scalar kernels' (identical results). */
typedef __attribute__((ext_vector_type(8))) unsigned short u16x8;

__device__ __forceinline__ u16x8 ld8(const bf16_t* p) { return *(const u16x8*)p; }
__device__ __forceinline__ void st8(bf16_t* p, u16x8 v) { *(u16x8*)p = v; }

__global__ void k_relu_bwd8(const bf16_t* __restrict__ y, const bf16_t* __restrict__ dy, bf16_t* __restrict__ out, size_t n8)
{
	for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n8; i += (size_t)gridDim.x * blockDim.x)
	{
		const u16x8 a = ld8(y + 8 * i), g = ld8(dy + 8 * i);
		u16x8 o;
#pragma unroll
		for (int k = 0; k < 8; k++) o[k] = bf2f(a[k]) > 0.0f ? g[k] : (unsigned short)0;
		st8(out + 8 * i, o);
	}
}

/* pixel row y of a W-wide image: groups j = px * G + c8 of 8 channels (G = C / 8 = 1 << gs) */
__global__ void k_pool2_bwd8(const bf16_t* __restrict__ dy, int gs, int W, bf16_t* __restrict__ dx, int acc)
{
	const int j = blockIdx.x * blockDim.x + threadIdx.x, G = 1 << gs, py = blockIdx.y;
	if (j >= W * G) return;
	const int px = j >> gs, c8 = j & (G - 1);
	const u16x8 d = ld8(dy + ((size_t)(py >> 1) * (W >> 1) + (px >> 1)) * (8 * G) + 8 * c8);
	bf16_t* o = dx + ((size_t)py * W + px) * (8 * G) + 8 * c8;
	const u16x8 prev = acc ? ld8(o) : u16x8{};
	u16x8 r;
#pragma unroll
	for (int k = 0; k < 8; k++)
	{
		float v = bf2f(d[k]) * 0.25f;
		if (acc) v += bf2f(prev[k]);
		r[k] = f2bf(v);
	}
	st8(o, r);
}

/* the gradient of an encoder level's second activation: the skip connection's gradient plus a
 * quarter of the pooled tensor's (k_pool2_bwd8, accumulating), then the ReLU gradient, in one pass
 * (images of more rows than a grid has: a block takes several) */
__global__ void k_pool2_bwd_relu8(const bf16_t* __restrict__ dy, const bf16_t* __restrict__ skip, const bf16_t* __restrict__ act, int gs, int H, int W,
	bf16_t* __restrict__ out)
{
	const int j = blockIdx.x * blockDim.x + threadIdx.x, G = 1 << gs;
	if (j >= W * G) return;
	const int px = j >> gs, c8 = j & (G - 1);
	for (int py = blockIdx.y; py < H; py += gridDim.y)
	{
		const size_t at = ((size_t)py * W + px) * (8 * G) + 8 * c8;
		const u16x8 d = ld8(dy + ((size_t)(py >> 1) * (W >> 1) + (px >> 1)) * (8 * G) + 8 * c8), prev = ld8(skip + at), a = ld8(act + at);
		u16x8 r;
#pragma unroll
		for (int k = 0; k < 8; k++)
		{
			float v = bf2f(d[k]) * 0.25f;
			v += bf2f(prev[k]);
			r[k] = bf2f(a[k]) > 0.0f ? f2bf(v) : (unsigned short)0;
		}
		st8(out + at, r);
	}
}

__global__ void k_pool2_8(const bf16_t* __restrict__ x, int gs, int W, bf16_t* __restrict__ y)
{
	const int w2 = W >> 1, j = blockIdx.x * blockDim.x + threadIdx.x, G = 1 << gs, py = blockIdx.y;
	if (j >= w2 * G) return;
	const int px = j >> gs, c8 = j & (G - 1), C = 8 * G;
	const bf16_t* b = x + ((size_t)(2 * py) * W + 2 * px) * C + 8 * c8;
	const u16x8 a = ld8(b), c = ld8(b + C), d = ld8(b + (size_t)W * C), e = ld8(b + (size_t)W * C + C);
	u16x8 r;
#pragma unroll
	for (int k = 0; k < 8; k++) r[k] = f2bf(((bf2f(a[k]) + bf2f(c[k])) + (bf2f(d[k]) + bf2f(e[k]))) * 0.25f);
	st8(y + ((size_t)py * w2 + px) * C + 8 * c8, r);
}

/* cat row: groups j = px * (G0 + G1) + g; the first G0 from the coarse pixel */
__global__ void k_upcat8(const bf16_t* __restrict__ coarse, int G0, const bf16_t* __restrict__ skip, int G1, int W, bf16_t* __restrict__ out)
{
	const int G = G0 + G1, j = blockIdx.x * blockDim.x + threadIdx.x, py = blockIdx.y;
	if (j >= W * G) return;
	const int px = j / G, g = j - px * G;
	const u16x8 v = g < G0 ? ld8(coarse + ((size_t)(py >> 1) * (W >> 1) + (px >> 1)) * (8 * G0) + 8 * g)
		: ld8(skip + ((size_t)py * W + px) * (8 * G1) + 8 * (g - G0));
	st8(out + ((size_t)py * W + px) * (8 * G) + 8 * g, v);
}

__global__ void k_upcat_bwd_coarse8(const bf16_t* __restrict__ dcat, int G0, int G1, int W, bf16_t* __restrict__ dcoarse)
{
	const int G = G0 + G1, w2 = W >> 1, j = blockIdx.x * blockDim.x + threadIdx.x, py = blockIdx.y;
	if (j >= w2 * G0) return;
	const int px = j / G0, g = j - px * G0, C = 8 * G;
	const bf16_t* b = dcat + ((size_t)(2 * py) * W + 2 * px) * C + 8 * g;
	const u16x8 a = ld8(b), c = ld8(b + C), d = ld8(b + (size_t)W * C), e = ld8(b + (size_t)W * C + C);
	u16x8 r;
#pragma unroll
	for (int k = 0; k < 8; k++) r[k] = f2bf((bf2f(a[k]) + bf2f(c[k])) + (bf2f(d[k]) + bf2f(e[k])));
	st8(dcoarse + ((size_t)py * w2 + px) * (8 * G0) + 8 * g, r);
}

__global__ void k_upcat_bwd_skip8(const bf16_t* __restrict__ dcat, int G0, int G1, int W, bf16_t* __restrict__ dskip)
{
	const int G = G0 + G1, j = blockIdx.x * blockDim.x + threadIdx.x, py = blockIdx.y;
	if (j >= W * G1) return;
	const int px = j / G1, g = j - px * G1;
	st8(dskip + ((size_t)py * W + px) * (8 * G1) + 8 * g, ld8(dcat + ((size_t)py * W + px) * (8 * G) + 8 * (G0 + g)));
}

static int log2_exact(int v) { int k = 0; while ((1 << k) < v) k++; return (1 << k) == v ? k : -1; }
static dim3 row_grid(int perRow, int rows) { return dim3((unsigned)((perRow + 255) / 256), (unsigned)rows); }

__global__ void k_relu_bwd(const bf16_t* __restrict__ y, const bf16_t* __restrict__ dy, bf16_t* __restrict__ out, size_t n)
{
	for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
		out[i] = bf2f(y[i]) > 0.0f ? dy[i] : (bf16_t)0;
}


hipError_t dn_relu_bwd(const bf16_t* y, const bf16_t* dy, bf16_t* dyPre, size_t n, hipStream_t s)
{
	if (!n) return hipSuccess;
	if (n % 8 == 0 && aligned16_3(y, dy, dyPre))
	{
		const size_t n8 = n / 8;
		const int blocks = (int)((n8 + 255) / 256 < 65536 ? (n8 + 255) / 256 : 65536);
		k_relu_bwd8<<<blocks, 256, 0, s>>>(y, dy, dyPre, n8);
		return hipGetLastError();
	}
	const int blocks = (int)((n + 255) / 256 < 65536 ? (n + 255) / 256 : 65536);
	k_relu_bwd<<<blocks, 256, 0, s>>>(y, dy, dyPre, n);
	return hipGetLastError();
}

__global__ void k_pool2(const bf16_t* __restrict__ x, int C, int H, int W, bf16_t* __restrict__ y)
{
	const int h2 = H / 2, w2 = W / 2;
	const size_t n = (size_t)h2 * w2 * C;
	for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
	{
		const int c = (int)(i % C);
		const size_t p = i / C;
		const int px = (int)(p % w2), py = (int)(p / w2);
		const size_t b = ((size_t)(2 * py) * W + 2 * px) * C + c;
		const float v = ((bf2f(x[b]) + bf2f(x[b + C])) + (bf2f(x[b + (size_t)W * C]) + bf2f(x[b + (size_t)W * C + C]))) * 0.25f;
		y[i] = f2bf(v);
	}
}

__global__ void k_pool2_bwd(const bf16_t* __restrict__ dy, int C, int H, int W, bf16_t* __restrict__ dx, int acc)
{
	const size_t n = (size_t)H * W * C;
	for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
	{
		const int c = (int)(i % C);
		const size_t p = i / C;
		const int px = (int)(p % W), py = (int)(p / W);
		float v = bf2f(dy[((size_t)(py / 2) * (W / 2) + px / 2) * C + c]) * 0.25f;
		if (acc) v += bf2f(dx[i]);
		dx[i] = f2bf(v);
	}
}

__global__ void k_upcat(const bf16_t* __restrict__ coarse, int C0, const bf16_t* __restrict__ skip, int C1, int H, int W, bf16_t* __restrict__ out)
{
	const int C = C0 + C1;
	const size_t n = (size_t)H * W * C;
	for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
	{
		const int c = (int)(i % C);
		const size_t p = i / C;
		const int px = (int)(p % W), py = (int)(p / W);
		out[i] = c < C0 ? coarse[((size_t)(py / 2) * (W / 2) + px / 2) * C0 + c] : skip[p * C1 + (c - C0)];
	}
}

__global__ void k_upcat_bwd_coarse(const bf16_t* __restrict__ dcat, int C0, int C1, int H, int W, bf16_t* __restrict__ dcoarse)
{
	const int C = C0 + C1, h2 = H / 2, w2 = W / 2;
	const size_t n = (size_t)h2 * w2 * C0;
	for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
	{
		const int c = (int)(i % C0);
		const size_t p = i / C0;
		const int px = (int)(p % w2), py = (int)(p / w2);
		const size_t b = ((size_t)(2 * py) * W + 2 * px) * C + c;
		dcoarse[i] = f2bf((bf2f(dcat[b]) + bf2f(dcat[b + C])) + (bf2f(dcat[b + (size_t)W * C]) + bf2f(dcat[b + (size_t)W * C + C])));
	}
}

__global__ void k_upcat_bwd_skip(const bf16_t* __restrict__ dcat, int C0, int C1, size_t pixels, bf16_t* __restrict__ dskip)
{
	const int C = C0 + C1;
	const size_t n = pixels * C1;
	for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
		dskip[i] = dcat[(i / C1) * C + C0 + (i % C1)];
}

static int grid_for(size_t n) { const size_t b = (n + 255) / 256; return (int)(b < 65536 ? (b ? b : 1) : 65536); }

hipError_t dn_pool2(const bf16_t* x, int C, int H, int W, bf16_t* y, hipStream_t s)
{
	if (H % 2 || W % 2) return hipErrorInvalidValue;
	if (!H || !W || !C) return hipSuccess;
	const int gs = C % 8 ? -1 : log2_exact(C / 8);
	if (gs >= 0 && aligned16(x) && aligned16(y) && H / 2 <= 65535)
		k_pool2_8<<<row_grid((W / 2) << gs, H / 2), 256, 0, s>>>(x, gs, W, y);
	else k_pool2<<<grid_for((size_t)H * W * C / 4), 256, 0, s>>>(x, C, H, W, y);
	return hipGetLastError();
}

hipError_t dn_pool2_bwd(const bf16_t* dy, int C, int H, int W, bf16_t* dx, int accumulate, hipStream_t s)
{
	if (H % 2 || W % 2) return hipErrorInvalidValue;
	if (!H || !W || !C) return hipSuccess;
	const int gs = C % 8 ? -1 : log2_exact(C / 8);
	if (gs >= 0 && aligned16(dy) && aligned16(dx) && H <= 65535)
		k_pool2_bwd8<<<row_grid(W << gs, H), 256, 0, s>>>(dy, gs, W, dx, accumulate);
	else k_pool2_bwd<<<grid_for((size_t)H * W * C), 256, 0, s>>>(dy, C, H, W, dx, accumulate);
	return hipGetLastError();
}

hipError_t dn_pool2_bwd_relu(const bf16_t* dy, const bf16_t* skip, const bf16_t* act, int C, int H, int W, bf16_t* out, hipStream_t s)
{
	if (H % 2 || W % 2 || H <= 0 || W <= 0) return hipErrorInvalidValue;
	const int gs = C <= 0 || C % 8 ? -1 : log2_exact(C / 8);
	if (gs < 0 || !aligned16_3(dy, skip, act) || !aligned16(out)) return hipErrorInvalidValue;
	k_pool2_bwd_relu8<<<row_grid(W << gs, H < 65535 ? H : 65535), 256, 0, s>>>(dy, skip, act, gs, H, W, out);
	return hipGetLastError();
}

hipError_t dn_upcat(const bf16_t* coarse, int C0, const bf16_t* skip, int C1, int H, int W, bf16_t* out, hipStream_t s)
{
	if (H % 2 || W % 2) return hipErrorInvalidValue;
	if (!H || !W || !(C0 + C1)) return hipSuccess;
	if (C0 > 0 && C1 > 0 && C0 % 8 == 0 && C1 % 8 == 0 && aligned16_3(coarse, skip, out) && H <= 65535)
		k_upcat8<<<row_grid(W * ((C0 + C1) / 8), H), 256, 0, s>>>(coarse, C0 / 8, skip, C1 / 8, W, out);
	else k_upcat<<<grid_for((size_t)H * W * (C0 + C1)), 256, 0, s>>>(coarse, C0, skip, C1, H, W, out);
	return hipGetLastError();
}

hipError_t dn_upcat_bwd(const bf16_t* dcat, int C0, int C1, int H, int W, bf16_t* dcoarse, bf16_t* dskip, hipStream_t s)
{
	if (H % 2 || W % 2) return hipErrorInvalidValue;
	if (!H || !W || !(C0 + C1)) return hipSuccess;
	if (C0 > 0 && C1 > 0 && C0 % 8 == 0 && C1 % 8 == 0 && aligned16_3(dcat, dcoarse, dskip) && H <= 65535)
	{
		k_upcat_bwd_coarse8<<<row_grid((W / 2) * (C0 / 8), H / 2), 256, 0, s>>>(dcat, C0 / 8, C1 / 8, W, dcoarse);
		k_upcat_bwd_skip8<<<row_grid(W * (C1 / 8), H), 256, 0, s>>>(dcat, C0 / 8, C1 / 8, W, dskip);
		return hipGetLastError();
	}
	k_upcat_bwd_coarse<<<grid_for((size_t)H * W * C0 / 4), 256, 0, s>>>(dcat, C0, C1, H, W, dcoarse);
	k_upcat_bwd_skip<<<grid_for((size_t)H * W * C1), 256, 0, s>>>(dcat, C0, C1, (size_t)H * W, dskip);
	return hipGetLastError();
}

__global__ void k_pack_input(const float4* __restrict__ rad, const float4* __restrict__ alb, const float4* __restrict__ nrm,
	const float* __restrict__ depth, size_t pixels, bf16_t* __restrict__ out)
{
	for (size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x; p < pixels; p += (size_t)gridDim.x * blockDim.x)
	{
		const float4 r = rad[p], a = alb[p], n = nrm[p];
		const float d = depth[p];
		auto pk = [](float lo, float hi) { return pack_bf(lo, hi); };
		uint4* o = (uint4*)(out + p * 16);
		o[0] = make_uint4(pk(r.x, r.y), pk(r.z, a.x), pk(a.y, a.z), pk(n.x, n.y));
		o[1] = make_uint4(pk(n.z, d), 0, 0, 0);
	}
}

hipError_t dn_pack_input(const float4* radiance, const float4* albedo, const float4* normal, const float* depth, int H, int W, bf16_t* out, hipStream_t s)
{
	k_pack_input<<<grid_for((size_t)H * W), 256, 0, s>>>(radiance, albedo, normal, depth, (size_t)H * W, out);
	return hipGetLastError();
}


__global__ void k_frame_input(const float4* __restrict__ acc, const uint4* __restrict__ feat, float invSpp, int w, int h, int Hp, int Wp,
	bf16_t* __restrict__ out)
{
	const size_t pixels = (size_t)Hp * Wp;
	for (size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x; p < pixels; p += (size_t)gridDim.x * blockDim.x)
	{
		const int x = (int)(p % (size_t)Wp), y = (int)(p / (size_t)Wp);
		uint4* o = (uint4*)(out + p * 16);
		if (x >= w || y >= h)
		{
			o[0] = make_uint4(0, 0, 0, 0), o[1] = make_uint4(0, 0, 0, 0);
			continue;
		}
		const size_t q = (size_t)x + (size_t)y * w;
		const float4 d = acc[q], i = acc[q + (size_t)w * h];
		const uint4 f = feat[q];
		const float3 a = feat_albedo(f.x), n = feat_normal(f.y);
		float depth = __uint_as_float(f.z);
		depth = __builtin_isfinite(depth) ? fminf(depth, 1.0e4f) : 1.0e4f;
		const float r[3] = { (d.x + i.x) * invSpp, (d.y + i.y) * invSpp, (d.z + i.z) * invSpp };
		const float al[3] = { a.x, a.y, a.z };
		float c[3];
		for (int k = 0; k < 3; k++) c[k] = log1pf(fmaxf(r[k], 0.0f) / fmaxf(al[k], DN_ALBEDO_FLOOR));
		const float dz = log1pf(depth) * 0.1f;
		auto pk = [](float lo, float hi) { return pack_bf(lo, hi); };
		o[0] = make_uint4(pk(c[0], c[1]), pk(c[2], a.x), pk(a.y, a.z), pk(n.x, n.y));
		o[1] = make_uint4(pk(n.z, dz), 0, 0, 0);
	}
}

hipError_t dn_frame_input(const float4* acc32, const uint4* features, float invSpp, int w, int h, int Hp, int Wp, bf16_t* out, hipStream_t s)
{
	if (w <= 0 || h <= 0 || Hp < h || Wp < w) return hipErrorInvalidValue;
	const size_t px = (size_t)Hp * Wp;
	k_frame_input<<<grid_for(px) < 4096 ? grid_for(px) : 4096, 256, 0, s>>>(acc32, features, invSpp, w, h, Hp, Wp, out);
	return hipGetLastError();
}

__global__ void k_frame_output(const float* __restrict__ net, int Wp, const uint4* __restrict__ feat, int w, int h, float4* __restrict__ image)
{
	const size_t pixels = (size_t)w * h;
	for (size_t q = blockIdx.x * (size_t)blockDim.x + threadIdx.x; q < pixels; q += (size_t)gridDim.x * blockDim.x)
	{
		const int x = (int)(q % (size_t)w), y = (int)(q / (size_t)w);
		const float* o = net + ((size_t)x + (size_t)y * Wp) * 16;
		const float3 a = feat_albedo(feat[q].x);
		const float al[3] = { a.x, a.y, a.z };
		float v[3];
		for (int k = 0; k < 3; k++) v[k] = sqrtf(sqrtf(expm1f(fmaxf(o[k], 0.0f)) * fmaxf(al[k], DN_ALBEDO_FLOOR)));
		image[q] = make_float4(v[0], v[1], v[2], 0.0f);
	}
}

hipError_t dn_frame_output(const float* out, int Hp, int Wp, const uint4* features, int w, int h, float4* image, hipStream_t s)
{
	if (w <= 0 || h <= 0 || Hp < h || Wp < w) return hipErrorInvalidValue;
	const size_t px = (size_t)w * h;
	k_frame_output<<<grid_for(px) < 4096 ? grid_for(px) : 4096, 256, 0, s>>>(out, Wp, features, w, h, image);
	return hipGetLastError();
}

__global__ void k_relmse(const float* __restrict__ out, int Cout, const float4* __restrict__ target, size_t pixels, float invN,
	bf16_t* __restrict__ dout, float* __restrict__ loss)
{
	__shared__ float red[256];
	float l = 0.0f;
	for (size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x; p < pixels; p += (size_t)gridDim.x * blockDim.x)
	{
		const float4 t4 = target[p];
		const float t[3] = { t4.x, t4.y, t4.z };
		for (int c = 0; c < Cout; c++)
		{
			if (c < 3)
			{
				const float d = out[p * Cout + c] - t[c], den = t[c] * t[c] + 0.01f;
				l += d * d / den;
				dout[p * Cout + c] = f2bf(2.0f * d / den * invN);
			}
			else dout[p * Cout + c] = 0;
		}
	}
	red[threadIdx.x] = l;
	__syncthreads();
	for (int k = 128; k > 0; k >>= 1)
	{
		if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
		__syncthreads();
	}
	if (threadIdx.x == 0) atomicAdd(loss, red[0] * invN);
}

/* The network's 16 output channels: one 16-byte read and two 16-byte writes per
 * pixel in place of 3 + 16 element accesses at a 64-byte stride; the same
 * per-pixel arithmetic and order of sums. 1088 x 1920: 89 -> 42 us. */
__global__ void __launch_bounds__(256) k_relmse16(const float4* __restrict__ out, const float4* __restrict__ target, size_t pixels, float invN,
	uint4* __restrict__ dout, float* __restrict__ loss)
{
	__shared__ float red[256];
	float l = 0.0f;
	for (size_t p = blockIdx.x * (size_t)blockDim.x + threadIdx.x; p < pixels; p += (size_t)gridDim.x * blockDim.x)
	{
		const float4 t4 = target[p], o4 = out[4 * p];
		const float t[3] = { t4.x, t4.y, t4.z }, o[3] = { o4.x, o4.y, o4.z };
		uint32_t g[3];
#pragma unroll
		for (int c = 0; c < 3; c++)
		{
			const float d = o[c] - t[c], den = t[c] * t[c] + 0.01f;
			l += d * d / den;
			g[c] = f2bf(2.0f * d / den * invN);
		}
		dout[2 * p] = make_uint4(g[0] | g[1] << 16, g[2], 0, 0);
		dout[2 * p + 1] = make_uint4(0, 0, 0, 0);
	}
	red[threadIdx.x] = l;
	__syncthreads();
	for (int k = 128; k > 0; k >>= 1)
	{
		if ((int)threadIdx.x < k) red[threadIdx.x] += red[threadIdx.x + k];
		__syncthreads();
	}
	if (threadIdx.x == 0) atomicAdd(loss, red[0] * invN);
}

hipError_t dn_relmse(const float* out, int Cout, const float4* target, int H, int W, bf16_t* dout, float* loss, hipStream_t s)
{
	const size_t pixels = (size_t)H * W;
	const int blocks = grid_for(pixels) < 1024 ? grid_for(pixels) : 1024;
	const float invN = 1.0f / (3.0f * (float)pixels);
	if (Cout == 16 && aligned16_3(out, target, dout)) k_relmse16<<<blocks, 256, 0, s>>>((const float4*)out, target, pixels, invN, (uint4*)dout, loss);
	else k_relmse<<<blocks, 256, 0, s>>>(out, Cout, target, pixels, invN, dout, loss);
	return hipGetLastError();
}

__device__ __forceinline__ void adam_element(const AdamTensor& T, size_t i, float lr, float b1, float b2, float eps, float c1, float c2)
{
	float w = T.p[i];
	if (T.g)
	{
		const float gi = T.g[i];
		const float mi = b1 * T.m[i] + (1.0f - b1) * gi, vi = b2 * T.v[i] + (1.0f - b2) * gi * gi;
		T.m[i] = mi, T.v[i] = vi;
		w -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
		T.p[i] = w;
	}
	if (T.wfwd) T.wfwd[i] = f2bf(w);
	if (T.wbwd)
	{
		const int ci = (int)(i % T.Cin), co = (int)((i / T.Cin) % T.Cout), tap = (int)(i / ((size_t)T.Cin * T.Cout));
		T.wbwd[((size_t)(8 - tap) * T.Cin + ci) * T.Cout + co] = f2bf(w);
	}
}

__global__ void k_adam(const AdamTensor T, float lr, float b1, float b2, float eps, float c1, float c2)
{
	for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < T.n; i += (size_t)gridDim.x * blockDim.x) adam_element(T, i, lr, b1, b2, eps, c1, c2);
}

/* All tensors of a network in one launch, a block of 256 elements each within
 * one tensor: 38 launches of 2.4-3.4 us became one of 7. */
static constexpr int ADAM_MAX = 48;
struct AdamBatch { AdamTensor t[ADAM_MAX]; uint32_t block0[ADAM_MAX]; int n; };
static_assert(sizeof(AdamBatch) <= 4000, "kernel argument size");

__global__ void __launch_bounds__(256) k_adam_batch(const AdamBatch B, float lr, float b1, float b2, float eps, float c1, float c2)
{
	int k = 0;
	while (k + 1 < B.n && B.block0[k + 1] <= blockIdx.x) k++;
	const AdamTensor& T = B.t[k];
	const size_t i = (size_t)(blockIdx.x - B.block0[k]) * 256 + threadIdx.x;
	if (i < T.n) adam_element(T, i, lr, b1, b2, eps, c1, c2);
}

hipError_t dn_adam(float* p, float* m, float* v, const float* g, size_t n, float lr, float b1, float b2, float eps, int t,
	bf16_t* wfwd, bf16_t* wbwd, int Cout, int Cin, hipStream_t s)
{
	if (wbwd && (Cout <= 0 || Cin <= 0 || n != (size_t)9 * Cout * Cin)) return hipErrorInvalidValue;
	const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
	const AdamTensor T = { p, m, v, g, wfwd, wbwd, n, Cout, Cin };
	k_adam<<<grid_for(n), 256, 0, s>>>(T, lr, b1, b2, eps, c1, c2);
	return hipGetLastError();
}

hipError_t dn_adam_batch(const AdamTensor* t, int n, float lr, float b1, float b2, float eps, int step, hipStream_t s)
{
	if (!t || n < 0) return hipErrorInvalidValue;
	for (int i = 0; i < n; i++)
		if (!t[i].p || !t[i].m || !t[i].v || t[i].n > ((size_t)1 << 31) ||
			(t[i].wbwd && (t[i].Cout <= 0 || t[i].Cin <= 0 || t[i].n != (size_t)9 * t[i].Cout * t[i].Cin))) return hipErrorInvalidValue;
	const float c1 = 1.0f - powf(b1, (float)step), c2 = 1.0f - powf(b2, (float)step);
	for (int i = 0; i < n;)
	{
		AdamBatch B;
		uint32_t blocks = 0;
		for (B.n = 0; i < n && B.n < ADAM_MAX && blocks < (1u << 30); i++)
			if (t[i].n) B.t[B.n] = t[i], B.block0[B.n++] = blocks, blocks += (uint32_t)((t[i].n + 255) / 256);
		if (blocks) k_adam_batch<<<blocks, 256, 0, s>>>(B, lr, b1, b2, eps, c1, c2);
	}
	return hipGetLastError();
}

} // namespace lh
