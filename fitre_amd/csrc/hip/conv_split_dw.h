// Weight gradient of 3x3 and 5x5 convolutions of stride 1 that keep the map's size, on the bf16 pipes (split_bf16.h).
//
//     dW[o][c][ta][tb] = sum_m delta[o][m] * x[c][m + (ta-P)*B + (tb-P)]
//
// A workgroup takes ONE tap row ta, 64 output and 64 input channels and a range of the reduction; a wave 32 x 32 channels and the
// KS taps of the row.  The reduction runs over the image rows at which the tap row is inside the image (the
// others are never touched), in groups of eight consecutive cells of a row -- or of two rows of maps at most four cells wide --
// the short last group of a row filled up with zeros.  Groups of delta and, ta - P rows away, of x are split while they are
// staged: LDS [part][group][channel][8 cells] holds the matrix fragments as they are read.  The fragment of tap tb is the
// group's word moved by tb - P cells: a funnel shift with the last (first) two cells of the group before (behind) it, which are
// zero at the end of a row.  Stages of four groups, double buffered.
//
// The five small products have accumulators of their own.  Added to the large ones, each of the six would round the whole sum, also
// where there is next to nothing to add, and gradients are full of that: 256 -> 256 channels, 8 x 8 maps, 256 images, inputs
// behind a ReLU, error against 64 bits with one accumulator / two / on the fp32 pipe 4.3e-7 / 1.4e-7 / 3.7e-7, and with one error
// in fifty not zero 1.2e-7 / 4.0e-8 / 6.4e-8; weight gradients of VGG-11's layers on 8 x 8 and 4 x 4 maps at 256 images 4.5e-7 to
// 5.8e-7 / 2.3e-7 to 3.8e-7 / 4.0e-7 to 5.5e-7.  What is left is the pipe's own: it adds eight products at a time and cuts each off below
// the last place of the largest, towards zero.  Where the errors of a channel are a few large ones of one sign among many small
// ones of the other, all of the small ones lose the same way: its second layer 1.6e-6, nearly all of it one number a
// channel, against 6.4e-7 on the fp32 pipe.
//
// Partial sums leave as [range][tap][o][c], whole rows of c; split_dw_reduce_kernel adds the ranges in double, in order.
#pragma once
#include "conv3x3.h"
#include "split_bf16.h"

namespace fitre {

constexpr int kSplitDwGroups = 4; // groups per stage: two bf16 MFMA steps
constexpr int kSplitDwTile = 64;  // output and input channels of a workgroup

// how a row is cut into groups
constexpr int kRowsPaired = 0; // B <= 4: two rows a group
constexpr int kRowsWhole = 1;  // B <= 8: a row a group
constexpr int kRowsCut = 2;    // two or four groups a row

struct ConvSplitDwParams {
	const float *x, *delta;
	const float *x2, *delta2; // a second pair over which the reduction continues (null: none)
	uint32_t xBytes, deltaBytes;
	int I, cin, J, A, B;      // output and input channels, positions, map
	int logGroups;            // groups a row, kRowsCut
	int stages, perSplit;     // of one pair, for the tap row with the most rows; of a range
	int cTiles;
	float *partial;           // [range][KS * KS][I][cin]
	FastDiv divLive[3];       // image rows a tap row |ta - P| rows off the middle is inside: A, A - 1, A - 2
	int samples;
};

// the tile by fp32 multiply-adds: eight output channels x 64 (input channel, tap) a wave at a time
template <int KS, int MODE>
__device__ __forceinline__ void split_dw_exact_tile(const ConvSplitDwParams &p, int o0, int c0, int ta, int stBeg, int stEnd, float *partial)
{
	constexpr int P = KS / 2, OT = kSplitDwTile, CT = kSplitDwTile, G = kSplitDwGroups, WAVES = kGemmThreads / 64;
	static_assert(CT % 64 == 0, "whole groups of 64 (input channel, tap)");
	const int lane = threadIdx.x & 63, off = ta - P, a0 = off < 0 ? -off : 0, live = p.A - (off < 0 ? -off : off);
	const int rows = p.samples * live;
	for (int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); g < OT / 8 * (CT * KS / 64); g += WAVES) {
		const int oBase = o0 + g % (OT / 8) * 8, e = g / (OT / 8) * 64 + lane;
		const int c = c0 + e % CT, tb = e / CT;
		if (oBase >= p.I) continue;
		const bool mine = c < p.cin && tb < KS;
		float s[8];
#pragma unroll
		for (int r = 0; r < 8; r++) s[r] = 0.f;
		for (int st = stBeg; st < stEnd; st++) {
			const bool second = st >= p.stages;
			const float *x = (second ? p.x2 : p.x) + (size_t)(mine ? c : 0) * p.J, *d = second ? p.delta2 : p.delta;
			const int q0 = (st - (second ? p.stages : 0)) * G;
			for (int k = 0; k < G * 8; k++) {
				const int q = q0 + k / 8, cell = k % 8;
				const int r = MODE == kRowsPaired ? 2 * q + cell / 4 : (MODE == kRowsWhole ? q : q >> p.logGroups);
				const int b = MODE == kRowsPaired ? cell % 4 : (MODE == kRowsWhole ? cell : (q & ((1 << p.logGroups) - 1)) * 8 + cell);
				if (r >= rows || b >= p.B) continue; // uniform
				const int n = r / live, a = a0 + r - n * live, bx = b + tb - P;
				const float xv = mine && (unsigned)bx < (unsigned)p.B ? x[(n * p.A + a + off) * p.B + bx] : 0.f;
#pragma unroll
				for (int i = 0; i < 8; i++) s[i] = fmaf(d[(size_t)(oBase + i < p.I ? oBase + i : p.I - 1) * p.J + (n * p.A + a) * p.B + b], xv, s[i]);
			}
		}
		if (!mine) continue;
		for (int i = 0; i < 8 && oBase + i < p.I; i++) partial[((size_t)(ta * KS + tb) * p.I + oBase + i) * p.cin + c] = s[i];
	}
}

// 3 x 3 windows take at most 180 registers, 5 x 5 ones 243: two workgroups find room on a compute unit and leave 144 of a SIMD's 512,
// or 16, to the bandwidth kernels of the layer below.  Whole passes, us, this tile against 128 output channels in eight waves with
// stages of eight groups, one workgroup on a compute unit: VGG-11 b256 1655 / 1700, VGG-16 b128 1900 / 1960, AlexNet b64 2730 /
// 2870.  Alone the larger tile is the faster one (256 -> 256 channels, 8 x 8 maps, 256 images, with the reduction 110 / 99 us;
// 64 -> 192, 27 x 27, 5 x 5 windows, 64 images 163 / 185), but nothing of the chain starts beside it before all of it has ended.
// Held to 168 registers for three workgroups: 1706 / 1998 / 2836.
template <int KS, int MODE>
__global__ void __launch_bounds__(kGemmThreads, 2)
conv_split_dw_kernel(const ConvSplitDwParams p)
{
	FITRE_RAISE_MATRIX_WAVE_PRIORITY();
	constexpr int P = KS / 2, T = kGemmThreads, OT = kSplitDwTile, CT = kSplitDwTile, G = kSplitDwGroups;
	constexpr int DLD = OT + 4, XLD = CT + 4; // 16-byte words a group; four spare ones spread the stores of the groups over the banks
	constexpr int DPART = G * DLD, XPART = G * XLD;
	static_assert(G == 4 && OT * G == T && CT * G == T, "two steps a stage; a thread stages one group of either");
	__shared__ u32x4 Ds[2][3 * DPART], Xs[2][3 * XPART];

	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int khalf = lane >> 5, l32 = lane & 31;
	const int wo = wave & 1, wc = wave >> 1;
	// an XCD takes consecutive (range, tile) indices: workgroups that read the same positions share its L2
	int bx, by, bz;
	{
		const unsigned groups = gridDim.x * gridDim.y * gridDim.z;
		const unsigned lin = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
		const unsigned xcd = lin & 7u, each = groups >> 3, extra = groups & 7u;
		const unsigned logical = xcd * each + (xcd < extra ? xcd : extra) + (lin >> 3);
		const unsigned tiles = gridDim.x * gridDim.y;
		bz = (int)(logical / tiles);
		const unsigned rem = logical - (unsigned)bz * tiles;
		by = (int)(rem / gridDim.x);
		bx = (int)(rem - (unsigned)by * gridDim.x);
	}
	const int ta = bx / p.cTiles, c0 = (bx - ta * p.cTiles) * CT, o0 = by * OT;
	const int off = ta - P, away = off < 0 ? -off : off, a0 = off < 0 ? -off : 0, live = p.A - away;
	const FastDiv divLive = p.divLive[away];
	const int rows = p.samples * live;
	const int stTotal = p.x2 ? 2 * p.stages : p.stages;
	const int stBeg = bz * p.perSplit, stEnd = stBeg + p.perSplit < stTotal ? stBeg + p.perSplit : stTotal;

	// this thread's group of a stage, and the channels whose groups it stages
	const int qs = tid % G, g = MODE == kRowsCut ? qs & ((1 << p.logGroups) - 1) : 0;
	const int valid = p.B - 8 * g; // cells of its group that are inside the row (kRowsPaired: of each of its two)
	const int dRow = o0 + tid / G, xRow = c0 + tid / G;
	const uint32_t dOff = dRow < p.I ? 4u * (uint32_t)dRow * (uint32_t)p.J : kGroupOutOfRange;
	const uint32_t xOff = xRow < p.cin ? 4u * (uint32_t)xRow * (uint32_t)p.J : kGroupOutOfRange;
	const int dLds = qs * DLD + tid / G, xLds = qs * XLD + tid / G;
	for (int i = tid; i < 3 * XPART; i += T) Xs[0][i] = Xs[1][i] = u32x4{ 0, 0, 0, 0 }; // the spare words are what lies past a row's end

	u32x4 dreg[2], xreg[2];
	v16f acc[KS], low[KS]; // the large products, and the five small ones
#pragma unroll
	for (int t = 0; t < KS; t++)
#pragma unroll
		for (int v = 0; v < 16; v++) acc[t][v] = low[t][v] = 0.f;

#define SPLIT_DW_ROW(R, OFFSET)                                                                                       \
	{                                                                                                                 \
		uint32_t n_, a_;                                                                                              \
		divLive.divmod((uint32_t)(R), n_, a_);                                                                        \
		OFFSET = 4 * (((int)n_ * p.A + a0 + (int)a_) * p.B + 8 * g);                                                  \
	}
#define SPLIT_DW_LOAD(ST)                                                                                             \
	{                                                                                                                 \
		const bool second_ = (ST) >= p.stages;                                                                        \
		const int q_ = ((ST) - (second_ ? p.stages : 0)) * G + qs;                                                    \
		const __amdgpu_buffer_rsrc_t dRs_ = make_rsrc(second_ ? p.delta2 : p.delta, p.deltaBytes), xRs_ = make_rsrc(second_ ? p.x2 : p.x, p.xBytes); \
		const int r_ = MODE == kRowsPaired ? 2 * q_ : (MODE == kRowsWhole ? q_ : q_ >> p.logGroups);                  \
		int at0_, at1_; /* bytes of the two halves of the group from the channel's first */                           \
		SPLIT_DW_ROW(r_, at0_);                                                                                       \
		at1_ = at0_ + 16;                                                                                             \
		const bool in0_ = r_ < rows, in1_ = MODE == kRowsPaired ? r_ + 1 < rows : in0_;                               \
		if constexpr (MODE == kRowsPaired) SPLIT_DW_ROW(r_ + 1, at1_);                                                \
		const int shift_ = 4 * off * p.B;                                                                             \
		const bool dIn_ = dOff != kGroupOutOfRange, xIn_ = xOff != kGroupOutOfRange;                                    \
		dreg[0] = __builtin_amdgcn_raw_buffer_load_b128(dRs_, (int)((dIn_ & in0_) ? dOff + at0_ : kGroupOutOfRange), 0, 0); \
		dreg[1] = __builtin_amdgcn_raw_buffer_load_b128(dRs_, (int)((dIn_ & in1_) ? dOff + at1_ : kGroupOutOfRange), 0, 0); \
		xreg[0] = __builtin_amdgcn_raw_buffer_load_b128(xRs_, (int)((xIn_ & in0_) ? xOff + at0_ + shift_ : kGroupOutOfRange), 0, 0); \
		xreg[1] = __builtin_amdgcn_raw_buffer_load_b128(xRs_, (int)((xIn_ & in1_) ? xOff + at1_ + shift_ : kGroupOutOfRange), 0, 0); \
	}
#define SPLIT_DW_STORE_ONE(REG, LDS, PARTWORDS)                                                                       \
	{                                                                                                                 \
		float v_[8];                                                                                                  \
		_Pragma("unroll") for (int i = 0; i < 8; i++)                                                                 \
		{                                                                                                             \
			const uint32_t bits_ = REG[i / 4][i % 4];                                                                 \
			v_[i] = (MODE == kRowsPaired ? i % 4 : i) < valid ? __builtin_bit_cast(float, bits_) : 0.f;               \
		}                                                                                                             \
		u32x4 part_[3];                                                                                               \
		split_eight(v_, part_);                                                                                       \
		_Pragma("unroll") for (int s = 0; s < 3; s++) (LDS)[s * (PARTWORDS)] = part_[s];                              \
	}
#define SPLIT_DW_STORE_DELTA(BUFFER) SPLIT_DW_STORE_ONE(dreg, &Ds[BUFFER][dLds], DPART)
#define SPLIT_DW_STORE_X(BUFFER) SPLIT_DW_STORE_ONE(xreg, &Xs[BUFFER][xLds], XPART)
// fragments of a step: part S of delta; part S of x and the cells beside it
#define SPLIT_DW_READ_A(TO, BUFFER, STEP, S) TO = Ds[BUFFER][(S) * DPART + (2 * (STEP) + khalf) * DLD + wo * 32 + l32]
#define SPLIT_DW_READ_X(BUFFER, STEP, S)                                                                              \
	{                                                                                                                 \
		const u32x4 *xw_ = &Xs[BUFFER][(2 * (STEP) + khalf) * XLD + wc * 32 + l32 + (S) * XPART];                     \
		word = *xw_;                                                                                                  \
		if constexpr (MODE == kRowsCut) {                                                                             \
			const int at_ = (2 * (STEP) + khalf) & ((1 << p.logGroups) - 1);                                          \
			const u32x4 *none_ = &Xs[BUFFER][CT + (S) * XPART];                                                       \
			last = (at_ == 0 ? none_ : xw_ - XLD)[0][3];                                                              \
			first = (at_ == (1 << p.logGroups) - 1 ? none_ : xw_ + XLD)[0][0];                                        \
		}                                                                                                             \
	}
#define SPLIT_DW_TAPS()                                                                                               \
	_Pragma("unroll") for (int t = 0; t < KS; t++)                                                                    \
	{                                                                                                                 \
		const int by_ = t - P;                                                                                        \
		if (by_ == 0) f[t] = word;                                                                                    \
		else if (by_ == -1)                                                                                           \
			f[t] = u32x4{ __builtin_amdgcn_alignbit(word[0], last, 16), __builtin_amdgcn_alignbit(word[1], word[0], 16), \
				          __builtin_amdgcn_alignbit(word[2], word[1], 16), __builtin_amdgcn_alignbit(word[3], word[2], 16) }; \
		else if (by_ == 1)                                                                                            \
			f[t] = u32x4{ __builtin_amdgcn_alignbit(word[1], word[0], 16), __builtin_amdgcn_alignbit(word[2], word[1], 16), \
				          __builtin_amdgcn_alignbit(word[3], word[2], 16), __builtin_amdgcn_alignbit(first, word[3], 16) }; \
		else if (by_ == -2) f[t] = u32x4{ last, word[0], word[1], word[2] };                                          \
		else f[t] = u32x4{ word[1], word[2], word[3], first };                                                        \
		if constexpr (MODE == kRowsPaired) { /* the second row starts in the middle */                                \
			if (by_ == -1) f[t][2] &= 0xffff0000u;                                                                    \
			else if (by_ == 1) f[t][1] &= 0x0000ffffu;                                                                \
		}                                                                                                             \
	}
#define SPLIT_DW_PRODUCTS(SUM, A)                                                                                     \
	_Pragma("unroll") for (int t = 0; t < KS; t++) SUM[t] = mfma_bf16(A, f[t], SUM[t]);
// vector instructions of the staging between the matrix instructions
#define SPLIT_DW_MIX(MFMAS)                                                                                           \
	_Pragma("unroll") for (int i = 0; i < (MFMAS); i++)                                                               \
	{                                                                                                                 \
		__builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                            \
		__builtin_amdgcn_sched_group_barrier(0x002, 9, 0);                                                            \
	}

	SPLIT_DW_LOAD(stBeg);
	__syncthreads(); // the zeros are in place
	SPLIT_DW_STORE_DELTA(0);
	SPLIT_DW_STORE_X(0);
	if (stBeg + 1 < stEnd) SPLIT_DW_LOAD(stBeg + 1);
	__syncthreads();

	// A phase multiplies one part of x with the parts of delta it is kept with, while the next phase's part of either is read.
	// The next stage is split and stored during the first step's last phase and the second's second, and the one after it requested
	// behind them; the barrier comes before the last phase, whose operands are in registers, so that the next stage's first fragments are read under it.
	u32x4 d0[2], d1, d2, word, f[KS];
	uint32_t last = 0, first = 0; // two cells of the group before, two of the one behind: zero at the end of a row
	SPLIT_DW_READ_A(d0[0], 0, 0, 0);
	SPLIT_DW_READ_X(0, 0, 2);
	for (int st = stBeg; st < stEnd; st++) {
		const int buffer = (st - stBeg) & 1;
#pragma unroll
		for (int step = 0; step < G / 2; step++) {
			const bool ends = step + 1 == G / 2;
			SPLIT_DW_TAPS();
			SPLIT_DW_READ_A(d1, buffer, step, 1);
			SPLIT_DW_READ_X(buffer, step, 1);
			SPLIT_DW_PRODUCTS(low, d0[step & 1]);
			__builtin_amdgcn_sched_barrier(0);
			SPLIT_DW_TAPS();
			SPLIT_DW_READ_A(d2, buffer, step, 2);
			SPLIT_DW_READ_X(buffer, step, 0);
			if (ends) SPLIT_DW_STORE_DELTA(buffer ^ 1);
			SPLIT_DW_PRODUCTS(low, d1);
			SPLIT_DW_PRODUCTS(low, d0[step & 1]);
			if (ends) SPLIT_DW_MIX(2 * KS);
			__builtin_amdgcn_sched_barrier(0);
			SPLIT_DW_TAPS();
			if (ends) {
				if (st + 2 < stEnd) SPLIT_DW_LOAD(st + 2);
				__syncthreads();
			}
			SPLIT_DW_READ_A(d0[(step + 1) & 1], ends ? buffer ^ 1 : buffer, ends ? 0 : step + 1, 0);
			SPLIT_DW_READ_X(ends ? buffer ^ 1 : buffer, ends ? 0 : step + 1, 2);
			if (!ends) SPLIT_DW_STORE_X(buffer ^ 1);
			SPLIT_DW_PRODUCTS(low, d2);
			SPLIT_DW_PRODUCTS(low, d1);
			SPLIT_DW_PRODUCTS(acc, d0[step & 1]);
			if (!ends) SPLIT_DW_MIX(3 * KS);
			__builtin_amdgcn_sched_barrier(0);
		}
	}
#undef SPLIT_DW_STORE_DELTA
#undef SPLIT_DW_STORE_X
#undef SPLIT_DW_READ_A
#undef SPLIT_DW_READ_X
#undef SPLIT_DW_TAPS
#undef SPLIT_DW_PRODUCTS
#undef SPLIT_DW_MIX
#undef SPLIT_DW_ROW
#undef SPLIT_DW_LOAD
#undef SPLIT_DW_STORE_ONE

	float *partial = p.partial + (size_t)bz * KS * KS * p.I * p.cin;
	bool suspect = false;
#pragma unroll
	for (int t = 0; t < KS; t++)
#pragma unroll
		for (int v = 0; v < 16; v++) {
			acc[t][v] += low[t][v];
			suspect |= split_sum_suspect(acc[t][v]);
		}
	if (__syncthreads_or(suspect)) {
		split_dw_exact_tile<KS, MODE>(p, o0, c0, ta, stBeg, stEnd, partial);
		return;
	}
	const int c = c0 + wc * 32 + l32;
	if (c >= p.cin) return;
#pragma unroll
	for (int t = 0; t < KS; t++)
#pragma unroll
		for (int v = 0; v < 16; v++) {
			const int o = o0 + wo * 32 + 8 * (v / 4) + 4 * khalf + (v % 4);
			if (o < p.I) partial[((size_t)(ta * KS + t) * p.I + o) * p.cin + c] = acc[t][v] * kSplitSumScale;
		}
}

// dW[o][c][tap] = sum over the ranges, in order.  64 (o, c) x four phases a workgroup; a phase adds every fourth range, the
// phases are added in order.  blockIdx.y: tap row.
template <int KS>
__global__ void __launch_bounds__(256) split_dw_reduce_kernel(const float *partial, int ranges, int products, float *dW)
{
	FITRE_RAISE_WAVE_PRIORITY();
	__shared__ double sums[4][KS][64];
	const int at = blockIdx.x * 64 + (threadIdx.x & 63), phase = threadIdx.x >> 6;
	const size_t range = (size_t)KS * KS * products;
	double s[KS];
#pragma unroll
	for (int t = 0; t < KS; t++) s[t] = 0.0;
	if (at < products) {
		const float *p = partial + (size_t)blockIdx.y * KS * products + at;
#pragma unroll 4
		for (int r = phase; r < ranges; r += 4)
#pragma unroll
			for (int t = 0; t < KS; t++) s[t] += (double)p[r * range + (size_t)t * products];
	}
#pragma unroll
	for (int t = 0; t < KS; t++) sums[phase][t][threadIdx.x & 63] = s[t];
	__syncthreads();
	if (phase == 0 && at < products)
#pragma unroll
		for (int t = 0; t < KS; t++)
			dW[(size_t)at * KS * KS + blockIdx.y * KS + t] = (float)(sums[0][t][threadIdx.x] + sums[1][t][threadIdx.x] + sums[2][t][threadIdx.x] + sums[3][t][threadIdx.x]);
}

} // namespace fitre
