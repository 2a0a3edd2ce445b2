// Tile engine for products of fp32 operands on the bf16 pipes (split_bf16.h):  C[i][j] = sum_r A(i, r) * B(r, j).
//
// 256 threads, 2 x 2 waves.  An operand fetches its part of a BK-deep slice straight from the tensor into registers, eight
// consecutive reduction indices of a row a time, splits them and stores one 16-byte word per part: LDS [part][8 indices][row] is
// the order the matrix fragments are read in.  Slices are double buffered and requested one slice ahead of that; the large
// products and the five small ones have accumulators of their own.
#pragma once
#include "conv3x3.h"
#include "split_bf16.h"

namespace fitre {

// a [C][N][2][2] tensor: four consecutive rows (or reduction indices) are the cells of one map
struct QuadParams {
	const float *p;
	uint32_t bytes;  // extent of the tensor
	int groupStride; // floats between consecutive channels: 4 * samples
	int rows;
};

// ROWS x BK of an operand: UNITS groups of eight indices of a row per thread
template <int ROWS, int BK>
struct SplitUnits {
	static constexpr int G = BK / 8, UNITS = ROWS * G / kGemmThreads;
	static constexpr int LD = ROWS + 4, PART = G * LD; // 16-byte words
	static_assert(ROWS * G % kGemmThreads == 0 && kGemmThreads % ROWS == 0, "whole units per thread");
	float v[UNITS][8];
	__device__ __forceinline__ void put(u32x4 *lds, int e, int group, int row) const
	{
		u32x4 part[3];
		split_eight(v[e], part);
#pragma unroll
		for (int s = 0; s < 3; s++) lds[s * PART + group * LD + row] = part[s];
	}
};

// The offsets of a thread's elements are the same in every slice: load() only moves the (uniform) base of the resource.
struct SplitSlices {
	const char *base;
	uint32_t bytes;
	__device__ __forceinline__ __amdgpu_buffer_rsrc_t at(size_t byteOffset) const
	{
		return make_rsrc((const float *)(base + byteOffset), byteOffset < bytes ? bytes - (uint32_t)byteOffset : 0u);
	}
};

// element(row, k) = p[k * ld + row]: lanes along the rows; zero behind kend, where the resource ends
template <int ROWS, int BK>
struct SplitRowContig {
	typedef SplitUnits<ROWS, BK> U;
	typedef PlainParams Params;
	static constexpr bool kZeroTail = true;
	SplitSlices mem;
	int ld, row, groupL;
	uint32_t off[U::UNITS][8];
	__device__ __forceinline__ void init(const Params &pr, int row0, int kend, int tid)
	{
		const size_t end = (size_t)kend * pr.ld * 4;
		mem = SplitSlices{ (const char *)pr.p, end < pr.bytes ? (uint32_t)end : pr.bytes };
		ld = pr.ld, row = tid % ROWS, groupL = tid / ROWS;
#pragma unroll
		for (int e = 0; e < U::UNITS; e++)
#pragma unroll
			for (int q = 0; q < 8; q++) { // (a slice of a short reduction may reach past 2^32 bytes: there is no such operand)
				const unsigned long long at = (unsigned long long)(8 * (groupL + kGemmThreads / ROWS * e) + q) * (unsigned)ld + (unsigned)(row0 + row);
				off[e][q] = row0 + row < pr.rows && at < (1ull << 30) ? 4u * (uint32_t)at : kOutOfRange;
			}
	}
	__device__ __forceinline__ void load(int k0, int, U &u) const
	{
		const __amdgpu_buffer_rsrc_t rs = mem.at((size_t)k0 * ld * 4);
#pragma unroll
		for (int e = 0; e < U::UNITS; e++)
#pragma unroll
			for (int q = 0; q < 8; q++) u.v[e][q] = buffer_load(rs, off[e][q]);
	}
	__device__ __forceinline__ void store(u32x4 *lds, const U &u, int, int) const
	{
#pragma unroll
		for (int e = 0; e < U::UNITS; e++) u.put(lds, e, groupL + kGemmThreads / ROWS * e, row);
	}
	static __device__ __forceinline__ float at(const Params &pr, int i, int k) { return pr.p[(size_t)k * pr.ld + i]; }
};

// element(row, k) = p[row * ld + k].  MASK: what lies behind kend is made zero.  One operand of a product is enough where the other's
// rows follow each other: a number of the matrix times zero is zero, or not finite and then found in the sum.
template <int ROWS, int BK, bool MASK>
struct SplitKContigT {
	typedef SplitUnits<ROWS, BK> U;
	typedef PlainParams Params;
	static constexpr bool kZeroTail = MASK;
	SplitSlices mem;
	int group, rowL;
	uint32_t off[U::UNITS];
	__device__ __forceinline__ void init(const Params &pr, int row0, int, int tid)
	{
		mem = SplitSlices{ (const char *)pr.p, pr.bytes };
		group = tid % U::G, rowL = tid / U::G;
#pragma unroll
		for (int e = 0; e < U::UNITS; e++) {
			const int row = row0 + rowL + kGemmThreads / U::G * e;
			off[e] = row < pr.rows ? 4u * (uint32_t)(row * pr.ld + 8 * group) : kSplitNowhere;
		}
	}
	__device__ __forceinline__ void load(int k0, int, U &u) const
	{
		const __amdgpu_buffer_rsrc_t rs = mem.at((size_t)k0 * 4);
#pragma unroll
		for (int e = 0; e < U::UNITS; e++)
#pragma unroll
			for (int h = 0; h < 2; h++) {
				const quad4f w = buffer_load4(rs, off[e] + 16u * h);
				u.v[e][4 * h] = w.x, u.v[e][4 * h + 1] = w.y, u.v[e][4 * h + 2] = w.z, u.v[e][4 * h + 3] = w.w;
			}
	}
	__device__ __forceinline__ void store(u32x4 *lds, U &u, int k0, int kend) const
	{
		if (MASK && k0 + BK > kend) {
#pragma unroll
			for (int e = 0; e < U::UNITS; e++)
#pragma unroll
				for (int q = 0; q < 8; q++) u.v[e][q] = k0 + 8 * group + q < kend ? u.v[e][q] : 0.f;
		}
#pragma unroll
		for (int e = 0; e < U::UNITS; e++) u.put(lds, e, group, rowL + kGemmThreads / U::G * e);
	}
	static __device__ __forceinline__ float at(const Params &pr, int i, int k) { return pr.p[(size_t)i * pr.ld + k]; }
};
template <int ROWS, int BK> using SplitKContig = SplitKContigT<ROWS, BK, false>;
template <int ROWS, int BK> using SplitKContigMasked = SplitKContigT<ROWS, BK, true>;

// element(row = n, k = (c, q)) = p[c * groupStride + 4 * row + q]  (2 x 2 maps; 16-byte aligned, whole channels a range)
template <int ROWS, int BK>
struct SplitQuadK {
	typedef SplitUnits<ROWS, BK> U;
	typedef QuadParams Params;
	static constexpr bool kZeroTail = true;
	SplitSlices mem;
	int row, groupL, groupStride;
	uint32_t off[U::UNITS][2];
	__device__ __forceinline__ void init(const Params &pr, int row0, int kend, int tid)
	{
		const size_t end = (size_t)(kend >> 2) * pr.groupStride * 4;
		mem = SplitSlices{ (const char *)pr.p, end < pr.bytes ? (uint32_t)end : pr.bytes };
		row = tid % ROWS, groupL = tid / ROWS, groupStride = pr.groupStride;
#pragma unroll
		for (int e = 0; e < U::UNITS; e++)
#pragma unroll
			for (int h = 0; h < 2; h++)
				off[e][h] = row0 + row < pr.rows ? 4u * (uint32_t)((2 * (groupL + kGemmThreads / ROWS * e) + h) * groupStride + 4 * (row0 + row)) : kSplitNowhere;
	}
	__device__ __forceinline__ void load(int k0, int, U &u) const
	{
		const __amdgpu_buffer_rsrc_t rs = mem.at((size_t)(k0 >> 2) * groupStride * 4);
#pragma unroll
		for (int e = 0; e < U::UNITS; e++)
#pragma unroll
			for (int h = 0; h < 2; h++) {
				const quad4f w = buffer_load4(rs, off[e][h]);
				u.v[e][4 * h] = w.x, u.v[e][4 * h + 1] = w.y, u.v[e][4 * h + 2] = w.z, u.v[e][4 * h + 3] = w.w;
			}
	}
	__device__ __forceinline__ void store(u32x4 *lds, const U &u, int, int) const
	{
#pragma unroll
		for (int e = 0; e < U::UNITS; e++) u.put(lds, e, groupL + kGemmThreads / ROWS * e, row);
	}
	static __device__ __forceinline__ float at(const Params &pr, int i, int k) { return pr.p[(size_t)(k >> 2) * pr.groupStride + 4 * (size_t)i + (k & 3)]; }
};

// C[i][j] of a finished sum, as the fp32 engine stores it
__device__ __forceinline__ void split_gemm_store(const OutParams &out, float *C, int i, int j, float val)
{
	float *dst = out.quadLd ? C + (size_t)(i >> 2) * out.quadLd + 4 * (size_t)j + (i & 3) : C + (size_t)i * out.ldc + j;
	if (!out.splitStride) {
		val *= out.alpha;
		if (out.biasI) val += out.biasI[i];
		if (out.biasJ) val += out.biasJ[j];
		if (out.beta != 0.f) val += out.beta * *dst;
	}
	*dst = val;
}

template <int BM, int BN, int BK, class OpA, class OpB>
__global__ void __launch_bounds__(kGemmThreads, 2)
split_gemm_kernel(const typename OpA::Params pa, const typename OpB::Params pb, const OutParams out, int I, int J, int R, int kChunk)
{
	static_assert(OpA::kZeroTail || OpB::kZeroTail, "one operand is zero behind the end of the reduction");
	constexpr int TM = BM / 64, TN = BN / 64;
	__shared__ u32x4 As[2][3 * OpA::U::PART], Bs[2][3 * OpB::U::PART];
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int khalf = lane >> 5, l32 = lane & 31, wm = wave >> 1, wn = wave & 1;
	const int i0 = blockIdx.y * BM, j0 = blockIdx.x * BN;
	const int kbeg = blockIdx.z * kChunk, kend = kbeg + kChunk < R ? kbeg + kChunk : R;

	OpA opA;
	OpB opB;
	opA.init(pa, i0, kend, tid);
	opB.init(pb, j0, kend, tid);
	v16f acc[TM][TN], low[TM][TN];
#pragma unroll
	for (int tm = 0; tm < TM; tm++)
#pragma unroll
		for (int tn = 0; tn < TN; tn++)
#pragma unroll
			for (int v = 0; v < 16; v++) acc[tm][tn][v] = low[tm][tn][v] = 0.f;

	// two slices on their way in registers (behind kend nothing, or nothing that counts, is read)
	typename OpA::U ua[2];
	typename OpB::U ub[2];
	opA.load(kbeg, kend, ua[0]);
	opB.load(kbeg, kend, ub[0]);
	__builtin_amdgcn_sched_barrier(0);
	opA.load(kbeg + BK, kend, ua[1]);
	opB.load(kbeg + BK, kend, ub[1]);
	__builtin_amdgcn_sched_barrier(0);
	opA.store(As[0], ua[0], kbeg, kend);
	opB.store(Bs[0], ub[0], kbeg, kend);
	__builtin_amdgcn_sched_barrier(0);
	opA.load(kbeg + 2 * BK, kend, ua[0]);
	opB.load(kbeg + 2 * BK, kend, ub[0]);
	__syncthreads();
	constexpr int STEPS = BK / 16, MFMAS = STEPS * TM * TN * 6, VECTOR = (OpA::U::UNITS + OpB::U::UNITS) * 54;
#define SPLIT_GEMM_PRODUCTS(SUM, PA, PB)                                                                              \
	_Pragma("unroll") for (int tm = 0; tm < TM; tm++)                                                                 \
		_Pragma("unroll") for (int tn = 0; tn < TN; tn++) SUM[tm][tn] = mfma_bf16(a[step][tm][PA], b[step][tn][PB], SUM[tm][tn]);
// slice K0 from buffer BUF, while slice K0 + BK, which register set BUF ^ 1 holds, is split and stored into the other buffer
#define SPLIT_GEMM_SLICE(K0, BUF)                                                                                     \
	{                                                                                                                 \
		u32x4 a[STEPS][TM][3], b[STEPS][TN][3];                                                                       \
		_Pragma("unroll") for (int step = 0; step < STEPS; step++)                                                    \
			_Pragma("unroll") for (int s = 0; s < 3; s++)                                                             \
			{                                                                                                         \
				_Pragma("unroll") for (int tm = 0; tm < TM; tm++)                                                     \
					a[step][tm][s] = As[BUF][s * OpA::U::PART + (2 * step + khalf) * OpA::U::LD + wm * (BM / 2) + tm * 32 + l32]; \
				_Pragma("unroll") for (int tn = 0; tn < TN; tn++)                                                     \
					b[step][tn][s] = Bs[BUF][s * OpB::U::PART + (2 * step + khalf) * OpB::U::LD + wn * (BN / 2) + tn * 32 + l32]; \
			}                                                                                                         \
		__builtin_amdgcn_sched_barrier(0);                                                                            \
		opA.store(As[(BUF) ^ 1], ua[(BUF) ^ 1], (K0) + BK, kend);                                                     \
		opB.store(Bs[(BUF) ^ 1], ub[(BUF) ^ 1], (K0) + BK, kend);                                                     \
		_Pragma("unroll") for (int step = 0; step < STEPS; step++)                                                    \
		{                                                                                                             \
			SPLIT_GEMM_PRODUCTS(acc, 0, 0);                                                                           \
			SPLIT_GEMM_PRODUCTS(low, 1, 0);                                                                           \
			SPLIT_GEMM_PRODUCTS(low, 0, 1);                                                                           \
			SPLIT_GEMM_PRODUCTS(low, 1, 1);                                                                           \
			SPLIT_GEMM_PRODUCTS(low, 2, 0);                                                                           \
			SPLIT_GEMM_PRODUCTS(low, 0, 2);                                                                           \
		}                                                                                                             \
		_Pragma("unroll") for (int i = 0; i < MFMAS; i++)                                                             \
		{                                                                                                             \
			__builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                        \
			__builtin_amdgcn_sched_group_barrier(0x002, (VECTOR + MFMAS - 1) / MFMAS, 0);                             \
		}                                                                                                             \
		__builtin_amdgcn_sched_barrier(0);                                                                            \
		opA.load((K0) + 3 * BK, kend, ua[(BUF) ^ 1]);                                                                 \
		opB.load((K0) + 3 * BK, kend, ub[(BUF) ^ 1]);                                                                 \
		__syncthreads();                                                                                              \
	}
	int k0 = kbeg;
	for (; k0 + BK < kend; k0 += 2 * BK) {
		SPLIT_GEMM_SLICE(k0, 0);
		SPLIT_GEMM_SLICE(k0 + BK, 1);
	}
	if (k0 < kend) SPLIT_GEMM_SLICE(k0, 0);
#undef SPLIT_GEMM_PRODUCTS
#undef SPLIT_GEMM_SLICE

	float *C = out.C + (size_t)blockIdx.z * out.splitStride;
	bool suspect = false;
#pragma unroll
	for (int tm = 0; tm < TM; tm++)
#pragma unroll
		for (int tn = 0; tn < TN; tn++)
#pragma unroll
			for (int v = 0; v < 16; v++) {
				acc[tm][tn][v] += low[tm][tn][v];
				suspect |= split_sum_suspect(acc[tm][tn][v]);
			}
	if (__syncthreads_or(suspect)) { // by fp32 multiply-adds
		for (int e = tid; e < BM * BN; e += kGemmThreads) {
			const int i = i0 + e / BN, j = j0 + e % BN;
			if (i >= I || j >= J) continue;
			float sum = 0.f;
			for (int k = kbeg; k < kend; k++) sum = fmaf(OpA::at(pa, i, k), OpB::at(pb, j, k), sum);
			split_gemm_store(out, C, i, j, sum);
		}
		return;
	}
#pragma unroll
	for (int tm = 0; tm < TM; tm++)
#pragma unroll
		for (int tn = 0; tn < TN; tn++) {
			const int j = j0 + wn * (BN / 2) + tn * 32 + l32;
			if (j >= J) continue;
#pragma unroll
			for (int v = 0; v < 16; v++) {
				const int i = i0 + wm * (BM / 2) + tm * 32 + 8 * (v / 4) + 4 * khalf + (v % 4);
				if (i < I) split_gemm_store(out, C, i, j, acc[tm][tn][v] * kSplitSumScale);
			}
		}
}

// ---- host side ------------------------------------------------------------------------------------------------------
constexpr int kSplitGemmTile = 64, kSplitGemmBK = 32;

// Reduction ranges of a product, at most mostSplits and each at most longest indices.  Measured, us: 4.5 for a launch, 0.55 a slice
// of 32 with a workgroup on every compute unit, 0.42 where they hold more, a reduction 4.5 and its traffic at 3 TB/s.  1000 x 784 x
// 512 unsplit 14.9 (fp32 engine 22.2), 1000 x 512 x 784 in two ranges 17.4 (24.6), 256 x 2048 x 2048 in four 25.6 (34.7), 64 x
// 4096 x 9216 in eight 43 (64), 4096^3 861 (1230).
inline GemmPlan split_gemm_plan(long I, long J, long R, long mostSplits, long longest, long cus)
{
	const long tiles = ((I + kSplitGemmTile - 1) / kSplitGemmTile) * ((J + kSplitGemmTile - 1) / kSplitGemmTile);
	GemmPlan best{};
	double bestT = 1e30;
	for (long s = 1; s <= mostSplits && (s == 1 || s <= R / (2 * kSplitGemmBK)); s++) {
		const long chunk = ((R + s - 1) / s + kSplitGemmBK - 1) / kSplitGemmBK * kSplitGemmBK, ranges = (R + chunk - 1) / chunk;
		if (chunk > longest && s < mostSplits) continue;
		const long perCu = (tiles * ranges + cus - 1) / cus;
		double t = 4.5 + (double)perCu * (double)(chunk / kSplitGemmBK) * (perCu > 1 ? 0.42 : 0.55);
		if (ranges > 1) t += 4.5 + (double)(ranges + 1) * (double)I * (double)J * 4.0 / 3.0e6;
		if (t < bestT) {
			bestT = t;
			best.splits = (int)ranges, best.kChunk = (int)chunk;
		}
	}
	if (bestT >= 1e30) { // no allowed number of ranges is short enough: the most there are
		const long chunk = ((R + mostSplits - 1) / mostSplits + kSplitGemmBK - 1) / kSplitGemmBK * kSplitGemmBK;
		best.kChunk = (int)chunk, best.splits = (int)((R + chunk - 1) / chunk);
	}
	best.bm = best.bn = kSplitGemmTile, best.bk = kSplitGemmBK, best.estimateUs = bestT;
	best.wsBytes = best.splits > 1 ? (size_t)best.splits * I * J * sizeof(float) : 0;
	return best;
}

// The plan in the place of an fp32 one: no more ranges (its workspace), and none more than four times as long.  A sum of K terms
// of either sign is off by 0.1 sqrt(K) 2^-24 of its norm here and by 0.3 sqrt(K) 2^-24 there, so that its error is no larger (of one
// sign: split_bf16.h).
inline GemmPlan split_gemm_plan_for(const GemmPlan &fp32, long I, long J, long R, long cus)
{
	return split_gemm_plan(I, J, R, fp32.splits, 4L * fp32.kChunk, cus);
}

// leftSplits (may be null): the partial results of a cut product are left in ws and counted there
template <template <int, int> class OpA, template <int, int> class OpB, class PA, class PB>
static int launch_split_gemm(const PA &pa, const PB &pb, const OutParams &out, int I, int J, int R, const GemmPlan &plan, void *ws, int kernelClass,
                             double flops, int *leftSplits = nullptr, int tileId = kTileSplit)
{
	typedef OpA<kSplitGemmTile, kSplitGemmBK> A;
	typedef OpB<kSplitGemmTile, kSplitGemmBK> B;
	const dim3 grid((unsigned)((J + kSplitGemmTile - 1) / kSplitGemmTile), (unsigned)((I + kSplitGemmTile - 1) / kSplitGemmTile), (unsigned)plan.splits);
	if (grid.y > 65535 || grid.z > 65535) return fail(FITRE_E_UNSUPPORTED, "gemm grid %u x %u x %u too large", grid.x, grid.y, grid.z);
	OutParams part = out, fin = out;
	part.splitStride = fin.splitStride = 0;
	if (plan.splits > 1) {
		part.C = (float *)ws;
		part.splitStride = (long)I * J;
		if (!out.quadLd) part.ldc = J;
	}
	{
		LaunchScope scope(kernelClass, flops, tileId);
		split_gemm_kernel<kSplitGemmTile, kSplitGemmTile, kSplitGemmBK, A, B><<<grid, kGemmThreads, 0, stream()>>>(pa, pb, part, I, J, R, plan.kChunk);
	}
	if (leftSplits) *leftSplits = plan.splits;
	if (plan.splits > 1 && !leftSplits) {
		if (out.quadLd) { // the partials are in the result's layout: a flat sum
			fin.quadLd = 0, fin.ldc = (long)I * J;
			launch_splitk_reduce((const float *)ws, plan.splits, 1, I * J, fin);
		} else {
			launch_splitk_reduce((const float *)ws, plan.splits, I, J, fin);
		}
	}
	return check_launch("split_gemm_kernel");
}

} // namespace fitre
