// The kernel of dense_product.hip:  C[i][j] = sum_r A(i, r) * B(j, r), j contiguous, and what is done to the sum.
#pragma once
#include "split_bf16.h"

namespace fitre {

constexpr int kDenseThreads = 512, kDenseWaves = kDenseThreads / 64;
constexpr int kDenseJ = 64, kDenseStep = 16; // columns of a tile; reduction indices of a step: the depth of one bf16 MFMA
constexpr int kDenseSets = 2;                              // steps whose numbers are on their way
constexpr int kDenseBatch = 8;
constexpr int kDenseLongest = 4096; // reduction indices of a product the fully connected family brings here

struct DenseOperand {
	const float *p, *p2; // p2: the second pair's, over which the reduction continues (null: none)
	uint32_t bytes;
	int ld, rows;
};

struct DenseItem {
	DenseOperand a, b;
	int R, then, act, vec, tilesJ;
	float alpha;
	const float *bias; // per j
	float *out, *raw, *also;
	const float *z, *x, *d;
	double *headSums;
	float *rowSums; // per j: alpha times the sum of B's first matrix over the reduction
};

struct DenseBatch {
	int count;
	int first[kDenseBatch + 1]; // tiles of the products before
	DenseItem item[kDenseBatch];
};

// 32 * BLOCKS rows of an operand: lane l has row l % 32 (of each block) and the reduction indices 8 (l / 32) .. + 7 of a step
template <bool KCONTIG, int BLOCKS>
struct DenseLoader {
	uint32_t off[KCONTIG ? BLOCKS : 8];
	__device__ __forceinline__ void init(const DenseOperand &o, int row0, int lane)
	{
		const int row = row0 + (lane & 31), k = 8 * (lane >> 5);
		if constexpr (KCONTIG) {
#pragma unroll
			for (int b = 0; b < BLOCKS; b++) off[b] = row + 32 * b < o.rows ? 4u * ((uint32_t)(row + 32 * b) * (uint32_t)o.ld + (uint32_t)k) : kSplitNowhere;
		} else { // rows past the last are other rows' numbers, and of no result that is kept
#pragma unroll
			for (int q = 0; q < 8; q++) {
				const unsigned long long at = (unsigned long long)(k + q) * (unsigned)o.ld + (unsigned)row;
				off[q] = at < (1ull << 30) - 64 ? 4u * (uint32_t)at : kSplitNowhere;
			}
		}
	}
	// zero behind the last index where rows follow each other in memory (KCONTIG: what comes next in memory), and of a step that is not live
	__device__ __forceinline__ void load(const DenseOperand &o, bool second, int k0, bool live, float (&v)[BLOCKS][8]) const
	{
		const size_t at = 4 * (KCONTIG ? (size_t)k0 : (size_t)k0 * (unsigned)o.ld);
		const __amdgpu_buffer_rsrc_t rs = make_rsrc((const float *)((const char *)(second ? o.p2 : o.p) + at), live && at < o.bytes ? o.bytes - (uint32_t)at : 0u);
#pragma unroll
		for (int b = 0; b < BLOCKS; b++) {
			if constexpr (KCONTIG) {
#pragma unroll
				for (int h = 0; h < 2; h++) {
					const quad4f w = buffer_load4(rs, off[b] + 16u * h);
					v[b][4 * h] = w.x, v[b][4 * h + 1] = w.y, v[b][4 * h + 2] = w.z, v[b][4 * h + 3] = w.w;
				}
			} else {
#pragma unroll
				for (int q = 0; q < 8; q++) v[b][q] = buffer_load(rs, off[q] + 128u * b);
			}
		}
	}
	static __device__ __forceinline__ float at(const DenseOperand &o, bool second, int row, int k)
	{
		const float *p = second ? o.p2 : o.p;
		return KCONTIG ? p[(size_t)row * o.ld + k] : p[(size_t)k * o.ld + row];
	}
};

// what follows the product, for element (i, j) at `at`; loss terms of a head go to `terms`
__device__ __forceinline__ float dense_follow(const DenseItem &p, float v, size_t at, float &also, double (&terms)[2])
{
	switch (p.then) {
	case FITRE_DENSE_ACTIVATE: return act_forward_value(p.act, v);
	case FITRE_DENSE_DERIVATIVE: return p.act == ACT_LINEAR ? v : act_backward_value(p.act, v, 0.f, p.z[at]);
	case FITRE_DENSE_ROP_BACKWARD: {
		const float z = p.z ? p.z[at] : 0.f;
		float f1 = 1.f, g = 0.f;
		if (p.act == ACT_LOGISTIC) f1 = (1.f - z) * z, g = 1.f - 2.f * z;
		else if (p.act == ACT_TANH) f1 = (1.f + z) * (1.f - z), g = -2.f * z;
		float r = f1 * v;
		if (p.x) r += p.x[at] * g * p.d[at];
		return r;
	}
	case FITRE_DENSE_LOGISTIC_HEAD: {
		const float y = p.d[at], out = act_forward_value(ACT_LOGISTIC, v), ind = v >= 0.f ? 1.f : 0.f, e = y - out;
		terms[0] += (double)(v * (y - ind) - logf(1.f + expf(v - 2.f * v * ind)));
		terms[1] += (double)(e * e);
		also = e;
		return out;
	}
	case FITRE_DENSE_LINEAR_HEAD: {
		const float e = p.d[at] - v;
		terms[0] += (double)(e * e);
		terms[1] += (double)(e * e);
		also = 2.f * e;
		return v;
	}
	default: return v;
	}
}

template <bool AK, bool BK, int TI>
__device__ __forceinline__ void dense_product_tile(const DenseItem &p, const int tile)
{
	__shared__ float part[kDenseWaves][TI * 32][64]; // [wave][32 x 32 block and register of the accumulator][lane]
	__shared__ double lds2[2][kDenseWaves];
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int it = tile / p.tilesJ, i0 = it * 32 * TI, j0 = (tile - it * p.tilesJ) * kDenseJ;
	const int steps = (p.R + kDenseStep - 1) / kDenseStep, total = p.a.p2 ? 2 * steps : steps;
	const int beg = total * wave / kDenseWaves, end = total * (wave + 1) / kDenseWaves;
	const bool sums = p.rowSums != nullptr && it == 0;

	DenseLoader<AK, TI> A;
	DenseLoader<BK, 2> B;
	A.init(p.a, i0, lane);
	B.init(p.b, j0, lane);
	float av[kDenseSets][TI][8], bv[kDenseSets][2][8];
	v16f acc[TI][2], low[TI][2]; // the large products, and the five small ones
#pragma unroll
	for (int b = 0; b < TI; b++)
#pragma unroll
		for (int t = 0; t < 2; t++)
#pragma unroll
			for (int v = 0; v < 16; v++) acc[b][t][v] = low[b][t][v] = 0.f;
	double rs[2] = { 0.0, 0.0 };
#define DENSE_LOAD(S, U)                                                                                              \
	{                                                                                                                 \
		const bool second_ = (S) >= steps;                                                                            \
		const int k_ = ((S) - (second_ ? steps : 0)) * kDenseStep;                                                    \
		A.load(p.a, second_, k_, (S) < end, av[U]);                                                                   \
		B.load(p.b, second_, k_, (S) < end, bv[U]);                                                                   \
	}
#define DENSE_PRODUCTS(SUM, PA, PB)                                                                                   \
	_Pragma("unroll") for (int h = 0; h < TI; h++)                                                                     \
		_Pragma("unroll") for (int t = 0; t < 2; t++) SUM[h][t] = mfma_bf16(a[h][PA], b[t][PB], SUM[h][t]);
#pragma unroll
	for (int u = 0; u < kDenseSets; u++) DENSE_LOAD(beg + u, u);
	for (int s0 = beg; s0 < end; s0 += kDenseSets) {
#pragma unroll
		for (int u = 0; u < kDenseSets; u++) { // (a step past the wave's last is one of zeros)
			const int s = s0 + u;
			if constexpr (AK && BK) { // nothing else makes what follows a row's last number zero
				const int k = (s >= steps ? s - steps : s) * kDenseStep;
				if (k + kDenseStep > p.R) {
#pragma unroll
					for (int h = 0; h < TI; h++)
#pragma unroll
						for (int q = 0; q < 8; q++) av[u][h][q] = k + 8 * (lane >> 5) + q < p.R ? av[u][h][q] : 0.f;
				}
			}
			if (sums && s < steps) {
#pragma unroll
				for (int t = 0; t < 2; t++)
#pragma unroll
					for (int q = 0; q < 8; q++) rs[t] += (double)bv[u][t][q];
			}
			u32x4 a[TI][3], b[2][3];
#pragma unroll
			for (int h = 0; h < TI; h++) split_eight(av[u][h], a[h]);
#pragma unroll
			for (int t = 0; t < 2; t++) split_eight(bv[u][t], b[t]);
			DENSE_LOAD(s + kDenseSets, u);
			DENSE_PRODUCTS(acc, 0, 0);
			DENSE_PRODUCTS(low, 1, 0);
			DENSE_PRODUCTS(low, 0, 1);
			DENSE_PRODUCTS(low, 1, 1);
			DENSE_PRODUCTS(low, 2, 0);
			DENSE_PRODUCTS(low, 0, 2);
		}
	}
#undef DENSE_LOAD
#undef DENSE_PRODUCTS

#pragma unroll
	for (int h = 0; h < TI; h++)
#pragma unroll
		for (int t = 0; t < 2; t++)
#pragma unroll
			for (int v = 0; v < 16; v++) part[wave][32 * h + 16 * t + v][lane] = acc[h][t][v] + low[h][t][v];
	__syncthreads();
	// four results of each block a thread: consecutive j of one i
	float val[TI][4];
	bool suspect = false;
	const int l0 = (tid & 15) * 4, v = (tid >> 4) & 15, j = j0 + 32 * (tid >> 8) + (l0 & 31);
	const int iBase = i0 + 8 * (v / 4) + 4 * (l0 >> 5) + (v % 4);
#pragma unroll
	for (int h = 0; h < TI; h++) {
		double sum[4] = { 0.0, 0.0, 0.0, 0.0 };
#pragma unroll
		for (int w = 0; w < kDenseWaves; w++) {
			const float4 f = *(const float4 *)&part[w][32 * h + (tid >> 4)][l0];
			sum[0] += (double)f.x, sum[1] += (double)f.y, sum[2] += (double)f.z, sum[3] += (double)f.w;
		}
#pragma unroll
		for (int q = 0; q < 4; q++) {
			val[h][q] = (float)(sum[q] * (double)kSplitSumScale);
			suspect |= iBase + 32 * h < p.a.rows && j + q < p.b.rows && !(fabs(sum[q]) < 0x1p128); // an infinity or a NaN among the partial sums
		}
	}
	const bool exact = __syncthreads_or(suspect);
	double terms[2] = { 0.0, 0.0 };
#pragma unroll
	for (int h = 0; h < TI; h++) {
		const int i = iBase + 32 * h;
		if (i >= p.a.rows || j >= p.b.rows) continue;
		if (exact) { // by fp32 multiply-adds
#pragma unroll
			for (int q = 0; q < 4; q++) {
				if (j + q >= p.b.rows) continue;
				float c = 0.f;
				for (int second = 0; second < (p.a.p2 ? 2 : 1); second++)
					for (int k = 0; k < p.R; k++)
						c = fmaf(DenseLoader<AK, TI>::at(p.a, second != 0, i, k), DenseLoader<BK, 2>::at(p.b, second != 0, j + q, k), c);
				val[h][q] = c;
			}
		}
		const size_t at = (size_t)i * p.b.rows + j;
		float out[4], also[4] = { 0.f, 0.f, 0.f, 0.f };
#pragma unroll
		for (int q = 0; q < 4; q++) {
			if (j + q >= p.b.rows) continue;
			val[h][q] *= p.alpha;
			if (p.bias) val[h][q] += p.bias[j + q];
			out[q] = dense_follow(p, val[h][q], at + q, also[q], terms);
			if (p.then < FITRE_DENSE_LOGISTIC_HEAD) also[q] = -out[q];
		}
		if (p.vec) {
			*(float4 *)(p.out + at) = make_float4(out[0], out[1], out[2], out[3]);
			if (p.raw) *(float4 *)(p.raw + at) = make_float4(val[h][0], val[h][1], val[h][2], val[h][3]);
			if (p.also) *(float4 *)(p.also + at) = make_float4(also[0], also[1], also[2], also[3]);
		} else {
#pragma unroll
			for (int q = 0; q < 4; q++) {
				if (j + q >= p.b.rows) continue;
				p.out[at + q] = out[q];
				if (p.raw) p.raw[at + q] = val[h][q];
				if (p.also) p.also[at + q] = also[q];
			}
		}
	}
	if (p.then >= FITRE_DENSE_LOGISTIC_HEAD) {
		terms[0] = wave_sum(terms[0]), terms[1] = wave_sum(terms[1]);
		if (lane == 0) lds2[0][wave] = terms[0], lds2[1][wave] = terms[1];
		__syncthreads();
		if (tid < 2) {
			double s = 0.0;
#pragma unroll
			for (int w = 0; w < kDenseWaves; w++) s += lds2[tid][w];
			p.headSums[2 * tile + tid] = s;
		}
	}
	if (sums) { // (the partial tiles have been read: the barrier of the suspects is behind everyone)
		double *r = (double *)&part[0][0][0];
#pragma unroll
		for (int t = 0; t < 2; t++) r[(wave * 2 + t) * 64 + lane] = rs[t];
		__syncthreads();
		if (tid < kDenseJ && j0 + tid < p.b.rows) {
			double s = 0.0;
#pragma unroll
			for (int w = 0; w < kDenseWaves; w++) s += r[(w * 2 + (tid >> 5)) * 64 + (tid & 31)] + r[(w * 2 + (tid >> 5)) * 64 + 32 + (tid & 31)];
			p.rowSums[j0 + tid] = (float)s * p.alpha;
		}
	}
}

template <bool AK, bool BK, int TI>
__global__ void __launch_bounds__(kDenseThreads)
dense_product_kernel(const DenseBatch b)
{
	// an XCD takes consecutive tiles: those that read the same rows share its L2
	const unsigned groups = gridDim.x, xcd = blockIdx.x & 7u, each = groups >> 3, extra = groups & 7u;
	const int block = (int)(xcd * each + (xcd < extra ? xcd : extra) + (blockIdx.x >> 3));
	int m = 0;
	while (m + 1 < b.count && block >= b.first[m + 1]) m++;
	m = __builtin_amdgcn_readfirstlane(m);
	dense_product_tile<AK, BK, TI>(b.item[m], block - b.first[m]);
}

} // namespace fitre
