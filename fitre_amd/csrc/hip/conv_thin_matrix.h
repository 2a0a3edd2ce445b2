// Forward convolution of layers with very few input channels and nine to sixteen output channels (LeNet: 6 -> 16 with 5 x 5 windows) on
// the fp32 matrix pipes, from LDS.
//
// A workgroup has an image, some small ones or a band of rows in LDS with its zero border, and everything else follows from two
// tables: the word of a position in it, and the word a reduction index (channel, tap) lies further on.  v_mfma_f32_16x16x4_f32 then
// takes sixteen channels x sixteen positions; a step is one LDS word a lane for the four rows of weights, one of the table, and
// one per sixteen positions.  The pipe multiplies at twice the rate of plain vector instructions, so a product of less than nine
// rows is better off with those (conv_thin_forward.h); where it is not bound by either, it is shorter here because no wave waits
// for a scalar load of its weights.  Vector kernel / here, us: 6 -> 16 channels, 14 x 14 maps, 5 x 5 windows 11.4 / 7.8 at 128 images,
// 20.6 / 17.2 at 1024 (with activation and pool 12.1 / 9.2, 23.2 / 22.4), 16 -> 16 59 / 32 at 1024, 12 -> 9, 10 x 10, 3 x 3 13.0 /
// 5.6 at 128; but 3 -> 6, 32 x 32 9.4 / 11.4 and 28 / 60.  Input and weight gradients in this form were no shorter: 13 / 17 and
// 38.5 / 37.8 for the first layer named, whose gradient has six rows.
#pragma once
#include "conv_thin.h"

namespace fitre {

typedef float v4f __attribute__((ext_vector_type(4)));
__device__ __forceinline__ v4f mfma_f32_16(float a, float b, v4f c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

constexpr int kThinMatLeastRows = 9;
constexpr int kTileThinMatrix = 12; // profile variant
constexpr int kThinMatRows = 16, kThinMatPitch = 17; // rows of a product; words between two reduction indices of the weights in LDS
constexpr int kThinMatWaves = 4, kThinMatThreads = 64 * kThinMatWaves;

struct ThinMatParams {
	const float *src, *w, *bias;
	float *out;
	int cred, rows, samples, srcA, srcB, outA, outB, pad;
	int K, groups16;                // cred * ks * ks, in whole groups of four steps
	int images, bands, bandRows;    // images of a workgroup, or bands an image is cut into and their output rows
	int PA, PB, rowsAtOnce;         // bordered rows and their length; how many of them a wave stages at once
	int posWords;                   // words between two rows of a result in LDS
	FastDiv divRows, divPA, divPB, divPos, divOutB, divKK, divKs, divRowK;
	// the steps behind the product
	int act, store;
	bool average, toFc;
	float *actOut, *poolOut;
	FastDiv divItems, divGroups;    // patches of a row of a result, and of an image row
	int groups;
};

// Bordered rows of `rows` (image, channel, row) to LDS, the lanes along them; r of row (.., r) is image row r + a0
template <int WAVES>
__device__ __forceinline__ void thin_stage_rows(const float *src, size_t plane, size_t image, int rows, int srcA, int srcB, int a0, int pad, int PB, int atOnce,
                                                const FastDiv &divRows, const FastDiv &divPA, const FastDiv &divPB, int wave, int lane, float *dst)
{
	uint32_t sub, col;
	divPB.divmod((uint32_t)lane, sub, col);
	const bool mine = atOnce > 1 ? (int)sub < atOnce : true;
	for (int c0 = atOnce > 1 ? (int)col : lane, first = 1; first || (atOnce == 1 && c0 < PB); c0 += 64, first = 0) {
		const int s = atOnce > 1 ? (int)sub : 0, b = c0 - pad;
		for (int r0 = wave * atOnce + s; r0 < rows; r0 += WAVES * atOnce * 8) {
			float v[8];
#pragma unroll
			for (int u = 0; u < 8; u++) {
				const int row = r0 + WAVES * atOnce * u;
				uint32_t im, rest, c, r;
				divRows.divmod((uint32_t)(row < rows ? row : 0), im, rest);
				divPA.divmod(rest, c, r);
				const int a = (int)r + a0;
				const bool ok = mine & (row < rows) & ((unsigned)a < (unsigned)srcA) & ((unsigned)b < (unsigned)srcB);
				v[u] = ok ? src[(size_t)c * plane + (size_t)im * image + a * srcB + b] : 0.f;
			}
#pragma unroll
			for (int u = 0; u < 8; u++) {
				const int row = r0 + WAVES * atOnce * u;
				if (mine && row < rows && c0 < PB) dst[row * PB + c0] = v[u];
			}
		}
	}
}

// The weights of a layer, [cout][K] in memory, as [reduction index][kThinMatPitch] and zero behind the last index, and the words its
// reduction indices lie behind a position in a bordered image
template <int THREADS>
__device__ __forceinline__ void thin_mat_tables(const float *w, int rows, int K, int K4, int plane, int PB, const FastDiv &divK, const FastDiv &divKK, const FastDiv &divKs,
                                                float *W, int *further)
{
	const int tid = threadIdx.x;
	for (int e0 = tid; e0 < rows * K; e0 += THREADS * 8) {
		float v[8];
#pragma unroll
		for (int u = 0; u < 8; u++) v[u] = e0 + THREADS * u < rows * K ? w[e0 + THREADS * u] : 0.f;
#pragma unroll
		for (int u = 0; u < 8; u++) {
			const int e = e0 + THREADS * u;
			if (e >= rows * K) break;
			uint32_t row, k;
			divK.divmod((uint32_t)e, row, k);
			W[(int)k * kThinMatPitch + (int)row] = v[u];
		}
	}
	for (int e = K * kThinMatPitch + tid; e < K4 * kThinMatPitch; e += THREADS) W[e] = 0.f;
	for (int k = tid; k < K4; k += THREADS) {
		uint32_t c, tap, ta, tb;
		divKK.divmod((uint32_t)k, c, tap);
		divKs.divmod(tap, ta, tb);
		further[k] = k < K ? (int)c * plane + (int)ta * PB + (int)tb : 0;
	}
}

// sixteen rows x TN blocks of sixteen positions, whose words in S are `at`: four steps at a time; their words are read while the
// four before are multiplied, and where they are while those before that
template <int TN>
__device__ __forceinline__ void thin_mat_multiply(const float *W, const int *further, const float *S, const int (&at)[TN], int K, int groups16, v4f (&acc)[TN])
{
	const int lane = threadIdx.x & 63, l16 = lane & 15, lk = lane >> 4, last = groups16 - 1;
	const float *wk = W + lk * kThinMatPitch + l16;
	const int *fk = further + lk;
	int f[4];
	float a[2][4], x[2][TN][4];
	auto where = [&](int g) {
#pragma unroll
		for (int q = 0; q < 4; q++) f[q] = fk[16 * g + 4 * q];
	};
	auto read = [&](int g, float (&aTo)[4], float (&xTo)[TN][4]) {
#pragma unroll
		for (int q = 0; q < 4; q++) {
			aTo[q] = wk[(16 * g + 4 * q) * kThinMatPitch];
#pragma unroll
			for (int u = 0; u < TN; u++) xTo[u][q] = S[f[q] + at[u]];
		}
		if (g == last) { // nothing behind the last reduction index
#pragma unroll
			for (int q = 0; q < 4; q++)
#pragma unroll
				for (int u = 0; u < TN; u++) xTo[u][q] = 16 * g + 4 * q + lk < K ? xTo[u][q] : 0.f;
		}
	};
	auto multiply = [&](const float (&aOf)[4], const float (&xOf)[TN][4]) {
#pragma unroll
		for (int q = 0; q < 4; q++)
#pragma unroll
			for (int u = 0; u < TN; u++) acc[u] = mfma_f32_16(aOf[q], xOf[u][q], acc[u]);
	};
#pragma unroll
	for (int u = 0; u < TN; u++) acc[u] = v4f{ 0.f, 0.f, 0.f, 0.f };
	where(0);
	read(0, a[0], x[0]);
	where(last < 1 ? last : 1);
	for (int g = 0; g < groups16; g += 2) {
		read(g + 1 < last ? g + 1 : last, a[1], x[1]);
		where(g + 2 < last ? g + 2 : last);
		multiply(a[0], x[0]);
		if (g + 1 > last) break;
		read(g + 2 < last ? g + 2 : last, a[0], x[0]);
		where(g + 3 < last ? g + 3 : last);
		multiply(a[1], x[1]);
	}
}

// TN: blocks of sixteen positions a wave has at once.  FOLD: the layer's activation and pool behind it.
template <bool FOLD, int TN>
__global__ void __launch_bounds__(kThinMatThreads) thin_matrix_kernel(const ThinMatParams p)
{
	extern __shared__ __align__(16) float thin_lds[];
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lk = lane >> 4;
	const int n0 = (int)blockIdx.x * p.images, images = p.samples - n0 < p.images ? p.samples - n0 : p.images;
	const int row0 = (int)blockIdx.y * p.bandRows, bandRows = p.outA - row0 < p.bandRows ? p.outA - row0 : p.bandRows;
	const int K4 = 16 * p.groups16, plane = p.PA * p.PB;
	float *W = thin_lds, *S = W + K4 * kThinMatPitch + K4;
	int *further = (int *)(W + K4 * kThinMatPitch);
	float *Y = S + p.images * p.cred * plane;

	const size_t srcPlane = (size_t)p.samples * p.srcA * p.srcB, srcImage = (size_t)p.srcA * p.srcB;
	thin_stage_rows<kThinMatWaves>(p.src + (size_t)n0 * srcImage, srcPlane, srcImage, images * p.cred * p.PA, p.srcA, p.srcB, row0 - p.pad, p.pad, p.PB,
	                               p.rowsAtOnce, p.divRows, p.divPA, p.divPB, wave, lane, S);
	thin_mat_tables<kThinMatThreads>(p.w, p.rows, p.K, K4, plane, p.PB, p.divRowK, p.divKK, p.divKs, W, further);
	__syncthreads();

	const int positions = images * bandRows * p.outB, tiles = (positions + 15) / 16;
	const size_t outPlane = (size_t)p.samples * p.outA * p.outB;
	for (int task = wave; task * TN < tiles; task += kThinMatWaves) {
		int at[TN];
		v4f acc[TN];
#pragma unroll
		for (int u = 0; u < TN; u++) {
			const int pos = (task * TN + u) * 16 + l16;
			uint32_t im, rest, r, b;
			p.divPos.divmod((uint32_t)(pos < positions ? pos : positions - 1), im, rest);
			p.divOutB.divmod(rest, r, b);
			at[u] = (int)im * p.cred * plane + (int)r * p.PB + (int)b;
		}
		thin_mat_multiply<TN>(W, further, S, at, p.K, p.groups16, acc);
#pragma unroll
		for (int u = 0; u < TN; u++) {
			const int pos = (task * TN + u) * 16 + l16;
			if (pos >= positions) continue;
#pragma unroll
			for (int v = 0; v < 4; v++) {
				const int i = 4 * lk + v;
				if (i >= p.rows) break;
				const float val = acc[u][v] + (p.bias ? p.bias[i] : 0.f);
				if constexpr (FOLD) {
					Y[i * p.posWords + pos] = val;
				} else {
					uint32_t im, rest;
					p.divPos.divmod((uint32_t)pos, im, rest);
					p.out[(size_t)i * outPlane + (size_t)(n0 + (int)im) * p.outA * p.outB + row0 * p.outB + (int)rest] = val;
				}
			}
		}
	}
	if constexpr (!FOLD) return;
	__syncthreads();
	// patches of two rows x four cells, (channel, image, row pair, group); outA and outB are even
	const int pairs = bandRows / 2, perRow = images * pairs * p.groups;
	for (int item = tid; item < p.rows * perRow; item += kThinMatThreads) {
		const int i = item / perRow, rest = item - i * perRow;
		uint32_t im = 0, cell = (uint32_t)rest, rp, g;
		if (p.bands == 1) p.divItems.divmod((uint32_t)rest, im, cell); // (a band is of one image)
		p.divGroups.divmod(cell, rp, g);
		const int n = n0 + (int)im, r = 2 * (int)rp, a = row0 + r, b = 4 * (int)g, left = p.outB - b;
		const float *y = Y + i * p.posWords + ((int)im * bandRows + r) * p.outB + b;
		const size_t to = (((size_t)i * p.samples + n) * p.outA + a) * p.outB + b;
		float v[2][4];
#pragma unroll
		for (int h = 0; h < 2; h++) {
#pragma unroll
			for (int j = 0; j < 4; j++) v[h][j] = j < left ? y[h * p.outB + j] : 0.f;
			thin_store_row(p.out + to + (size_t)h * p.outB, v[h], p.store, left);
#pragma unroll
			for (int j = 0; j < 4; j++) v[h][j] = act_forward_value(p.act, v[h][j]);
			thin_store_row(p.actOut + to + (size_t)h * p.outB, v[h], p.store, left);
		}
		const int poolA = p.outA / 2, poolB = p.outB / 2;
#pragma unroll
		for (int q = 0; q < 2; q++) {
			if (2 * q >= left) break;
			const float top = pool2x2(p.average, v[0][2 * q], v[0][2 * q + 1], v[1][2 * q], v[1][2 * q + 1]);
			const int oa = a / 2, ob = 2 * (int)g + q;
			if (p.toFc) p.poolOut[((size_t)n * p.rows + i) * (poolA * poolB) + (size_t)ob * poolA + oa] = top;
			else p.poolOut[(((size_t)i * p.samples + n) * poolA + oa) * poolB + ob] = top;
		}
	}
}

// ---- host side ------------------------------------------------------------------------------------------------------
constexpr int kThinMatLdsFloats = 16384; // 64 KB: two workgroups on a compute unit

struct ThinMatPlan {
	ThinMatParams p;
	int groupsX, tn;
	size_t lds;
};
// fold: with the layer's activation and pool, in bands of whole row pairs
static inline bool thin_mat_plan(const fitre_conv_shape *s, bool fold, ThinMatPlan &plan)
{
	const int rows = s->outChannels, cred = s->inChannels, samples = s->samples, outA = s->outA, outB = s->outB, ks = s->ksize;
	ThinMatParams p{};
	p.cred = cred, p.rows = rows, p.samples = samples, p.srcA = s->inA, p.srcB = s->inB, p.outA = outA, p.outB = outB, p.pad = s->padding;
	p.K = cred * ks * ks, p.groups16 = (p.K + 15) / 16;
	if (rows > kThinMatRows) return false;
	const int cells = outA * outB, cus = device_compute_units(), unit = fold ? 2 : 1, units = (outA + unit - 1) / unit;
	// 256 positions keep the four waves' blocks full; images are cut while there are fewer than two workgroups a compute unit
	p.images = cells < 256 ? 256 / cells : 1;
	while (p.images > 1 && samples / p.images < 2 * cus) p.images--;
	if (p.images > samples) p.images = samples;
	int bands = 1;
	if (p.images == 1) {
		bands = (2 * cus + samples - 1) / samples;
		if (bands > units) bands = units;
		if (bands > 1 && bands > cells / 64) bands = cells / 64 > 1 ? cells / 64 : 1;
	}
	const int fixed = 16 * p.groups16 * (kThinMatPitch + 1);
	for (;;) {
		p.bandRows = (units + bands - 1) / bands * unit;
		if (p.bandRows > outA) p.bandRows = outA;
		p.bands = (outA + p.bandRows - 1) / p.bandRows;
		p.PA = p.bandRows + ks - 1, p.PB = outB + ks - 1;
		const int positions = p.images * p.bandRows * outB;
		p.posWords = ((positions + 63) & ~63) + 4;
		const int words = fixed + p.images * cred * p.PA * p.PB + (fold ? rows * p.posWords : 0);
		plan.lds = sizeof(float) * (size_t)words;
		if (words <= kThinMatLdsFloats) break;
		if (p.images > 1) p.images--;
		else if (bands < units) bands++;
		else return false;
	}
	p.rowsAtOnce = p.PB <= 64 ? 64 / p.PB : 1;
	p.divRowK = FastDiv((uint32_t)p.K), p.divRows = FastDiv((uint32_t)(cred * p.PA)), p.divPA = FastDiv((uint32_t)p.PA), p.divPB = FastDiv((uint32_t)p.PB);
	p.divPos = FastDiv((uint32_t)(p.bandRows * outB)), p.divOutB = FastDiv((uint32_t)outB);
	p.divKK = FastDiv((uint32_t)(ks * ks)), p.divKs = FastDiv((uint32_t)ks);
	p.groups = (outB + 3) / 4;
	p.divItems = FastDiv((uint32_t)((p.bandRows + unit - 1) / unit * p.groups)), p.divGroups = FastDiv((uint32_t)p.groups);
	const int tiles = (p.images * p.bandRows * outB + 15) / 16, each = (tiles + kThinMatWaves - 1) / kThinMatWaves;
	plan.tn = each >= 4 ? 4 : (each >= 2 ? 2 : 1);
	plan.groupsX = (samples + p.images - 1) / p.images;
	plan.p = p;
	return true;
}

template <bool FOLD>
static void launch_thin_matrix(const ThinMatPlan &plan)
{
	const dim3 grid((unsigned)plan.groupsX, (unsigned)plan.p.bands);
	if (plan.tn == 4) thin_matrix_kernel<FOLD, 4><<<grid, kThinMatThreads, plan.lds, stream()>>>(plan.p);
	else if (plan.tn == 2) thin_matrix_kernel<FOLD, 2><<<grid, kThinMatThreads, plan.lds, stream()>>>(plan.p);
	else thin_matrix_kernel<FOLD, 1><<<grid, kThinMatThreads, plan.lds, stream()>>>(plan.p);
}

} // namespace fitre
