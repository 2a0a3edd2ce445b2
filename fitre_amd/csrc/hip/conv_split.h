// 3x3 and 5x5 convolutions of stride 1 that keep the map's size, forward and input gradient, on the bf16 pipes (split_bf16.h).
//
//     out[i][m] = sum_{c, ta, tb} Wsel(i, c, ta, tb) * src[c][m + (ta-P)*B + (tb-P)]      (zero outside the image)
//
// Weights are split once per call into the order the matrix fragments are read in (split_weights_kernel) and go from L2
// straight into registers, one coalesced 16-byte load per fragment, a tap ahead of their use.  The raw source window of
// sixteen channels is split while it is staged and sits in LDS as [part][half of the channels][cell][8 channels], cells in
// the zero-padded order (every image row followed by P zero cells, every image by P zero rows): the fragment of tap
// (ta, tb) is the lane's own 16-byte word + an offset that is the same for all lanes, and one conversion serves KS*KS taps.
// The window is double buffered: one barrier per sixteen channels.
#pragma once
#include "conv3x3.h"
#include "split_bf16.h"

namespace fitre {

constexpr int kSplitCB = 16; // reduction channels per block: the depth of one bf16 MFMA

struct ConvSplitParams {
	const float *src, *w;    // [cred][N][A][B]; the layer's own [Cout][Cin][KS][KS]
	const u32x4 *wp;         // split weights
	const float *src2, *w2;  // a second pair over which the reduction continues (null: none)
	const u32x4 *wp2;
	uint32_t srcBytes;
	int I, cred, J, A, B;
	int dx;                  // the input gradient: which way w is read where the tile is computed by fp32 multiply-adds
	int perSplit;            // channel blocks per split
	int rowGroups;           // groups of 32 output channels of the split weights
	int before;              // cells of the padded window before the tile's first position
	int late;                // whole images added to a position so that those of the halo before the tensor are not negative
	FastDiv divB, divA;
};

// ---- weights ------------------------------------------------------------------------------------------------------
// [channel block][tap][32 rows][part][half of the channels][row][8 channels] of bf16; rows past I are zero.  A workgroup makes one (channel block, 32 rows): its floats go through LDS, read in memory order.
// DX: rows are the layer's input channels, the reduction runs over its output channels, windows are flipped.
template <int KS, bool DX>
__device__ __forceinline__ void split_weights_block(const float *w, int I, int cred, int rowGroups, u32x4 *wp, int rb, int cb)
{
	constexpr int T = KS * KS, LD = DX ? 32 * T + 1 : kSplitCB * T + 1, ROWS = DX ? kSplitCB : 32;
	constexpr int SPAN = DX ? 32 * T : kSplitCB * T; // floats in a row, consecutive in memory
	__shared__ float L[ROWS * LD];
	const int i0 = rb * 32, c0 = cb * kSplitCB;
	const int rowLen = (DX ? I : cred) * T, col0 = (DX ? i0 : c0) * T, row0 = DX ? c0 : i0;
	const int live = (I - i0 < 32 ? I - i0 : 32) * T; // DX: floats of a row inside the tensor
	constexpr int N = ROWS * SPAN / 256;
	float v[N]; // every load is under way before the first is waited for: 10 -> 4 us where the weights come from memory
#pragma unroll
	for (int k = 0; k < N; k++) {
		const int e = threadIdx.x + 256 * k, r = e / SPAN, x = e - r * SPAN;
		v[k] = (DX ? x < live : i0 + r < I) ? w[(size_t)(row0 + r) * rowLen + col0 + x] : 0.f;
	}
#pragma unroll
	for (int k = 0; k < N; k++) {
		const int e = threadIdx.x + 256 * k, r = e / SPAN;
		L[r * LD + e - r * SPAN] = v[k];
	}
	__syncthreads();
	for (int u = threadIdx.x; u < T * 64; u += 256) {
		const int tap = u >> 6, half = (u >> 5) & 1, row = u & 31;
		float x[8];
#pragma unroll
		for (int q = 0; q < 8; q++) {
			const int c = half * 8 + q;
			x[q] = DX ? L[c * LD + row * T + (T - 1 - tap)] : L[row * LD + c * T + tap];
		}
		u32x4 part[3];
		split_eight(x, part);
		u32x4 *dst = wp + ((size_t)(cb * T + tap) * rowGroups + rb) * 192 + (u & 63);
#pragma unroll
		for (int s = 0; s < 3; s++) dst[s * 64] = part[s];
	}
}

// one layer's; blockIdx.z: a pair's second weights, whose parts follow the first's
template <int KS, bool DX>
__global__ void __launch_bounds__(256)
split_weights_kernel(const float *w, const float *w2, int I, int cred, int rowGroups, u32x4 *wp)
{
	if (blockIdx.z) w = w2, wp += (size_t)gridDim.y * KS * KS * rowGroups * 192;
	split_weights_block<KS, DX>(w, I, cred, rowGroups, wp, blockIdx.x, blockIdx.y);
}

// several layers': a pass has the copies of all of them made at once, beside its first steps
constexpr int kSplitWeightsBatch = 16;
struct SplitWeightsBatch {
	int count;
	int first[kSplitWeightsBatch + 1]; // blocks of the layers before
	int I[kSplitWeightsBatch], cred[kSplitWeightsBatch], rowGroups[kSplitWeightsBatch];
	const float *w[kSplitWeightsBatch];
	u32x4 *wp[kSplitWeightsBatch];
};
template <int KS, bool DX>
__global__ void __launch_bounds__(256) split_weights_batch_kernel(const SplitWeightsBatch b)
{
	int m = 0;
	while (m + 1 < b.count && (int)blockIdx.x >= b.first[m + 1]) m++;
	const int block = (int)blockIdx.x - b.first[m], groups = b.rowGroups[m], cb = block / groups;
	split_weights_block<KS, DX>(b.w[m], b.I[m], b.cred[m], groups, b.wp[m], block - cb * groups, cb);
}

// ---- the product --------------------------------------------------------------------------------------------------
// A wave owns 32 channels x 128 positions: the waves of a workgroup share the source window in LDS, and no two of them load the
// same weights.  128 x 128 per workgroup, or 64 x 256 for products of at most 64 channels.
template <int WM> struct ConvSplitTile {
	static constexpr int WN = 4 / WM, IT = 32 * WM, JT = 128 * WN;
};
inline int conv_split_halo(int P, int B) { return P * (B + 1); }
inline int conv_split_before(int P, int A, int B)
{
	const int halo = conv_split_halo(P, B);
	return halo + (halo + B - 1) / B * P + (halo + A * B - 1) / (A * B) * P * (B + P);
}
inline int conv_split_window(int P, int A, int B, int jt)
{
	const int halo = conv_split_halo(P, B), span = jt - 1 + halo;
	return conv_split_before(P, A, B) + span + 1 + ((span + B - 1) / B + 1) * P + (span + A * B - 1) / (A * B) * P * (B + P);
}

// whole images added to a position so that the halo before position 0 has an index too
inline int conv_split_late(int P, int A, int B) { return (conv_split_halo(P, B) + A * B - 1) / (A * B) * A * B; }

// the kernel a shape takes: waves along the channels, cells of the window there is LDS for (twice, 12 bytes and 16 channels each,
// for one workgroup per compute unit at least), (cell, half) pairs a thread stages
struct ConvSplitVariant {
	int ks, wm, cells, xe;
};
constexpr ConvSplitVariant kConvSplitVariants[] = {
	{ 3, 4, 240, 2 }, { 3, 4, 320, 2 }, { 3, 4, 512, 3 }, { 3, 2, 400, 3 }, { 5, 4, 424, 2 }, { 5, 2, 520, 3 },
};
inline const ConvSplitVariant *conv_split_variant(int ks, int I, int A, int B)
{
	const int wm = I <= 64 ? 2 : 4, P = ks / 2, jt = 128 * (4 / wm);
	for (const ConvSplitVariant &v : kConvSplitVariants)
		if (v.ks == ks && v.wm == wm && conv_split_window(P, A, B, jt) <= v.cells && 2 * (jt + 2 * conv_split_halo(P, B)) <= kGemmThreads * v.xe)
			return &v;
	return nullptr;
}

__device__ __forceinline__ uint32_t conv_split_cell(const ConvSplitParams &p, int P, uint32_t m)
{
	uint32_t q, b, n, a;
	p.divB.divmod(m, q, b);
	p.divA.divmod(q, n, a);
	return (n * (uint32_t)(p.A + P) + a) * (uint32_t)(p.B + P) + b;
}

// the tile by fp32 multiply-adds, for sums the split may not have carried: eight channels x 64 positions a wave at a time
template <int KS, int IT, int JT>
__device__ __forceinline__ void conv_split_exact_tile(const ConvSplitParams &p, const OutParams &out, int i0, int j0, int cbBeg, int cbEnd, float *C)
{
	constexpr int P = KS / 2, T = KS * KS;
	const int lane = threadIdx.x & 63;
	const int cbHalf = p.cred / kSplitCB;
	for (int g = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); g < IT / 8 * (JT / 64); g += 4) {
		const int iBase = i0 + g % (IT / 8) * 8, j = j0 + g / (IT / 8) * 64 + lane;
		if (iBase >= p.I) continue;
		uint32_t q, b, n, a;
		p.divB.divmod((uint32_t)j, q, b);
		p.divA.divmod(q, n, a);
		float s[8];
#pragma unroll
		for (int r = 0; r < 8; r++) s[r] = 0.f;
		for (int c = cbBeg * kSplitCB; c < cbEnd * kSplitCB; c++) {
			const bool second = c >= cbHalf * kSplitCB;
			const int cc = second ? c - cbHalf * kSplitCB : c;
			const float *src = (second ? p.src2 : p.src) + (size_t)cc * p.J, *w = second ? p.w2 : p.w;
			for (int t = 0; t < T; t++) {
				const int da = t / KS - P, db = t % KS - P;
				const bool in = j < p.J && (unsigned)((int)a + da) < (unsigned)p.A && (unsigned)((int)b + db) < (unsigned)p.B;
				const float x = in ? src[j + da * p.B + db] : 0.f;
#pragma unroll
				for (int r = 0; r < 8; r++) {
					const int i = iBase + r < p.I ? iBase + r : p.I - 1;
					s[r] = fmaf(w[p.dx ? ((size_t)cc * p.I + i) * T + (T - 1 - t) : ((size_t)i * p.cred + cc) * T + t], x, s[r]);
				}
			}
		}
		if (j >= p.J) continue;
		for (int r = 0; r < 8 && iBase + r < p.I; r++)
			C[(size_t)(iBase + r) * out.ldc + j] = s[r] + (!out.splitStride && out.biasI ? out.biasI[iBase + r] : 0.f);
	}
}

// CELLS: cells of the padded window there is room for.  XE: (cell, half) pairs a thread stages.
template <int KS, int WM, int CELLS, int XE>
__global__ void __launch_bounds__(kGemmThreads, 2 * 192 * (CELLS + 1) <= 160 * 1024 ? 2 : 1)
conv_split_kernel(const ConvSplitParams p, const OutParams out)
{
	FITRE_RAISE_MATRIX_WAVE_PRIORITY();
	constexpr int P = KS / 2, T = KS * KS, TN = 4;
	constexpr int WN = ConvSplitTile<WM>::WN, IT = ConvSplitTile<WM>::IT, JT = ConvSplitTile<WM>::JT;
	constexpr int HALF = CELLS + 1, PART = 2 * HALF, BUF = 3 * PART; // in 16-byte words; cell CELLS takes what has no place
	__shared__ u32x4 Bs[2 * BUF];

	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int khalf = lane >> 5, l32 = lane & 31;
	const int i0 = blockIdx.y * IT, j0 = blockIdx.x * JT;
	const int halo = P * (p.B + 1), win = JT + 2 * halo, pitch = p.B + P;
	const int cbHalf = p.cred / kSplitCB, cbTotal = p.src2 ? 2 * cbHalf : cbHalf;
	const int cbBeg = blockIdx.z * p.perSplit, cbEnd = cbBeg + p.perSplit < cbTotal ? cbBeg + p.perSplit : cbTotal;
	const uint32_t ref = conv_split_cell(p, P, (uint32_t)(j0 + p.late));

	for (int i = tid; i < 2 * BUF; i += kGemmThreads) Bs[i] = u32x4{ 0, 0, 0, 0 };

	// what this thread stages, the same for every block: cell x of the window, eight of the sixteen channels
	uint32_t sOff[XE];
	int sLds[XE];
#pragma unroll
	for (int e = 0; e < XE; e++) {
		const int u = tid + kGemmThreads * e, half = u >= win, x = u - (half ? win : 0);
		const int m = j0 - halo + x;
		const bool has = x < win, inside = has & (m >= 0) & (m < p.J);
		sOff[e] = inside ? 4u * ((uint32_t)(half * 8) * (uint32_t)p.J + (uint32_t)m) : kOutOfRange;
		sLds[e] = half * HALF + (has ? (int)(conv_split_cell(p, P, (uint32_t)(m + p.late)) - ref) + p.before : CELLS);
	}
	float sreg[XE][8];
	v16f acc[TN], low[TN]; // the large products, and the five small ones
#pragma unroll
	for (int tn = 0; tn < TN; tn++)
#pragma unroll
		for (int v = 0; v < 16; v++) acc[tn][v] = low[tn][v] = 0.f;

	int bCell[TN]; // 16-byte words, tap (0, 0)
#pragma unroll
	for (int tn = 0; tn < TN; tn++) {
		const uint32_t m = (uint32_t)(j0 + wave % WN * 128 + tn * 32 + l32);
		bCell[tn] = (int)(conv_split_cell(p, P, m + p.late) - ref) + p.before - P * pitch - P + khalf * HALF;
	}
	// this wave's 32 rows of the split weights: 192 words per (block, tap)
	const size_t rowWords = (size_t)(blockIdx.y * WM + wave / WN) * 192, tapWords = (size_t)p.rowGroups * 192;

#define SPLIT_LOAD_WINDOW(CB)                                                                                         \
	{                                                                                                                 \
		const bool second_ = (CB) >= cbHalf;                                                                          \
		const size_t shift_ = (size_t)(((CB) - (second_ ? cbHalf : 0)) * kSplitCB) * p.J;                             \
		const __amdgpu_buffer_rsrc_t rs_ = make_rsrc((second_ ? p.src2 : p.src) + shift_, p.srcBytes - (uint32_t)(4 * shift_)); \
		_Pragma("unroll") for (int e = 0; e < XE; e++)                                                                \
			_Pragma("unroll") for (int q = 0; q < 8; q++)                                                             \
				sreg[e][q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_, (int)sOff[e], 4 * q * p.J, 0)); \
	}
#define SPLIT_STORE_WINDOW(BUFFER, E)                                                                                 \
	{                                                                                                                 \
		u32x4 part_[3];                                                                                               \
		split_eight(sreg[E], part_);                                                                                  \
		_Pragma("unroll") for (int s = 0; s < 3; s++) Bs[(BUFFER) * BUF + s * PART + sLds[E]] = part_[s];             \
	}
// the four products of part PA of the weights and part PB of the source
#define SPLIT_PRODUCTS(SUM, PA, PB)                                                                                   \
	_Pragma("unroll") for (int tn = 0; tn < TN; tn++) SUM[tn] = mfma_bf16(a[cur][PA], b[tn][PB], SUM[tn]);
#define SPLIT_READ_PART(S)                                                                                            \
	_Pragma("unroll") for (int tn = 0; tn < TN; tn++) b[tn][S] = bNext[bCell[tn] + (S) * PART];
#define SPLIT_READ_WEIGHTS(SET, FROM)                                                                                 \
	_Pragma("unroll") for (int s = 0; s < 3; s++) a[SET][s] = (FROM)[s * 64 + lane];

	SPLIT_LOAD_WINDOW(cbBeg);
	__syncthreads(); // the zeros are in place
#pragma unroll
	for (int e = 0; e < XE; e++) SPLIT_STORE_WINDOW(0, e);
	__syncthreads();

	u32x4 a[2][3], b[TN][3];
	const u32x4 *wBlock = (cbBeg >= cbHalf ? p.wp2 + (size_t)(cbBeg - cbHalf) * T * tapWords : p.wp + (size_t)cbBeg * T * tapWords) + rowWords;
	SPLIT_READ_WEIGHTS(0, wBlock);
	const u32x4 *bNext = Bs;
	SPLIT_READ_PART(2);
	SPLIT_READ_PART(1);
	SPLIT_READ_PART(0);

	for (int cb = cbBeg; cb < cbEnd; cb++) {
		const int buffer = (cb - cbBeg) & 1;
		const bool more = cb + 1 < cbEnd;
		const int nb = more ? cb + 1 : cb; // (the last block's is staged once more, and not read)
		const u32x4 *wNext = (nb >= cbHalf ? p.wp2 + (size_t)(nb - cbHalf) * T * tapWords : p.wp + (size_t)nb * T * tapWords) + rowWords;
		// A tap's fragments are read while the tap before it is multiplied: the weights into the other register set, a part
		// of the source into the registers whose last product has been issued.  The next block's window arrives during the
		// first taps and is split and stored during the last ones.
#pragma unroll
		for (int t = 0; t < T; t++) {
			const int cur = t & 1, nxt = cur ^ 1;
			const u32x4 *wTap = t + 1 < T ? wBlock + (size_t)(t + 1) * tapWords : wNext;
			bNext = Bs + buffer * BUF + (t + 1) / KS * pitch + (t + 1) % KS;
			SPLIT_READ_WEIGHTS(nxt, wTap);
			if (t == 0) SPLIT_LOAD_WINDOW(nb);
			SPLIT_PRODUCTS(low, 0, 2);
			__builtin_amdgcn_sched_barrier(0);
			if (t + 1 < T) SPLIT_READ_PART(2);
			if (t >= T - XE) SPLIT_STORE_WINDOW(buffer ^ 1, t - (T - XE));
			SPLIT_PRODUCTS(low, 0, 1);
			SPLIT_PRODUCTS(low, 1, 1);
			if (t >= T - XE) {
#pragma unroll
				for (int i = 0; i < 8; i++) {
					__builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
					__builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
				}
			}
			__builtin_amdgcn_sched_barrier(0);
			if (t + 1 < T) SPLIT_READ_PART(1);
			SPLIT_PRODUCTS(low, 2, 0);
			SPLIT_PRODUCTS(low, 1, 0);
			SPLIT_PRODUCTS(acc, 0, 0);
			__builtin_amdgcn_sched_barrier(0);
			if (t + 1 < T) SPLIT_READ_PART(0);
		}
		// an odd number of taps leaves the next block's first fragments in the other half
		if constexpr (T & 1) {
#pragma unroll
			for (int s = 0; s < 3; s++) a[0][s] = a[1][s];
		}
		wBlock = wNext;
		__syncthreads();
		bNext = Bs + (buffer ^ 1) * BUF;
		SPLIT_READ_PART(2);
		SPLIT_READ_PART(1);
		SPLIT_READ_PART(0);
	}
#undef SPLIT_PRODUCTS
#undef SPLIT_READ_PART
#undef SPLIT_READ_WEIGHTS
#undef SPLIT_LOAD_WINDOW
#undef SPLIT_STORE_WINDOW

	const bool split = out.splitStride != 0;
	float *C = out.C + (size_t)blockIdx.z * out.splitStride;
	bool suspect = false;
#pragma unroll
	for (int tn = 0; tn < TN; tn++)
#pragma unroll
		for (int v = 0; v < 16; v++) {
			acc[tn][v] += low[tn][v];
			suspect |= split_sum_suspect(acc[tn][v]);
		}
	if (__syncthreads_or(suspect)) {
		conv_split_exact_tile<KS, IT, JT>(p, out, i0, j0, cbBeg, cbEnd, C);
		return;
	}
#pragma unroll
	for (int tn = 0; tn < TN; tn++) {
		const int j = j0 + wave % WN * 128 + tn * 32 + l32;
		if (j >= p.J) continue;
#pragma unroll
		for (int v = 0; v < 16; v++) {
			const int i = i0 + wave / WN * 32 + 8 * (v / 4) + 4 * khalf + (v % 4);
			if (i >= p.I) continue;
			float val = acc[tn][v] * kSplitSumScale;
			if (!split && out.biasI) val += out.biasI[i];
			C[(size_t)i * out.ldc + j] = val;
		}
	}
}

// ---- 4 x 4 maps ------------------------------------------------------------------------------------------------------
// The columns of a matrix block are one cell of 32 images, so that the 44 of 144 (cell, tap) pairs that reach outside a map are
// left out: a workgroup owns 32 channels x 32 images, a wave a quadrant of the map and its 25 live pairs.  Quadrants are seen
// mirrored so that each has the map's corner at local cell (0, 0): what is live is then known at compile time, and only the
// addresses of cells and taps differ.  The nine source cells of a quadrant stay in registers for a block of sixteen channels;
// weights stream as above.  One workgroup per compute unit with up to 512 registers a lane.  512 -> 512 channels, 256 images, two
// ranges: 80 us in the window form, 67 in this.
constexpr int kCellSplitImages = 32, kCellSplitRows = 32;
__global__ void __launch_bounds__(kGemmThreads, 1)
conv_split_cell_kernel(const ConvSplitParams p, const OutParams out)
{
	FITRE_RAISE_MATRIX_WAVE_PRIORITY();
	constexpr int T = 9, LDN = 33, HALF = 16 * LDN, PART = 2 * HALF, BUF = 3 * PART; // 16-byte words: [part][half][cell][image]
	constexpr int XE = 4, ROW = 20;                                                  // results: floats between two images' maps in LDS
	static_assert(kCellSplitRows * kCellSplitImages * ROW <= 2 * BUF * 4, "the results fit the buffers");
	__shared__ u32x4 Bs[2 * BUF];

	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int khalf = lane >> 5, l32 = lane & 31, qa = wave >> 1, qb = wave & 1;
	const int n0 = blockIdx.x * kCellSplitImages, i0 = blockIdx.y * kCellSplitRows, j0 = n0 * 16;
	const int cbHalf = p.cred / kSplitCB, cbTotal = p.src2 ? 2 * cbHalf : cbHalf;
	const int cbBeg = blockIdx.z * p.perSplit, cbEnd = cbBeg + p.perSplit < cbTotal ? cbBeg + p.perSplit : cbTotal;

	// position tid or tid + 256 of the 512, either half of the channels
	uint32_t sOff[XE];
	int sLds[XE];
#pragma unroll
	for (int e = 0; e < XE; e++) {
		const int pos = tid + 256 * (e & 1), half = e >> 1;
		sOff[e] = j0 + pos < p.J ? 4u * ((uint32_t)(half * 8) * (uint32_t)p.J + (uint32_t)(j0 + pos)) : kOutOfRange;
		sLds[e] = half * HALF + (pos & 15) * LDN + (pos >> 4);
	}
	float sreg[XE][8];
	v16f acc[4], low[4];
#pragma unroll
	for (int c = 0; c < 4; c++)
#pragma unroll
		for (int v = 0; v < 16; v++) acc[c][v] = low[c][v] = 0.f;
	const size_t rowWords = (size_t)blockIdx.y * 192, tapWords = (size_t)p.rowGroups * 192;

#define CELL_LOAD(CB)                                                                                                 \
	{                                                                                                                 \
		const bool second_ = (CB) >= cbHalf;                                                                          \
		const size_t shift_ = (size_t)(((CB) - (second_ ? cbHalf : 0)) * kSplitCB) * p.J;                             \
		const __amdgpu_buffer_rsrc_t rs_ = make_rsrc((second_ ? p.src2 : p.src) + shift_, p.srcBytes - (uint32_t)(4 * shift_)); \
		_Pragma("unroll") for (int e = 0; e < XE; e++)                                                                \
			_Pragma("unroll") for (int q = 0; q < 8; q++)                                                             \
				sreg[e][q] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs_, (int)sOff[e], 4 * q * p.J, 0)); \
	}
#define CELL_STORE(BUFFER, E)                                                                                         \
	{                                                                                                                 \
		u32x4 part_[3];                                                                                               \
		split_eight(sreg[E], part_);                                                                                  \
		_Pragma("unroll") for (int s = 0; s < 3; s++) Bs[(BUFFER) * BUF + s * PART + sLds[E]] = part_[s];             \
	}
#define CELL_READ(BUFFER)                                                                                             \
	_Pragma("unroll") for (int r = 0; r < 3; r++)                                                                     \
		_Pragma("unroll") for (int c = 0; c < 3; c++)                                                                 \
			_Pragma("unroll") for (int s = 0; s < 3; s++)                                                             \
				b[r][c][s] = Bs[(BUFFER) * BUF + s * PART + khalf * HALF + ((qa ? 3 - r : r) * 4 + (qb ? 3 - c : c)) * LDN + l32];
#define CELL_READ_WEIGHTS(SET, BLOCK, TAP)                                                                            \
	{                                                                                                                 \
		const int tap_ = (qa ? 2 - (TAP) / 3 : (TAP) / 3) * 3 + (qb ? 2 - (TAP) % 3 : (TAP) % 3);                     \
		_Pragma("unroll") for (int s = 0; s < 3; s++) a[SET][s] = (BLOCK)[(size_t)tap_ * tapWords + s * 64 + lane];   \
	}
#define CELL_PRODUCTS(SUM, PA, PB)                                                                                    \
	_Pragma("unroll") for (int c = 0; c < 4; c++)                                                                     \
		if ((c >> 1) + t / 3 >= 1 && (c & 1) + t % 3 >= 1)                                                            \
			SUM[c] = mfma_bf16(a[t & 1][PA], b[(c >> 1) + t / 3 >= 1 ? (c >> 1) + t / 3 - 1 : 0][(c & 1) + t % 3 >= 1 ? (c & 1) + t % 3 - 1 : 0][PB], SUM[c]);

	u32x4 a[2][3], b[3][3][3];
	const u32x4 *wBlock = (cbBeg >= cbHalf ? p.wp2 + (size_t)(cbBeg - cbHalf) * T * tapWords : p.wp + (size_t)cbBeg * T * tapWords) + rowWords;
	CELL_READ_WEIGHTS(0, wBlock, 0);
	CELL_LOAD(cbBeg);
#pragma unroll
	for (int e = 0; e < XE; e++) CELL_STORE(0, e);
	__syncthreads();
	for (int cb = cbBeg; cb < cbEnd; cb++) {
		const int buffer = (cb - cbBeg) & 1;
		const int nb = cb + 1 < cbEnd ? cb + 1 : cb; // (the last block's is staged once more, and not read)
		const u32x4 *wNext = (nb >= cbHalf ? p.wp2 + (size_t)(nb - cbHalf) * T * tapWords : p.wp + (size_t)nb * T * tapWords) + rowWords;
		CELL_READ(buffer);
#pragma unroll
		for (int t = 0; t < T; t++) {
			if (t + 1 < T) CELL_READ_WEIGHTS((t + 1) & 1, wBlock, t + 1) else CELL_READ_WEIGHTS((t + 1) & 1, wNext, 0);
			if (t == 0) CELL_LOAD(nb);
			__builtin_amdgcn_sched_barrier(0);
			if (t >= T - XE) CELL_STORE(buffer ^ 1, t - (T - XE));
			CELL_PRODUCTS(low, 0, 2);
			CELL_PRODUCTS(acc, 0, 0);
			CELL_PRODUCTS(low, 0, 1);
			CELL_PRODUCTS(low, 1, 1);
			CELL_PRODUCTS(low, 2, 0);
			CELL_PRODUCTS(low, 1, 0);
			if (t >= T - XE) {
#pragma unroll
				for (int i = 0; i < 12; i++) {
					__builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
					__builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
				}
			}
			__builtin_amdgcn_sched_barrier(0);
		}
#pragma unroll
		for (int s = 0; s < 3; s++) a[0][s] = a[1][s]; // nine taps: the next block's first fragments are in the other set
		wBlock = wNext;
		__syncthreads();
	}
#undef CELL_LOAD
#undef CELL_STORE
#undef CELL_READ
#undef CELL_READ_WEIGHTS
#undef CELL_PRODUCTS

	const bool split = out.splitStride != 0;
	float *C = out.C + (size_t)blockIdx.z * out.splitStride;
	bool suspect = false;
#pragma unroll
	for (int c = 0; c < 4; c++)
#pragma unroll
		for (int v = 0; v < 16; v++) {
			acc[c][v] += low[c][v];
			suspect |= split_sum_suspect(acc[c][v]);
		}
	if (__syncthreads_or(suspect)) {
		conv_split_exact_tile<3, kCellSplitRows, kCellSplitImages * 16>(p, out, i0, j0, cbBeg, cbEnd, C);
		return;
	}
	// through LDS, whose maps leave as 16-byte groups along the positions
	float *R = (float *)Bs;
#pragma unroll
	for (int c = 0; c < 4; c++) {
		const int cell = (qa ? 3 - (c >> 1) : (c >> 1)) * 4 + (qb ? 3 - (c & 1) : (c & 1));
#pragma unroll
		for (int v = 0; v < 16; v++) R[((8 * (v / 4) + 4 * khalf + (v % 4)) * kCellSplitImages + l32) * ROW + cell] = acc[c][v] * kSplitSumScale;
	}
	__syncthreads();
	for (int e = tid; e < kCellSplitRows * kCellSplitImages * 4; e += kGemmThreads) {
		const int row = e / (kCellSplitImages * 4), n = e / 4 % kCellSplitImages, quarter = e % 4, i = i0 + row;
		if (i >= p.I || j0 + n * 16 >= p.J) continue;
		float4 val = *(const float4 *)&R[(row * kCellSplitImages + n) * ROW + 4 * quarter];
		if (!split && out.biasI) {
			const float bias = out.biasI[i];
			val.x += bias, val.y += bias, val.z += bias, val.w += bias;
		}
		*(float4 *)&C[(size_t)i * out.ldc + j0 + n * 16 + 4 * quarter] = val;
	}
}

} // namespace fitre
