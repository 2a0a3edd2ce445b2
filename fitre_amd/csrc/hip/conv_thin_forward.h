// Forward convolution of layers with very few channels (LeNet: 3 -> 6 and 6 -> 16 with 5 x 5 windows), with the
// activation and a 2 x 2 pool of a layer without batch norm in the same launch.
//
// Bound: vector multiply-adds at a large batch, launches and load latency at a small one.  On the tile engine six output
// channels are a tenth of a 64-row tile: 104 us for the first layer at batch 1024, 0.7 GFLOP.  Here the images of a
// workgroup sit in LDS with their zero border, a thread owns a patch of 2 x 4 output cells for COG output channels, and the
// words of a bordered row (two 16-byte reads for a 5-wide window) feed up to 8 * 5 * COG multiply-adds whose other
// operand, the weight, is uniform over the wave and comes through scalar loads.  The patch is also what a 2 x 2 pool needs:
// two pooled cells, so the activation and the pool (and the linear layers' order of the last layer's output) come from
// registers instead of three further launches.  From nine output channels on the plan launches conv_thin_matrix.h.  Rows of LDS are as long as the border needs or a little longer, where that
// spreads sixteen neighbouring lanes' 16-byte reads over the banks.
// Measured, a whole forward and backward pass, before and after: LeNet with batch norm at batch 1024 488 -> 362 us, without at
// batch 128 176 -> 149, with average pools at batch 16 175 -> 145.
#pragma once
#include "conv_thin_matrix.h"

namespace fitre {

struct ThinFwdParams {
	const float *x, *w, *bias;
	float *y;
	int cin, cout, samples, inA, inB, outA, outB, pad;
	int images;             // images of a workgroup
	int rowPairs, groups;   // output patches of an image: pairs of rows x groups of four columns
	int chunks, chunk;      // waves' worth of patches of a workgroup's images, evenly
	int coGroups;           // groups of COG output channels
	int PA, PB;             // bordered image in LDS
	int store;              // 4: rows are whole 16-byte groups, 2: whole 8-byte groups, 1: neither
	FastDiv divImage, divPlane, divPB, divItems, divGroups;
	// the layer's activation and pool (FOLD)
	int act;
	bool average, toFc;
	float *actOut, *poolOut;
};

// Words of a bordered image below which a workgroup's images are staged together.  Of the time one by one, 1 to 1024 images:
// 0.2 at 96 words, 0.35 at 288, 0.7 at 768, 0.83 to 0.87 at 1152; 0.94 to 1.05 at 1296, 1.0 to 1.04 at 1680 and 1.0 to 1.06
// at 3456 (LeNet's two), as every word is divided once more.
constexpr int kThinFwdSmallImage = 1280;

template <int KS, int COG, bool FOLD>
__global__ void __launch_bounds__(256) thin_forward_kernel(const ThinFwdParams p, const float *__restrict__ x, const float *__restrict__ w)
{
	extern __shared__ __align__(16) float thin_lds[];
	constexpr int WORDS = (KS + 3 + 3) & ~3; // words of a bordered row under four neighbouring windows, in whole 16-byte groups
	const int tid = threadIdx.x;
	const int n0 = (int)blockIdx.x * p.images;
	const int images = (p.samples - n0 < p.images) ? p.samples - n0 : p.images;
	const int cells = p.inA * p.inB;
	const size_t iplane = (size_t)p.samples * cells;
	const int plane = p.PA * p.PB, image = p.cin * plane;
	// eight words of a thread on the way at once: of one image after the other, or of all images where one is a fraction of that
	auto stage = [&](auto several, const float *src, float *dst, int words) {
		for (int base = tid; base < words; base += 256 * 8) {
			float v[8];
#pragma unroll
			for (int u = 0; u < 8; u++) {
				const int i = base + 256 * u;
				uint32_t im = 0, at = (uint32_t)(i < words ? i : 0), c, q, r, col;
				if constexpr (decltype(several)::value) p.divImage.divmod(at, im, at);
				p.divPlane.divmod(at, c, q);
				p.divPB.divmod(q, r, col);
				const int a = (int)r - p.pad, b = (int)col - p.pad;
				const bool ok = (i < words) & ((unsigned)a < (unsigned)p.inA) & ((unsigned)b < (unsigned)p.inB);
				v[u] = ok ? src[(size_t)c * iplane + (size_t)im * cells + a * p.inB + b] : 0.f;
			}
#pragma unroll
			for (int u = 0; u < 8; u++)
				if (base + 256 * u < words) dst[base + 256 * u] = v[u];
		}
	};
	const float *src = x + (size_t)n0 * cells;
	if (image < kThinFwdSmallImage) stage(std::true_type{}, src, thin_lds, images * image);
	else
		for (int im = 0; im < images; im++) stage(std::false_type{}, src + (size_t)im * cells, thin_lds + im * image, image);
	__syncthreads();
	const int lane = tid & 63, wave = tid >> 6;
	const int perImage = p.rowPairs * p.groups, items = images * perImage;
	for (int task = wave + 4 * (int)blockIdx.y; task < p.chunks * p.coGroups; task += 4 * (int)gridDim.y) {
		const int cg = __builtin_amdgcn_readfirstlane(task / p.chunks), part = task - cg * p.chunks;
		const int item = part * p.chunk + lane;
		const bool live = lane < p.chunk && item < items;
		uint32_t im, cell, rp, g;
		p.divItems.divmod((uint32_t)(live ? item : 0), im, cell);
		p.divGroups.divmod(cell, rp, g);
		const float *d0 = thin_lds + (int)im * image + (2 * (int)rp) * p.PB + 4 * (int)g;
		float acc[COG][2][4];
		const float *wc[COG];
#pragma unroll
		for (int c = 0; c < COG; c++) {
			const int co = cg * COG + c < p.cout ? cg * COG + c : p.cout - 1; // a channel past the end repeats the last one and is not stored
			wc[c] = w + (size_t)co * p.cin * (KS * KS);
#pragma unroll
			for (int j = 0; j < 4; j++) acc[c][0][j] = acc[c][1][j] = 0.f;
		}
		for (int ci = 0; ci < p.cin; ci++) {
#pragma unroll
			for (int r = 0; r <= KS; r++) { // bordered row r is window row r of the patch's first row, r - 1 of its second
				const float4 *drow = reinterpret_cast<const float4 *>(d0 + ci * plane + r * p.PB);
				float d[WORDS];
#pragma unroll
				for (int q = 0; q < WORDS / 4; q++) {
					const float4 v4 = drow[q];
					d[4 * q] = v4.x, d[4 * q + 1] = v4.y, d[4 * q + 2] = v4.z, d[4 * q + 3] = v4.w;
				}
#pragma unroll
				for (int c = 0; c < COG; c++) {
					const float *wk = wc[c] + ci * (KS * KS);
#pragma unroll
					for (int tb = 0; tb < KS; tb++) {
						if (r < KS) {
							const float w0 = wk[r * KS + tb];
#pragma unroll
							for (int j = 0; j < 4; j++) acc[c][0][j] = fmaf(w0, d[tb + j], acc[c][0][j]);
						}
						if (r > 0) {
							const float w1 = wk[(r - 1) * KS + tb];
#pragma unroll
							for (int j = 0; j < 4; j++) acc[c][1][j] = fmaf(w1, d[tb + j], acc[c][1][j]);
						}
					}
				}
			}
		}
		if (!live) continue;
		const int n = n0 + (int)im, a = 2 * (int)rp, b = 4 * (int)g, left = p.outB - b;
#pragma unroll
		for (int c = 0; c < COG; c++) {
			const int co = cg * COG + c;
			if (co >= p.cout) break;
			const float bias = p.bias ? p.bias[co] : 0.f;
			const size_t at = (((size_t)co * p.samples + n) * p.outA + a) * p.outB + b;
#pragma unroll
			for (int h = 0; h < 2; h++) {
#pragma unroll
				for (int j = 0; j < 4; j++) acc[c][h][j] += bias;
				if (a + h < p.outA) thin_store_row(p.y + at + (size_t)h * p.outB, acc[c][h], p.store, left);
			}
			if constexpr (FOLD) { // outA and outB are even
#pragma unroll
				for (int h = 0; h < 2; h++) {
#pragma unroll
					for (int j = 0; j < 4; j++) acc[c][h][j] = act_forward_value(p.act, acc[c][h][j]);
					thin_store_row(p.actOut + at + (size_t)h * p.outB, acc[c][h], p.store, left);
				}
				const int poolA = p.outA / 2, poolB = p.outB / 2;
#pragma unroll
				for (int q = 0; q < 2; q++) {
					if (2 * q >= left) break;
					const float v = pool2x2(p.average, acc[c][0][2 * q], acc[c][0][2 * q + 1], acc[c][1][2 * q], acc[c][1][2 * q + 1]);
					const int oa = (int)rp, ob = 2 * (int)g + q;
					if (p.toFc) p.poolOut[((size_t)n * p.cout + co) * (poolA * poolB) + (size_t)ob * poolA + oa] = v;
					else p.poolOut[(((size_t)co * p.samples + n) * poolA + oa) * poolB + ob] = v;
				}
			}
		}
	}
}

constexpr int kThinFwdLdsFloats = 15360; // 60 KB of images per workgroup
// Words per bordered row: what the rightmost patch reads, and up to 28 more where sixteen neighbouring patches' reads then
// touch fewer banks twice.
static inline int thin_fwd_row_words(int groups, int words)
{
	const int least = 4 * (groups - 1) + words;
	int best = least, bestClash = 1 << 20;
	for (int row = least; row < least + 32; row += 4) {
		int used[16] = { 0 }, clash = 0; // sixteen-byte bank groups
		for (int i = 0; i < 16; i++) {
			const int bank = (((i / groups) * 2 * row + 4 * (i % groups)) / 4) & 15;
			clash += used[bank]++;
		}
		if (clash < bestClash) bestClash = clash, best = row;
	}
	return best;
}
struct ThinFwdPlan {
	int rowPairs, groups, PA, PB, imageFloats;
	int images, chunks, chunk, cog, coGroups; // as the parameters of the kernel
	int groupsX, groupsY;
};
// false: not for this kernel.  Up to sixteen channels on either side (alexnet's 3 -> 96 and VGG's 3 -> 64 first layers are the
// tile engine's).  Layer on the engine / here, 128 images: 24 -> 24 channels 33 / 35 us, 32 -> 32 36 / 60 (14 x 14 maps), so
// sixteen in is where the engine's rows fill; with three in, 32 x 32 maps, 5 x 5 windows 3 -> 16 22 / 12, 3 -> 32 36 / 22,
// 3 -> 64 41 / 35, so sixteen out is on the safe side.
static inline bool thin_fwd_plan(const fitre_conv_shape *s, ThinFwdPlan &p)
{
	if (s->stride != 1 || (s->ksize != 3 && s->ksize != 5) || s->padding >= s->ksize || s->inChannels > kThinMaxChannels ||
	    s->outChannels > kThinMaxChannels || s->outA < 1 || s->outB < 1)
		return false;
	p.rowPairs = (s->outA + 1) / 2, p.groups = (s->outB + 3) / 4;
	const int words = (s->ksize + 6) & ~3;
	p.PA = 2 * p.rowPairs + s->ksize - 1, p.PB = thin_fwd_row_words(p.groups, words);
	p.imageFloats = s->inChannels * p.PA * p.PB;
	if (p.imageFloats > kThinFwdLdsFloats) return false;
	const int perImage = p.rowPairs * p.groups;
	// small maps: as many images as fill a wave
	p.images = perImage < 64 ? 64 / perImage : 1;
	if (p.images > kThinFwdLdsFloats / p.imageFloats) p.images = kThinFwdLdsFloats / p.imageFloats;
	if (p.images > s->samples) p.images = s->samples;
	p.groupsX = (s->samples + p.images - 1) / p.images;
	const int items = p.images * perImage;
	p.chunks = (items + 63) / 64, p.chunk = (items + p.chunks - 1) / p.chunks;
	// channels of a wave: one until every SIMD has two waves (a wave is a serial chain of cin * k^2 * 8 multiply-adds a
	// channel), then two, and four where they divide the channels and every SIMD has sixteen, for half the LDS reads.  One /
	// two / four, 5 x 5 windows: 8 -> 8 on 14 x 14 maps 15.2 / 18.5 / 25.4 us at 128 images, 30.2 / 26.2 / 37.4 at 2048, 83 / 78 / 98
	// at 8192; on 32 x 32 44.3 / 41.7 / 37.7 at 512, 137 / 129 / 130 at 2048; 3 -> 6 on 32 x 32 9.0 / 9.2 / 12.1 at 128, 26.9 / 26.4 /
	// 28.8 at 1024.  The line of four was drawn at sixteen channels (342 / 324 / 319 at 8192), which the matrix form takes now;
	// at four and eight it is the better one in few places on either side of that line.
	const int cus = device_compute_units();
	const long waves1 = (long)p.groupsX * p.chunks * s->outChannels;
	p.cog = waves1 <= 8L * cus ? 1 : 2;
	if (waves1 >= 64L * cus && s->outChannels % 4 == 0) p.cog = 4;
	p.coGroups = (s->outChannels + p.cog - 1) / p.cog;
	// the tasks of a workgroup's images over further workgroups while the chip has room: each stages the images again
	p.groupsY = (p.chunks * p.coGroups + 3) / 4;
	const int room = (4 * cus + p.groupsX - 1) / p.groupsX;
	if (p.groupsY > room) p.groupsY = room;
	return true;
}
// Microseconds of such a launch while the chip has room: loads of eight words a thread to stage the images, then the taps of
// a wave's channels one after the other.  Fitted to 2365 launches of the vector kernel (windows of 3 and 5, 1 to 16 channels in, 4
// to 16 out, maps of 5 to 28, 1 to 1024 images): 0.5 us off on average, 2.1 at most.  The matrix form, which runs from nine channels out
// on, takes less (16 -> 16 channels on 14 x 14 maps 21.6 / 14.0 us at 32 images, 29.0 / 15.0 at 256).
static inline double thin_fwd_us(const fitre_conv_shape *s, const ThinFwdPlan &p)
{
	const int loads = p.imageFloats < kThinFwdSmallImage ? (p.images * p.imageFloats + 2047) / 2048 : p.images * ((p.imageFloats + 2047) / 2048);
	const int taps = s->inChannels * s->ksize * s->ksize;
	const int tasks = (p.chunks * p.coGroups + 4 * p.groupsY - 1) / (4 * p.groupsY);
	return 2.9 + 1.05 * loads + 0.012 * taps * (1 + tasks * p.cog);
}
// Where the kernel is the shorter way.  Two chains compete at a small batch: its own, and the tile engine's, which a plan that is
// cut over its reduction makes shorter (such an estimate holds within a fifth; an uncut plan takes 1.7 times its estimate).
// 5 x 5 windows on 14 x 14 maps, engine / kernel: 6 -> 8 channels 18.5 / 10.7 us at 32 images, 18.8 / 11.5 at 256; 8 -> 8
// 15.3 / 15.1 at 8, 13.6 / 15.1 at 32; 16 -> 8 13.9 / 21.4 at 32, 37.2 / 21.7 at 256.  Of 400 layers of four to eight channels out, as
// above, the choice is wrong by more than 3 % for ten, by 9 % at most.  Of 400 of nine to sixteen, whose estimate is too long, none
// comes here wrongly, but 65 stay on the engine that are shorter here (8 -> 10 at 8 images 13.8 / 8.6, 16 -> 16 at 32 14.3 / 14.0;
// 2.7 times at most).  sparedUs: launches behind the engine's that the kernel's epilogue makes unnecessary.  A workspace that does not
// hold the engine's ranges leaves it the long chain (16 -> 16 channels, 32 images: 14.3 us cut, 38 uncut, 14.0 here).
constexpr double kThinFwdFoldUs = 3.0;
static inline bool thin_fwd_chosen(const fitre_conv_shape *s, double sparedUs, const void *ws, size_t wsBytes, ThinFwdPlan &plan)
{
	if (!thin_fwd_plan(s, plan)) return false;
	const GemmPlan engine =
	    plan_gemm(s->outChannels, (long)s->samples * s->outA * s->outB, (long)s->inChannels * s->ksize * s->ksize, false, 0, true);
	if (engine.splits > 1 && (!ws || wsBytes < engine.wsBytes)) return true;
	return thin_fwd_us(s, plan) < engine.estimateUs * (engine.splits > 1 ? 1.0 : 1.7) + sparedUs;
}

// fold: the fields act .. poolOut of the parameters, or null
static int launch_thin_forward(const fitre_conv_shape *s, const ThinFwdPlan &plan, const float *x, const float *w, const float *bias, float *y,
                               const ThinFwdParams *fold)
{
	ThinFwdParams p{};
	if (fold) p = *fold;
	p.x = x, p.w = w, p.bias = bias, p.y = y;
	p.cin = s->inChannels, p.cout = s->outChannels, p.samples = s->samples;
	p.inA = s->inA, p.inB = s->inB, p.outA = s->outA, p.outB = s->outB, p.pad = s->padding;
	p.images = plan.images, p.rowPairs = plan.rowPairs, p.groups = plan.groups, p.chunks = plan.chunks, p.chunk = plan.chunk;
	p.coGroups = plan.coGroups, p.PA = plan.PA, p.PB = plan.PB;
	const int imageFloats = plan.imageFloats, perImage = p.rowPairs * p.groups, cog = plan.cog;
	p.divImage = FastDiv((uint32_t)imageFloats);
	p.divPlane = FastDiv((uint32_t)(p.PA * p.PB));
	p.divPB = FastDiv((uint32_t)p.PB);
	p.divItems = FastDiv((uint32_t)perImage);
	p.divGroups = FastDiv((uint32_t)p.groups);
	const uintptr_t at = (uintptr_t)y | (fold ? (uintptr_t)p.actOut : 0);
	p.store = (s->outB % 4 == 0 && (at & 15) == 0) ? 4 : ((s->outB % 2 == 0 && (at & 7) == 0) ? 2 : 1);
	const dim3 grid((unsigned)plan.groupsX, (unsigned)plan.groupsY);
	const size_t lds = sizeof(float) * (size_t)p.images * imageFloats;
	ThinMatPlan m;
	const bool matrix = s->outChannels >= kThinMatLeastRows && thin_mat_plan(s, fold != nullptr, m);
	LaunchScope scope(FITRE_KC_CONV_FWD, conv_flops(s), matrix ? kTileThinMatrix : 0);
	if (matrix) {
		m.p.src = x, m.p.w = w, m.p.bias = bias, m.p.out = y, m.p.store = p.store;
		if (fold) {
			m.p.act = fold->act, m.p.average = fold->average, m.p.toFc = fold->toFc, m.p.actOut = fold->actOut, m.p.poolOut = fold->poolOut;
			launch_thin_matrix<true>(m);
		} else {
			launch_thin_matrix<false>(m);
		}
		return check_launch("thin_matrix_kernel");
	}
	auto launch = [&](auto kernel) { kernel<<<grid, 256, lds, stream()>>>(p, x, w); };
	auto pick = [&](auto ks) {
		constexpr int KS = decltype(ks)::value;
		if (fold) {
			if (cog == 1) launch(thin_forward_kernel<KS, 1, true>);
			else if (cog == 2) launch(thin_forward_kernel<KS, 2, true>);
			else launch(thin_forward_kernel<KS, 4, true>);
		} else {
			if (cog == 1) launch(thin_forward_kernel<KS, 1, false>);
			else if (cog == 2) launch(thin_forward_kernel<KS, 2, false>);
			else launch(thin_forward_kernel<KS, 4, false>);
		}
	};
	if (s->ksize == 5) pick(std::integral_constant<int, 5>{});
	else pick(std::integral_constant<int, 3>{});
	return check_launch("thin_forward_kernel");
}

} // namespace fitre
