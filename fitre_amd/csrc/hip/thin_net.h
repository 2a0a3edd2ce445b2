// The forward pass of a whole small network in one launch: convolutions of few channels with their activation and 2 x 2 pool, a run of
// linear layers, softmax and the loss terms (LeNet; functions/cnn_forward.cu:49-383 queues every one of these steps).
//
// Bound: launches and load latency.  An image of LeNet is 0.65 million multiply-adds, 4 us of one compute unit's vector
// instructions, and takes five launches of 4 to 16 us one after the other.  A workgroup of sixteen waves takes one image through all of it: layers in
// LDS, convolutions on the fp32 matrix pipes in the form of conv_thin_matrix.h, the reduction of a linear output dealt over the
// threads its layer's width leaves.  Everything that is waited for from memory -- the image and the convolutions' weights -- is
// asked for at once; the code is kept short, as every line of it is fetched once per launch.  Forward pass of LeNet with the wait for
// its loss, launches / this, us: 49 / 45 at 1 image, 56 / 45 at 8, 59 / 46 at 128, 64 / 49 at 256, 77 / 64 at 512, 89 / 87 at 700, 94 /
// 104 at 1024: two images on a compute unit at once, and from there on a third waits (net_fits).
#pragma once
#include "conv_thin_matrix.h"
#include "linear_forward.h"

namespace fitre {

constexpr int kNetConvs = 3, kNetLinears = 4, kNetThreads = 1024, kNetWaves = kNetThreads / 64;
constexpr int kNetBlocks = 2;      // blocks of sixteen positions a wave has at once
constexpr int kNetMaxClasses = 64; // one lane each

// All LDS traffic of the workgroup before it: what is on its way to memory is not waited for.
__device__ __forceinline__ void net_barrier()
{
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
	__builtin_amdgcn_s_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

struct NetConv {
	int cin, cout, outA, outB, pad, K, groups16;
	int PA, PB, rowsAtOnce;         // its bordered input
	int weights, source;            // words of LDS: tables, bordered input
	int posWords, act;
	bool average;
	const float *w, *bias;
	float *y, *actOut, *poolOut;
	FastDiv divK, divKK, divKs, divOutB, divPositions, divPooled, divPoolB;
};
struct NetLinear {
	int in, out, act, logWidth;
	const float *W, *bias;
	float *pre, *post;
};
struct NetParams {
	int convs, linears, samples, inA, inB, classes;
	int results;                    // words of LDS: a convolution's output, then the linear layers' inputs and parts
	const float *x, *target;
	float *probs, *errors, *nll;
	FastDiv divRows, divPA, divPB;  // staging of the image
	NetConv c[kNetConvs];
	NetLinear l[kNetLinears];
};

// one convolution layer: products to Y, then the tensors of the layer and the next one's bordered input (last: the linear layers' order)
__device__ __forceinline__ void net_conv(const NetConv &p, const NetConv &next, bool last, int n, int samples, float *lds, float *Y, float *features)
{
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, lk = lane >> 4;
	const float *W = lds + p.weights, *S = lds + p.source;
	const int *further = (const int *)(W + 16 * p.groups16 * kThinMatPitch);
	const int positions = p.outA * p.outB, tiles = (positions + 15) / 16;
#pragma unroll 1
	for (int task = wave; task * kNetBlocks < tiles; task += kNetWaves) {
		int at[kNetBlocks];
		v4f acc[kNetBlocks];
#pragma unroll
		for (int u = 0; u < kNetBlocks; u++) {
			const int pos = (task * kNetBlocks + u) * 16 + l16;
			uint32_t r, b;
			p.divOutB.divmod((uint32_t)(pos < positions ? pos : positions - 1), r, b);
			at[u] = (int)r * p.PB + (int)b;
		}
		thin_mat_multiply<kNetBlocks>(W, further, S, at, p.K, p.groups16, acc);
#pragma unroll
		for (int u = 0; u < kNetBlocks; u++) {
			const int pos = (task * kNetBlocks + u) * 16 + l16;
#pragma unroll
			for (int v = 0; v < 4; v++)
				if (4 * lk + v < p.cout && pos < positions) Y[(4 * lk + v) * p.posWords + pos] = acc[u][v];
		}
	}
	net_barrier();
	const size_t image = (size_t)n * positions, plane = (size_t)samples * positions;
#pragma unroll 1
	for (int e = tid; e < p.cout * positions; e += kNetThreads) {
		uint32_t i, pos;
		p.divPositions.divmod((uint32_t)e, i, pos);
		float v = Y[(int)i * p.posWords + (int)pos];
		if (p.bias) v += p.bias[i];
		p.y[i * plane + image + pos] = v;
		v = act_forward_value(p.act, v);
		p.actOut[i * plane + image + pos] = v;
		Y[(int)i * p.posWords + (int)pos] = v;
	}
	net_barrier();
	const int poolA = p.outA / 2, poolB = p.outB / 2, pooled = poolA * poolB;
	float *N = lds + next.source;
#pragma unroll 1
	for (int e = tid; e < p.cout * pooled; e += kNetThreads) {
		uint32_t i, cell, oa, ob;
		p.divPooled.divmod((uint32_t)e, i, cell);
		p.divPoolB.divmod(cell, oa, ob);
		const float *y = Y + (int)i * p.posWords + 2 * (int)oa * p.outB + 2 * (int)ob;
		const float top = pool2x2(p.average, y[0], y[1], y[p.outB], y[p.outB + 1]);
		if (last) {
			const int f = (int)i * pooled + (int)ob * poolA + (int)oa;
			p.poolOut[(size_t)n * p.cout * pooled + f] = top;
			features[f] = top;
		} else {
			p.poolOut[((size_t)i * samples + n) * pooled + cell] = top;
			N[((int)i * next.PA + (int)oa + next.pad) * next.PB + (int)ob + next.pad] = top;
		}
	}
	net_barrier();
}

__global__ void __launch_bounds__(kNetThreads, 8) thin_net_forward_kernel(const NetParams p)
{
	extern __shared__ __align__(16) float thin_lds[];
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n = (int)blockIdx.x;
	const size_t cells = (size_t)p.inA * p.inB;
	const NetConv &c0 = p.c[0];
	thin_stage_rows<kNetWaves>(p.x + n * cells, (size_t)p.samples * cells, 0, c0.cin * c0.PA, p.inA, p.inB, -c0.pad, c0.pad, c0.PB, c0.rowsAtOnce, p.divRows,
	                           p.divPA, p.divPB, wave, lane, thin_lds + c0.source);
#pragma unroll 1
	for (int l = 0; l < p.convs; l++) {
		const NetConv &c = p.c[l];
		float *W = thin_lds + c.weights;
		thin_mat_tables<kNetThreads>(c.w, c.cout, c.K, 16 * c.groups16, c.PA * c.PB, c.PB, c.divK, c.divKK, c.divKs, W, (int *)(W + 16 * c.groups16 * kThinMatPitch));
		if (l > 0) // the borders
			for (int e = tid; e < c.cin * c.PA * c.PB; e += kNetThreads) thin_lds[c.source + e] = 0.f;
	}
	float *Y = thin_lds + p.results;
	net_barrier();
	const NetConv &top = p.c[p.convs - 1];
	float *in = Y + top.cout * top.posWords; // the linear layers' inputs, behind the last convolution's results
#pragma unroll 1
	for (int l = 0; l < p.convs; l++) net_conv(p.c[l], p.c[l + 1 < p.convs ? l + 1 : l], l + 1 == p.convs, n, p.samples, thin_lds, Y, in);
	float *out = thin_lds, *part = thin_lds + kFwdTailMaxOut; // (the tables and images have been read)
#pragma unroll 1
	for (int f = 0; f < p.linears; f++) {
		const NetLinear &l = p.l[f];
		const int m = tid & ((1 << l.logWidth) - 1), mine = tid >> l.logWidth, parts = kNetThreads >> l.logWidth;
		float acc = 0.f;
		if (m < l.out) {
			const float *w = l.W + m;
#pragma unroll 1
			for (int k0 = mine; k0 < l.in; k0 += 16 * parts) {
				float wv[16];
#pragma unroll
				for (int u = 0; u < 16; u++) {
					const int k = k0 + u * parts;
					wv[u] = k < l.in ? w[(size_t)k * l.out] : 0.f;
				}
#pragma unroll
				for (int u = 0; u < 16; u++) {
					const int k = k0 + u * parts;
					if (k < l.in) acc = fmaf(wv[u], in[k], acc);
				}
			}
		}
		part[tid] = acc;
		net_barrier();
		if (tid < l.out) {
			float v = 0.f;
#pragma unroll 4
			for (int q = 0; q < parts; q++) v += part[(q << l.logWidth) + tid];
			if (l.bias) v += l.bias[tid];
			const float y = act_forward_value(l.act, v);
			l.pre[(size_t)n * l.out + tid] = v;
			l.post[(size_t)n * l.out + tid] = y;
			out[tid] = y;
		}
		net_barrier();
		in = out;
		out = out == thin_lds ? part + kNetThreads : thin_lds;
	}
	if (wave == 0) { // as softmax_ce_kernel
		const bool mine = lane < p.classes;
		const float v = mine ? in[lane] : -FLT_MAX, mx = wave_max(v);
		const float s = wave_sum(mine ? expf(v - mx) : 0.f), inv = 1.f / s;
		const int label = (int)p.target[n]; // 1-based
		if (mine) {
			const float q = expf(v - mx) * inv + 1e-10f;
			p.probs[(size_t)n * p.classes + lane] = q;
			if (p.errors) p.errors[(size_t)n * p.classes + lane] = (lane + 1 == label ? q - 1.f : q) * (1.f / (float)p.samples);
			if (lane + 1 == label) p.nll[n] = -logf(q);
		}
		if (lane == 0 && (label < 1 || label > p.classes)) p.nll[n] = 0.f;
	}
}

// ---- host side ------------------------------------------------------------------------------------------------------
constexpr int kNetLdsFloats = 16384; // 64 KB
// shapes and LDS of the parameters (the pointers are the caller's to fill in); words: of LDS
static inline bool net_plan(int convs, const fitre_thin_net_layer *c, int linears, const fitre_fc_forward_layer *l, int n, int classes, NetParams &p, int &words)
{
	if (convs < 1 || convs > kNetConvs || linears < 0 || linears > kNetLinears || n < 1 || classes < 1 || classes > kNetMaxClasses) return false;
	p.convs = convs, p.linears = linears, p.samples = n, p.classes = classes, p.inA = c[0].shape.inA, p.inB = c[0].shape.inB;
	int at = 0, results = 0;
	for (int i = 0; i < convs; i++) {
		const fitre_conv_shape &s = c[i].shape;
		if (s.samples != n || s.stride != 1 || (s.ksize != 3 && s.ksize != 5) || s.padding < 0 || s.padding >= s.ksize || s.inChannels < 1 || s.outChannels < 1 ||
		    s.inChannels > kThinMatRows || s.outChannels > kThinMatRows || s.outA < 2 || s.outB < 2 || s.outA % 2 || s.outB % 2 || s.outA > 64 || s.outB > 64 ||
		    s.outA != s.inA + 2 * s.padding - s.ksize + 1 || s.outB != s.inB + 2 * s.padding - s.ksize + 1)
			return false;
		if (i > 0 && (s.inChannels != c[i - 1].shape.outChannels || s.inA != c[i - 1].shape.outA / 2 || s.inB != c[i - 1].shape.outB / 2)) return false;
		NetConv &q = p.c[i];
		q.cin = s.inChannels, q.cout = s.outChannels, q.outA = s.outA, q.outB = s.outB, q.pad = s.padding;
		q.K = s.inChannels * s.ksize * s.ksize, q.groups16 = (q.K + 15) / 16;
		q.PA = s.inA + 2 * s.padding, q.PB = s.inB + 2 * s.padding, q.rowsAtOnce = q.PB <= 64 ? 64 / q.PB : 1;
		q.weights = at, at += 16 * q.groups16 * (kThinMatPitch + 1);
		q.source = at, at += q.cin * q.PA * q.PB;
		q.posWords = ((s.outA * s.outB + 63) & ~63) + 4;
		q.divK = FastDiv((uint32_t)q.K), q.divKK = FastDiv((uint32_t)(s.ksize * s.ksize)), q.divKs = FastDiv((uint32_t)s.ksize);
		q.divOutB = FastDiv((uint32_t)s.outB), q.divPositions = FastDiv((uint32_t)(s.outA * s.outB));
		q.divPooled = FastDiv((uint32_t)(s.outA / 2 * (s.outB / 2))), q.divPoolB = FastDiv((uint32_t)(s.outB / 2));
		const int need = q.cout * q.posWords + (i + 1 == convs ? q.cout * (s.outA / 2) * (s.outB / 2) : 0);
		if (need > results) results = need;
	}
	const int least = kFwdTailMaxOut + kNetThreads + kFwdTailMaxOut; // a linear layer's outputs, its parts, and the next one's outputs
	p.results = at < least ? least : at;
	words = p.results + results;
	const NetConv &f = p.c[0], &top = p.c[convs - 1];
	p.divRows = FastDiv((uint32_t)(f.cin * f.PA)), p.divPA = FastDiv((uint32_t)f.PA), p.divPB = FastDiv((uint32_t)f.PB);
	const int features = top.cout * (top.outA / 2) * (top.outB / 2);
	if (linears > 0 && (l[0].in != features || !fitre_hip_fc_tail_forward_fits(linears, l, n))) return false;
	if ((linears > 0 ? l[linears - 1].out : features) != classes) return false;
	return words <= kNetLdsFloats;
}
// two workgroups fit a compute unit; see above for more images than that
static inline bool net_fits(int n) { return n <= 2 * device_compute_units(); }

} // namespace fitre
