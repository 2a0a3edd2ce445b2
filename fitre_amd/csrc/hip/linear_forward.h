// The forward pass of a run of small fully connected layers in one launch: z_f = W_f z_{f-1} + b_f, its copy before the
// activation and the activation itself (functions/cnn_forward.cu:250-340 queues a product, a copy and an activation per
// layer), for as many layers as follow each other.
//
// Bound: load latency and the number of dependent launches -- LeNet's 400-120-84-10 at batch 128 is 7.5 million
// multiply-adds, nine launches and 53 us as products on 32 x 32 tiles, each tile walking the whole reduction alone on
// 16 workgroups; VGG's 512-10 at batch 256 was one such launch of 26 us on eight workgroups.  The layers do not couple
// samples, so a workgroup owns four samples and takes them through all layers: their inputs sit in LDS as one 16-byte
// group per input, the reduction of an output is dealt over as many of the 1024 threads as the layer's width leaves, and
// a thread has eight weights of its own on the way at a time (consecutive threads, consecutive outputs: whole rows of W).
// The parts of an output are added in part order, so the order of every sum is fixed by the layer's width.
// Measured, a whole forward and backward pass, before and after: LeNet batch 128 217 -> 184 us, batch 16 209 -> 181,
// the CIFAR AlexNet at batch 100 663 -> 640 (its upper two layers), VGG-11 at batch 256 2277 -> 2265.
#pragma once
#include "common.h"
#include "fitre_nn.h"

namespace fitre {

constexpr int kFwdTailLayers = 4;
constexpr int kFwdTailThreads = 1024;
constexpr int kFwdTailSamples = 4;
constexpr int kFwdTailMaxIn = 2048;   // 32 KB of LDS for a layer's inputs
constexpr int kFwdTailMaxOut = 1024;  // one output per thread at most
// A workgroup reads every weight: with more of them than this the layers are better taken one by one, over the whole chip.
constexpr long kFwdTailMaxWeights = 98304;
// and with more multiply-adds than this the matrix cores are the better unit
constexpr double kFwdTailMaxWork = 1.3e8;

struct FwdTailLayer {
	int in, out, act;
	int logWidth; // threads per part of the reduction = 1 << logWidth >= out
	const float *W, *bias;
	float *pre, *post;
};
struct FwdTailParams {
	int layers, samples;
	const float *x; // in x samples
	FwdTailLayer l[kFwdTailLayers];
};

__global__ void __launch_bounds__(kFwdTailThreads) fc_tail_forward_kernel(const FwdTailParams p)
{
	__shared__ float4 zs[kFwdTailMaxIn];         // the four samples' values of one input
	__shared__ float4 part[kFwdTailThreads];     // [part][output]
	const int tid = threadIdx.x;
	const int n0 = (int)blockIdx.x * kFwdTailSamples;
	const int live = (p.samples - n0 < kFwdTailSamples) ? p.samples - n0 : kFwdTailSamples;
	{
		const int in = p.l[0].in;
		const float *x0 = p.x + (size_t)n0 * in;
		for (int k = tid; k < in; k += kFwdTailThreads) {
			float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
			v.x = x0[k];
			if (live > 1) v.y = x0[(size_t)in + k];
			if (live > 2) v.z = x0[2 * (size_t)in + k];
			if (live > 3) v.w = x0[3 * (size_t)in + k];
			zs[k] = v;
		}
	}
	for (int f = 0; f < p.layers; f++) {
		const FwdTailLayer &l = p.l[f];
		const int in = l.in, out = l.out;
		const int m = tid & ((1 << l.logWidth) - 1), mine = tid >> l.logWidth, parts = kFwdTailThreads >> l.logWidth;
		__syncthreads(); // the inputs are there, and the previous layer's parts have been read
		float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
		if (m < out) {
			const float *w = l.W + m;
			for (int k0 = mine; k0 < in; k0 += 8 * parts) {
				float wv[8];
#pragma unroll
				for (int u = 0; u < 8; u++) {
					const int k = k0 + u * parts;
					wv[u] = k < in ? w[(size_t)k * out] : 0.f;
				}
#pragma unroll
				for (int u = 0; u < 8; u++) {
					const int k = k0 + u * parts;
					if (k < in) {
						const float4 z = zs[k];
						acc.x = fmaf(wv[u], z.x, acc.x);
						acc.y = fmaf(wv[u], z.y, acc.y);
						acc.z = fmaf(wv[u], z.z, acc.z);
						acc.w = fmaf(wv[u], z.w, acc.w);
					}
				}
			}
		}
		part[tid] = acc;
		__syncthreads();
		// one thread per (sample, output); out <= 1024, so at most four rounds
		const float *flat = reinterpret_cast<const float *>(part);
		float *next = reinterpret_cast<float *>(zs);
		for (int i = tid; i < out * kFwdTailSamples; i += kFwdTailThreads) {
			const int s = i / out, o = i - s * out;
			float v = 0.f;
			for (int q = 0; q < parts; q++) v += flat[(size_t)(((q << l.logWidth) + o) * kFwdTailSamples + s)];
			if (l.bias) v += l.bias[o];
			const float y = act_forward_value(l.act, v);
			if (s < live) {
				const size_t at = (size_t)(n0 + s) * out + o;
				l.pre[at] = v;
				l.post[at] = y;
			}
			next[o * kFwdTailSamples + s] = y; // this layer's inputs have been read: the barrier above
		}
	}
}

} // namespace fitre
