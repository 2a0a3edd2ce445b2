/*
 * cnnForward / cnnBackward / computeCNNGradient: the model-level passes of the
 * gradient path, as C host code over the C-ABI device layer.
 *
 * Data flow and z / dx contents follow functions/cnn_forward.cu:49-383,
 * functions/cnn_backward.cu:76-857 and functions/cnn_gradient.cu:13-64 of the
 * reference; what differs is below the layer calls: no patch matrices, no
 * ones-vector products, no staging copies -- the dx slots themselves are the
 * working buffers of the backward pass.
 */
#include <stdio.h>
#include <stdint.h>
#include <stdlib.h>
#include "fitre_cnn.h"
#include "fitre_hip.h"
#include "sweep.h"

#define HIP_CALL(expr)                                                                               \
	do {                                                                                             \
		int rc_ = (expr);                                                                            \
		if (rc_ != FITRE_OK) {                                                                       \
			fprintf(stderr, "%s:%d: %s -> error %d: %s\n", __FILE__, __LINE__, #expr, rc_,           \
			        fitre_hip_last_error());                                                         \
			exit(-1);                                                                                \
		}                                                                                            \
	} while (0)

static int has_bn(const CONV_LAYER *c) { return c->batchNorm != PERFORM_NO_BATCH_NORM; }

static fitre_conv_shape conv_shape(const CONV_LAYER *l, int samples)
{
	fitre_conv_shape s;
	s.samples = samples;
	s.inChannels = l->inChannels;
	s.outChannels = l->outChannels;
	s.inA = l->width; /* A = image column index, B = image row index (fastest) */
	s.inB = l->height;
	s.outA = l->outWidth;
	s.outB = l->outHeight;
	s.ksize = l->kSize;
	s.stride = l->stride;
	s.padding = l->padding;
	return s;
}

static size_t max_sz(size_t a, size_t b) { return a > b ? a : b; }

/* extent of the feature map handed to the first FC layer */
static void feature_extent(const CNN_MODEL *model, int *extA, int *extB)
{
	const CONV_LAYER *c = &model->convLayer[model->cLayers - 1];
	const POOL_LAYER *p = &model->poolLayer[model->cLayers - 1];
	if (p->type != NO_POOL) {
		*extA = p->outWidth;
		*extB = p->outHeight;
	} else {
		*extA = c->outWidth;
		*extB = c->outHeight;
	}
}

/* A sweep writes a batch's hits, a real an image, to the front of this (input_path.c) while the weight copies behind it are kept. */
static size_t forward_ws_bytes(const CNN_MODEL *model, int batch)
{
	size_t need = max_sz(256, sizeof(real) * (size_t)batch);
	for (int i = 0; i < model->cLayers; i++) {
		const CONV_LAYER *c = &model->convLayer[i];
		fitre_conv_shape s = conv_shape(c, batch);
		int extA, extB;
		feature_extent(model, &extA, &extB);
		/* the last layer's output is left in the linear layers' order */
		need = max_sz(need, i == model->cLayers - 1 ? fitre_hip_conv_bn_act_pool_fc_workspace(&s, has_bn(c), extA, extB)
		                                            : fitre_hip_conv_bn_act_pool_workspace(&s, has_bn(c)));
	}
	for (int i = 0; i < model->lLayers; i++)
		need = max_sz(need, fitre_hip_gemm_workspace(model->fcLayer[i].out, batch, model->fcLayer[i].in));
	return need;
}

/* cnnBackward carves two workspaces from devPtr: one for the chain that produces each layer's
 * delta (pool / activation / batch norm / input gradient, lane 0) and one for the weight gradients,
 * which run beside that chain on lane 1. */
/* The chain workspace has two parts that are live at the same time: the input gradient's split partials,
 * which the pool / activation pass of the layer below sums while it reads them, and that pass's
 * batch-norm sums. */
static size_t backward_dx_ws_bytes(const CNN_MODEL *model, int batch)
{
	size_t need = 256;
	for (int i = 1; i < model->cLayers; i++) {
		fitre_conv_shape s = conv_shape(&model->convLayer[i], batch);
		need = max_sz(need, fitre_hip_conv_input_grad_workspace(&s));
	}
	for (int i = 0; i < model->lLayers; i++) {
		const FC_LAYER *f = &model->fcLayer[i];
		need = max_sz(need, fitre_hip_gemm_workspace(f->in, batch, f->out));
	}
	if (model->cLayers > 0) {
		/* the first linear layer's delta in the convolution layout, until the last convolution layer has read it */
		int extA, extB;
		feature_extent(model, &extA, &extB);
		need = max_sz(need, sizeof(real) * (size_t)extA * extB * batch * model->convLayer[model->cLayers - 1].outChannels);
	}
	return (need + 255) & ~(size_t)255;
}

static size_t backward_bn_ws_bytes(const CNN_MODEL *model, int batch)
{
	size_t need = 256;
	for (int i = 0; i < model->cLayers; i++) {
		const CONV_LAYER *c = &model->convLayer[i];
		need = max_sz(need, fitre_hip_batch_norm_workspace(c->outChannels, (long)batch * c->outWidth * c->outHeight));
	}
	return (need + 255) & ~(size_t)255;
}

static size_t backward_chain_ws_bytes(const CNN_MODEL *model, int batch)
{
	return backward_dx_ws_bytes(model, batch) + backward_bn_ws_bytes(model, batch);
}

/* the linear layers as the fused tail sees them (shapes only; tail_layers fills in the pointers); 0 when they do not fit it */
static int tail_shapes(const CNN_MODEL *model, int n, fitre_fc_tail_layer *tail)
{
	if (model->lLayers < 2 || model->lLayers > 4) return 0; /* one layer alone: the two per-layer launches are the shorter way */
	for (int f = 0; f < model->lLayers; f++) {
		fitre_fc_tail_layer t = { model->fcLayer[f].in, model->fcLayer[f].out, model->fcLayer[f].actFun, NULL, NULL, NULL, NULL, NULL, NULL, NULL };
		tail[f] = t;
	}
	return fitre_hip_fc_tail_fits(model->lLayers, tail, n);
}

static size_t backward_side_ws_bytes(const CNN_MODEL *model, int batch)
{
	size_t need = 256;
	fitre_fc_tail_layer tail[4];
	if (tail_shapes(model, batch, tail)) need = max_sz(need, fitre_hip_fc_tail_workspace(model->lLayers, tail, batch));
	size_t held = 0; /* layers whose reduction is held back until the end of the pass keep their blocks: a slice each */
	for (int i = 0; i < model->cLayers; i++) {
		fitre_conv_shape s = conv_shape(&model->convLayer[i], batch);
		need = max_sz(need, fitre_hip_conv_weight_grad_workspace(&s));
		held += fitre_hip_thin_reduce_bytes(&s);
		if (!has_bn(&model->convLayer[i]))
			need = max_sz(need, fitre_hip_channel_sum_workspace(model->convLayer[i].outChannels,
			                                                    (long)batch * model->convLayer[i].outWidth * model->convLayer[i].outHeight));
	}
	for (int i = 0; i < model->lLayers; i++) {
		const FC_LAYER *f = &model->fcLayer[i];
		need = max_sz(need, fitre_hip_linear_weight_grad_workspace(f->in, f->out, batch));
	}
	return ((need + 255) & ~(size_t)255) + held;
}

/* Rearranged weight copies that some input gradients multiply by (fitre_hip_conv_input_grad_prepare): made at the
 * start of the pass on a lane of their own, one buffer per layer that has one. */
static size_t backward_prepared_bytes(const CNN_MODEL *model, int batch)
{
	size_t need = 0;
	for (int i = 1; i < model->cLayers; i++) {
		fitre_conv_shape s = conv_shape(&model->convLayer[i], batch);
		need += (fitre_hip_conv_input_grad_prepared_bytes(&s) + 255) & ~(size_t)255;
	}
	return need;
}

static size_t backward_ws_bytes(const CNN_MODEL *model, int batch)
{
	return backward_chain_ws_bytes(model, batch) + backward_side_ws_bytes(model, batch) + backward_prepared_bytes(model, batch);
}

int fitreBackwardUnsupportedLayer(const CNN_MODEL *model)
{
	for (int c = 1; c < model->cLayers; c++)
		if (model->convLayer[c].stride != 1) return c + 1;
	return 0;
}

/* weight copies of the forward convolutions, one buffer per layer that has one, behind the workspace */
static size_t forward_prepared_bytes(const CNN_MODEL *model, int batch)
{
	size_t need = 0;
	for (int i = 1; i < model->cLayers; i++) {
		fitre_conv_shape s = conv_shape(&model->convLayer[i], batch);
		need += (fitre_hip_conv_forward_prepared_bytes(&s) + 255) & ~(size_t)255;
	}
	return need;
}

long cnnForwardMemRequired(CNN_MODEL *model)
{
	const size_t need = ((forward_ws_bytes(model, model->batchSize) + 255) & ~(size_t)255) + forward_prepared_bytes(model, model->batchSize);
	return (long)((need + sizeof(real) - 1) / sizeof(real));
}

/* Queues the copies of every layer that has one and returns how many there are: a launch for each kind of copy (windows of 3 and of 5,
 * sixteen layers to a launch; the dense form of 2 x 2 maps, eight).  One by one they were 5 to 8 us each, and their launches held up the
 * pass behind them.  Forward pass with its copies together / each in front of its layer, us: VGG-11 593 / 605 at 256 images, 322 /
 * 344 at 77, VGG-16 707 / 741 at 128, AlexNet, which has four, 969 / 974 at 64 and 338 / 346 at 8.  make == 0: they are there, and
 * only found again.  The buffers are laid out for the model's batch size; a layer of a shorter one that finds no room makes its own.
 * lane != 0: on that lane, behind whatever the caller has queued on lane 0 (a weight update, say); nothing is ordered where there is
 * no copy to make.  (The forward pass's on lane 2, beside its first layer, were no shorter, as both are bound by memory there, and
 * AlexNet at 64 images 1 % longer.) */
static int prepare_weights(const CNN_MODEL *model, const real *weights, int n, int inputGrad, char *at, const char *end, const void **prepared, int make,
                           int lane)
{
	fitre_conv_shape shapes[MAX_LAYERS];
	const real *w[MAX_LAYERS];
	void *to[MAX_LAYERS];
	int count = 0;
	at += -(uintptr_t)at & 15;
	if (at > end) at = (char *)end;
	for (int c = 1; c < model->cLayers; c++) {
		fitre_conv_shape shape = conv_shape(&model->convLayer[c], n);
		const size_t bytes = inputGrad ? fitre_hip_conv_input_grad_prepared_bytes(&shape) : fitre_hip_conv_forward_prepared_bytes(&shape);
		prepared[c] = NULL;
		if (bytes == 0 || bytes > (size_t)(end - at) || (inputGrad && !has_bn(&model->convLayer[c - 1]))) continue;
		shapes[count] = shape, w[count] = weights + model->wOffsets[c], to[count] = at;
		prepared[c] = at;
		count++;
		at += (bytes + 255) & ~(size_t)255;
		if (at > end) at = (char *)end;
	}
	if (count && make) {
		if (lane) {
			HIP_CALL(fitre_hip_lane_wait(lane, 0));
			HIP_CALL(fitre_hip_lane_select(lane));
		}
		HIP_CALL(fitre_hip_conv_prepare_weights(count, shapes, w, to, inputGrad));
		if (lane) HIP_CALL(fitre_hip_lane_select(0));
	}
	return count;
}

long cnnBackwardMemRequired(CNN_MODEL *model)
{
	return (long)((backward_ws_bytes(model, model->batchSize) + sizeof(real) - 1) / sizeof(real));
}

/* the linear layers from l up as the fused forward launches see them */
static int forward_rest(const CNN_MODEL *model, const real *weights, real *z, int n, int l, fitre_fc_forward_layer *rest)
{
	const int nc = model->cLayers, left = model->lLayers - l;
	for (int k = 0; k < left && left <= 4; k++) {
		const FC_LAYER *g = &model->fcLayer[l + k];
		real *post = z + model->zOffsets[l + k + 1 + nc];
		fitre_fc_forward_layer t = { g->in, g->out, g->actFun, weights + model->wOffsets[l + k + nc],
			                         (model->bias == 0) ? NULL : weights + model->bOffsets[l + k + nc], post + (long)g->out * n, post };
		rest[k] = t;
	}
	return left;
}

/* a network of few channels without batch norm (LeNet): every layer, softmax and loss in one launch; 0 where it is none */
static int forward_in_one_launch(const CNN_MODEL *model, const DEVICE_DATASET *data, real *z, real *probs, real *errors, int n, real *loss)
{
	fitre_thin_net_layer conv[3];
	fitre_fc_forward_layer rest[4];
	const int nc = model->cLayers;
	if (nc > 3 || model->lLayers > 4) return 0;
	for (int l = 0; l < nc; l++) {
		const CONV_LAYER *cv = &model->convLayer[l];
		const POOL_LAYER *pl = &model->poolLayer[l];
		real *slab = z + model->zOffsets[l + 1];
		if (has_bn(cv) || (pl->type != MAX_POOL && pl->type != AVG_POOL) || pl->pSize != 2 || pl->stride != 2 || pl->padding != 0 ||
		    pl->outWidth * 2 != cv->outWidth || pl->outHeight * 2 != cv->outHeight || cv->outputOffset != cv->poolOffset)
			return 0;
		fitre_thin_net_layer t = { conv_shape(cv, n), model->actFuns[l], pl->type == AVG_POOL, data->weights + model->wOffsets[l],
			                       (model->bias == 0) ? NULL : data->weights + model->bOffsets[l], slab, slab + cv->activationOffset,
			                       slab + cv->poolOffset };
		conv[l] = t;
	}
	forward_rest(model, data->weights, z, n, 0, rest);
	if (!fitre_hip_thin_net_forward_fits(nc, conv, model->lLayers, rest, n, data->numClasses)) return 0;
	HIP_CALL(fitre_hip_thin_net_forward(nc, conv, model->lLayers, rest, n, data->currentBatch, data->sampledTrainY, data->numClasses, probs, errors, loss));
	return 1;
}

/* loss NULL: added to the totals of a sweep, and nothing is waited for */
static void forward_pass(CNN_MODEL *model, DEVICE_DATASET *data, SCRATCH_AREA *scratch, real *z, real *probs, real *errors, int curBatchSize,
                         EVAL_TYPE forTesting, int sameWeights, real *loss)
{
	const int *wOffsets = model->wOffsets, *bOffsets = model->bOffsets, *zOffsets = model->zOffsets;
	const real *weights = data->weights;
	const int nc = model->cLayers, n = curBatchSize;
	void *ws = (void *)scratch->nextDevPtr;
	const size_t wsBytes = (forward_ws_bytes(model, model->batchSize) + 255) & ~(size_t)255;

	if (forTesting != MODEL_TRAIN && forTesting != MODEL_TRAIN_ACCURACY && forTesting != MODEL_TEST_ACCURACY) {
		fprintf(stderr, "Unknown EVAL_TYPE... \n\n");
		exit(-1);
	}
	if (nc < 1 || n < 1 || n > model->batchSize) {
		fprintf(stderr, "cnnForward: needs at least one convolution layer and 1 <= batch (%d) <= model batch (%d)\n", n,
		        model->batchSize);
		exit(-1);
	}

	if (forward_in_one_launch(model, data, z, probs, errors, n, loss)) return;
	const void *prepared[MAX_LAYERS] = { NULL };
	prepare_weights(model, weights, n, 0, (char *)ws + wsBytes, (char *)ws + sizeof(real) * (size_t)cnnForwardMemRequired(model), prepared, !sameWeights, 0);
	for (int l = 0; l < nc; l++) {
		const CONV_LAYER *cv = &model->convLayer[l];
		const POOL_LAYER *pl = &model->poolLayer[l];
		const real *in = (l == 0) ? data->currentBatch : z + zOffsets[l] + model->convLayer[l - 1].outputOffset;
		real *slab = z + zOffsets[l + 1];
		real *actOut = slab + cv->activationOffset;
		fitre_conv_shape shape = conv_shape(cv, n);

		const real *bias = (model->bias == 0) ? NULL : weights + bOffsets[l];
		real *bnOut = has_bn(cv) ? slab + cv->batchNormOffset : NULL;
		/* convolution, batch norm (where the layer has it), activation and pooling in as few passes as the shapes allow; the
		 * last layer's output leaves in the linear layers' order: [C][N][a*B+b] -> [N][C][b*A+a] */
		HIP_CALL(fitre_hip_conv_bn_act_pool_forward_prepared(
		    &shape, in, weights + wOffsets[l], prepared[l], bias, slab, bnOut, bnOut ? bnOut + cv->meansOffset : NULL,
		    bnOut ? bnOut + cv->variancesOffset : NULL, bnOut ? bnOut + cv->runningMeansOffset : NULL,
		    bnOut ? bnOut + cv->runningVariancesOffset : NULL, (real)BATCH_NORM_EPSILON, (real)BATCH_NORM_MOMENTUM,
		    forTesting == MODEL_TRAIN, model->actFuns[l], actOut, pl->type, pl->pSize, pl->stride, pl->padding, pl->outWidth,
		    pl->outHeight, (pl->type != NO_POOL) ? slab + cv->poolOffset : NULL, l == nc - 1, ws, wsBytes));
	}

	const CONV_LAYER *last = &model->convLayer[nc - 1];
	const real *feat = z + zOffsets[nc] + last->outputOffset;

	int outputOffset = last->outputOffset;
	for (int l = 0; l < model->lLayers; l++) {
		if (l != 0) outputOffset = 0;
		const FC_LAYER *f = &model->fcLayer[l];
		/* the layers from here up in one launch, where they are small enough (LeNet's three, VGG's one, the upper two of the
		 * CIFAR AlexNet) */
		fitre_fc_forward_layer rest[4];
		const int left = forward_rest(model, weights, z, n, l, rest);
		if (left <= 4 && fitre_hip_fc_tail_forward_fits(left, rest, n)) {
			HIP_CALL(fitre_hip_fc_tail_forward(left, rest, n, z + zOffsets[l + nc] + outputOffset));
			break;
		}
		real *out = z + zOffsets[l + 1 + nc];
		const long count = (long)f->out * n;
		/* W z + b, then the saved copy behind it, then the activation in place */
		HIP_CALL(fitre_hip_gemm(0, 0, f->out, n, f->in, 1.f, weights + wOffsets[l + nc], f->out,
		                        z + zOffsets[l + nc] + outputOffset, f->in, 0.f, out, f->out,
		                        (model->bias == 0) ? NULL : weights + bOffsets[l + nc], ws, wsBytes));
		HIP_CALL(fitre_hip_copy_d2d(out + count, out, sizeof(real) * (size_t)count));
		HIP_CALL(fitre_hip_activation_forward(f->actFun, out, out, count));
	}

	const real *logits = (model->lLayers == 0) ? feat : z + zOffsets[model->lLayers + nc];
	if (loss) HIP_CALL(fitre_hip_softmax_cross_entropy(logits, data->sampledTrainY, n, data->numClasses, probs, errors, loss));
	else HIP_CALL(fitre_hip_softmax_cross_entropy_add(logits, data->sampledTrainY, n, data->numClasses, probs, errors));
}

real cnnForward(CNN_MODEL *model, DEVICE_DATASET *data, SCRATCH_AREA *scratch, real *z, real *probs, real *errors,
                int s, int curBatchSize, EVAL_TYPE forTesting)
{
	(void)s;
	real loss = 0;
	forward_pass(model, data, scratch, z, probs, errors, curBatchSize, forTesting, 0, &loss);
	HIP_CALL(fitre_hip_sync());
	return loss;
}

void fitre_forward_batch(CNN_MODEL *model, DEVICE_DATASET *data, SCRATCH_AREA *scratch, real *z, real *probs, real *errors, int n, EVAL_TYPE mode,
                         int sameWeights)
{
	forward_pass(model, data, scratch, z, probs, errors, n, mode, sameWeights, NULL);
}

/* Multiply-adds of the convolution layers' two gradient products: what decides whether a pass is long enough for
 * the lanes to pay.  Ordering two lanes costs the host two runtime calls per dependency, a few microseconds each:
 * a pass of LeNet at batch 128 (1.5e8, kernels of 5 to 17 us) takes the same time either way (0.092 ms) and stays on
 * one lane; LeNet with batch norm at batch 1024 (1.2e9) takes 0.217 ms on two lanes against 0.227 on one, AlexNet
 * at batch 64 2.82 against 2.90 ms, VGG-11 with batch norm at batch 256 1.37 against 1.52 ms.  (While the largest
 * weight-gradient kernels filled the register file, two lanes lost on networks with little pooling / batch-norm
 * traffic per multiply-add, such as AlexNet, and a second limit kept those on one lane; the kernels of the delta
 * chain now find room beside every weight gradient and the limit is gone.) */
static double backward_conv_work(const CNN_MODEL *model, int n)
{
	double macs = 0;
	for (int c = 0; c < model->cLayers; c++) {
		const CONV_LAYER *l = &model->convLayer[c];
		macs += 2.0 * n * l->outHeight * l->outWidth * (double)l->outChannels * l->inChannels * l->kSize * l->kSize;
	}
	return macs;
}
#define LANE_WORK_THRESHOLD 1.0e9
/* The chain's bandwidth-bound steps (pooling, activation, batch norm: about 28 bytes per activation with batch norm, 16
 * without) of layer c - 1 run beside the weight gradient of layer c on lane 1, and the next input gradient waits for
 * them.  Where they are many per multiply-add of that weight gradient, it is planned for fewer compute units and the
 * chain has the rest of the chip to itself (fitre_hip_weight_grad_share).  Measured on VGG-11 with batch norm at batch
 * 256, bytes per thousand FLOP / best share: layer 1 49 / six eighths, layer 2 24 and layer 4 12 / seven or six
 * eighths (equal within the noise), layers 3 and 5 6 and 3 / the whole chip; the pass 1.32 against 1.37 ms.  A pass with
 * few such bytes overall (AlexNet at batch 64: about 400 FLOP per byte against 140) keeps the whole chip for every weight
 * gradient: 2.82 against 3.00 ms with the shares.  These were fp32 kernels; with the bf16 ones (conv_split_dw.h) the optimum is
 * flat, forward and backward of VGG-11 at 256 / VGG-16 at 128 images in us, this rule against: the whole chip for all 1823 / 2298,
 * 1845 / 2280; limits of half as much 1826 / 2296, 1825 / 2311; an eighth less for all 1809 / 2260, 1858 / 2321.  The share
 * depends on the network alone, not on whether the lanes are in use, so that one lane and two give the same bits. */
static double elementwise_bytes(const CONV_LAYER *l, int n)
{
	return (double)n * l->outHeight * l->outWidth * l->outChannels * (has_bn(l) ? 28.0 : 16.0);
}
static double backward_flop_per_elementwise_byte(const CNN_MODEL *model, int n)
{
	double bytes = 0;
	for (int c = 0; c < model->cLayers; c++) bytes += elementwise_bytes(&model->convLayer[c], n);
	return bytes > 0 ? 2.0 * backward_conv_work(model, n) / bytes : 0.0;
}
#define SHARE_INTENSITY_LIMIT 250.0
static int backward_shares_chip(const CNN_MODEL *model, int n)
{
	return backward_conv_work(model, n) >= LANE_WORK_THRESHOLD && backward_flop_per_elementwise_byte(model, n) < SHARE_INTENSITY_LIMIT;
}
/* eighths of the compute units the weight gradient of layer c is planned for */
static int weight_grad_eighths(const CNN_MODEL *model, int n, int c)
{
	if (c < 1) return 8;
	const CONV_LAYER *l = &model->convLayer[c];
	const double flops = 2.0 * n * l->outHeight * l->outWidth * (double)l->outChannels * l->inChannels * l->kSize * l->kSize;
	const double perKiloFlop = 1000.0 * elementwise_bytes(&model->convLayer[c - 1], n) / flops;
	return perKiloFlop >= 40.0 ? 6 : (perKiloFlop >= 10.0 ? 7 : 8);
}
/* -1: by the limit above (fitted on LeNet, VGG-11 and AlexNet); 0: one lane; 1: lanes, whatever the network */
static int g_backward_lanes = -1;
void fitreSetBackwardLanes(int mode) { g_backward_lanes = mode < 0 ? -1 : (mode ? 1 : 0); }
int fitreBackwardUsesLanes(CNN_MODEL *model, int batchSize)
{
	if (g_backward_lanes >= 0) return g_backward_lanes;
	return backward_conv_work(model, batchSize) >= LANE_WORK_THRESHOLD;
}
#define LANE_SELECT(lane_) do { if (lanes) HIP_CALL(fitre_hip_lane_select(lane_)); } while (0)
#define LANE_WAIT(waiter_, signaller_) do { if (lanes) HIP_CALL(fitre_hip_lane_wait(waiter_, signaller_)); } while (0)

void cnnBackward(CNN_MODEL *model, DEVICE_DATASET *data, real *devPtr, real *z, real *gradient, real *dx, real *delta,
                 real *delta_new, int offset, int batchSize, real *hostPtr)
{
	(void)offset;
	(void)hostPtr;
	const int *wOffsets = model->wOffsets, *bOffsets = model->bOffsets, *zOffsets = model->zOffsets;
	const real *weights = data->weights;
	const int n = batchSize, nc = model->cLayers;
	const int lanes = fitreBackwardUsesLanes(model, n);
	void *ws = (void *)devPtr; /* input-gradient partials (and the FC products' splits) */
	const size_t wsBytes = backward_dx_ws_bytes(model, model->batchSize);
	void *bnWs = (void *)((char *)devPtr + wsBytes);
	const size_t bnBytes = backward_bn_ws_bytes(model, model->batchSize);
	void *sideWs = (void *)((char *)bnWs + bnBytes);
	const size_t sideBytes = backward_side_ws_bytes(model, model->batchSize);
	char *const preparedWs = (char *)sideWs + sideBytes;
	const char *preparedEnd = preparedWs + backward_prepared_bytes(model, model->batchSize);
	const void *prepared[MAX_LAYERS] = { NULL };
	int preparedPending = 0;

	if (nc < 1 || n < 1 || n > model->batchSize) {
		fprintf(stderr, "cnnBackward: needs at least one convolution layer and 1 <= batch (%d) <= model batch (%d)\n", n,
		        model->batchSize);
		exit(-1);
	}
	if (fitreBackwardUnsupportedLayer(model)) {
		fprintf(stderr, "cnnBackward: convolution layer %d has stride %d; only the first layer may be strided (the input "
		                "gradient is implemented for stride 1)\n",
		        fitreBackwardUnsupportedLayer(model), model->convLayer[fitreBackwardUnsupportedLayer(model) - 1].stride);
		exit(-1);
	}
	const CONV_LAYER *last = &model->convLayer[nc - 1];
	const int sharesChip = backward_shares_chip(model, n);

	/* Weight copies of the layers whose input gradient reads one: they depend on the weights only, so lane 2 makes
	 * them while the chain works through the linear layers. */
	preparedPending = prepare_weights(model, weights, n, 1, preparedWs, preparedEnd, prepared, 1, lanes ? 2 : 0);

	/* Linear layers, top down.  The delta of a layer (after its activation derivative) is written once, into the
	 * layer's dx slot -- the snapshot the Hessian-vector product and the KFAC factors read -- and everything that
	 * follows reads it there: the chain (lane 0) never writes a buffer that lane 1 still reads, so it never waits
	 * for lane 1.  The last product leaves the first convolution-side delta in the chain workspace, already in
	 * the convolution layout [C][N][a*B+b] (the reference permutes it separately, functions/cnn_backward.cu:330-348);
	 * the workspace is free until the last convolution layer's input gradient, which is queued behind the pass
	 * that reads this tensor. */
	real *features = (real *)ws;
	int extA, extB;
	feature_extent(model, &extA, &extB);
	fitre_fc_tail_layer tail[4];
	const int fusedTail = tail_shapes(model, n, tail);
	/* a pass on one lane: the weight gradients of small layers, the linear ones' too, wait for one launch at its end */
	if (!lanes) HIP_CALL(fitre_hip_weight_grads_defer());
	int tailFoldedPool = 0;
	if (fusedTail) {
		/* small layers (LeNet's 400-120-84-10): the whole tail in two launches on the chain's lane -- every delta into its
		 * slot, every weight and bias gradient, and the first convolution-side delta */
		for (int f = 0; f < model->lLayers; f++) {
			const FC_LAYER *l = &model->fcLayer[f];
			real *zl = z + zOffsets[f + nc + 1];
			tail[f].W = weights + wOffsets[f + nc];
			tail[f].zPre = zl + l->offset, tail[f].zPost = zl;
			tail[f].zin = z + zOffsets[f + nc] + ((f == 0) ? last->outputOffset : 0);
			tail[f].slot = dx + zOffsets[f + nc + 1];
			tail[f].dW = gradient + wOffsets[f + nc];
			tail[f].db = (model->bias != 0) ? gradient + bOffsets[f + nc] : NULL;
		}
		const POOL_LAYER *pl = &model->poolLayer[nc - 1];
		if (!has_bn(last) && (pl->type == MAX_POOL || pl->type == AVG_POOL) && pl->pSize == 2 && pl->stride == 2 && pl->padding == 0 && pl->width == 2 * extA &&
		    pl->height == 2 * extB && pl->outWidth == extA && pl->outHeight == extB) {
			/* the top convolution layer's pool and activation steps ride on the launch that produces their delta */
			const real *slabT = z + zOffsets[nc];
			real *dslabT = dx + zOffsets[nc];
			HIP_CALL(fitre_hip_fc_tail_backward_pool_type_act(model->lLayers, tail, n, delta, extA, extB, features, pl->type, model->actFuns[nc - 1],
			                                                  slabT, slabT + last->activationOffset, dslabT, dslabT + last->activationOffset,
			                                                  sideWs, sideBytes));
			tailFoldedPool = 1;
		} else {
			HIP_CALL(fitre_hip_fc_tail_backward(model->lLayers, tail, n, delta, extA, extB, features, sideWs, sideBytes));
		}
	}
	for (int f = fusedTail ? -1 : model->lLayers - 1; f >= 0; f--) {
		const FC_LAYER *l = &model->fcLayer[f];
		real *zl = z + zOffsets[f + nc + 1];
		real *slot = dx + zOffsets[f + nc + 1];
		const real *zin = z + zOffsets[f + nc] + ((f == 0) ? last->outputOffset : 0);

		/* delta .* f'(.) of the output layer; the layers below get theirs from the epilogue of the product above them.
		 * Without an activation it is the caller's delta as it stands: the product reads it there and leaves the copy in
		 * the slot on its way. */
		const real *cur_delta = slot;
		real *snapshot = NULL;
		if (f == model->lLayers - 1) {
			if (l->actFun == CNN_ACT_NONE || l->actFun == ACT_LINEAR) {
				cur_delta = delta;
				snapshot = slot;
			} else {
				HIP_CALL(fitre_hip_activation_backward(l->actFun, delta, zl + l->offset, zl, slot, (long)l->out * n));
			}
		}
		if (!snapshot) LANE_WAIT(1, 0);
		/* the chain goes straight on: delta of the layer below = f'(.) .* (W' * delta) */
		if (f > 0) {
			const FC_LAYER *below = &model->fcLayer[f - 1];
			real *zb = z + zOffsets[f + nc];
			HIP_CALL(fitre_hip_linear_input_grad(l->in, l->out, n, weights + wOffsets[f + nc], cur_delta, below->actFun,
			                                     zb + below->offset, zb, 0, 0, dx + zOffsets[f + nc], NULL, ws, wsBytes, snapshot));
		} else {
			HIP_CALL(fitre_hip_linear_input_grad(l->in, l->out, n, weights + wOffsets[f + nc], cur_delta, -1, NULL, NULL, extA, extB,
			                                     features, delta_new, ws, wsBytes, snapshot));
		}
		if (snapshot) LANE_WAIT(1, 0); /* lane 1 reads the slot the product has just filled */
		/* beside it, on lane 1, what nothing later in this pass reads: dW = delta * z', db = delta * 1 */
		LANE_SELECT(1);
		HIP_CALL(fitre_hip_linear_weight_grad(l->in, l->out, n, slot, zin, gradient + wOffsets[f + nc],
		                                      (model->bias != 0) ? gradient + bOffsets[f + nc] : NULL, sideWs, sideBytes));
		LANE_SELECT(0);
	}
	if (model->lLayers == 0) HIP_CALL(fitre_hip_fc_to_conv(delta, last->outChannels, n, extA, extB, features));

	/* delta as the layer above left it: a plain tensor, or the unsummed split partials of its input
	 * gradient (summed by the pool / activation pass below while it reads them) */
	fitre_split_view dview = { features, 1, 0 };
	/* The weight gradients of layers with very few channels end in a short reduction launch each: they are held back and
	 * made as one launch at the end of the pass.  Until then such a layer's blocks stay in a slice of lane 1's workspace of
	 * their own, and the layers after it work in what follows the slices. */
	size_t sideHeld = 0;
	HIP_CALL(fitre_hip_thin_reduce_defer(1));
	int poolFolded = tailFoldedPool;
	for (int c = nc - 1; c >= 0; c--) {
		const CONV_LAYER *l = &model->convLayer[c];
		const POOL_LAYER *p = &model->poolLayer[c];
		const real *slab = z + zOffsets[c + 1];
		real *dslab = dx + zOffsets[c + 1];
		const long perChannel = (long)n * l->outWidth * l->outHeight;
		const int act = model->actFuns[c];

		if (p->type != MAX_POOL && p->type != AVG_POOL && p->type != NO_POOL) {
			fprintf(stderr, "Unknown Pool Function... \n");
			exit(-1);
		}
		const real *actIn = has_bn(l) ? slab + l->batchNormOffset : slab;
		const real *actOut = slab + l->activationOffset;
		/* With batch norm and ReLU the fused pass derives the activation output from its input. */
		const int fusedRelu = has_bn(l) && act == CNN_ACT_RELU;
		if (c == nc - 1 && p->type == NO_POOL) {
			/* The forward pass rewrote this layer's activation output into the FC layout in place;
			 * rebuild it from the activation input (the reference reads the permuted buffer,
			 * functions/cnn_backward.cu:574-580). */
			if (!fusedRelu) HIP_CALL(fitre_hip_activation_forward(act, actIn, delta_new, perChannel * l->outChannels));
			actOut = delta_new;
		}
		const real *cur;
		if (poolFolded) {
			/* the layer above's input gradient went on through this layer's pool and activation in its own launch */
			poolFolded = 0;
			cur = dslab + l->activationOffset;
		} else if (has_bn(l)) {
			/* pool backward -> dx slab + 0; times f'(.) -> dx slab + activationOffset; batch-norm backward ->
			 * dx slab + batchNormOffset, its column sums being the bias gradient */
			HIP_CALL(fitre_hip_pool_act_bn_backward(p->type, act, dview.base, dview.splits, dview.stride, actIn,
			                                        fusedRelu ? NULL : actOut,
			                                        slab + l->batchNormOffset + l->variancesOffset, l->outChannels, n, p->width,
			                                        p->height, p->pSize, p->stride, p->padding, p->outWidth, p->outHeight,
			                                        (real)BATCH_NORM_EPSILON, dslab, dslab + l->activationOffset,
			                                        dslab + l->batchNormOffset,
			                                        (model->bias != 0) ? gradient + bOffsets[c] : NULL, bnWs, bnBytes));
			cur = dslab + l->batchNormOffset;
		} else {
			/* pool backward -> dx slab + 0; times f'(.) -> dx slab + activationOffset */
			HIP_CALL(fitre_hip_pool_act_backward(p->type, act, dview.base, actIn, actOut, l->outChannels, n, p->width, p->height,
			                                     p->pSize, p->stride, p->padding, p->outWidth, p->outHeight, dslab,
			                                     dslab + l->activationOffset));
			cur = dslab + l->activationOffset; /* its channel sums (the bias gradient) are taken on lane 1, below */
		}

		const real *input = (c == 0) ? data->currentBatch : z + zOffsets[c] + model->convLayer[c - 1].outputOffset;
		fitre_conv_shape shape = conv_shape(l, n);
		/* The weight gradient, whose result nothing later reads, goes to lane 1 as soon as this layer's delta is
		 * complete: it shares the matrix pipes with the input gradient below, and its kernels leave registers
		 * free on every SIMD, on which the bandwidth-bound kernels of the layer below (split reduction, pooling,
		 * batch norm) run while it keeps the pipes busy.  Queued only behind the input gradient it started 10 us
		 * after that had ended, with no matrix kernel running in between (measured: the pass 0.8 % longer). */
		const int beside = fitre_hip_conv_weight_grad_runs_beside(&shape);
		if (beside) LANE_WAIT(1, 0);
		if (c != 0) {
			if (has_bn(&model->convLayer[c - 1])) {
				if (prepared[c] && preparedPending) { /* the chain's first use of a copy lane 2 made */
					LANE_WAIT(0, 2);
					preparedPending = 0;
				}
				HIP_CALL(fitre_hip_conv_input_grad_split_prepared(&shape, cur, weights + wOffsets[c], prepared[c], delta, ws, wsBytes,
				                                                  &dview));
			} else {
				const CONV_LAYER *lb = &model->convLayer[c - 1];
				const POOL_LAYER *pb = &model->poolLayer[c - 1];
				if ((pb->type == MAX_POOL || pb->type == AVG_POOL) && pb->pSize == 2 && pb->stride == 2 && pb->padding == 0 && pb->width == 2 * shape.inA &&
				    pb->height == 2 * shape.inB && pb->outWidth == shape.inA && pb->outHeight == shape.inB &&
				    fitre_hip_conv_input_grad_folds_pool(&shape)) {
					const real *slabB = z + zOffsets[c];
					real *dslabB = dx + zOffsets[c];
					HIP_CALL(fitre_hip_conv_input_grad_pool_type_act(&shape, cur, weights + wOffsets[c], delta, pb->type, model->actFuns[c - 1],
					                                                 slabB, slabB + lb->activationOffset, dslabB,
					                                                 dslabB + lb->activationOffset, ws, wsBytes));
					poolFolded = 1;
				} else {
					HIP_CALL(fitre_hip_conv_input_grad(&shape, cur, weights + wOffsets[c], delta, ws, wsBytes));
				}
				dview.base = delta, dview.splits = 1, dview.stride = 0;
			}
		}
		/* A weight gradient the device layer does not want beside other matrix kernels (none by now) stays in line; its
		 * workspace is lane 1's, so the lanes are ordered around it. */
		if (!beside) LANE_WAIT(1, 0);
		if (beside) {
			LANE_SELECT(1);
		} else {
			LANE_WAIT(0, 1);
		}
		/* without batch norm the bias gradient is taken here as well (with batch norm it is a by-product of its
		 * backward pass above); nothing in the chain reads either */
		HIP_CALL(fitre_hip_weight_grad_share(sharesChip ? weight_grad_eighths(model, n, c) : 8));
		HIP_CALL(fitre_hip_conv_weight_bias_grad(&shape, input, cur, gradient + wOffsets[c],
		                                         (!has_bn(l) && model->bias != 0) ? gradient + bOffsets[c] : NULL,
		                                         (char *)sideWs + sideHeld, sideBytes - sideHeld));
		sideHeld += fitre_hip_thin_reduce_bytes(&shape);
		if (c == 0) HIP_CALL(fitre_hip_thin_reduce_defer(0)); /* every held reduction, on the lane their blocks were made on */
		if (beside) LANE_SELECT(0);
	}
	HIP_CALL(fitre_hip_weight_grad_share(8));
	HIP_CALL(fitre_hip_sync());
}

real evaluateCNNModel(CNN_MODEL *model, DEVICE_DATASET *data, SCRATCH_AREA *scratch, real *z, real *probs,
                      real *lossFuncErrors, int offset, int curBatchSize)
{
	return cnnForward(model, data, scratch, z, probs, lossFuncErrors, offset, curBatchSize, MODEL_TRAIN);
}

real computeCNNGradient(CNN_MODEL *model, DEVICE_DATASET *data, SCRATCH_AREA *scratch, real *z, real *dx, real *probs,
                        real *lossFuncErrors, real *gradient, int offset, int curBatchSize, real weightDecay)
{
	real *oldDevPtr = scratch->nextDevPtr;
	real *oldHostPtr = scratch->nextHostPtr;
	real *oldPagePtr = scratch->nextPageLckPtr;

	real *errors = scratch->nextDevPtr;
	real *errors_1 = errors + model->maxDeltaSize;
	real *nextDevPtr = errors_1 + model->maxDeltaSize;
	scratch->nextDevPtr = nextDevPtr;

	real lossVal = evaluateCNNModel(model, data, scratch, z, probs, lossFuncErrors, offset, curBatchSize);

	HIP_CALL(fitre_hip_copy_d2d(errors, lossFuncErrors, sizeof(real) * (size_t)data->numClasses * curBatchSize));
	cnnBackward(model, data, nextDevPtr, z, gradient, dx, errors, errors_1, offset, curBatchSize, scratch->nextHostPtr);

	if (weightDecay != 0) HIP_CALL(fitre_hip_axpy(model->pSize, weightDecay, data->weights, gradient));
	HIP_CALL(fitre_hip_sync());

	scratch->nextDevPtr = oldDevPtr;
	scratch->nextHostPtr = oldHostPtr;
	scratch->nextPageLckPtr = oldPagePtr;
	return lossVal;
}

real computeAccuracy(real *probs, real *target, int rows, int numClasses, real *devPtr, real *pageLckPtr)
{
	HIP_CALL(fitre_hip_accuracy_hits(probs, target, rows, numClasses, devPtr));
	HIP_CALL(fitre_hip_dot(rows, devPtr, devPtr, pageLckPtr)); /* complete on return */
	return (real)((*pageLckPtr * 100.) / (real)rows);
}

void computeCrossEntropyError(real *probs, int rows, int num_classes, real *target, real *errors)
{
	HIP_CALL(fitre_hip_cross_entropy_error(probs, target, rows, num_classes, errors));
	HIP_CALL(fitre_hip_sync());
}

void getMultinomialDistSample(real *probs, int samples, int numClasses, real *distClasses, real *devPtr)
{
	HIP_CALL(fitre_hip_random_uniform(devPtr, samples));
	HIP_CALL(fitre_hip_multinomial_classes(probs, devPtr, samples, numClasses, distClasses));
	HIP_CALL(fitre_hip_sync());
}

void computeDistributionErrors(real *probs, real *distTarget, real *distError, int rows, int num_classes, real *devPtr,
                               real *hostPtr)
{
	(void)hostPtr;
	getMultinomialDistSample(probs, rows, num_classes, distTarget, devPtr);
	computeCrossEntropyError(probs, rows, num_classes, distTarget, distError);
}
