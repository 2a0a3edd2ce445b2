"""The passes of this framework that a trainer's time goes into, as cases to be measured.

A case names a pass, a network of the model builders and its sizes; the passes are called as a C program calls them,
through the boundary of include/fitre_*.h, on device memory that torch holds:

  gradient   computeCNNGradient: forward pass, loss and flat gradient of one mini-batch
  step       its two halves, cnnForward and cnnBackward, as the trust-region loop calls them, for networks with kinks
  evaluate   computeTestGeneralizationErrors: loss and accuracy over a test set in batches, a short one at the end
  hessian    cnnHv: one Hessian-vector product at the point of the last gradient
  curvature  computeOmegaZAndLambdaDelta + computeNaturalGradient: factors, damped inverses, natural gradient
  dense      computeGradient + gaussNewtonHessianVec of the fully connected family

exact() says what they should return, from plain torch arithmetic in 64 bits on the inputs that prepare() made.  It covers
losses, probabilities, gradients, Hessian-vector products and, where no running statistics are in it, the activation store.

A ReLU at zero and two equal cells under a max pool send whole gradient entries elsewhere when a forward pass differs in
its last bit, which says nothing about the pass.  So in "step", "hessian" and "curvature" what the backward side reads
as z is a float64 forward pass made by torch and rounded, the same for every implementation, and the forward pass of a
step writes a z of its own beside it.

Networks: "lenet" (5x5 convolutions, max pools), "lenet_avg" (the same with average pools and swish), "alexnet_cifar"
(two 5x5 layers of 64 channels, 3/2 pools), "vgg11" / "vgg13" / "vgg16" (3x3 layers, 32x32 images), "alexnet" (224x224
images, three large linear layers), "autoencoder" (linear layers only).
"""
import ctypes as C

import torch
import torch.nn.functional as F

from fitre_amd import lib as L
from fitre_amd import structs as S
from fitre_amd.harness import build_alexnet, build_lenet, build_vgg11, input_dims, num_classes

ACTS = {"none": S.CNN_ACT_NONE, "softplus": S.CNN_ACT_SOFTPLUS, "elu": S.CNN_ACT_ELU, "relu": S.CNN_ACT_RELU, "swish": S.CNN_ACT_SWISH}
AUTOENCODER = (784, 512, 256, 64, 256, 512, 784)  # 28x28 images squeezed to 64 numbers and back
DAMPING = 1e-3
CIFAR10_STATISTICS = ((0.4914, 0.4822, 0.4465), (0.2470, 0.2435, 0.2616))  # means and deviations of the input pipeline
DEVICE = "cuda:0"


# ---------------------------------------------------------------- cases
def step(net, batch, filled=None, act="relu", bn=True, bias=True, name=None, do="step"):
    case = dict(do=do, net=net, batch=batch, filled=filled or batch, act=act, bn=bn, bias=bias)
    return dict(case, name=name) if name else case


def listed():
    return [
        # the smallest step: a few images, every launch and every host microsecond shows
        step("lenet_avg", 16, act="swish", bn=False, name="lenet_avg_b16", do="gradient"),
        # LeNet at its two benchmark batches, without and with batch norm
        step("lenet", 128, bn=False, name="lenet_b128"),
        step("lenet", 1024, bn=True, name="lenet_bn_b1024"),
        # the 5x5 network for 32x32 images, at a batch of no round size
        step("alexnet_cifar", 100, act="swish", bn=True, name="alexnet_cifar_b100"),
        # the headline network and batch
        step("vgg11", 256, name="vgg11_b256"),
        # the same network with the readers' activation, its buffers laid out for 256 images and 77 of them filled: the
        # end of an epoch
        step("vgg11", 256, filled=77, act="swish", name="vgg11_swish_77_of_256"),
        # a deep member of the family: 32x32 maps of 64 channels
        step("vgg16", 128, act="swish", name="vgg16_b128"),
        # large images, a thousand classes, linear layers of 4096
        step("alexnet", 64, bn=False, name="alexnet_224_b64"),
        # the accuracy sweep after an epoch: input pipeline, forward passes, a last batch of 232
        dict(do="evaluate", net="vgg11", batch=256, images=1000, act="relu", bn=True, bias=True, name="vgg11_test_1000"),
        # the trust-region step's other two parts: curvature along a direction, factors + inverses + natural gradient
        dict(do="hessian", net="vgg11", batch=256, filled=256, act="relu", bn=True, bias=True, name="vgg11_hv_b256"),
        dict(do="curvature", net="vgg11", batch=256, filled=256, act="relu", bn=True, bias=True, name="vgg11_kfac_b256"),
        # gradient and Gauss-Newton product of an autoencoder on a thousand images
        dict(do="dense", net="autoencoder", points=1000, name="autoencoder_1000"),
    ]


def _log_int(rng, low, high):
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    do = rng.choice(["step"] * 6 + ["evaluate", "hessian", "curvature", "dense"])
    act = rng.choice(["relu", "relu", "swish", "elu", "softplus"])
    if do == "dense":
        return dict(do=do, net="autoencoder", points=_log_int(rng, 100, 2000))
    if do == "evaluate":
        return dict(do=do, net="vgg11", batch=256, images=_log_int(rng, 100, 1000), act=act, bn=True, bias=True)
    if do in ("hessian", "curvature"):
        net = rng.choice(["lenet", "vgg11"])
        batch = _log_int(rng, 32, 256)
        return dict(do=do, net=net, batch=batch, filled=batch, act=act, bn=True, bias=True)
    net = rng.choice(["lenet_avg", "lenet", "alexnet_cifar", "vgg11", "vgg11", "vgg13", "vgg16", "alexnet"])
    low, high = dict(lenet_avg=(8, 1024), lenet=(8, 1024), alexnet_cifar=(16, 256), alexnet=(8, 64)).get(net, (16, 256 if net == "vgg11" else 128))
    batch = _log_int(rng, low, high)
    filled = batch if net == "lenet_avg" or rng.random() < 0.8 else max(1, int(batch * rng.uniform(0.3, 1.0)))
    if net not in ("lenet", "vgg11", "alexnet"):
        act = "swish"  # what their builders set
    bn = net != "alexnet" and rng.random() < 0.7
    bias = net in ("vgg13", "vgg16") or rng.random() < 0.8
    return step(net, batch, filled, act, bn, bias, do="gradient" if net == "lenet_avg" else "step")


# ---------------------------------------------------------------- models
def _model(case):
    net, batch, bn, bias, act = case["net"], case["batch"], int(case["bn"]), int(case["bias"]), ACTS[case["act"]]
    m = S.CNN_MODEL()
    if net == "lenet":
        return build_lenet(batch, bn=bool(bn), act=act, fc_act=act, bias=bias)
    if net == "lenet_avg":
        L.cnn.readLenetCNN(C.byref(m), 3, 32, 32, batch, bias, bn)
    elif net == "alexnet_cifar":
        L.cnn.readAlexNetCNN(C.byref(m), batch, 32, 32, 10, bias, bn)
    elif net == "vgg11":
        return build_vgg11(batch, bn=bool(bn), act=act, bias=bias)
    elif net == "alexnet":
        return build_alexnet(batch, act=act, fc_act=act, bias=bias)
    else:
        getattr(L.cnn, "read" + net.upper())(C.byref(m), batch, 32, 32, 10, 3, bias, bn, S.CIFAR10)
    return m


def _autoencoder(points):
    m = S.NN_MODEL()
    sizes, acts = AUTOENCODER, [S.ACT_LOGISTIC] * (len(AUTOENCODER) - 1)
    acts[len(acts) // 2 - 1] = S.ACT_LINEAR  # the code layer
    L.cnn.fitre_build_nn(C.byref(m), (C.c_int * len(sizes))(*sizes), (C.c_int * len(acts))(*acts), len(acts), S.MODEL_TYPE_MSE, points)
    for set_offsets in (L.cnn.initRZOffsets, L.cnn.initSampledZOffsets, L.cnn.initSampledROffsets):
        set_offsets(C.byref(m), points)
    return m


def _weights(model, gen):
    """He-normal weights and small biases in the flat layout."""
    w = torch.zeros(model.pSize, device=DEVICE)
    layers = [(model.convLayer[i].inChannels * model.convLayer[i].kSize ** 2, model.convLayer[i].outChannels) for i in range(model.cLayers)]
    layers += [(model.fcLayer[i].in_, model.fcLayer[i].out) for i in range(model.lLayers)]
    for i, (fan_in, out) in enumerate(layers):
        a = model.wOffsets[i]
        w[a:a + fan_in * out].normal_(0.0, (2.0 / fan_in) ** 0.5, generator=gen)
        if model.bias:
            w[model.bOffsets[i]:model.bOffsets[i] + out].normal_(0.0, 0.02, generator=gen)
    return w


def _images(count, channels, height, width, gen):
    """Images with neighbouring pixels alike, as photographs are: coarse noise blown up, and fine noise on it."""
    coarse = torch.randn(count, channels, -(-height // 8), -(-width // 8), device=DEVICE, generator=gen)
    x = coarse.repeat_interleave(8, 2).repeat_interleave(8, 3)[:, :, :height, :width]
    return 0.8 * x + 0.6 * torch.randn(count, channels, height, width, device=DEVICE, generator=gen)


class _State:
    """What a trainer keeps: the model record, its device buffers and the records that point at them."""

    def __init__(self, case, seed):
        L.check(L.hip.fitre_hip_init(0))
        self.case = case
        self.gen = torch.Generator(DEVICE).manual_seed(seed)
        self.reals = []

    def hold(self, t):
        self.reals.append(t)
        return t.data_ptr()

    def space(self, reals):
        return self.hold(torch.empty(max(int(reals), 64), device=DEVICE))


def _cnn_state(case, seed):
    st = _State(case, seed)
    m = st.model = _model(case)
    n = st.n = case.get("filled", case["batch"])
    c, h, w = input_dims(m)
    k = num_classes(m)
    st.weights = _weights(m, st.gen)
    st.z, st.dx, st.grad = (torch.zeros(s, device=DEVICE) for s in (m.zSize, m.zSize, m.pSize))
    st.probs, st.errors = torch.zeros(k * case["batch"], device=DEVICE), torch.zeros(max(k * case["batch"], m.maxDeltaSize), device=DEVICE)
    st.labels = torch.randint(1, k + 1, (n,), device=DEVICE, generator=st.gen).float()
    d = st.data = S.DEVICE_DATASET()
    d.weights, d.numClasses, d.datasetType = st.weights.data_ptr(), k, S.CIFAR10
    d.features, d.height, d.width = c * h * w, h, w
    d.sampledTrainY = st.labels.data_ptr()
    if case["do"] != "evaluate":
        st.batch = _images(n, c, h, w, st.gen).transpose(0, 1).contiguous()  # [C][N][W][H]
        d.currentBatch = st.batch.data_ptr()
    need = 2 * m.maxDeltaSize + max(L.cnn.cnnForwardMemRequired(C.byref(m)), L.cnn.cnnBackwardMemRequired(C.byref(m))) + 1024
    st.scratch = S.SCRATCH_AREA()
    st.scratch.devWorkspace = st.scratch.nextDevPtr = st.space(need)
    L.cnn.initBatchNormData(C.byref(m), st.z.data_ptr(), m.zOffsets)
    return st


def _activate(code, x):
    if code == S.CNN_ACT_RELU:
        return torch.relu(x)
    if code == S.CNN_ACT_SWISH:
        return x * torch.sigmoid(x)
    if code == S.CNN_ACT_ELU:
        return F.elu(x)
    return F.softplus(x, threshold=700.0) if code == S.CNN_ACT_SOFTPLUS else x


def _unfolded(x, c, wm):
    """The convolution of c as a product with laid-out patches, some images at a time: [N][Cout][A][B]."""
    some = max(1, (1 << 27) // (wm.shape[1] * c.outWidth * c.outHeight))
    parts = []
    for a in range(0, x.shape[0], some):
        cols = F.unfold(x[a:a + some], c.kSize, padding=c.padding, stride=c.stride).transpose(0, 1)
        parts.append((wm @ cols.reshape(wm.shape[1], -1)).reshape(c.outChannels, -1, c.outWidth, c.outHeight).transpose(0, 1))
    return torch.cat(parts)


def _network(st, w, x, put=lambda at, t: None, running=None):
    """Logits of the network in float64 for images x [N][C][A][B] and flat weights w.  put(at, t) is told every stage of the
    activation store (the slabs of include/fitre_nn.h); running: the store whose running statistics normalise."""
    m, n = st.model, x.shape[0]

    def bias(i, out):
        return w[m.bOffsets[i]:m.bOffsets[i] + out] if m.bias else torch.zeros(out, dtype=torch.float64, device=DEVICE)

    for i in range(m.cLayers):
        c, p, slab = m.convLayer[i], m.poolLayer[i], m.zOffsets[i + 1]
        k = c.inChannels * c.kSize ** 2
        wm = w[m.wOffsets[i]:m.wOffsets[i] + k * c.outChannels].reshape(c.outChannels, k)
        y = _unfolded(x, c, wm) + bias(i, c.outChannels).reshape(1, -1, 1, 1)
        put(slab, y.transpose(0, 1))
        if c.batchNorm:
            at = slab + c.batchNormOffset
            mean, var = y.mean((0, 2, 3)), y.var((0, 2, 3), unbiased=False)
            if running is not None:
                mean, var = (running[at + o:at + o + c.outChannels].double() for o in (c.runningMeansOffset, c.runningVariancesOffset))
            y = (y - mean.reshape(1, -1, 1, 1)) / torch.sqrt(var.reshape(1, -1, 1, 1) + 1e-5)
            put(at, y.transpose(0, 1))
            put(at + c.meansOffset, mean)
            put(at + c.variancesOffset, var)
        x = _activate(m.actFuns[i], y)
        put(slab + c.activationOffset, x.transpose(0, 1))
        if p.type == S.MAX_POOL:  # the cell that is taken is the largest of the rounded ones
            at = F.max_pool2d(x.detach().float(), p.pSize, p.stride, p.padding, return_indices=True)[1]
            x = x.flatten(2).gather(2, at.flatten(2)).reshape(at.shape)
        elif p.type == S.AVG_POOL:
            x = F.avg_pool2d(x, p.pSize, p.stride, p.padding)
        if p.type != S.NO_POOL:
            put(slab + c.poolOffset, x.transpose(0, 1))
    x = x.transpose(2, 3).reshape(n, -1)  # the linear layers read [N][C][B][A], written over the last slab's output
    put(m.zOffsets[m.cLayers] + m.convLayer[m.cLayers - 1].outputOffset, x)
    for i in range(m.lLayers):
        f, at = m.fcLayer[i], m.zOffsets[m.cLayers + i + 1]
        a = m.wOffsets[m.cLayers + i]
        x = x @ w[a:a + f.in_ * f.out].reshape(f.in_, f.out) + bias(m.cLayers + i, f.out)
        put(at + f.offset, x)
        x = _activate(f.actFun, x)
        put(at, x)
    return x


def _store(z):
    """put() of _network that writes into z, rounded to its type."""
    def put(at, t):
        z[at:at + t.numel()] = t.detach().reshape(-1).to(z.dtype)
    return put


def _fill_z(st):
    """The activation store, probabilities and loss errors of a training forward pass, from float64 arithmetic."""
    p = torch.softmax(_network(st, st.weights.double(), st.batch.double().transpose(0, 1), _store(st.z)), 1)
    st.probs[:p.numel()] = p.reshape(-1).float()
    p[torch.arange(st.n), st.labels.long() - 1] -= 1
    st.errors[:p.numel()] = (p / st.n).reshape(-1).float()


def _forward(st, z):
    return L.cnn.cnnForward(C.byref(st.model), C.byref(st.data), C.byref(st.scratch), z.data_ptr(), st.probs.data_ptr(), st.errors.data_ptr(), 0,
                            st.n, S.MODEL_TRAIN)


def _backward(st):
    """cnnBackward on a copy of the loss errors, which it overwrites."""
    m, delta = st.model, st.scratch.nextDevPtr
    L.check(L.hip.fitre_hip_copy_d2d(delta, st.errors.data_ptr(), 4 * st.data.numClasses * st.n))
    L.cnn.cnnBackward(C.byref(m), C.byref(st.data), delta + 8 * m.maxDeltaSize, st.z.data_ptr(), st.grad.data_ptr(), st.dx.data_ptr(), delta,
                      delta + 4 * m.maxDeltaSize, 0, st.n, None)


def prepare(case, seed):
    if case["do"] == "dense":
        return _prepare_dense(case, seed)
    st = _cnn_state(case, seed)
    m, d = st.model, st.data
    if case["do"] == "evaluate":
        images, n = case["images"], case["batch"]
        x = _images(images, 3, 32, 32, st.gen).mul_(64).add_(128).clamp_(0, 255).round_().reshape(images, -1)
        y = torch.randint(1, 11, (images,), device=DEVICE, generator=st.gen).float()
        st.test_x, st.test_y = x, y
        d.testSetX, d.testSetY, d.testSizeX, d.testSizeY = x.data_ptr(), y.data_ptr(), images, images
        st.both = torch.zeros(2 * n * 3072, device=DEVICE)  # a batch as it is stored, and as the network reads it
        d.sampledTrainX = st.both.data_ptr()
        st.batch_labels = torch.zeros(n, device=DEVICE)
        d.sampledTrainY = st.batch_labels.data_ptr()
        st.page = torch.zeros(64).pin_memory()
        st.scratch.pageLckWorkspace = st.scratch.nextPageLckPtr = st.page.data_ptr()
        # running statistics as a few training passes leave them
        st.batch = _images(n, 3, 32, 32, st.gen).transpose(0, 1).contiguous()
        d.currentBatch, d.sampledTrainY = st.batch.data_ptr(), st.hold(torch.ones(n, device=DEVICE))
        st.n = n
        for _ in range(5):
            _forward(st, st.z)
        d.sampledTrainY = st.batch_labels.data_ptr()
    if case["do"] in ("step", "hessian", "curvature"):
        _fill_z(st)
    if case["do"] == "step":
        st.new_z = torch.zeros_like(st.z)
        L.cnn.initBatchNormData(C.byref(m), st.new_z.data_ptr(), m.zOffsets)
    if case["do"] in ("hessian", "curvature"):
        _backward(st)
    if case["do"] == "hessian":
        st.v = torch.randn(m.pSize, device=DEVICE, generator=st.gen).mul_(1e-2)
        st.hv = torch.zeros(m.pSize, device=DEVICE)
        st.ws = st.space(L.cnn.cnnHvMemRequired(C.byref(m)))
    if case["do"] == "curvature":
        info = st.info = S.KFAC_CURVATURE_INFO()
        L.cnn.computeKFACStorageIndices(C.byref(m), C.byref(info))
        last = m.cLayers + m.lLayers
        st.ngrad = torch.zeros(m.pSize, device=DEVICE)
        info.regLambda, info.dampGamma = DAMPING, 0.0
        info.OmegaZInv, info.LambdaGInv = st.space(info.OmegaZOffsets[last]), st.space(info.LambdaGOffsets[last])
        info.gradient, info.nGradient = st.grad.data_ptr(), st.ngrad.data_ptr()
        st.ws = st.space(max(L.cnn.kfacInverseMemRequired(C.byref(m), st.n), L.cnn.kfacNaturalGradientMemRequired(C.byref(m))) + 64)
    return st


def _prepare_dense(case, seed):
    st = _State(case, seed)
    n = case["points"]
    m = st.model = _autoencoder(n)
    st.weights = torch.zeros(m.pSize, device=DEVICE)
    for i in range(m.numLayers):
        count = m.layerSizes[i] * m.layerSizes[i + 1]
        st.weights[m.wOffsets[i]:m.wOffsets[i] + count].normal_(0.0, (1.0 / m.layerSizes[i]) ** 0.5, generator=st.gen)
    st.x = torch.sigmoid(2 * _images(n, 1, 28, 28, st.gen)).reshape(n, 784).contiguous()
    st.v = torch.randn(m.pSize, device=DEVICE, generator=st.gen).mul_(1e-2)
    st.z, st.dx, st.grad = (torch.zeros(s, device=DEVICE) for s in (m.zSize, m.rFullSize, m.pSize))
    d = st.data = S.DEVICE_DATASET()
    d.features = 784
    d.trainSetX = d.trainSetY = st.x.data_ptr()  # the images are their own targets
    d.trainSizeX = d.trainSizeY = n
    need = 2 * (L.cnn.nnGradientMemRequired(C.byref(m), n) + m.zSize + m.rFullSize + 4096)
    st.scratch = S.SCRATCH_AREA()
    st.scratch.devWorkspace = st.scratch.nextDevPtr = st.space(need)
    st.hv = torch.zeros(L.cnn.nnHessianVecMemRequired(C.byref(m), C.byref(d), S.FULL_DATASET), device=DEVICE)
    st.hv_scratch = S.SCRATCH_AREA()
    st.hv_scratch.devWorkspace = st.hv_scratch.nextDevPtr = st.hv.data_ptr()
    st.loss, st.error = C.c_float(), C.c_float()
    return st


# ---------------------------------------------------------------- one pass
def run(st):
    do, m = st.case["do"], st.model
    if do == "gradient":
        loss = L.cnn.computeCNNGradient(C.byref(m), C.byref(st.data), C.byref(st.scratch), st.z.data_ptr(), st.dx.data_ptr(), st.probs.data_ptr(),
                                        st.errors.data_ptr(), st.grad.data_ptr(), 0, st.n, 5e-4)
        return dict(loss=loss, probs=st.probs, errors=st.errors, gradient=st.grad, z=st.z, dx=st.dx)
    if do == "step":
        loss = _forward(st, st.new_z)
        _backward(st)
        return dict(loss=loss, probs=st.probs, errors=st.errors, gradient=st.grad, z=st.new_z, dx=st.dx)
    if do == "evaluate":
        loss, accuracy = C.c_float(), C.c_float()
        L.cnn.computeTestGeneralizationErrors(C.byref(m), C.byref(st.data), C.byref(st.scratch), st.z.data_ptr(), st.probs.data_ptr(),
                                              st.errors.data_ptr(), C.byref(loss), C.byref(accuracy))
        return dict(loss=loss.value, accuracy=accuracy.value, probs=st.probs, z=st.z)
    if do == "hessian":
        L.cnn.cnnHv(C.byref(m), C.byref(st.data), st.z.data_ptr(), st.probs.data_ptr(), st.errors.data_ptr(), st.dx.data_ptr(), st.v.data_ptr(),
                    st.hv.data_ptr(), 0, st.n, st.ws, None, 0.0)
        return dict(hv=st.hv)
    if do == "curvature":
        L.cnn.computeOmegaZAndLambdaDelta(C.byref(st.info), C.byref(m), C.byref(st.data), st.n, None, st.z.data_ptr(), st.dx.data_ptr(), None,
                                          m.zOffsets, m.zztOffsets, st.ws)
        L.cnn.computeNaturalGradient(C.byref(m), C.byref(st.info), st.ws, None)
        return dict(natural_gradient=st.ngrad)
    L.cnn.computeGradient(C.byref(m), C.byref(st.data), C.byref(st.scratch), st.weights.data_ptr(), st.z.data_ptr(), st.dx.data_ptr(),
                          st.grad.data_ptr(), C.byref(st.loss), C.byref(st.error), S.FULL_DATASET)
    L.cnn.gaussNewtonHessianVec(C.byref(m), C.byref(st.data), st.z.data_ptr(), st.dx.data_ptr(), st.v.data_ptr(), st.weights.data_ptr(),
                                C.byref(st.hv_scratch), S.FULL_DATASET)
    return dict(loss=st.loss.value, error=st.error.value, gradient=st.grad, z=st.z, dx=st.dx, gauss_newton=st.hv[:m.pSize])


# ---------------------------------------------------------------- the same in 64 bits
def _padded(t, like):
    out = torch.zeros(like.numel(), dtype=torch.float64, device=DEVICE)
    out[:t.numel()] = t.detach().reshape(-1)
    return out


def exact(case, seed):
    do = case["do"]
    if do == "curvature":
        return None  # factors, damping and inverses of nine layers by the rules of the framework: its tests' oracle has them
    st = prepare(case, seed)
    if do == "dense":
        return _exact_dense(st)
    if do == "evaluate":
        return _exact_evaluate(st)
    w = st.weights.double().requires_grad_()
    z = torch.zeros(st.z.numel(), dtype=torch.float64, device=DEVICE)
    logits = _network(st, w, st.batch.double().transpose(0, 1), _store(z))
    labels = st.labels.long() - 1
    loss = F.cross_entropy(logits, labels)
    if do == "hessian":
        g, = torch.autograd.grad(loss, w, create_graph=True)
        return dict(hv=torch.autograd.grad((g * st.v.double()).sum(), w)[0])
    g, = torch.autograd.grad(loss, w)
    if do == "gradient":
        g = g + 5e-4 * st.weights.double()
    p = torch.softmax(logits.detach(), 1)
    errors = p.clone()
    errors[torch.arange(st.n), labels] -= 1
    # a probability below the smallest float makes the 32-bit loss a matter of how it is clamped
    loss = loss.item() if p.min().item() > 1e-30 else None
    return dict(loss=loss, probs=_padded(p, st.probs), errors=_padded(errors / st.n, st.errors), gradient=g,
                z=None if case["bn"] else z, dx=None)


def _exact_evaluate(st):
    """Batches through the running statistics that prepare() left; probabilities of the last, short one."""
    d, n, total = st.data, st.case["batch"], st.data.testSizeX
    x, y = st.test_x.double().reshape(total, 3, 32, 32), st.test_y.long() - 1
    mean, std = (torch.tensor(t, dtype=torch.float64, device=DEVICE).reshape(1, 3, 1, 1) for t in CIFAR10_STATISTICS)
    x = (x / 255 - mean) / std
    w, running, loss, hits = st.weights.double(), st.z.clone(), 0.0, 0
    probs = st.probs.double()  # the rows past the last batch are what was there before
    for a in range(0, total, n):
        logits, labels = _network(st, w, x[a:a + n], running=running), y[a:a + n]
        loss += F.cross_entropy(logits, labels, reduction="sum").item()
        hits += (logits.argmax(1) == labels).sum().item()
        probs[:logits.numel()] = torch.softmax(logits, 1).reshape(-1)
    return dict(loss=loss / total, accuracy=100.0 * hits / total, probs=probs, z=None)


def _exact_dense(st):
    """Loss, gradient and Gauss-Newton product; the last keeps the reference's term of the top layer, -(1/n) of the product of
    that layer's direction and the errors, back-propagated through the layers below."""
    m, n, x, v = st.model, st.x.shape[0], st.x.double(), st.v.double()
    z = torch.zeros(st.z.numel(), dtype=torch.float64, device=DEVICE)

    def layers(w, top):
        h = x
        for i in range(top):
            a, b, size = m.wOffsets[i], m.bOffsets[i], m.layerSizes[i + 1]
            h = h @ w[a:a + m.layerSizes[i] * size].reshape(m.layerSizes[i], size) + w[b:b + size]
            if i + 1 == m.numLayers:
                return h
            h = torch.sigmoid(h) if m.actFuns[i] == S.ACT_LOGISTIC else h
            _store(z)(m.zOffsets[i + 1], h)
        return h

    w, top = st.weights.double().requires_grad_(), m.numLayers
    logits = layers(w, top)
    out = torch.sigmoid(logits)
    _store(z)(m.zOffsets[top], out)
    loss = -(x * logits - F.softplus(logits)).sum() / n
    g, = torch.autograd.grad(loss, w, retain_graph=True)
    u = torch.zeros_like(logits, requires_grad=True)
    jt, = torch.autograd.grad(logits, w, u, create_graph=True)  # J'u, whose derivative by u takes v to Jv
    jv, = torch.autograd.grad(jt, u, v)
    out = out.detach()
    gn, = torch.autograd.grad(logits, w, out * (1 - out) * jv / n)
    size = m.layerSizes[top]
    below = layers(w, top - 1)
    a = m.wOffsets[top - 1]
    vw = v[a:a + m.layerSizes[top - 1] * size].reshape(-1, size)
    gn = gn - torch.autograd.grad(below, w, (x - out) @ vw.t() / n)[0]
    return dict(loss=loss.item(), error=((x - out) ** 2).sum().item() / n, gradient=g, z=z, dx=None, gauss_newton=gn)


# ---------------------------------------------------------------- what a pass cannot do without
def _live_macs(layer, n):
    """Multiply-adds of one convolution product whose window tap lies inside the image."""
    def live(size, out):
        return sum(1 for o in range(out) for t in range(layer.kSize) if 0 <= o * layer.stride - layer.padding + t < size)
    return float(n) * layer.inChannels * layer.outChannels * live(layer.height, layer.outHeight) * live(layer.width, layer.outWidth)


def work(case):
    if case["do"] == "dense":
        m, n = _autoencoder(case["points"]), case["points"]
        macs = [float(n) * m.layerSizes[i] * m.layerSizes[i + 1] for i in range(m.numLayers)]
        # gradient: forward, dW, dX; product: R-forward (one product more, of VW), R-dW, R-dX
        flops = 2.0 * (6 * sum(macs) + sum(macs[1:]))
        return dict(bytes=4.0 * (n * 784 + 4 * m.pSize + m.zSize + m.rFullSize), flops=flops)
    m = _model(case)
    n = case.get("filled", case.get("images"))
    conv = [_live_macs(m.convLayer[i], n) for i in range(m.cLayers)]
    fc = [float(n) * m.fcLayer[i].in_ * m.fcLayer[i].out for i in range(m.lLayers)]
    share = n / float(case["batch"])
    inputs = n * float(input_dims(m)[0] * input_dims(m)[1] * input_dims(m)[2])
    if case["do"] == "evaluate":
        return dict(bytes=4.0 * (inputs + n + m.pSize + m.zSize * share), flops=2.0 * (sum(conv) + sum(fc)))
    if case["do"] in ("gradient", "step"):
        products = 3 * sum(conv) - conv[0] + 3 * sum(fc)
        return dict(bytes=4.0 * (inputs + n + 2 * m.pSize + 2 * m.zSize * share), flops=2.0 * products)
    if case["do"] == "hessian":
        # R{forward}, R{dW} and R{dX} are two products each; the image itself has no R part
        products = 6 * (sum(conv) + sum(fc)) - 4 * conv[0]
        return dict(bytes=4.0 * (inputs + 3 * m.pSize + 2 * m.zSize * share), flops=2.0 * products)
    flops = 0.0
    for i in range(m.cLayers + m.lLayers):
        if i < m.cLayers:
            l = m.convLayer[i]
            order, out, positions = l.inChannels * l.kSize ** 2 + m.bias, l.outChannels, float(n) * l.outHeight * l.outWidth
        else:
            order, out, positions = m.fcLayer[i - m.cLayers].in_ + m.bias, m.fcLayer[i - m.cLayers].out, float(n)
        inner = min(float(order), positions)  # a factor of few positions is inverted at their number
        flops += (inner ** 2 * max(order, positions) + inner ** 3) + (float(out) ** 2 * positions + float(out) ** 3)
        flops += 2.0 * (float(out) ** 2 * order + 2 * float(out) * order * inner if inner < order else float(out) ** 2 * order + float(out) * float(order) ** 2)
    return dict(bytes=4.0 * (m.pSize * 2 + 2 * m.zSize * share), flops=flops)


def tolerance(case):
    """Moving every weight by a relative 2^-23 (one more rounding of each) moves the outputs of these cases by up to 2.5e-6
    in norm (the deep batch-normalised networks) and 1.2e-4 in single entries; the stored activations differ from float64
    ones by up to 1e-6.  Four times that."""
    return {"rel": 1e-5, "max": 5e-4}
