"""What the host code asks of the device layer, in which order and with which buffers: on the CPU, with a layer that notes the calls."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CNN = os.path.join(ROOT, "fitre_amd", "libfitre_cnn.so")

# every other call does nothing and returns 0: no workspace, not supported, done
NOTED = r"""
#include <stdio.h>
#include <stddef.h>
#define NOTE(...) do { printf(__VA_ARGS__); fflush(stdout); } while (0)
size_t fitre_hip_conv_input_grad_prepared_bytes(const void *s) { (void)s; return 256; }
size_t fitre_hip_conv_forward_prepared_bytes(const void *s) { (void)s; return 256; }
int fitre_hip_lane_wait(int waiter, int signaller) { NOTE("wait %d %d\n", waiter, signaller); return 0; }
int fitre_hip_lane_select(int lane) { NOTE("lane %d\n", lane); return 0; }
int fitre_hip_conv_prepare_weights(int count, const void *s, const void *const *w, void *const *to, int grad)
{
	(void)s, (void)w;
	NOTE("copies %d", grad);
	for (int i = 0; i < count; i++) NOTE(" %zu", (size_t)to[i]);
	NOTE("\n");
	return 0;
}
int fitre_hip_dense_product_fits(int ta, int tb, int m, int n, int k) { (void)ta, (void)tb, (void)m, (void)n, (void)k; return 1; }
int fitre_hip_output_terms(int term, const void *target, const void *out, long n, float scale, void *to)
{
	(void)target, (void)out, (void)scale;
	NOTE("terms %d %ld %zu\n", term, n, (size_t)to);
	return 0;
}
int fitre_hip_accuracy_add(const void *p, const void *t, int rows, int classes, void *hits)
{
	(void)p, (void)t, (void)classes;
	NOTE("hits %zu %d\n", (size_t)hits, rows);
	return 0;
}
"""


@pytest.fixture(scope="module")
def noting(tmp_path_factory):
    """noting(script): the calls that a script of Python makes, as lists of words."""
    where = tmp_path_factory.mktemp("layer")
    asked = subprocess.run(["nm", "-D", "--undefined-only", CNN], check=True, capture_output=True, text=True).stdout.split()
    names = sorted(n for n in asked if n.startswith("fitre_hip_") and " %s(" % n not in NOTED)
    source, lib = where / "layer.c", str(where / "layer.so")
    source.write_text(NOTED + "".join("long %s(void) { return 0; }\n" % n for n in names))
    subprocess.run(["gcc", "-shared", "-fPIC", "-fno-builtin", "-o", lib, str(source)], check=True)

    def run(script):
        head = "import ctypes as C\nC.CDLL(%r, mode=C.RTLD_GLOBAL)  # before the libraries: its names are found first\n" % lib
        head += "from fitre_amd import lib as L, structs as S\nfrom fitre_amd.harness import build_alexnet, build_vgg11\n"
        out = subprocess.run([sys.executable, "-c", head + script], cwd=ROOT, check=True, capture_output=True, text=True, timeout=300).stdout
        return [line.split() for line in out.splitlines()]

    return run


@pytest.mark.parametrize("build", ["build_alexnet(8)", "build_vgg11(8)"])
def test_lane_2_is_ordered_only_where_it_has_copies_to_make(noting, build):
    """The backward pass of a network without batch norm reads no copies (its layers take the plain input gradients): no lane waits for any."""
    calls = noting("""
m, data = %s, S.DEVICE_DATASET()
L.cnn.fitreSetBackwardLanes(1)
data.weights, data.currentBatch = 1 << 30, 2 << 30
assert L.cnn.cnnBackwardMemRequired(C.byref(m)) > 0
p = lambda i: C.c_void_p(i << 34)
L.cnn.cnnBackward(C.byref(m), C.byref(data), p(1), p(2), p(3), p(4), p(5), p(6), 0, 8, None)
""" % build)
    copies = [i for i, c in enumerate(calls) if c[0] == "copies"]
    if "vgg" in build:
        at, = copies
        assert calls[at][1] == "1" and calls[at - 2:at] == [["wait", "2", "0"], ["lane", "2"]] and calls[at + 1] == ["lane", "0"]
        assert calls.count(["wait", "0", "2"]) == 1  # the chain, in front of its first use of one
    else:
        assert not copies and not any("2" in c[1:] for c in calls if c[0] in ("wait", "lane"))
        assert ["lane", "1"] in calls  # on two lanes


def test_hits_of_a_sweep_stay_clear_of_the_weight_copies(noting):
    """Two batches of 100 images and one of 50, the copies of the first kept for the second, with layers that need no workspace of their own."""
    calls = noting("""
m, data, scratch, p = build_vgg11(100), S.DEVICE_DATASET(), S.SCRATCH_AREA(), lambda i: C.c_void_p(i << 34)
data.testSizeX, data.features, data.numClasses, data.datasetType = 250, 3072, 10, S.CIFAR10
scratch.nextDevPtr, scratch.nextPageLckPtr = 1 << 34, 2 << 34
loss, accuracy = C.c_float(), C.c_float()
L.cnn.computeTestGeneralizationErrors(C.byref(m), C.byref(data), C.byref(scratch), p(3), p(4), p(5), C.byref(loss), C.byref(accuracy))
print("room", 4 * L.cnn.cnnForwardMemRequired(C.byref(m)))
""")
    room = int(calls[-1][1])
    assert [c[0] for c in calls if c[0] in ("copies", "hits")] == ["copies", "hits", "hits", "copies", "hits"]
    copies = [int(w) for c in calls if c[0] == "copies" for w in c[2:]]
    assert len(copies) == 14 and all(c[1] == "0" for c in calls if c[0] == "copies")
    hits = [(int(c[1]), int(c[2])) for c in calls if c[0] == "hits"]
    assert [rows for _, rows in hits] == [100, 100, 50]
    assert all(at + 4 * rows <= min(copies) and at >= 1 << 34 for at, rows in hits) and max(copies) + 256 <= (1 << 34) + room


@pytest.mark.parametrize("targets", [9, 10, 11])
def test_error_term_of_other_than_one_target_a_point(noting, targets):
    """It is as long as the targets are; the dx slot of the last layer, where the fused sweep has it, as the points are."""
    calls = noting("""
import sys
m, data, scratch, p = S.NN_MODEL(), S.DEVICE_DATASET(), S.SCRATCH_AREA(), lambda i: C.c_void_p(i << 34)
L.cnn.fitre_build_nn(C.byref(m), (C.c_int * 3)(6, 5, 4), (C.c_int * 2)(S.ACT_TANH, S.ACT_SOFTMAX), 2, S.MODEL_TYPE_CLASSIFICATION, 10)
L.cnn.initRZOffsets(C.byref(m), 10)
data.features, data.trainSizeX, data.trainSizeY = 6, 10, %d
scratch.nextDevPtr = 1 << 34
loss, error = C.c_float(), C.c_float()
L.cnn.computeGradient(C.byref(m), C.byref(data), C.byref(scratch), p(2), p(3), p(4), p(5), C.byref(loss), C.byref(error), S.FULL_DATASET)
print("slot", (4 << 34) + 4 * m.rZOffsets[1], 4 * (m.rFullSize - m.rZOffsets[1]))
""" % targets)
    slot, size = map(int, calls[-1][1:])
    error = [c for c in calls if c[0] == "terms"][-1]  # behind the terms of the loss
    assert int(error[2]) == 4 * targets and size == 160
    assert int(error[3]) == (slot if targets == 10 else 1 << 34)
