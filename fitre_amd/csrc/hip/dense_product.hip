// Products of the fully connected family with the steps that follow them, one launch each.
//
// A pass over a thousand points of a small network is a chain of products of 10^7 to 10^9 multiply-adds, each of which the general
// engine cuts into ranges, sums in a second launch and hands to elementwise launches: the chain, not the arithmetic, is what it
// waits for.  Here a workgroup owns a whole 32 x 64 tile of the result.  Its eight waves share the reduction: each loads its part
// of both panels from memory straight into the order the matrix fragments have, splits it (split_bf16.h) and multiplies, with
// no LDS and no barrier in the loop, and every number of a panel is split once per workgroup.  The eight partial tiles meet in LDS,
// are added in wave order in double, and what follows the product -- bias, activation, derivative, loss -- is done to the sum.
//
// Bound: the vector instructions that split the numbers (162 a wave and step against 384 cycles of matrix instructions) and, of the 7
// us that the shortest product takes, the latency of its first loads, of LDS and of its stores.  Product and reduction on the
// engine / here, us: 512 x 1000 x 784 18.6 / 12.6, op(A) transposed 18.8 / 13.9, weight gradient 512 x 784 x 1000 19.4 / 13.0; 64 x
// 1000 x 256 13.5 / 7.1.  Gradient and Gauss-Newton product of a 784-512-256-64-256-512-784 autoencoder: 120 launches and 782 us
// for 1000 points with the engine, 25 and 359 here; 100 points 687 / 302, 2000 893 / 490.
#include "dense_product.h"

using namespace fitre;

static long dense_tiles(int M, int N, int blocks) { return (long)((N + 32 * blocks - 1) / (32 * blocks)) * ((M + kDenseJ - 1) / kDenseJ); }

// offsets into an operand are 32 bits of bytes, with room for a step past its end
static bool dense_operands_fit(int M, int N, int K)
{
	const double most = (double)(1 << 29);
	return M > 0 && N > 0 && K > 0 && (double)M * K < most && (double)N * K < most && (double)M * N < most;
}

// Blocks of 32 columns of C a tile has.  Two take 1.35 times as long as one, so that they are the better choice where single ones do
// not fit the chip at once: 784 x 1000 x 512, op(A) transposed, 21.0 us (416 tiles) / 16.0 (208), 512 x 2000 x 784 23.2 / 18.6; 512 x
// 1000 x 784 (256 tiles) 12.6 / 17.0.  Products of two operands whose rows lie across the reduction have no registers for two.
static int dense_high(bool ak, long tiles) { return ak && tiles > lane_compute_units() ? 2 : 1; }

extern "C" {

// The engine's larger tiles take over where the chip is full several times: 784 x 8000 x 512 60.9 / 88.4 us, 512 x 784 x 8000 75.8 /
// 69.2 but 64 x 256 x 8000 13.8 / 59.5 (the few tiles walk the reduction alone).  Whole passes, us: 2400 points of the autoencoder above
// 1027 / 666, a 33-17-33 network with 4096 464 / 135, 2048-1024-512-1024-2048 with 1000 1018 / 726; with more than these every layer of a
// network on the engine is as good.
int fitre_hip_dense_product_fits(int transA, int transB, int M, int N, int K)
{
	if (!dense_operands_fit(M, N, K) || (transA && transB)) return 0;
	const long cus = lane_compute_units(), tiles = dense_tiles(M, N, 1);
	return dense_tiles(M, N, dense_high(!transB, tiles)) <= (transB ? 4 : 2) * cus && K <= kDenseLongest;
}

long fitre_hip_dense_product_tiles(int M, int N)
{
	const long tiles = M > 0 && N > 0 ? dense_tiles(M, N, 1) : 0;
	return dense_tiles(M, N, dense_high(true, tiles));
}

int fitre_hip_dense_products(const fitre_dense_product *p, int count)
{
	FITRE_NEED_INIT();
	FITRE_REQUIRE(p && count >= 1 && count <= kDenseBatch, "fitre_hip_dense_products: %d products", count);
	DenseBatch b{};
	double flops = 0.0;
	long blocks = 0, tiles = 0;
	const bool ak = !p[0].transB, bk = p[0].transA == 1;
	for (int i = 0; i < count; i++) tiles += p[i].M > 0 && p[i].N > 0 ? dense_tiles(p[i].M, p[i].N, 1) : 0;
	const int high = dense_high(ak, tiles);
	for (int i = 0; i < count; i++) {
		const fitre_dense_product &q = p[i];
		FITRE_REQUIRE(q.A && q.B && q.C, "fitre_hip_dense_products: null pointer");
		FITRE_REQUIRE((q.A2 == nullptr) == (q.B2 == nullptr), "fitre_hip_dense_products: half of a second pair");
		FITRE_REQUIRE(dense_operands_fit(q.M, q.N, q.K), "fitre_hip_dense_products: shape %d x %d x %d", q.M, q.N, q.K);
		FITRE_REQUIRE(q.transA == p[0].transA && q.transB == p[0].transB && (q.transA == 0 || q.transA == 1) && (q.transB == 0 || q.transB == 1),
		              "fitre_hip_dense_products: transpose flags");
		FITRE_REQUIRE(!(q.transA && q.transB), "fitre_hip_dense_products: both operands transposed");
		FITRE_REQUIRE(!(q.transA && q.rowSums), "fitre_hip_dense_products: row sums of a transposed operand");
		FITRE_REQUIRE(q.then >= FITRE_DENSE_STORE && q.then <= FITRE_DENSE_LINEAR_HEAD, "fitre_hip_dense_products: step %d", q.then);
		FITRE_REQUIRE(q.then == FITRE_DENSE_STORE || q.then >= FITRE_DENSE_LOGISTIC_HEAD || act_known(q.act), "fitre_hip_dense_products: activation %d", q.act);
		FITRE_REQUIRE((q.then != FITRE_DENSE_DERIVATIVE && q.then != FITRE_DENSE_ROP_BACKWARD) || q.z || q.act == ACT_LINEAR,
		              "fitre_hip_dense_products: the derivative needs z");
		FITRE_REQUIRE((q.then != FITRE_DENSE_DERIVATIVE && q.then != FITRE_DENSE_ROP_BACKWARD) || !act_needs_zin(q.act),
		              "fitre_hip_dense_products: activation %d has no derivative by its output", q.act);
		FITRE_REQUIRE(!q.x || q.d, "fitre_hip_dense_products: x without d");
		FITRE_REQUIRE((q.then != FITRE_DENSE_LOGISTIC_HEAD && q.then != FITRE_DENSE_LINEAR_HEAD) || (q.d && q.also && q.headSums),
		              "fitre_hip_dense_products: a head needs targets, errors and sums");
		// engine rows i are the columns of C, op(B) by columns; engine columns j its rows, op(A) by rows
		DenseItem &t = b.item[i];
		t.a = DenseOperand{ q.B, q.B2, (uint32_t)(4u * (uint32_t)q.N * (uint32_t)q.K), q.transB ? q.N : q.K, q.N };
		t.b = DenseOperand{ q.A, q.A2, (uint32_t)(4u * (uint32_t)q.M * (uint32_t)q.K), q.transA ? q.K : q.M, q.M };
		t.R = q.K;
		t.alpha = q.alpha, t.bias = q.bias, t.then = q.then, t.act = q.act;
		t.out = q.C, t.raw = q.raw, t.also = q.also, t.z = q.z, t.x = q.x, t.d = q.d;
		t.headSums = q.headSums, t.rowSums = q.rowSums;
		t.vec = q.M % 4 == 0 && ((((uintptr_t)q.C | (uintptr_t)q.raw | (uintptr_t)q.also | (uintptr_t)q.z | (uintptr_t)q.x | (uintptr_t)q.d)) & 15) == 0;
		t.tilesJ = (q.M + kDenseJ - 1) / kDenseJ;
		b.first[i] = (int)blocks;
		blocks += dense_tiles(q.M, q.N, high);
		FITRE_REQUIRE(blocks < (1 << 30), "fitre_hip_dense_products: too many tiles");
		flops += 2.0 * (double)q.M * q.N * q.K * (q.A2 ? 2 : 1);
	}
	b.first[count] = (int)blocks;
	b.count = count;
	LaunchScope scope(FITRE_KC_FC_GEMM, flops, kTileSplit);
#define DENSE_LAUNCH(AK, BK)                                                                                          \
	(high == 2 ? dense_product_kernel<AK, BK, 2><<<(unsigned)blocks, kDenseThreads, 0, stream()>>>(b)                  \
	           : dense_product_kernel<AK, BK, 1><<<(unsigned)blocks, kDenseThreads, 0, stream()>>>(b))
	if (ak && !bk) DENSE_LAUNCH(true, false);
	else if (ak && bk) DENSE_LAUNCH(true, true);
	else dense_product_kernel<false, false, 1><<<(unsigned)blocks, kDenseThreads, 0, stream()>>>(b);
#undef DENSE_LAUNCH
	return check_launch("dense_product_kernel");
}

} // extern "C"
