// Host-side entry points of the gfx950 pass kernels (hmi_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "hmi_pass.h"

namespace hmi {

// Largest dynamic LDS the generic pass may request (gfx950: 160 KiB per workgroup).
constexpr int kGenericMaxLds = 160 * 1024;
// pass outputs above this size use non-temporal stores (larger than the MALL), and their loads
// too when a side of the pass walks the column axis (pass_args::stream)
constexpr long long kStreamBytes = 256LL << 20;
enum : int { kStreamStores = 1, kStreamLoadsStores = 3, kHalvedTile = 4 };

using fast_launcher = hipError_t (*)(const pass_args &, long long nblocks, hipStream_t);

// A compiled uniform pass: length n, E elements per thread, T lines per block.
struct fast_kernel_info {
    bool dbl;
    int n, E, T, PS;
    int radix[8];
    int nstages;
    fast_launcher launch;
};

// Real-to-real passes in complex<double> of 256 and more points, 8 elements per thread, exchange the
// parts one after the other through a tile of half the size (kHalvedTile): their loads and stores move
// half the bytes of a complex tile, so the pass is bound by latency, and its LDS holds a CU to half the
// waves that its registers would allow.  256^3 double DCT-II / III pair 465 -> 438 us, the results bit for
// bit the same; above the Infinity Cache with the streaming form of the pass (512 x 256 x 512, the
// contiguous axis 244 us with non-temporal loads and stores, 231 with stores only).  The complex passes
// stay as they are (512^3 complex<double> 768 -> 787 us per pass, 256^3 109 -> 108), and so do launches whose
// blocks all fit the CUs at once, 16 waves in each, where the additional barriers only cost (12 x 256 x 32
// 16.6 us whole, 19.0 in halves).
constexpr bool halved_tile(int n, int e, int bytes) { return n >= 256 && bytes == 16 && e <= 8; }
constexpr bool halved_launch(long long nblocks, int threads) { return nblocks * threads > 256LL * 16 * 64; }

// wide = the pass walks the column axis on load or store (needs 128-byte column
// chunks); otherwise the variant with the fewest lines per block is returned.
const fast_kernel_info *find_fast_kernel(int n, bool dbl, bool wide);

// Runtime-length pass (hmi_generic.h): at most kMixedThreads threads per block; plans whose radices
// all stay within kLightRadix run builds of their own with fewer registers.
constexpr int kMixedThreads = 512;
constexpr int kLightRadix = 10;
constexpr long long kMixedTile = 16 * 1024;  // bytes a tile aims at
// Fused two-axis pass: longest side (longer axes keep the compile-time and matrix-core passes), LDS
// bytes of a plane and of a block's planes.  A plane that fills the LDS alone, one block per CU, still
// beats two passes where there are enough of them (min_planes): complex<double> 16 x 100^3 286 -> 236 us,
// 90 x 100 x 108 32 -> 28 us, complex<float> 4 x (120, 120, 64) 38 -> 30 us.
constexpr int kPlaneMaxSide = 256;
constexpr long long kPlaneBytes = kGenericMaxLds, kPlaneTile = 32 * 1024;
// Launches of fewer blocks, of all lines of a batch, take smaller tiles on more CUs (r2c 20 x 14 x 12 float:
// 14.3 -> 13.1 us a call, 60 x 60 x 40 pair 30.7 -> 28.0 us).  One line per block wastes its lanes: sized by
// one transform's lines, 206 x (64, 1, 14) double cosine 43.5 us and by the batch's 16.2, 1386 x (3, 7, 1) double
// c2r 14.2 and 7.7.
constexpr long long kFewBlocks = 256;
hipError_t launch_mixed_f32(const pass_args &a, const mixed_plan &g, int threads, long long nblocks, size_t lds_bytes,
                            hipStream_t s);
hipError_t launch_mixed_f64(const pass_args &a, const mixed_plan &g, int threads, long long nblocks, size_t lds_bytes,
                            hipStream_t s);
inline hipError_t launch_mixed(bool dbl, const pass_args &a, const mixed_plan &g, int threads, long long nblocks,
                               size_t lds_bytes, hipStream_t s) {
    return (dbl ? launch_mixed_f64 : launch_mixed_f32)(a, g, threads, nblocks, lds_bytes, s);
}

// Fused pass over the two fastest axes (hmi_plane.h).
hipError_t launch_plane_f32(const plane_args &a, int threads, long long nblocks, size_t lds_bytes, hipStream_t s);
hipError_t launch_plane_f64(const plane_args &a, int threads, long long nblocks, size_t lds_bytes, hipStream_t s);

// Compile-time tile of the batched kernel for one length: lines per tile and LDS bytes
// for each precision, and the complex-unit size of its stage twiddle table.
struct batch_kernel_info {
    int n, lines_f32, lines_f64;
    int radix[8];
    int nstages;
    size_t lds_f32, lds_f64;
};
// Returns the tile id for length n (or -1: the runtime-plan tile runs it).
int find_batch_kernel(int n, batch_kernel_info *info);
// Register class of a tile id: 0 for the compile-time tiles with at most 12 elements per
// thread and the staged tiles, 1 for 14 to 16, 2 for the others and the runtime-plan tile (-1).  Each class has its
// own build of the batched kernel, so light tiles are not held to heavy tiles' register count.
constexpr int kBatchClasses = 3;
int batch_kernel_class(int kid);
// Compile date and time of the kernels (stamps the autotuner's cache: choices timed with other
// kernels are not reused).
const char *kernels_build_stamp();

// One phase (one axis) of a batch of mixed-size c2c transforms (see batch_args), for the
// work items of one register class.
hipError_t launch_batched(bool dbl, int cls, const batch_args &b, int nblocks, size_t lds_bytes, hipStream_t s);

// Fused phases of a batch (fft_batch_fused, hmi_plane.h): the x-y phase for planes that fit the LDS, the
// column-block z phase.  Work items of three sizes, each with its own launch: kFusedLds[k] bytes of LDS
// and kFusedThreads[k] threads per block.
constexpr int kFusedSizes = 3;
constexpr int kFusedLds[kFusedSizes] = {40 * 1024, 80 * 1024, kGenericMaxLds};
constexpr int kFusedThreads[kFusedSizes] = {256, 512, 512};
constexpr int xy_row_stride(int n0) { return n0 | 1; }
hipError_t launch_batch_fused_f32(bool xy, const batch_args &b, int threads, int nblocks, size_t lds_bytes, hipStream_t s);
hipError_t launch_batch_fused_f64(bool xy, const batch_args &b, int threads, int nblocks, size_t lds_bytes, hipStream_t s);

// Precision forms of the c2c passes: plain FP32/FP64 vector ALU, or the 512-point
// complex<float> pass on the matrix cores with split-precision operands.
enum : int { kPrecPlain = 0, kSplitF16 = 1, kSplitBF16 = 2 };
// 512-point complex<float> c2c pass on MFMA (nblocks = number of 16-line tiles, one
// 1024-thread block each); a.tw = the bytes of
// mfma512_operand_table(prec, conj): the W512 table and the split DFT-matrix operands of the
// forward transform, or their conjugates for the backward one (the kernel conjugates nothing).
hipError_t launch_mfma512(int prec, const pass_args &a, long long nblocks, hipStream_t s);
std::vector<unsigned char> mfma512_operand_table(int prec, bool conj);

// Permutation of a box between two layouts (heFFTe's in-node reshape).
// a = source-fastest axis, b = destination-fastest axis (or any other axis
// when both sides are fastest along a, same_fast = 1), c = remaining axis.
struct permute_args {
    long long n_a, n_b, n_c, nbatch;
    long long si_a, si_b, si_c, bs_in;
    long long so_a, so_b, so_c, bs_out;
    long long ntile_a, ntile_b;
    int same_fast;
};

hipError_t launch_permute(int elem_bytes, const void *src, void *dst, const permute_args &p, hipStream_t s);

// Static device workspace of the no-allocation entry point (hmi_scratch.hip): kScratchBytes per
// GPU, held until the process ends.  scratch_address() returns its device address on the current
// device (resolved with hipGetSymbolAddress on the first call per device; throws on failure).
constexpr size_t kScratchBytes = 64ull << 20;
void *scratch_address();

}  // namespace hmi
