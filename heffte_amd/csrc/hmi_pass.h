// Host/device description of one FFT pass: a batched 1D c2c transform of
// length n along one axis of a 3D array, reading one layout and writing another.
//
// A pass sees its data as lines (the FFT axis, stride sa) indexed by a column
// (stride sc), a third axis b1 (stride sb1) and the batch b2 (stride sb2), with
// independent strides on the input and on the output side.  The layout
// permutation heFFTe performs with reshape3d_transpose
// (include/heffte_reshape3d.h:443-487) is therefore folded into the strides of
// the load or of the store of a pass, and the scale of apply_scale
// (include/heffte_fft3d.h:662-678) into its store.
#pragma once
#include <cstdint>

namespace hmi {

enum : int { kMaxStages = 24 };

// Pass modes of the uniform kernel.  The real-data modes run a complex FFT of
// half the line length: kModeR2C reads 2N reals as N complex pairs and unpacks
// the half spectrum (N + 1 bins) after the FFT; kModeC2R packs the N + 1 bins
// into N complex values before an inverse FFT and writes 2N reals.
//
// The real-to-real modes compute one axis of rtransform<cos/sin> through an
// N-point complex FFT (Makhoul's reordering):
//   kModeDCT2 (forward cos): v[n] = x[2n], v[N-1-n] = x[2n+1]; Y[k] = 2 Re(e^{-i pi k/2N} V[k])
//   kModeDCT3 (backward cos): W[k] = e^{i pi k/2N} (x[k] - i x[N-k]), w = IDFT(W);
//                             y[2m] = 2 Re w[m], y[2m+1] = 2 Re w[N-1-m]
//   kModeDST2 / kModeDST3: the same with the sine identities
//     DST-II(x)[k] = DCT-II((-1)^n x[n])[N-1-k],  DST-III(x)[n] = (-1)^n DCT-III(x[N-1-.])[n]
//
// DCT-I (rtransform<cos1>) runs the kernel's FFT length F = 2(N-1) on the even extension
// E[j] = x[j] (j <= N-1), x[F-j] (j > N-1), imaginary parts zero, and stores y[k] = Re X[k]
// for k < N (store_len = N): kModeDCT1 forward (REDFT00), kModeDCT1B backward (2 REDFT00).
enum : int {
    kModeC2C = 0, kModeR2C = 1, kModeC2R = 2, kModeDCT2 = 3, kModeDCT3 = 4, kModeDST2 = 5, kModeDST3 = 6,
    kModeDCT1 = 7, kModeDCT1B = 8
};

struct pass_args {
    const void *in;
    void *out;
    const void *tw;  // twiddle table of the pass (real2 of the pass precision)
    long long in_sa, in_sc, in_sb1, in_sb2;
    long long out_sa, out_sc, out_sb1, out_sb2;
    int ncol;      // number of columns
    int nb1;       // extent of the third axis
    int nbatch;    // number of transforms in the batch
    int nlines;    // ncol * nb1 * nbatch: lines are numbered column-fastest, then b1, then batch
    int load_colfast;   // 1: consecutive threads walk the column axis on load
    int store_colfast;  // 1: ... on store
    int conj;      // 1: backward transform (conjugate on load and on store)
    int in_real;   // 1: input elements are real scalars (imaginary part 0)
    int out_real;  // 1: store only the real part
    int store_len; // positions >= store_len along the FFT axis are not stored (r2c half spectrum)
    int herm_load; // 1: positions > n/2 are read as conj(x[n - pos]) (c2r Hermitian extension)
    int mode;      // kModeC2C, kModeR2C or kModeC2R (uniform kernel only)
    int stream;    // non-temporal data accesses (outputs larger than the MALL): 0 none,
                   // kStreamStores (1) stores only, kStreamLoadsStores (3) loads and stores
    const void *mul;  // non-null: every loaded element is first multiplied by the element of this
                      // array at the same offset (same layout and type as in; plain c2c loads only)
    double scale;  // multiplies every stored value (cast to the pass precision)
    // First step of an axis split in two passes (n4 = n * n2 points, plain c2c store only):
    // non-null tw4 = table of w_n4^m (m < n4); the value stored at position k of a line is first
    // multiplied by w_n4^(j k), j = the line's index along dimension tw4_dim (0 column, 1 b1,
    // 2 batch), which runs over the n2 interleaved sub-sequences.
    const void *tw4;
    int tw4_dim;
};

// Runtime radix plan of the batched kernel's runtime-plan tile (any length).
struct generic_plan {
    int n;
    int nstages;
    int lines;                 // lines per block
    int radix[kMaxStages];
    int twoff[kMaxStages];     // offset (complex units) of stage twiddles w_{Ls R}^{p k}
    int rootoff[kMaxStages];   // offset of w_R^j, j < R (used by radices without a hard-coded butterfly)
};

// Division of x < 2^31 by a fixed divisor d: q = umulhi(2 x, mul) >> shift, with 2^(shift-1) < d <=
// 2^shift and mul = ceil(2^(31 + shift) / d); exact, since x (mul d - 2^(31 + shift)) < 2^(31 + shift).
struct fast_div {
    unsigned mul, shift;
};

// Radix plan of the runtime-length pass (fft_generic): an in-place decimation in frequency over one
// LDS tile.  n = r_0 r_1 ... r_{S-1}; after stage s the remaining sub-transforms have m_s =
// n / (r_0 ... r_s) points.  Stage s runs the butterflies of the elements base + j + p m_s
// (p < r_s, j < m_s) of each of the n / (r_s m_s) blocks, twiddles output q by w_{r_s m_s}^{j q} and
// leaves it at base + j + q m_s; frequency k_0 + r_0 k_1 + r_0 r_1 k_2 + ... ends at position
// k_0 m_0 + k_1 m_1 + ...  Element (line l, position i) of a tile sits at
// i pitch + (i / m_0) pad + l.
//
// Prime factors from 17 to 61 (to 107 beside other factors, max_direct) are direct stages, behind the
// others: an output pair (q, p - q) sums the (p - 1) / 2 input pairs (k, p - k) against the table w_p^t.
// The last stage takes them from LDS to global memory; a length with two or three such factors runs the
// earlier ones from one LDS buffer to a second one.
//
// Lines of len points whose length has a larger prime factor run as a chirp convolution (Bluestein,
// 1970): j k = (j^2 + k^2 - (k - j)^2) / 2, so X_k = c_k sum_j (x_j c_j) conj(c_{k-j}) with c_j =
// exp(-i pi j^2 / len), a cyclic convolution of n >= 2 len - 1 points, n with radices up to 16.  The
// stages above transform x_j c_j, the last one multiplies by the transform of conj(c) (in position
// order, times 1 / n) and conjugates, and the transposed stages S-1 ... 0 lead back to natural order.
enum : int { kMixedStages = 6 };
// Radices up to kLightRadix, all up to 16, and 3, 5, 7 and 9 with exact constants of radix 9.
enum : int { kSetLight = 0, kSetFull = 1, kSetOdd = 2 };
struct mixed_plan {
    int n, nst;
    int len;                         // points of a line (n, unless chirp)
    int chirp, direct;               // direct: number of direct stages
    int set;                         // build of the kernels that runs it (kSetLight, ...)
    int spread;                      // one-stage lengths: elementwise load and store (set by a launch)
    int log2t, pitch, pad;           // lines per tile 2^log2t, LDS strides (elements)
    int radix[kMixedStages];
    int m0;                          // the first stage's twiddles w_n^{j q}: table[j (r_0 - 1) + q - 1]
    int last;                        // r_{S-1}
    int postoff;                     // real-data twiddles (modes other than kModeC2C)
    int root0, root_last;            // w_p^t, t < p, of a direct first and last stage
    int chirpoff;                    // c_j, j < len, then the transform of conj(c) in position order
    fast_div by_r[kMixedStages];     // / r_s
    fast_div by_m0, by_last;         // / m_0, / (n / r_{S-1})
    fast_div by_n, by_ncol, by_nb1;  // line and element numbering
};

// Stages 1 to S - 1 of the plan, at the start of its device table (kMixedHead bytes; the twiddles
// follow): the kernel walks them with a run-time index, which a kernel argument would not allow
// without a copy to scratch memory.
struct mixed_stage {
    int radix, m, twoff;
    fast_div by_m, by_k0;            // / m_s, / (r_1 ... r_{s-1}): block number -> k_0
    int root;                        // w_r^t, t < r, of a direct stage
};
enum : int { kMixedHead = 192 };
static_assert(sizeof(mixed_stage) * (kMixedStages - 1) <= kMixedHead, "the stages fit the table head");

// Fused pass over the two fastest axes of a box (fft_plane): planes of n0 x n1 elements back to back,
// `planes` of them per block, the same layout on both sides.
struct plane_args {
    const void *in;
    void *out;
    const void *mul;              // as pass_args::mul
    const void *tw0, *tw1;        // runtime-length tables of n0 and n1
    mixed_plan g0, g1;            // their radix plans (tile fields unused)
    int n0, n1, nplanes, planes;
    int rp, ps;                   // LDS strides of rows and planes (elements); rp is odd
    unsigned rows, cols;          // planes n1, planes n0
    fast_div by_rows, by_cols, by_n0;
    int conj;
    double scale;
};

// Batched mixed-size transforms (one phase = one axis of every transform).
// Every transform is a c2c box in order (0, 1, 2) at its own element offset.
struct batch_xform {
    long long in_off, out_off;  // element offsets from the batch's input / output base
    int n[3];
    int size_id[3];             // index of the radix plan of each axis length
};

struct batch_item {
    int xform;  // transform
    int tile;   // tile of lines along the phase axis
};

// How the fused phases run one transform: planes per x-y work item, columns per z work item.
struct batch_fused {
    int planes, width;
    fast_div by_rows, by_cols, by_n0, by_width;
};

struct batch_args {
    const void *in;
    void *out;
    const void *tw;               // concatenated twiddle tables of every length
    const batch_xform *xforms;
    const batch_item *items;
    const generic_plan *plans;    // one per distinct length
    const int *twoff;             // table offset (complex units) of each length
    const int *kid;               // compile-time tile of each length (-1: runtime radix plan)
    int nitems;
    int axis;       // 0, 1 or 2
    int from_in;    // 1: read the input arrays (first phase), 0: read the output arrays in place
    int conj;       // backward transform
    int scaling;    // 0 none, 1 full (1/N of each transform), 2 symmetric; applied by the last phase
    // fused phases: one entry per transform; runtime-length radix plans and tables (byte offsets into
    // mtab) of each length
    const batch_fused *fused;
    const mixed_plan *mplans;
    const unsigned char *mtab;
    const int *mtoff;
};

}  // namespace hmi
