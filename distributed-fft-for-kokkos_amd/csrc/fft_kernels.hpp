// Host-visible launch interface of the HIP kernels.
#pragma once

#include <hip/hip_runtime.h>

#include "device_common.hpp"

namespace dfft {

enum LineKind : int32_t { kC2C = 0, kR2C = 1, kC2R = 2 };

// One batched 1-D transform pass along logical axis `axis`: every line of the
// index space (all axes but `axis`) is read through descriptor `in`,
// transformed and written through `out`.  The two descriptors may describe
// different distributions (that is how the exchange between topologies is
// fused into the first and last pass of a plan).
struct LinePass {
  DDesc in, out;
  int32_t axis;
  int32_t nbatch;                       // ndim - 1
  int32_t batch_axis[kMaxDim - 1];      // slowest ... fastest
  int32_t batch_ext[kMaxDim - 1];
  FastDiv batch_div[kMaxDim - 1];
  int32_t nlines;                       // lines processed by this launch
  int32_t line_begin;                   // first line (index space of all lines)
  int32_t kind;                         // LineKind
  int32_t n;                            // transform length (real length for R2C/C2R)
  int32_t inverse;                      // 1: exponent +2 pi i jk/n
  int32_t lines_fast;                   // 1: consecutive lanes walk across lines
  int32_t lines_per_block;              // 0: launcher heuristic
  int32_t values_per_thread;            // 0: default (8); compile-time kernels exist for 4, 8, 16,
                                        // the runtime-radix kernel takes it as an upper bound
  int32_t line_bytes;                   // LDS bytes from a line's buffer to the next (set by launchers)
  int32_t fit_block;                    // 1: lines_per_block is a default the launcher may halve to fit
  const void* tw;                       // exp(-2 pi i e / n), e in [0, n), Real precision
  double scale;
  // 1: an R2C (forward) or C2R (inverse) pass on the power-of-two kernels with
  // 8 values per lane transforms two real lines per complex FFT (lines 2q and
  // 2q+1 of the pass); other lengths run real lines one by one
  int32_t paired;
  // pad_real > 0: batch axis pad_axis is enumerated over a padded extent
  // (batch_ext, the row pitch of a padded array) and lines whose index along
  // it is >= pad_real are skipped, so blocks of lines start on aligned rows
  int32_t pad_axis;
  int32_t pad_real;
  // 1: consecutive blocks step along the slower batch axes first (the block
  // grid, rows of blocks along the fastest batch axis, is walked column by
  // column), spreading concurrent blocks over more of the array
  int32_t swizzle;
  // 1: blocks are renumbered so each of the 8 XCDs (which take workgroups
  // round-robin) walks one contiguous range of lines
  int32_t xcd_remap;
  // 1: global loads and stores of the line data are nontemporal (streaming
  // arrays larger than the caches; measured 5-13 % faster per pass at 512^3)
  int32_t nontemporal;
  // 1 (FP64 fast kernels, FP32 ones of length >= 1024): the radix stages
  // exchange real parts, then imaginary parts, through a line buffer of
  // reals, halving the LDS of a line (more resident blocks per CU for a few
  // more barriers)
  int32_t split_lds;
  // 1 (FP32 C2C lanes-across-lines passes whose consecutive lines are
  // adjacent elements of one row): two lines per lane, one 16-byte access
  // per element pair; ignored where the lines are not adjacent
  int32_t dual_lines;
  // two-lines-per-lane passes only: bit 0 set when the input side's line
  // pairs are loaded as two 8-byte elements instead of one aligned 16-byte
  // pair -- an input with odd rows under a padded enumeration, whose pair at
  // a row's end has its second line in the padding (that element is then not
  // loaded)
  int32_t dual_split;
  // FP64 R2C passes only (pair kernel): 1 = the line of field f (array axis 0,
  // six fields) is the pointwise product u_I * u_J of two of
  // the three fields that the input descriptor holds along that axis, (I, J)
  // = (0,0) (0,1) (0,2) (1,1) (1,2) (2,2) for f = 0..5 -- the products of the
  // divergence-form Navier-Stokes right-hand side formed as the lines load
  int32_t products;
  // band > 0: a pass over the kept modes |k| <= band of a dealiased field
  // (FP64, band_pass_supported lengths; launch_band_pass).  Index i of batch
  // axis j stands for i + (i > band ? band_shift[j] : 0) (the kept indices of
  // a whole spectral axis wrap around), inverse lines read the positions
  // beyond the band as zeros, forward lines store none of them.
  int32_t band;
  int32_t band_shift[kMaxDim - 1];
  // Weight of the interior half-spectrum entries (0 < k < n/2) of an R2C /
  // C2R line, applied to the values a C2R line loads or an R2C line stores;
  // 0 means 1.  Adjoint transforms use 1/2 (C2R) and 2 (R2C).
  double herm_weight;
  // long_n1 > 0: lines too long for one LDS buffer, n = n1 * n2, run as two
  // launches through long_scratch (complex, nlines * n values): first the n2
  // sub-lines of stride n2 and length n1 of every line, each output k1
  // multiplied by exp(-2 pi i i2 k1 / n); then the n1 contiguous sub-lines of
  // length n2, whose output k2 is element k1 + n1 k2 of the line
  int32_t long_n1;
  const void* long_tw1;  // exp(-2 pi i e / n1)
  const void* long_tw2;  // exp(-2 pi i e / n2)
  void* long_scratch;
};

// The form of a line pass that the register kernels read (fast_pass).  A wave
// has to know its lines' addresses before it can issue its first load, and
// evaluating a DDesc costs some sixty dependent scalar loads and branches (a
// LinePass spans 26 cache lines), 4 to 6 us before the first line load.  Here
// the few fields of a side lie together, nothing branches on an axis, and a
// single-rank side is three strides.  Round trips, DDesc -> this: 64^3 C2C
// 42.5 -> 34 us, 50x42x36 R2C FP32 61 -> 51 us, 256^3 R2C FP64 336 -> 307 us,
// 384^3 R2C FP64 1.50 -> 1.32 ms, 1024^3 R2C FP64 20.5 -> 19.8 ms.
struct SideAxis {  // one storage axis of a multi-rank side; index 0 of extent 1 if unused
  int32_t sel0, sel1, sel2;  // all ones for the batch axis it holds, else 0 (line axis: none)
  int32_t base;              // ext / ntopo (line axis: 0)
  int32_t split;             // rem * (base + 1): indices below it lie in ranks one longer
  int32_t rem;
  int32_t rstride;
  uint32_t m_small, m_xor;   // multiplier of the division by base, and what turns it into that by base + 1
  uint32_t l_small, l_xor;   // likewise the shift
  int32_t line_len;          // of the line axis: its extent, else 0
  int64_t line_sel;          // all ones for the line axis
};
struct Side {
  char* ptr;          // single rank: its buffer
  int64_t stride[3];  // single rank: elements between neighbours along each batch axis
  int64_t line;       // single rank: elements between neighbours of a line
  int32_t multi;      // more than one rank
  int32_t shift;      // log2 of the element size in bytes
  SideAxis ax[kMaxDim];  // storage axes, fastest first
};
struct FastPass {
  int32_t nlines, line_begin, kind, n;
  int32_t inverse, lines_fast, lines_per_block, xcd_remap;
  int32_t swizzle, pad_real;  // pad_real: lines whose index along the fastest batch axis is >= it are padding
  int32_t band, dual_split;
  int32_t line_bytes;
  int32_t ext[3];         // batch axes, slowest first; unused ones come first with extent 1
  int32_t band_shift[3];
  FastDiv div[3];
  FastDiv bdiv;           // lines_per_block
  const void* tw;
  double scale, herm_weight;
  Side in, out;
  char* in_ptr[kMaxRanks];   // multi-rank sides only
  char* out_ptr[kMaxRanks];
};
FastPass fast_pass(const LinePass& p, bool fp64);

// Element-wise permuted copy between two distributions of the same logical
// array (one-GPU form of pack -> all-to-all -> unpack, and of local
// transposes).  Iterates the destination in its storage order.
struct RemapArgs {
  DDesc src, dst;
  int64_t total;
  int32_t iter_axis[kMaxDim];  // slowest ... fastest
  int32_t iter_ext[kMaxDim];
  FastDiv iter_div[kMaxDim];
};

// Grouped line pass (one launch for the same pass of many transforms, line
// lengths 16, 32, 64, 96, 128, 160, 256 in any mix).  kGroupThreads lanes per
// block; launches of contiguous lines (lanes along the line) may use fewer
// (64 or 128: smaller blocks, cheaper barriers, more blocks per CU).
constexpr int kGroupThreads = 256;
constexpr size_t kGenericLdsMax = 160 * 1024;  // LDS of one gfx950 workgroup
constexpr size_t kGroupLds = 64 * 1024;  // dynamic LDS of a grouped launch, at most
// lines per block, LDS bytes from line to line and dynamic LDS bytes of the
// grouped kernel for length n in blocks of `lanes` lanes (64, 128 or
// kGroupThreads, across the lines or along them) with at most lds_cap bytes of
// LDS per block; false if n has no grouped kernel
struct GroupShape {
  int lines_per_block = 0;
  int line_bytes = 0;
  size_t lds_bytes = 0;
};
bool group_line_shape(int n, bool fp64, size_t lds_cap, int lanes, bool across, GroupShape* g);
// the same for FP32 lines taken two per lane (false if n has no such kernel)
bool group_dual_shape(int n, size_t lds_cap, GroupShape* g);
// true if the staged instance is the better one for contiguous lines of n: a
// lane of more than 16 values leaves 8 lanes to a line, 64 bytes per access
// (fields of 160^3 there and back 1884 -> 1755 us); elsewhere its registers (168
// against 90) cost more than the wider accesses give (128^3 1304 -> 1366 us)
bool group_stage_pays(int n);
// true if two adjacent lines per lane apply to pass p with that many lines per
// block (FP32 C2C, lanes across lines, consecutive lines adjacent row
// elements on both sides, 16-byte aligned rank buffers; grouped passes)
bool dual_lines_apply(const LinePass& p, int lines_per_block);
// grid of the persistent grouped launch: resident blocks of the whole device
int group_grid(size_t lds_bytes, bool fp64, bool dual, int lanes);
// dual: the launch holds only members with dual_lines set (FP32, kGroupThreads
// lanes); lanes: lanes per block of a one-line launch; stage (FP32 one-line):
// contiguous aligned lines move 16 bytes per lane through LDS
hipError_t launch_group_pass(const FastPass* items, const int32_t* first_block, int count, int total_blocks,
                             int grid, size_t lds_bytes, bool fp64, bool nontemporal, bool dual, int lanes,
                             bool stage, hipStream_t s);
bool has_fast_line_kernel(int n);
// true if a line of length n runs as one pass: the fast set, or the generic
// kernel (one line of n complex values, twice, in at most 160 KB of LDS)
bool line_length_single_pass(int n, bool fp64);
// n1 of a two-pass split n = n1 * n2 with both factors single-pass lengths
// (the divisor nearest sqrt(n), n1 <= n2), 0 if n has none
int long_line_split(int n, bool fp64);
// single pass or a two-pass split
bool line_length_supported(int n, bool fp64);
// true where the plan runs length n by Bluestein's algorithm: no other kernel
// runs it, or a measured cost model puts Bluestein well below the generic
// kernel (large prime factors)
bool bluestein_preferred(int n, bool fp64);
hipError_t launch_line_pass(const LinePass& p, bool fp64, hipStream_t s);
// Bluestein steps of pass p over an (nlines, 2^log2m) complex scratch (see
// fft_kernels.hip); chirp: exp(-pi i e / n), e in [0, 2n), FP64; filt: the
// m-point transform of the chirp filter divided by m, FP64
hipError_t launch_bluestein_pre(const LinePass& p, int log2m, const void* chirp, void* s1, bool fp64, hipStream_t s);
hipError_t launch_bluestein_mul(int64_t total, int log2m, const void* filt, void* buf, bool fp64, hipStream_t s);
hipError_t launch_bluestein_post(const LinePass& p, int log2m, const void* chirp, const void* s1, bool fp64,
                                 hipStream_t s);
// an FP64 R2C pass with p.products set (paired lines, lengths 8..1024 powers
// of two); hipErrorNotSupported for other passes
hipError_t launch_products_pass(const LinePass& p, hipStream_t s);
bool products_pass_supported(int n);
// a pass with p.band set (and products, if set too): C2C lines, R2C / C2R
// lines (of a power of two in pairs), undistributed line axis
hipError_t launch_band_pass(const LinePass& p, hipStream_t s);
bool band_pass_supported(int n);
hipError_t launch_remap(const RemapArgs& a, int esize, hipStream_t s);

// Reference-exact pack/unpack of one rank's local array (mapped by `map`)
// into/out of a (P, e_0..e_{D-1}) LayoutRight buffer, or, with layout_left,
// a LayoutLeft array into/out of an (e_0..e_{D-1}, P) LayoutLeft buffer.
struct PackArgs {
  int32_t ndim;
  int32_t layout_left;
  int32_t nprocs;
  int32_t axis;           // logical axis split (pack) / merged (unpack)
  int32_t merged_size;    // local extent of that axis
  int32_t map[kMaxDim];
  int64_t local_ext[kMaxDim];   // storage extents of the local array
  int64_t buf_ext[kMaxDim + 1]; // (P, e_0..e_{D-1}), or (e_0..e_{D-1}, P) with layout_left
  int64_t total;                // elements of the buffer
  const char* src;
  char* dst;
};
hipError_t launch_pack(const PackArgs& a, int esize, bool unpack, hipStream_t s);

// Device-local all-to-all of P buffers of shape (P, block): recv[q][p] = send[p][q].
struct All2AllArgs {
  int32_t nprocs;
  int64_t block_bytes;
  const char* send[kMaxRanks];
  char* recv[kMaxRanks];
};
hipError_t launch_all2all(const All2AllArgs& a, hipStream_t s);

}  // namespace dfft
