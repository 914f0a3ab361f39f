// Plan runtime: the one-GPU replacement of the reference's SlabPlan /
// PencilPlan / SharedPlan behind the InternalPlan boundary
// (KokkosFFT_Distributed_InternalPlan.hpp:22-143).
#pragma once

#include <hip/hip_runtime.h>

#include <map>
#include <memory>
#include <string>
#include <vector>

#include "dfft.h"
#include "fft_kernels.hpp"
#include "planner.hpp"
#include "vendor.hpp"

namespace dfft {

struct PassSpec {
  int axis;
  int kind;  // LineKind
  int n;     // transform length
  // launch shape (0 / -1: Plan::default_shape); set by options or the autotuner
  int lines_per_block = 0;
  int values_per_thread = 0;
  int lines_fast = -1;
  int nontemporal = -1;  // -1: by shape
  int paired = 1;        // R2C / C2R: two real lines per complex FFT where the length has such a kernel
  int xcd = -1;          // XCD-contiguous block numbering (-1: by shape)
  int swz = 0;           // column-major walk of the block grid
  int split = 1;         // exchanges in real / imaginary halves (half the LDS; FP64, FP32 n >= 1024)
  int dual = 1;          // FP32 C2C: two adjacent lines per lane (16-byte accesses) where they apply
  int lin = 1;           // passes that write the user's arrays enumerate real lines only (0: padded scratch rows)
};

// device table exp(-2 pi i e / n), e in [0, n): evaluated in long double,
// rounded once to FP64 (both precisions form butterfly powers from it in FP64)
void* upload_twiddles(int n);

class Plan {
 public:
  explicit Plan(const dfft_desc& d);
  ~Plan();
  Plan(const Plan&) = delete;
  Plan& operator=(const Plan&) = delete;

  void execute(void* const* in, void* const* out, int direction, hipStream_t stream);
  // throws DFFT_ERROR_MISMATCH unless every rank's in/out allocation can hold
  // the local array that execute(direction) reads/writes (checked at the C
  // boundary; internal callers pass the plan's own buffers)
  void check_buffers(void* const* in, void* const* out, int direction) const;
  // adjoint of execute(direction) under the real inner product Re sum conj(a) b
  // of each side: in has the shape of that direction's output, out of its input
  void execute_adjoint(void* const* in, void* const* out, int direction, hipStream_t stream);
  // Dealiased fields (4-D views, field axis first and not distributed, R2C
  // over axes 1..3): only modes |k| <= cut along each axis are kept.
  // band_supported: FP64, fused executor, LayoutRight, power-of-two lengths
  // 8..1024 (their real lines run in pairs whatever the plan's own passes do)
  // and even 2^a 3^b 5^c from 36 to 384 (one by one).  execute_band(FORWARD) writes the kept modes
  // of the spectra and leaves the others as they are; execute_band(BACKWARD)
  // transforms spectra whose other modes count as zeros, whatever the arrays
  // hold there.  Same results as execute on the masked spectra.
  // packed: the spectral side is one array of all ranks in the layout of the
  // plan's scratch (its one pointer first in the table): (fields, n, n,
  // band_row(cut)) elements, entry (f, x, y, z) of the global spectrum at that
  // index, nothing beyond the cutoff touched.
  bool band_supported(int cut) const;
  static int32_t band_row(int cut) { return (cut + 8) / 8 * 8; }
  void execute_band(void* const* in, void* const* out, int direction, int cut, bool packed, hipStream_t stream);
  // Forward execute of a 6-field R2C plan over such views whose input fields
  // are the products u_i u_j of the 3 velocity fields in `u3` (per rank: 3
  // fields shaped like the plan's input blocks), (i, j) = (0,0) (0,1) (0,2)
  // (1,1) (1,2) (2,2): the products are formed as the first (R2C) pass loads
  // its lines, so the 6 product fields are never stored.  cut > 0: as
  // execute_band.  products_supported(cut) says whether this plan can (FP64,
  // fused executor, an R2C first pass of a power-of-two length 8..1024, or with
  // cut > 0 band_supported).
  bool products_supported(int cut) const;
  void execute_forward_products(void* const* u3, void* const* out, int cut, bool packed, hipStream_t stream);
  // execute with a HIP event pair around every launch; durations in ms
  std::vector<float> execute_timed(void* const* in, void* const* out, int direction, hipStream_t stream);
  int num_passes(int direction) const;
  // tuning knobs: "chunk" (planes per chunk of the first two passes, 0 = off),
  // "pad" (scratch rows padded to 128-byte multiples: -1 auto, 0 off, 1 on),
  // "fwd.<i>.lpb|vpt|lf|nt|pair|xcd|swz|split|dual|lin", "bwd.<i>.…" (lines
  // per block, values per thread, lanes-across-lines, nontemporal accesses,
  // two real lines per complex FFT in an R2C / C2R pass of a power of two
  // with 8 values per thread, XCD-contiguous
  // blocks, column-major block walk, LDS exchanges in real/imaginary halves,
  // two adjacent FP32 lines per lane, the last pass enumerated over the real
  // elements) of pass i
  void set_option(const std::string& key, long value);
  long get_option(const std::string& key) const;
  // measure candidate launch shapes and chunk sizes on the caller's arrays
  // (their contents are overwritten) and keep the fastest
  void autotune(void* const* in, void* const* out, hipStream_t stream);
  // the same for the passes of execute_band on a packed spectral side (contents
  // are overwritten), whose launch shapes are kept apart
  void autotune_band(void* const* in, void* const* out, int cut, hipStream_t stream);

  const std::string& name() const { return name_; }
  std::size_t nranks() const { return P_; }
  const Vec& in_local(std::size_t r) const { return in_local_.at(r); }
  const Vec& out_local(std::size_t r) const { return out_local_.at(r); }
  void local_starts(std::size_t r, int which, Vec& ext, Vec& st) const;
  const std::vector<BlockAnalyses>& analyses() const { return analyses_; }
  std::size_t max_buffer_size() const { return max_buffer_size_; }
  std::size_t workspace_bytes() const { return workspace_bytes_; }

 private:
  void allocate();
  void release();
  DDesc user_desc(const Vec& ext, const Vec& topo, Layout tl, void* const* ptrs) const;
  // the plan scratch holding an array of extents `ext` with elements of
  // `elem_bytes` bytes; LayoutRight rows are padded to 128-byte multiples
  DDesc scratch_desc(const Vec& ext, void* p, std::size_t elem_bytes) const;
  std::size_t scratch_elems(const Vec& ext, std::size_t elem_bytes) const;  // incl. padding
  LinePass make_pass(const PassSpec& s, const DDesc& in, const DDesc& out, bool inverse, double scale,
                     int slow_axis = -1) const;
  // restricts pass i of a direction to the kept modes
  void band_pass(LinePass& p, std::size_t i, bool forward, int cut) const;
  static void packed_stores(LinePass& p, const PassSpec& s);
  DDesc band_array(int cut, void* p) const;
  // launch shape of a pass where its spec leaves it open
  void default_shape(LinePass& p, const PassSpec& s) const;
  float time_direction(void* const* in, void* const* out, bool forward, hipStream_t s, int reps);
  void plan_fused();
  void run_fused(void* const* in, void* const* out, bool forward, hipStream_t s);
  void run_blockwalk(void* const* in, void* const* out, bool forward, hipStream_t s);
  const void* twiddles(int n) const;
  double norm_scale(bool forward) const;
  double exec_scale(bool forward) const { return adj_scale_ >= 0.0 ? adj_scale_ : norm_scale(forward); }

  dfft_desc d_{};
  TopologyType kind_ = TopologyType::Shared;
  std::string name_;
  std::size_t P_ = 1;
  std::size_t rank_ = 3;
  Vec gin_, gout_, axes_, in_topo_, out_topo_, fft_extents_;
  Layout in_tl_ = Layout::Right, out_tl_ = Layout::Right, view_layout_ = Layout::Right;
  bool real_ = false, fp64_ = true;
  int device_ = 0;
  std::vector<Vec> in_local_, out_local_;
  std::vector<BlockAnalyses> analyses_;
  std::size_t max_buffer_size_ = 0;
  void* scratch_ = nullptr;
  // lines longer than one LDS buffer: complex scratch of the two-launch
  // transform (nlines * n values of a pass)
  void* long_scratch_ = nullptr;
  std::size_t long_bytes_ = 0;
  // lengths with a prime factor beyond one LDS line: Bluestein through two
  // m-point transforms of an (nlines, m) scratch pair
  struct Bluestein {
    int m = 0, log2m = 0;
    void* chirp = nullptr;  // exp(-pi i e / n), e in [0, 2n), FP64
    void* filt = nullptr;   // m-point transform of the chirp filter / m, FP64
  };
  std::map<int, Bluestein> blue_;
  void* blue_s_[2] = {nullptr, nullptr};
  std::size_t blue_bytes_ = 0;
  void setup_bluestein(int n, std::size_t max_lines);
  LinePass dense_pass(int rows, int m, void* src, void* dst, bool inverse, bool fp64) const;
  // a line pass through the kernel its length needs (Bluestein included)
  hipError_t launch_pass(const LinePass& p, hipStream_t s);
  std::vector<void*> walk_bufs_[2];  // block-walk ping-pong local arrays per rank
  std::unique_ptr<VendorFFT> vendor_;  // DFFT_EXEC_VENDOR: rocFFT over the gathered global array
  std::size_t workspace_bytes_ = 0;
  std::map<int, void*> tw_;
  std::vector<PassSpec> fwd_, bwd_;
  std::vector<PassSpec> band_fwd_, band_bwd_;  // launch shapes of the passes over kept modes
  int chunk_[2] = {0, 0};  // planes per chunk, forward / backward (0 = no chunking)
  int pad_ = -1;           // scratch row padding: -1 auto (<= 1/16 extra), 0 off, 1 on
  // set only while execute_adjoint runs: scale of the adjoint direction and
  // the interior half-spectrum weight of its R2C / C2R line pass
  double adj_scale_ = -1.0;
  double adj_herm_ = 0.0;
  // timing hooks (set only by execute_timed)
  std::vector<hipEvent_t>* timing_ = nullptr;
  void mark(hipStream_t s);
};

}  // namespace dfft
