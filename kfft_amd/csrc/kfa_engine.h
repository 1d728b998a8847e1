// Host side of the gfx950 transform engine: plans, device tables, execution.
//
// A Plan1D computes batched 1D complex DFTs of one length in one precision.
// Its shape is chosen at plan time:
//   Direct    one LDS pass (length fits a workgroup's LDS, all radices <= 31)
//   FourStep  N = N1*N2: column pass of length N1 with the W_N^(n2 k1) twiddle
//             fused into its store, then a row pass of length N2 whose store
//             writes the transposed (natural-order) result
//   Rader     prime N: gather x[g^n] fused into a forward FFT of N-1, then an
//             FFT of N-1 whose load multiplies by the precomputed FFT(b) and
//             whose store scatters to X[g^-m] adding x[0]
//   Bluestein anything else: chirp-multiplied, zero-padded FFT of a smooth
//             M >= 2N-1, pointwise product with FFT(chirp kernel), FFT back,
//             chirp-multiplied truncated store
// Direction is chosen per call; the inverse is conj(F(conj(x))), applied by the
// first pass's load and the last pass's store.  Twiddles, chirps and Rader
// kernels are generated on the GPU in double precision and rounded once.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <functional>
#include <memory>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "kfa_common.h"

namespace kfa {

// --------------------------------------------------------------------- runtime
void set_error(const std::string& msg);
const char* last_error();
bool hip_ok(hipError_t e, const char* what);
hipStream_t default_stream();
bool runtime_init();
// While set on the calling thread, executions allocate nothing: the two-pass
// path runs its groups on the caller's stream only (no second stream or
// events) and the fused FP64 on-chip kernel (which owns buffers) is not used.
void set_no_alloc(bool on);
bool no_alloc();
// The radix-16 arithmetic (KFA_FAST_MFMA_* bits, 0: vector units) of every
// execution on the calling thread that does not choose its own (Fuse::dft):
// set by the entry points of plans created with a split-operand flag.
void set_split_dft(uint32_t dft);
uint32_t split_dft_default();

// device bytes held by every DevBuf of the process
size_t device_bytes_held();
// what the device memory budget leaves (no budget: SIZE_MAX)
size_t device_room();

struct DevBuf {
    void* p = nullptr;
    size_t bytes = 0;
    DevBuf() = default;
    DevBuf(const DevBuf&) = delete;
    DevBuf& operator=(const DevBuf&) = delete;
    ~DevBuf();
    bool alloc(size_t n);  // exact size, contents undefined
    bool ensure(size_t n); // grow-only
    void release();
};

// A read-only device table shared by every plan that needs the same one (stage
// twiddles by length and radices, four-step factors by length): plans of a ragged
// batch's thousands of lengths then read a few tables that stay in the caches.
struct SharedTab {
    std::shared_ptr<DevBuf> buf;
    void* p = nullptr;
    // the table of (kind, a, b), made by `make` (allocation and launches on the
    // default stream, complete when this returns) unless some plan holds it
    bool get(uint32_t kind, uint32_t a, uint32_t b, const std::function<bool(DevBuf&)>& make);
};

// ------------------------------------------------------------------ addressing
// How instance b and element e of a transform's input or output are addressed
// (see KfaIo): b_lo = b % C, b_hi = b / C,
//   address = b_hi*dist_hi + b_lo*dist_lo + e*stride.
struct Layout {
    void* ptr = nullptr;
    int64_t dist_hi = 0, dist_lo = 0, stride = 1;
    uint32_t C = 1;
    uint32_t flags = 0; // KFA_IO_REAL / KFA_IO_REAL_PAIRS
    const int64_t* inst = nullptr; // device table of instance offsets (replaces dist_hi)
    // output side: super twiddles of a real-input rebuild fused into the store
    // (the transform is the half-length complex FFT of a real-input forward; the
    // output holds n/2+1 bins).  Only where Plan1D::fuses_real_post().
    const void* real_post = nullptr;
    // input side: inverse super twiddles of the inverse rebuild fused into the load
    // (bins 0..n of each row).  Only where Plan1D::fuses_real_pre().
    const void* real_pre = nullptr;
};

// Extra operations a caller fuses into a transform (used by the real-FFT,
// convolution and 2D layers).
struct Fuse {
    const void* pw_in = nullptr; // pointwise multiply on load, same layout as the input
    bool pw_in_f64 = false;
    bool onchip = false;         // allow the fused on-chip two-pass kernel
    uint32_t dft = 0;            // KFA_FAST_MFMA_F16 / _BF16: split-operand radix-16 stages
};

// -------------------------------------------------------------- LDS pass plans
struct LdsPass {
    uint32_t L = 0;
    int prec = 8; // bytes per real component
    int maxe = 16;
    uint32_t tpi = 0, nstages = 0, inst_stride = 0;
    uint32_t tw_count = 0; // stage twiddle entries (sum over stages s >= 1 of ns (R - 1))
    KfaStage st[KFA_MAX_STAGES] = {};
    SharedTab tw; // stage twiddles

    bool plan(uint32_t L, int prec, uint32_t max_radix = 16);
    // the stages and their twiddles only (for shaped passes of lengths beyond the
    // general pass)
    bool plan_stages(uint32_t L, int prec, uint32_t max_radix = 16);
    uint32_t pick_ipw(bool jfast) const;
    uint32_t lds_bytes(uint32_t ipw) const;
};

// Radix list for L (empty when L has a prime factor > 31).  max_radix below 16
// fuses fewer radix-2 levels per stage (8s or 4s) and splits 9s into 3s;
// KFA_MAXR_SPLIT (plans of the split-operand precision form) prefers radix 16
// wherever the power of two allows one (2^5 as 16 x 2 rather than 8 x 4), for
// lengths that are not powers of two (those run the shaped passes' order).
constexpr uint32_t KFA_MAXR_SPLIT = 32;
std::vector<uint32_t> radix_list(uint32_t L, uint32_t max_radix = 16);
bool lds_capable(uint32_t L, int prec);

class Plan1D;

// A smooth length executed as one LDS pass, a four-step pair of passes, or
// (lengths beyond a pair) three passes: a column pass of N1 followed, per
// transform, by an inner two-pass plan of N2 with a transposed store.
struct SubFft {
    uint32_t L = 0;
    int prec = 8;
    bool four = false;
    bool three = false;
    std::shared_ptr<Plan1D> inner; // three passes: the plan of the rows (length N2)
    uint32_t maxr = 16; // radix cap of the passes (16: the default radices)
    LdsPass direct;
    uint32_t N1 = 0, N2 = 0; // four-step: column length N1, row length N2
    LdsPass col, row;
    LdsPass big; // stages of the long one-pass row form (big.L == 0: none), which plain
                 // rows take; everything else takes the form above
    SharedTab tw4_hi, tw4_lo; // W_L^(hi S) and W_L^lo, FP64 (S = 2^tw4_shift)
    uint32_t tw4_shift = 0;
    SharedTab tw4_full; // W_L^m, m < L, compute precision (fast four-step passes)
    // with the tables of the real rebuilds (a convolution's inner transform has none)
    bool rebuilds = true;
    // real-input rebuild fused into pass B (power-of-two halves): W_2L^a, a < N1,
    // and W_2N2^e, e <= N2, compute precision
    SharedTab rp_row, rp_elem;
    // inverse rebuild fused into pass A's load: W_2N1^n1, n1 < N1, in two parts, and
    // W_2L^n2 - 1, n2 < N2 (two-pass lengths with a compiled column form, N1 = 64 to 1024)
    SharedTab rq_row, rq_col;
    // pass A's store twiddle from the two short tables instead of tw4_full
    // (lengths whose full table exceeds 1 MiB); FP32 copies of tw4_hi / tw4_lo
    bool tw4_split = false;
    SharedTab tw4s_hi, tw4s_lo;
    bool mixed_four = false; // a shaped two-pass form with a mixed-radix half

    bool plan(uint32_t L, int prec, bool force_four = false, uint32_t max_radix = 16);
    // scratch (in complex elements) needed for `batch` instances
    size_t scratch_elems(uint64_t batch) const;
    // Run with fully described first-load and last-store descriptors.  For
    // four-step the load/store must have C == 1 (contiguous instances).
    // `dft` (KFA_FAST_MFMA_* bits) selects the radix-16 arithmetic of the fast passes
    hipError_t run(const KfaIo& load, const KfaIo& store, double scale, double scale_post,
                   uint64_t batch, void* scratch, hipStream_t s, bool onchip = false,
                   uint32_t dft = 0) const;
    hipError_t run_big(const KfaIo& load, const KfaIo& store, double scale, uint64_t batch,
                       hipStream_t s) const;
    hipError_t run_four_fast(const KfaIo& load, const KfaIo& store, double scale, uint64_t batch,
                             void* scratch, uint32_t nt, hipStream_t s, uint32_t dft) const;
    // three passes over plain contiguous complex instances (conjugation on the
    // load, conjugation and scaling on the store)
    hipError_t run_three(const KfaIo& load, const KfaIo& store, double scale, uint64_t batch,
                         void* scratch, hipStream_t s, uint32_t dft) const;
    // y = IDFT(DFT(x) * h), unnormalised, with the load's / store's element
    // operations (the store's CONJ1 completes the inverse): one pass, or three
    // for four-step lengths, where hperm holds h[k1 + N1 k2] at [k1][k2] and
    // scratch holds batch x L values.  dc_out: the last pass also stores Rader's
    // X[0] (hipErrorNotSupported, with nothing stored, where it cannot)
    hipError_t run_conv(const KfaIo& load, const KfaIo& store, double scale, double scale_post,
                        uint64_t batch, const void* h, const void* hperm, void* scratch,
                        hipStream_t s, void* dc = nullptr, uint32_t dft = 0,
                        bool dc_out = false) const;
    // both passes on columns of row-major matrices (C = columns, dist_lo = 1): the
    // shaped column passes walk the columns with the lanes
    hipError_t run_four_cols(const KfaIo& load, const KfaIo& store, double scale, uint64_t batch,
                             void* scratch, uint32_t nt, hipStream_t s, uint32_t dft) const;
    // fused on-chip variant of the two passes (N1 == N2 == 256, library stream only)
    hipError_t run_fused(const KfaIo& load, const KfaIo& store, double scale, uint64_t batch,
                         hipStream_t s) const;
    // non-zero if a fused launch since the last check timed out waiting (syncs the stream)
    int fused_error() const;
    // shaped two-pass form whose transposing pass can hold rows k1 and N1 - k1 in
    // one workgroup (the real-input rebuild fused into its store, KFA_IO_RPOST)
    bool rpost_two_pass() const;
    mutable std::mutex fused_mu;
    mutable DevBuf fused_ctr, fused_ring;
    mutable uint64_t fused_T = 0;
    mutable bool fused_used = false;

    // Single-pass form of L = 65536 in FP32 (kfa_pair_impl.h): pairs of
    // workgroups on one XCD exchange a quarter of the data through L2, so the
    // intermediate never makes an HBM round trip.  Tables: W_L^(k1 m) [32][2048]
    // and the step-B twiddles; err: sticky error word of the launches.
    bool pair = false;
    DevBuf pair_tw4, pair_twb, pair_err;
    mutable std::atomic<bool> pair_used{false}; // a launch since the last error check
    // pairs of a launch over `batch` transforms (0: the form does not apply)
    uint32_t pair_count(uint64_t batch) const;
    size_t pair_scratch_bytes(uint64_t batch) const;
    hipError_t run_pair(const KfaIo& load, const KfaIo& store, double scale, uint64_t batch,
                        void* scratch, hipStream_t s, uint32_t dft) const;
    // non-zero if a launch since the last check left its error word set (syncs the device)
    int pair_error() const;
};

// XCDs that host workgroups of an ordinary grid (probed once with XCC_ID), 0
// when the mapping cannot be established; the fused path's queue count (0 when
// KFFT_AMD_FUSED=0); compute units of the device
uint32_t xcd_queues();
uint32_t fused_queues();
uint32_t num_cus();

// a one- or two-pass plan (three_ok: or three passes) exists for L
bool subfft_capable(uint32_t L, int prec, bool three_ok = true);

// Bluestein's convolution length for n: the smallest 2,3,5-smooth length from
// 2n - 1 with a plan, or (pow2) the smallest power of two
uint32_t blue_length(uint32_t n, int prec, bool pow2);

enum class Kind { Identity, Direct, Rader, Bluestein };

// Plan shape choices beyond the default (the autotuner's search space):
// maxr caps the radix of the LDS stages (stage fusion: 16, 8 or 4), four forces
// the two-pass four-step form where a one-pass plan would fit.
struct PlanVariant {
    uint32_t maxr = 16;
    bool four = false;
    bool pow2_m = false; // Bluestein: a power-of-two convolution length (else 2,3,5-smooth)
    uint32_t key() const { return maxr | (four ? 0x100u : 0u) | (pow2_m ? 0x200u : 0u); }
};

// the plan shape of an ordinary (not ragged) transform of n points
PlanVariant default_variant(uint32_t n, int prec);

class Plan1D {
  public:
    Plan1D(uint32_t n, int prec, PlanVariant v = PlanVariant()) : n_(n), prec_(prec), var_(v) {}
    bool build();
    uint32_t n() const { return n_; }
    int prec() const { return prec_; }
    Kind kind() const { return kind_; }
    // `onchip`: describe the form a KFFT_FLAG_GPU_ONCHIP plan runs
    const char* describe(bool onchip = false) const;

    // scratch bytes for a batch of `batch` instances
    size_t scratch_bytes(uint64_t batch) const;
    // what a batch counts against a fixed amount of scratch: as scratch_bytes, Bluestein
    // at its shortest convolution length, whichever one the plan runs
    size_t scratch_charge(uint64_t batch) const;
    // the largest equal groups a batch splits into whose scratch_bytes stay within `room`
    // (one transform at least)
    uint64_t group_within(uint64_t batch, size_t room) const;
    // Execute `batch` transforms.  `scale` multiplies every output (1/N for a
    // normalised inverse).  Column layouts (C > 1) are supported by Direct and
    // by Rader/Bluestein whose inner length is Direct.
    hipError_t execute(const Layout& in, const Layout& out, uint64_t batch, bool inverse,
                       double scale, void* scratch, hipStream_t s, const Fuse* fuse = nullptr) const;
    // column layouts (C > 1) with any fused element operations
    bool supports_columns() const;
    // column layouts of plain complex data (no real / mapped / pointwise element operations)
    bool supports_plain_columns() const;
    bool two_pass() const { return sub_.four || sub_.three; }
    bool three_pass() const { return sub_.three; }
    // points a transform moves through its passes (a convolution round counts twice)
    double work_points() const {
        const double inner = (double)std::max<uint32_t>(1, sub_.L);
        const double passes = sub_.three ? 3.0 : sub_.four ? 2.0 : 1.0;
        return inner * passes * (kind_ == Kind::Rader || kind_ == Kind::Bluestein ? 2.0 : 1.0);
    }
    // LDS bytes one instance of the plan's largest pass occupies
    size_t pass_inst_bytes() const;
    // one LDS pass over the whole transform: the real-input rebuild can be fused
    // into its store (Layout::real_post)
    bool fuses_real_post() const { return kind_ == Kind::Direct && !sub_.four && !sub_.three; }
    // a length whose (first) compiled pass has the inverse rebuild in its load
    bool fuses_real_pre() const;
    // outside the ragged executor, plain rows of this length run a shaped pass
    // (kfa_fast_impl.h), which has no fused rebuild
    bool shaped_rows() const;
    // shaped two-pass form with the rebuild fused into its second pass (plain
    // contiguous rows, outside the ragged executor)
    bool fuses_real_post_shaped() const { return kind_ == Kind::Direct && sub_.rpost_two_pass(); }
    int async_error() const {
        const int a = sub_.fused_error(), b = sub_.pair_error();
        return a ? a : b;
    }

  private:
    uint32_t n_;
    int prec_;
    PlanVariant var_;
    Kind kind_ = Kind::Identity;
    SubFft sub_;  // Direct: the transform; Rader: length n-1; Bluestein: length M
    uint32_t M_ = 0; // Bluestein: the convolution length
    mutable std::atomic<uint32_t> Mmin_{0}; // the shortest one
    DevBuf qidx_, pidx_, bhat_; // Rader
    DevBuf chirp_, hhat_;       // Bluestein
    DevBuf hperm_;              // four-step inner length: the FFT(h) / FFT(b) table at
                                // [k1][k2] holding index k1 + N1 k2 (convolution pass)
    mutable std::string desc_;

    hipError_t bluestein_steps(const Layout& in, const Layout& out, uint64_t batch, bool inverse,
                               double scale, void* scratch, hipStream_t s, uint32_t dft) const;
};

// -------------------------------------------------------------- plan registry
// Plans are cached by (n, precision) and shared; they are immutable after build.
std::shared_ptr<Plan1D> get_plan(uint32_t n, int prec, PlanVariant v = PlanVariant());

// Column convolution: b = scale * inverse DFT (unnormalised) of the columns' DFT(a)
// DFT(b), y rows of `cols` columns (row distance pitch) in one pass;
// hipErrorNotSupported where y is not compiled.  The table is the caller's to keep.
struct ColumnConv {
    uint32_t y = 0;
    int prec = 0;
    LdsPass pass;
    bool plan(uint32_t y, int prec); // false: not supported (or its table failed)
    // blocked: columns in blocks of four (KFA_IO_BLK4 rows), else rows of `pitch`
    hipError_t run(const void* a, void* b, bool blocked, uint64_t pitch, uint64_t cols,
                   double scale, hipStream_t s) const;
};

// Super twiddles of the real-input transform: st[i] = exp(-+ i pi ((i+1)/h + 1/2)).
bool make_real_twiddles(DevBuf& out, uint32_t h, int prec, bool inverse);

size_t elem_bytes(int prec); // bytes of one complex value

// ------------------------------------------------------------ ragged executor
// A batch of transforms of uneven lengths run as one persistent launch
// (kfa_ragged.hip).  Item kinds: complex (forward or inverse, n outputs) and
// real-input forward (n/2+1 outputs for even n, n for odd n).  Offsets are in
// bytes from the base pointers given to run().
enum { RAGGED_COMPLEX = 0, RAGGED_REAL = 1 };

struct RaggedItem {
    uint32_t n = 0, kind = RAGGED_COMPLEX;
    uint64_t in_off = 0, out_off = 0;
};

// plan shape of one length class: plan variant and largest instances per tile
// (0: the executor's default)
struct RaggedChoice {
    PlanVariant v;
    uint32_t ipw_cap = 0;
    bool operator==(const RaggedChoice& o) const {
        return v.key() == o.v.key() && ipw_cap == o.ipw_cap;
    }
};

// Default LDS budget of an executor workgroup: the LDS that lets as many
// workgroups stay resident per CU as the executor's registers do (three for
// FP32, two for FP64).
uint32_t ragged_lds_budget(int prec);

struct RaggedOptions {
    // LDS per workgroup that tiles and one-pass plans must fit (0: the default of
    // the precision, ragged_lds_budget)
    uint32_t lds_budget = 0;
    uint32_t ipw_cap = 0;            // largest instances per tile (0: as many as fit)
    uint32_t wgs_per_cu = 0;         // resident workgroups per CU (0: occupancy limit)
    uint32_t parts_per_queue = 4;    // split of the work of a queue into groups (balance)
    uint32_t lds_floor = 0;          // least dynamic LDS per workgroup (fixes the occupancy)
    bool graph = true;               // replay the launch sequence as a captured hipGraph
    // per-class choice (autotuner or cost model); default shapes when empty
    std::function<RaggedChoice(uint32_t n, uint32_t kind, uint32_t count)> choose;
};

// Cost-model inputs of one length class under one plan choice (COST_FEATURES
// values): exponents of 2, 3, 5, 7, {11, 13} and {17..31} in the inner
// transform length (the length itself, p - 1 for Rader, the choice's M for
// Bluestein), Rader and Bluestein flags, log2 of the length, the inner length
// and the batch, real input, FP64, the radix cap (one-hot 16 / 8 / 4), forced
// four-step, instances per tile, and whether the inner transform runs as one
// pass.  All scaled to about [0, 1].
constexpr int COST_FEATURES = 19;
// ln of the predicted speed-up a choice needs over the default shape before the
// tuned planner takes it (25%: the default shapes are close to the optimum of the
// choices, and smaller margins let prediction errors pick slower shapes)
constexpr float COST_MARGIN = 0.2231f;
// points that a class is timed with at least, and a batch ranked by the model holds
constexpr uint64_t COST_MIN_POINTS = 1ull << 22;
void cost_features(uint32_t n, uint32_t kind, uint32_t count, int prec, const RaggedChoice& c,
                   float* out);
// the choices the autotuner searches for one class, and whether one applies to
// a class (forced four-step needs a two-pass split of the inner length)
std::vector<RaggedChoice> tune_candidates();
// the plan shape of a class that nothing tuned (lds_budget 0: the executor's): what an
// untuned ragged plan runs and the tuner starts from
RaggedChoice ragged_default(uint32_t n, uint32_t kind, int prec, uint32_t lds_budget = 0);
bool choice_applies(uint32_t n, uint32_t kind, int prec, const RaggedChoice& c);
// Time `count` transforms of one class under one choice as a ragged batch: the
// class is replicated to at least 2^22 points and run at the occupancy of a
// mixed batch (68 KiB LDS per workgroup), so that it uses the GPU as it would
// inside a large batch, and the time is charged per `count` transforms
// (microseconds, best of `reps`), or a negative value when the choice does not
// apply to the length.
double tune_measure(uint32_t n, uint32_t kind, uint32_t count, int prec, const RaggedChoice& c,
                    uint32_t reps);

class RaggedPlan {
  public:
    RaggedPlan(int prec, bool inverse, bool norm) : prec_(prec), inverse_(inverse), norm_(norm) {}
    ~RaggedPlan();
    bool build(const std::vector<RaggedItem>& items, const RaggedOptions& opt);
    // asynchronous on s; in / out are device pointers
    hipError_t run(const void* in, void* out, hipStream_t s);
    // non-zero if the last run's dependency waits timed out (synchronises)
    int error();
    const char* describe() const { return desc_.c_str(); }
    size_t records() const { return nrec_; }
    size_t tickets() const { return ntick_; }

  private:
    int prec_;
    bool inverse_, norm_;
    RaggedOptions opt_;
    std::vector<std::shared_ptr<Plan1D>> plans_;
    std::vector<std::unique_ptr<DevBuf>> tables_; // real-FFT super twiddles
    DevBuf tbl_, scratch_, blob_, tq_, tq_off_, ctr_, patch_off_, patch_which_, patch_delta_;
    uint32_t nq_ = 0, nrec_ = 0, npatch_ = 0, lds_ = 0, groups_ = 0;
    size_t ntick_ = 0, ctr_words_ = 0;
    RagArgs args_ = {};
    hipGraph_t graph_ = nullptr;
    hipGraphExec_t exec_ = nullptr;
    hipStream_t cap_ = nullptr;  // capture stream (private, so no other work is captured)
    hipStream_t last_ = nullptr; // stream of the last run
    // completion of the last run: a run on any stream waits for it before it
    // patches the shared argument blob and clears the shared counters
    hipEvent_t done_ = nullptr;
    bool pending_ = false;
    const void* g_in_ = nullptr;
    void* g_out_ = nullptr;
    std::string desc_;
    std::mutex mu_;
    hipError_t enqueue(const void* in, void* out, hipStream_t s);
    hipError_t run_locked(const void* in, void* out, hipStream_t s);
};

} // namespace kfa
