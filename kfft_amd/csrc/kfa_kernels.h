// Host launchers of the gfx950 kernels (kfa_kernels.hip).  `prec` is the
// size in bytes of one real component: 8 (double) or 4 (float).
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "kfa_common.h"

namespace kfa {

#define KFA_RAG_THREADS 256 // threads per workgroup of the ragged executor
// bin pairs of a real-input rebuild per task (2048: 8 per thread; 256-pair tasks
// spent as long on their ticket, arguments and dependency wait as on the data)
#define KFA_RAG_POST_PAIRS 2048
// (log2 length, use) of the shaped tiles the executor holds: plain passes of every
// power of two up to 4096, Bluestein's one-pass convolutions from 64 and the three
// passes of its longer ones (64 x 128 to 512 x 512)
#define KFA_RAG_MIXES(X)                                                                           \
    X(4, KFA_USE_PLAIN) X(5, KFA_USE_PLAIN) X(6, KFA_USE_PLAIN) X(7, KFA_USE_PLAIN)                \
    X(8, KFA_USE_PLAIN) X(9, KFA_USE_PLAIN) X(10, KFA_USE_PLAIN) X(11, KFA_USE_PLAIN)              \
    X(12, KFA_USE_PLAIN) X(6, KFA_USE_ONE_BLUE) X(7, KFA_USE_ONE_BLUE) X(8, KFA_USE_ONE_BLUE)      \
    X(9, KFA_USE_ONE_BLUE) X(10, KFA_USE_ONE_BLUE) X(11, KFA_USE_ONE_BLUE)                         \
    X(12, KFA_USE_ONE_BLUE) X(6, KFA_USE_A1_BLUE) X(7, KFA_USE_A1_BLUE) X(8, KFA_USE_A1_BLUE)      \
    X(9, KFA_USE_A1_BLUE) X(6, KFA_USE_A2_BLUE) X(7, KFA_USE_A2_BLUE) X(8, KFA_USE_A2_BLUE)        \
    X(9, KFA_USE_A2_BLUE) X(6, KFA_USE_MID) X(7, KFA_USE_MID) X(8, KFA_USE_MID) X(9, KFA_USE_MID)

// The launches one plan execution would make, recorded instead of launched
// (the ragged executor turns them into tasks of one persistent launch).  While
// a recorder is current on the calling thread, launch_fft, launch_gather_first,
// launch_rader_dc and launch_real_post append their arguments; the planner
// avoids every other launcher.
struct RecOp {
    uint32_t type, prec, maxe, lds;
    uint64_t tiles; // workgroup tiles (FFT: fixed later from the executor's shape)
    uint32_t gx;
    std::vector<unsigned char> args;
};
struct Recorder {
    std::vector<RecOp> ops;
    hipError_t add(uint32_t type, int prec, int maxe, uint32_t lds, uint64_t tiles, uint32_t gx,
                   const void* args, size_t bytes);
};
Recorder*& recorder(); // current recorder of this thread (null: launch)

// dft: KFA_FAST_MFMA_F16 / _BF16 bits select the split-operand radix-16 stages
// of the FP32 pass (0: vector units; the FP64 pass ignores them)
hipError_t launch_fft(int prec, int maxe, const KfaFftArgs& a, uint32_t lds_bytes, hipStream_t s,
                      uint32_t dft = 0);
hipError_t launch_fft_f64(int maxe, const KfaFftArgs& a, uint32_t lds_bytes, hipStream_t s);
// the general pass of a compiled length (hipErrorNotSupported: not compiled, or
// a radix schedule other than the default one)
hipError_t launch_fft_ct_f64(const KfaFftArgs& a, uint32_t lds_bytes, hipStream_t s);
hipError_t launch_fft_ct_f32(const KfaFftArgs& a, uint32_t lds_bytes, hipStream_t s);
hipError_t launch_fft_f32(int maxe, const KfaFftArgs& a, uint32_t lds_bytes, hipStream_t s,
                          int dk);
// compile-time shaped power-of-two passes; mode: 0 row, 1 column, 2 row-in/column-out,
// 3 column with the inverse real rebuild in the load (64 to 1024 points)
hipError_t launch_fast_f64(uint32_t L, int mode, const FastArgs& a, hipStream_t s);
hipError_t launch_fast_f32(uint32_t L, int mode, const FastArgs& a, hipStream_t s);
// compile-time shaped mixed-radix row passes (kfa_mixed_impl.h) for the
// lengths of KFA_MIXED_LENGTHS; hipErrorNotSupported for any other length or
// for flags they do not take (split forms, real rebuild)
#define KFA_MIXED_LENGTHS(X)                                                                       \
    X(60) X(100) X(120) X(240) X(300) X(360) X(480) X(600) X(720) X(960) X(1000) X(1008) X(1200)   \
    X(1500) X(2000) X(2080) X(2400) X(3000) X(4000) X(4160) X(5000) X(6000)
// sub-lengths of two-pass transforms with the column (mode 1) and transposing
// (mode 2) forms as well
#define KFA_MIXED_SUB_LENGTHS(X)                                                                   \
    X(27) X(45) X(48) X(65) X(75) X(80) X(81) X(96) X(100) X(120) X(125) X(160) X(200) X(243)
// lengths whose general pass (every fused load / store operation, convolution
// rounds) also has a compiled stage schedule (launch_fft picks it where the
// pass's radices are the default ones)
#define KFA_GEN_LENGTHS(X) X(256) X(512) X(1024) X(2048) X(4096) X(1008) X(2080)
// lengths of the shaped pass behind the general pass's fused load / store
// operations and convolution rounds (launch_mixgen; hipErrorNotSupported for
// other lengths, other radix schedules or a real-input rebuild)
#define KFA_MIXGEN_LENGTHS(X)                                                                      \
    X(64) X(128) X(256) X(512) X(1024) X(2048) X(4096) X(1000) X(1008) X(2080) X(4160)
inline bool mixgen_len(uint32_t L, int prec) {
    switch (L) {
#define KFA_MIXGEN_CASE(N) case N:
        KFA_MIXGEN_LENGTHS(KFA_MIXGEN_CASE)
#undef KFA_MIXGEN_CASE
        return true;
    default:
        return prec == 4 && L == 8192;
    }
}
// those of them whose gathered and scattered passes are compiled for a two-pass Rader
// convolution, X[0] included: column lengths N1 <= N2, p - 1 = N1 N2 in the most square
// split (of the primes up to 2^22, 128 to 1024 occur).  Against the tile for all uses and
// two kernels around it, FP64: 256 (114689 x 146) 858 -> 776 us, 1000 (1008001 x 16) 1162
// -> 1137, 1008 (1032193 x 16) 1007 -> 973, the same in FP32 within 1%; left out, slower:
// 128 (17921 x 936) 610 and 661, 512 (262657 x 63) 1311 and 1350, FP32 883 and 916, 1024
// (1053697 x 15) 1028 and 1220.
constexpr bool rader_cols_len(uint32_t L) { return L == 256 || L == 1000 || L == 1008; }
hipError_t launch_mixgen_f64(const KfaFftArgs& a, hipStream_t s);
hipError_t launch_mixgen_f32(const KfaFftArgs& a, hipStream_t s);
// mode: 0 rows, 1 columns, 2 row-in / column-out (as launch_fast)
hipError_t launch_mixed_f64(uint32_t L, int mode, const FastArgs& a, hipStream_t s);
hipError_t launch_mixed_f32(uint32_t L, int mode, const FastArgs& a, hipStream_t s);
inline bool mixed_sub_len(uint32_t L) {
    switch (L) {
#define KFA_MIXED_CASE(N) case N:
        KFA_MIXED_SUB_LENGTHS(KFA_MIXED_CASE)
#undef KFA_MIXED_CASE
        return true;
    default:
        return false;
    }
}
// lengths with the shaped row pass (both lists)
inline bool mixed_len(uint32_t L) {
    switch (L) {
#define KFA_MIXED_CASE(N) case N:
        KFA_MIXED_LENGTHS(KFA_MIXED_CASE)
#undef KFA_MIXED_CASE
        return true;
    default:
        return mixed_sub_len(L);
    }
}
// lengths of the long one-pass rows (kfa_bigrow_impl.h): those that measured faster
// there from 256 rows on, two passes -> one, about 16 million points: FP64 5120
// 172 -> 128 us, 6144 212 -> 126, 6250 485 -> 164, 6400 187 -> 133, 6561 222 -> 160,
// 7680 223 -> 117, 8192 186 -> 121; FP32 10000 237 -> 146, 10240 187 -> 129, 15360
// 195 -> 142.  Left out: FP64 5000 and 6000 (one whole-value pass already: 164, 159
// and 145, 135, but 256 rows 18 and 22) and FP32 9600, 12000, 12288, 12500 and 16384
// (210, 177; 230, 284; 194, 170; 253, 246; 186, 179, and slower at 300 rows), whose
// rows leave few registers for two workgroups.  Other smooth lengths from 4097 on are
// not compiled and were not tried; they keep two passes.
#define KFA_BIGROW_F64(X) X(5120) X(6144) X(6250) X(6400) X(6561) X(7680) X(8192)
#define KFA_BIGROW_F32(X) X(10000) X(10240) X(15360)
hipError_t launch_bigrow_f64(const KfaFftArgs& a, hipStream_t s);
hipError_t launch_bigrow_f32(const KfaFftArgs& a, hipStream_t s);
inline bool bigrow_len(uint32_t L, int prec) {
    switch (L) {
#define KFA_BIGROW_CASE(N) case N:
        KFA_BIGROW_F64(KFA_BIGROW_CASE)
        return prec == 8;
        KFA_BIGROW_F32(KFA_BIGROW_CASE)
        return prec == 4;
#undef KFA_BIGROW_CASE
    default:
        return false;
    }
}
// column lengths of the one-pass column convolution (kfa_colconv_impl.h), heights in
// common use and their padded ones; hipErrorNotSupported for others, which keep the
// separate passes.  All measured against those on 1024 wide images, the whole
// convolution FP64 256 rows 60 -> 50 us, 1000 121 -> 66, 2160 192 -> 104, 3000 175 -> 141,
// 4000 255 -> 232, 4160 206 -> 184 (the least gains at 256, 2400 and up but for 4096),
// FP32 56 -> 46, 102 -> 63, 158 -> 71, 133 -> 87, 155 -> 133, 132 -> 103.
#define KFA_COLCONV_LENGTHS(X)                                                                     \
    X(256) X(480) X(512) X(720) X(960) X(1000) X(1024) X(1200) X(1440) X(1920) X(2000) X(2048)     \
    X(2080) X(2160) X(2400) X(3000) X(4000) X(4096) X(4160)
// where the one pass is the faster: from 65 columns on for the FP64 lengths whose tiles
// spill most and hold two columns (4000 and 4160 rows by 33 columns 114 and 88 us, 105 and
// 80 in separate passes; by 65 107 and 79, 107 and 82); at any width for the others
// (9 columns: 1000 rows FP64 63 us, 85 separate; 2080 68, 85; 4160 FP32 65, 79)
inline bool colconv_wide(uint32_t L, int prec, uint64_t cols) {
    return prec == 4 || (L != 4000 && L != 4160) || cols > 64;
}
hipError_t launch_colconv_f64(uint32_t L, const ColConvArgs& a, hipStream_t s);
hipError_t launch_colconv_f32(uint32_t L, const ColConvArgs& a, hipStream_t s);
inline bool colconv_len(uint32_t L) {
    switch (L) {
#define KFA_COLCONV_CASE(N) case N:
        KFA_COLCONV_LENGTHS(KFA_COLCONV_CASE)
#undef KFA_COLCONV_CASE
        return true;
    default:
        return false;
    }
}
// instances per workgroup of the shaped transposing pass of length L (0: none)
uint32_t fast_tout_ipw_f64(uint32_t L);
uint32_t fast_tout_ipw_f32(uint32_t L);
// fused on-chip two-pass transform of N*N points (N = 256)
hipError_t launch_fused_f32(uint32_t N, const FusedArgs& f, uint32_t groups, hipStream_t s);
hipError_t launch_fused_f64(uint32_t N, const FusedArgs& f, uint32_t groups, hipStream_t s);
// single-pass 65536-point FP32 transform by pairs of workgroups (2 a.npairs
// workgroups); dft: KFA_FAST_MFMA_* bits or 0
hipError_t launch_pair_f32(const PairArgs& a, uint32_t dft, hipStream_t s);
hipError_t launch_xcc_probe(uint32_t* out, uint32_t groups, hipStream_t s);
hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t s);
// ragged executor: allow `lds` bytes of dynamic LDS and report resident
// workgroups per CU; launch the persistent grid; patch caller pointers
hipError_t ragged_prepare(int prec, uint32_t lds, int* occupancy);
hipError_t launch_ragged(int prec, const RagArgs& r, uint32_t groups, uint32_t lds, hipStream_t s);
hipError_t launch_ragged_patch(void* blob, const uint64_t* off, const uint32_t* which,
                               const int64_t* delta, uint32_t n, const void* in, void* out,
                               hipStream_t s);
// lengths of the shaped row passes (one instance of 8192 fills a 512-thread
// workgroup) and of the shaped column / transposing passes of the two-pass
// transforms (which need several instances per workgroup to coalesce)
inline bool fast_len(uint32_t L) { return L >= 16 && L <= 8192 && (L & (L - 1)) == 0; }
inline bool fast_len_split(uint32_t L) { return L >= 16 && L <= 4096 && (L & (L - 1)) == 0; }
hipError_t launch_stage_twiddles(int prec, void* tw, const KfaFftArgs& a, hipStream_t s);
hipError_t launch_twiddle_table(void* out_d, uint64_t count, uint64_t step, uint64_t M,
                                hipStream_t s);
hipError_t launch_twiddle_2d(void* out_d, uint64_t rows, uint64_t cols, uint64_t M,
                             hipStream_t s);
hipError_t launch_twiddle_indexed(void* out_d, const uint32_t* idx, uint64_t count, uint64_t M,
                                  int conjugate, hipStream_t s);
hipError_t launch_bluestein_tables(void* chirp_d, void* h_d, uint64_t N, uint64_t M,
                                   hipStream_t s);
hipError_t launch_convert_from_f64(int prec, void* dst, const void* src_d, uint64_t n,
                                   double scale, hipStream_t s);
hipError_t launch_real_post(int prec, const void* Z, int64_t z_dist, void* X, int64_t xdh,
                            int64_t xdl, int64_t xs, uint32_t C, uint32_t h, uint64_t batch,
                            const void* st, int expand, int conj_out, hipStream_t s,
                            const int64_t* ztbl = nullptr, const int64_t* xtbl = nullptr);
// pw: null, or a factor in X's layout that multiplies the spectrum as it is read;
// blk: bins in blocks of four columns (KFA_IO_BLK4), xs the blocks' distance
hipError_t launch_real_pre(int prec, const void* X, int64_t xdh, int64_t xdl, int64_t xs,
                           uint32_t C, void* Z, int64_t z_dist, uint32_t h, uint64_t batch,
                           const void* st, const void* pw, hipStream_t s, int blk = 0);
// Bluestein steps of a three-pass inner length (one transform):
//   pre:  y[j] = conj?(x[j stride]) c[j] for j < n, 0 for n <= j < M (x real or complex)
//   mul_conj: y = conj(y * h)
//   post: out[k stride] = conj?(conj(y[k]) c[k] scale) for k < n (real: the real part)
hipError_t launch_bluestein_pre(int prec, const void* x, int64_t stride, bool real_in, bool conj_in,
                                const void* chirp, void* y, uint32_t n, uint32_t M, hipStream_t s);
hipError_t launch_mul_conj(int prec, void* y, const void* h, uint64_t n, hipStream_t s);
hipError_t launch_bluestein_post(int prec, const void* y, const void* chirp, void* out,
                                 int64_t stride, bool real_out, bool conj_out, double scale,
                                 uint32_t n, hipStream_t s);
hipError_t launch_transpose(int elem_bytes, const void* in, void* out, uint32_t x, uint32_t y,
                            uint32_t nmat, hipStream_t s);
hipError_t launch_hadamard(int prec, void* acc, const void* other, uint64_t n, hipStream_t s);
// fftshift (forward) / ifftshift (inverse) of a y x x row-major matrix of
// elem_bytes-sized elements in place; tmp (x*y elements) is needed unless
// shift_in_place(x, y)
bool shift_in_place(uint32_t x, uint32_t y);
hipError_t launch_shift(int elem_bytes, void* buf, void* tmp, uint32_t x, uint32_t y, bool inverse,
                        hipStream_t s);
// out[i] = |in[i]| of n complex values of the precision
hipError_t launch_magnitude(int prec, const void* in, void* out, uint64_t n, hipStream_t s);
// per-block FP64 sums of n reals of the precision into partial[blocks]
hipError_t launch_partial_sum(int prec, const void* in, uint64_t n, double* partial, uint32_t blocks,
                              hipStream_t s);
hipError_t launch_hadamard_real(int prec, void* acc, const void* other, uint64_t n,
                                hipStream_t s);
hipError_t launch_copy(int prec, const void* in, void* out, uint64_t n, int conj_, double scale,
                       hipStream_t s);
// refinement step of the precision form: FP32 -> FP64 copy, r = x - z, y += d
hipError_t launch_widen(const void* in_f32, void* out_f64, uint64_t n, hipStream_t s);
hipError_t launch_residual(const void* x_f32, const void* z_f64, void* r_f32, uint64_t n,
                           hipStream_t s);
hipError_t launch_accumulate(void* y_f32, const void* d_f32, uint64_t n, hipStream_t s);
hipError_t launch_gather_first(int prec, int real_in, const void* in, int64_t dist_hi,
                               int64_t dist_lo, uint32_t C, void* out, uint64_t batch,
                               hipStream_t s, const int64_t* tbl = nullptr);

hipError_t launch_rader_dc(int prec, const void* x0, int x0_real, const void* A, uint32_t L,
                           void* out, int64_t dh, int64_t dl, uint32_t C, int real_out, int conj_,
                           double scale, uint64_t batch, hipStream_t s,
                           const int64_t* tbl = nullptr);

} // namespace kfa
