// Shared host/device definitions of the gfx950 transform engine.
//
// One kernel family (k_fft) runs a batched length-L complex FFT entirely in a
// workgroup: a cooperative load moves the workgroup's instances from HBM into
// LDS, the radix stages run LDS to LDS (Stockham autosort), and a cooperative
// store writes them back.  Planner-built pass descriptors (KfaFftArgs) describe how element e of
// instance b is addressed on each side and which fused element operations
// (conjugation, pointwise products, four-step twiddles, Rader gather/scatter,
// Bluestein chirps, real in/out) apply on the way in and out.
#pragma once
#include <stdint.h>

#define KFA_MAX_STAGES 24
#define KFA_MAX_RADIX 32

// I/O flags (KfaIo::flags)
#define KFA_IO_REAL 0x0001u       // real data: load imag=0 / store real part
#define KFA_IO_REAL_PAIRS 0x0002u // store complex as two reals at 2*ph, 2*ph+1 (stride in reals)
#define KFA_IO_CONJ1 0x0004u      // conjugate right after load / right before store ops
#define KFA_IO_CONJ2 0x0008u      // conjugate at the end of load ops / after scaling on store
#define KFA_IO_PW 0x0010u         // pointwise multiply by pw[...]
#define KFA_IO_PW_LAYOUT 0x0020u  // pw indexed like the data (else by logical index)
#define KFA_IO_SCALE 0x0040u      // multiply by KfaFftArgs::scale (store)
#define KFA_IO_TW4 0x0080u        // four-step twiddle W_N^(b_lo * e) (store)
#define KFA_IO_ADDX0 0x0100u      // add the instance's aux value (Rader x[0]) after all ops (store)
#define KFA_IO_RPOST 0x0200u      // real-input rebuild on store: Z = FFT_L of 2L reals read as L
                                  // complex values; writes bins X[0..L] (pw: super twiddles
                                  // st[i] = exp(-i pi ((i+1)/L + 1/2)), compute precision)
#define KFA_IO_MAP 0x0800u        // element permutation map[logical]
#define KFA_IO_PW_F64 0x1000u     // pw table is double precision complex
#define KFA_IO_SCALE_POST 0x2000u // multiply by KfaFftArgs::scale_post after ADDX0
#define KFA_IO_AUX_REAL 0x4000u   // aux (x[0] source) is a real array
#define KFA_IO_INST 0x8000u       // instance bases from a table: base = inst[b_hi] + b_lo*dist_lo
// (input side, set by the shaped general pass's launcher only) the maps of both
// sides, map[lg] for lg < L, are also in LDS as 16-bit values behind the tile's
// instance slots: the input's at [0, L), the output's at [L, 2L)
#define KFA_IO_LMAP 0x10000u

// (output of a real rebuild, input of the inverse one) bins in blocks of four
// columns: bin e at base + (e / 4) * stride + e mod 4, so that consecutive rows'
// blocks are adjacent
#define KFA_IO_BLK4 0x20000u
// (load) the inverse of the real-input rebuild: the instance holds bins X[0..L] of
// a real transform of 2L points, the pass transforms Z (pw: inverse super
// twiddles, as k_real_pre)
#define KFA_IO_RPRE 0x40000u

// Addressing of element e of instance b on one side of a pass:
//   b_lo = b % C, b_hi = b / C
//   lg   = b_lo * lo_mul + e * e_mul              (logical index)
//   ph   = (flags & MAP) ? map[lg] : lg           (physical index)
//   addr = b_hi * dist_hi + b_lo * dist_lo + ph * stride   (in elements)
//   (KFA_IO_INST: inst[b_hi] replaces b_hi * dist_hi; ragged batches)
// lg >= valid loads zero / skips the store.
struct KfaIo {
    uint64_t ptr;
    int64_t dist_hi, dist_lo, stride;
    uint64_t map;
    uint64_t pw;
    uint64_t aux; // ADDX0: x[0] values, indexed by b_hi*aux_dist + b_lo*aux_dist_lo
    int64_t aux_dist, aux_dist_lo;
    uint64_t inst; // KFA_IO_INST: int64 element offset of every instance
    uint32_t C, lo_mul, e_mul, valid;
    uint32_t flags;
    // KFA_IO_MAP on contiguous complex rows (C = 1, stride 1): the permuted
    // positions of an instance lie in [row_lo, row_span) and, on the store side,
    // fill it; a pass whose tile holds row_span elements per instance may move
    // the rows through LDS contiguously and permute there (0: no such bound)
    uint32_t row_span, row_lo, pad0;
};

// One LDS stage: radix, ns (product of the earlier radices), offset of its
// twiddles, and ns_magic = ceil(2^32 / ns) (0 for ns = 1): for b, ns < 2^16,
// b / ns = umulhi(b, ns_magic) exactly (the rounding error times b stays
// below 2^32), which replaces a runtime division per butterfly.
struct KfaStage {
    uint32_t radix, ns, tw_off, ns_magic;
};

struct KfaFftArgs {
    KfaIo in, out;
    uint64_t tw;               // per-stage twiddles, complex of the compute precision
    uint64_t tw4_hi, tw4_lo;   // four-step twiddle tables, complex double
    double scale, scale_post;
    uint64_t batch;            // number of instances
    uint32_t tw4_n, tw4_shift; // four-step length and log2 of the low table size
    // convolution pass (Bluestein, Rader): after the stages, element e of
    // instance b is multiplied by mid_pw[(b mod mid_rows) * L + e] (compute
    // precision) and conjugated, and the stages run again (0: an ordinary pass).
    // mid_dc (if set) receives the first round's element 0 of the instances with
    // b mod mid_rows == 0, at index b / mid_rows (Rader's A[0]).
    uint64_t mid_pw;
    uint64_t mid_dc;
    // Rader's last pass (dc_out != 0; the shaped tiles compiled for it only): also
    // store X[0] = x[0] + A[0] of every instance, A[0] from dc_src (two-pass inner
    // length) or from the tile's own first round
    uint64_t dc_src;
    uint32_t dc_out, dc_pad;
    uint32_t mid_rows;
    // workgroup -> tile order (k_fft): 0 in dispatch order; n > 1: workgroups are
    // dealt round-robin to n XCDs, and XCD x runs a contiguous range of tiles, so
    // the tiles of one transform share that XCD's L2 (scattered Rader gathers)
    uint32_t xcds;
    uint32_t L, nstages;
    uint32_t tpi, ipw;         // threads per instance, instances per workgroup
    uint32_t in_jfast;         // cooperative load: consecutive threads on consecutive instances
    uint32_t out_jfast;        // cooperative store: same for the store side
    uint32_t inst_stride;      // LDS elements per instance (padded, odd)
    uint32_t tw_lds;           // FP64: stage twiddles copied into LDS after the instances at
                               // the start of a tile (entries; 0: stages read them from memory)
    KfaStage st[KFA_MAX_STAGES];
};

// Uses of a pass.  The shaped general passes are compiled per use: only the IO
// flags the use can carry (in / out masks; KFA_IOM_PART: fewer valid elements than
// the pass's) and only its rounds (conv: the convolution's second one) have code,
// which halves the registers and the code of a tile against one that asks.
#define KFA_IOM_ANY 0xffffffffu
#define KFA_IOM_PART 0x80000000u
enum KfaUse {
    KFA_USE_ANY = 0,   // whatever the arguments say
    KFA_USE_PLAIN,     // rows or columns, four-step twiddle or real rebuild in the store
    KFA_USE_A1_BLUE,   // Bluestein, two-pass inner length: chirped, zero-padded columns
    KFA_USE_MID,       // two-pass convolution's middle rows
    KFA_USE_A2_BLUE,   // Bluestein: columns back, chirped, truncated
    KFA_USE_ONE_BLUE,  // Bluestein in one pass
    KFA_USE_A1_RADER,  // Rader, two-pass inner length: gathered columns
    KFA_USE_A2_RADER,  // Rader: columns back, scattered
    KFA_USE_ONE_RADER, // Rader in one pass
    KFA_USE_RPRE,      // inverse real rows: the inverse rebuild in the load
    KFA_USE_ROWS,      // plain complex rows (long lengths, exchange in halves)
    KFA_USES
};
constexpr uint32_t kfa_use_in(int u) {
    return u == KFA_USE_PLAIN      ? KFA_IO_CONJ1 | KFA_IO_REAL | KFA_IO_INST
           : u == KFA_USE_A1_BLUE || u == KFA_USE_ONE_BLUE
               ? KFA_IO_PW | KFA_IO_CONJ1 | KFA_IO_REAL | KFA_IO_INST | KFA_IOM_PART
           : u == KFA_USE_MID      ? 0u
           : u == KFA_USE_A2_BLUE || u == KFA_USE_A2_RADER ? KFA_IO_CONJ1
           : u == KFA_USE_RPRE ? KFA_IO_RPRE | KFA_IO_CONJ1 | KFA_IO_BLK4
           : u == KFA_USE_ROWS ? KFA_IO_CONJ1
           : u == KFA_USE_A1_RADER || u == KFA_USE_ONE_RADER
               ? KFA_IO_MAP | KFA_IO_CONJ1 | KFA_IO_REAL | KFA_IO_LMAP
               : KFA_IOM_ANY;
}
constexpr uint32_t kfa_use_out(int u) {
    return u == KFA_USE_PLAIN
               ? KFA_IO_CONJ2 | KFA_IO_SCALE | KFA_IO_TW4 | KFA_IO_INST | KFA_IO_RPOST | KFA_IO_BLK4
           : u == KFA_USE_A1_BLUE || u == KFA_USE_A1_RADER ? KFA_IO_TW4
           : u == KFA_USE_MID  ? KFA_IO_TW4 | KFA_IO_CONJ2
           : u == KFA_USE_RPRE || u == KFA_USE_ROWS ? KFA_IO_CONJ2 | KFA_IO_SCALE
           : u == KFA_USE_A2_BLUE || u == KFA_USE_ONE_BLUE
               ? KFA_IO_CONJ1 | KFA_IO_CONJ2 | KFA_IO_PW | KFA_IO_SCALE | KFA_IO_INST | KFA_IOM_PART
           : u == KFA_USE_A2_RADER || u == KFA_USE_ONE_RADER
               ? KFA_IO_MAP | KFA_IO_CONJ1 | KFA_IO_CONJ2 | KFA_IO_SCALE | KFA_IO_ADDX0 |
                     KFA_IO_SCALE_POST | KFA_IO_AUX_REAL | KFA_IO_REAL
               : KFA_IOM_ANY;
}
constexpr bool kfa_use_conv(int u) {
    return u == KFA_USE_MID || u == KFA_USE_ONE_BLUE || u == KFA_USE_ONE_RADER;
}
inline uint32_t kfa_io_needs(const KfaIo& io) {
    return io.flags | (io.valid == 0xffffffffu ? 0u : KFA_IOM_PART);
}
// the first use that covers a pass
inline int kfa_use_of(const KfaFftArgs& a) {
    const uint32_t in = kfa_io_needs(a.in), out = kfa_io_needs(a.out);
    for (int u = KFA_USE_PLAIN; u < KFA_USES; ++u)
        if (kfa_use_conv(u) == (a.mid_pw != 0) && !(in & ~kfa_use_in(u)) &&
            !(out & ~kfa_use_out(u)))
            return u;
    return KFA_USE_ANY;
}

// LDS padding: one spare element every 2^KFA_PAD_SHIFT elements keeps the
// stride-R writes of a Stockham stage off a single bank group.
#define KFA_PAD_SHIFT_F64 4
#define KFA_PAD_SHIFT_F32 4

// Arguments of the compile-time shaped power-of-two passes (kfa_fast_impl.h).
#define KFA_FAST_CONJ_IN 1u
#define KFA_FAST_CONJ_OUT 2u
#define KFA_FAST_SCALE 4u
#define KFA_FAST_TW4 8u
#define KFA_FAST_NT_IN 16u  // non-temporal (streaming) loads of the input
#define KFA_FAST_NT_OUT 32u // non-temporal (streaming) stores of the output
#define KFA_FAST_TW4_HI 256u    // four-step twiddle indexed by (instance / out_C) mod pad
#define KFA_FAST_MFMA_F16 64u   // radix-16 stages as split FP16 matrix products (FP32 data)
#define KFA_FAST_MFMA_BF16 128u // radix-16 stages as split BF16 matrix products (FP32 data)
// pass B of a real-input transform's half-length two-pass transform (TOUT): the
// workgroup holds rows a and N1 - a (row 0 with N1/2) and stores the real-input
// spectrum X[0..h] (h = N1 * L) instead of Z; the rebuild's twiddle
// st[k - 1] = exp(-i pi (k / h + 1/2)) for k = a + N1 e is -i W_2h^a W_2L^e,
// from rpost_st (W_2h^a, a < N1) and rpost_w2 (W_2L^e, e <= L)
#define KFA_FAST_RPOST 512u
// pass-A store twiddle W_N^m (m = col * k < N) as the product of two short
// tables, tw4[m >> tw4_shift] = W_N^(m & ~(S - 1)) and tw4_lo[m & (S - 1)] =
// W_N^(m mod S), S = 2^tw4_shift, in place of the N-entry [k][col] table
#define KFA_FAST_TW4_SPLIT 1024u

struct FastArgs {
    const void* in;
    void* out;
    const void* tw;  // stage twiddles (same layout as LdsPass)
    const void* tw4; // tw4[k * out_C + col] = W_N^(col * k), compute precision (pass A)
    int64_t in_hi, in_lo, in_stride;
    int64_t out_hi, out_lo, out_stride;
    uint64_t batch;
    uint32_t in_C, out_C;
    uint32_t flags;
    uint32_t pad; // KFA_FAST_TW4_HI: the four-step row length N2 (twiddle table stride)
    double scale;
    const void* rpost_st; // KFA_FAST_RPOST: W_2h^a, a < N1 (compute precision)
    uint32_t xcds;        // > 1: XCD-contiguous tile order (as KfaFftArgs::xcds)
    uint32_t tw4_shift;   // KFA_FAST_TW4_SPLIT: log2 of the low table's size
    const void* rpost_w2; // KFA_FAST_RPOST: W_2L^e, e <= L (compute precision)
    const void* tw4_lo;   // KFA_FAST_TW4_SPLIT: W_N^j, j < 2^tw4_shift (compute precision)
};


// Arguments of the column convolution (kfa_colconv_impl.h): element n of column x
// of both matrices at n * pitch + x, or (blk != 0: blocks of four columns) at
// (x / 4) * blk + 4 n + x mod 4; the result over b
struct ColConvArgs {
    const void* a;
    void* b;
    const void* tw; // stage twiddles of the column length (LdsPass layout)
    uint64_t pitch, cols, blk;
    double scale;
    uint32_t xcds, pad; // > 1: XCD-contiguous tile order (as KfaFftArgs::xcds)
};

// Arguments of the per-instance helper kernels (kfa_aux_dev.h); a non-zero
// table replaces the instance distance (ragged batches).
struct GatherArgs { // out[b] = x_b[0]
    uint64_t in, out, tbl;
    int64_t dist_hi, dist_lo;
    uint64_t batch;
    uint32_t C, comps;
};
struct DcArgs { // Rader X[0] = scale * (x0 + conj?(A[0]))
    uint64_t x0, A, out, tbl;
    int64_t dh, dl;
    double scale;
    uint64_t batch;
    uint32_t L, C, x0_real, real_out, conj_, pad;
};
struct RealPostArgs { // real-input rebuild, X from Z = FFT_h(x as complex)
    uint64_t Z, X, st, ztbl, xtbl;
    int64_t z_dist, xdh, xdl, xs;
    uint64_t batch;
    uint32_t C, h, expand, conj_out;
};

// Ragged executor (kfa_ragged.hip): one recorded launch of a length group.
#define KFA_REC_FFT 1u
#define KFA_REC_GATHER 2u
#define KFA_REC_DC 3u
#define KFA_REC_REAL_POST 4u
// a general pass of a power-of-two length L <= 4096 with the default radix
// schedule, run as the compile-time shaped tile (4096 / L instances per task)
#define KFA_REC_MIX 5u
// One task: a tile of a record.  A ticket holds all that its dispatch needs, so a
// workgroup reads one line of a stream its neighbours read too, then the
// arguments (a record beside it would be one more dependent cache miss).
struct RagTicket {
    uint64_t args;      // byte offset of the launch arguments in the blob
    uint32_t tile;      // tile of the record
    uint32_t rec;       // the record (its completion counter)
    int32_t dep;        // record that must be complete first (same queue), -1 none
    uint32_t dep_tiles; // its tile count
    uint32_t type;      // KFA_REC_*; KFA_REC_MIX | use << 8 | log2 length << 16
    uint32_t gx;        // REAL_POST: bin pairs per instance (h/2 + 1)
};
struct RagArgs {
    const unsigned char* blob;
    const RagTicket* tq;    // tickets, queue by queue
    const uint32_t* tq_off; // first ticket of each queue (nq + 1 entries)
    uint32_t* ctr;          // queue tickets (16 words apart), then done[records], then error
    uint32_t nq, nrec, spin_limit, pad;
};
// bytes past the last record's arguments that the blob reserves (a task touches
// the lines of the largest argument structure whatever its type)
#define KFA_RAG_BLOB_PAD 1024u

// Arguments of the single-pass 65536-point transform by pairs of workgroups
// (kfa_pair_impl.h).  inbox and ctr are scratch of the caller: 2 npairs x 16384
// complex values, and 64 npairs words that are zero at the launch.
struct PairArgs {
    const void* in;
    void* out;
    int64_t in_dist, out_dist; // elements between consecutive transforms
    const void* tw4;           // [32][2048]: W_65536^(k1 m)
    const void* twb;           // [128][16]: W_2048^(m_lo q2), then [8][16]: W_128^(m0 q1)
    void* inbox;
    uint32_t* ctr;
    uint32_t* err; // sticky error word: 1 a wait timed out, 2 an XCD id beyond nxcd
    uint64_t T;    // transforms (below 2^32 - 1)
    uint32_t npairs, nxcd, flags, spin_limit; // flags: KFA_FAST_CONJ_IN / CONJ_OUT / SCALE
    float scale;
    uint32_t stagger_groups, stagger_cycles; // start pairs in groups, this many cycles apart
    uint32_t spx;                            // pair slots per XCD (npairs = nxcd * spx)
};

// Arguments of the fused on-chip two-pass transform (kfa_fused_impl.h).
struct FusedArgs {
    const void* in;
    void* out;
    int64_t in_dist, out_dist; // elements between transforms
    void* ring;                // nq * S slots of N1*N2 elements
    const void* tw_col;        // stage twiddles of the N1 pass
    const void* tw_row;        // stage twiddles of the N2 pass
    const void* tw4;           // [k1][n2] four-step twiddles
    uint32_t* ctr;             // tickets (16 words apart), doneA[T], doneB[T], error
    uint64_t T;                // transforms in this launch
    uint32_t S, nq;
    uint32_t flags; // KFA_FAST_CONJ_IN / CONJ_OUT / SCALE
    uint32_t spin_limit;
    double scale;
};
