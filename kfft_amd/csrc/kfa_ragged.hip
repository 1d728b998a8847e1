// Ragged executor: a batch of transforms of uneven lengths in one persistent
// launch fed by per-XCD device work queues.
//
// The host records, for every length group, the launches its plan would make
// (general LDS passes, Rader gathers and DC terms, real-input rebuilds) and
// turns each launch into a record with `tiles` workgroup tasks.  Records of a
// group form a chain: every task of record r waits until all tiles of the
// record before it in the chain are done.  A group and all of its records
// belong to one queue, and a workgroup serves the queue of the XCD it runs on
// (hardware register XCC_ID), so every intermediate a chain writes is read
// back on the same XCD, through the same L2.  Tickets of a queue are ordered
// level by level (all first records, then all second records, ...), so a task
// only ever waits for tasks dequeued before it by running workgroups; the
// wait is bounded and raises an error flag instead of hanging.
#include "kfa_aux_dev.h"
#include "kfa_fft_impl.h"
#include "kfa_kernels.h"
#include "kfa_mixed_impl.h"
#include "kfa_sync.h"

namespace kfa {

// One tile of a record as a function of its own: inlined into the ticket loop, all
// the tiles' index arithmetic and addresses would share one register allocation
// (hundreds of spilled registers).  Per task the time goes to the tile itself
// (35,000-70,000 cycles of a 4096-point tile at three workgroups per CU, by use, read
// from the clock in an instrumented build; dependency wait, ticket and completion
// together about 5,000): waves wait for 69% of their time.  20,000 mixed
// transforms (16 to 65536 points, FP32): 12.3 ms with inlined tiles reading their
// arguments as vector loads and their data element by element, 9.7 with scalar
// arguments, tiles as functions and batched loads, 6.7 with tiles compiled per use,
// 6.4 with power-of-two Bluestein lengths, 6.0 with queues balanced by the plans' work.
template <typename T>
__device__ __attribute__((noinline)) void rag_fft(uint64_t args, uint32_t tile, uint32_t lds) {
    const KfaFftArgs& A = const_args<KfaFftArgs>(uniform64(args));
    fft_tile<T, 32, DFT_VALU, 0, true>(A, (uint64_t)__builtin_amdgcn_readfirstlane(tile) * A.ipw,
                                       lds_at<cx<T>>(__builtin_amdgcn_readfirstlane(lds)),
                                       threadIdx.x);
}
template <typename T, int N, int U>
__device__ __attribute__((noinline)) void rag_mix(uint64_t args, uint32_t tile, uint32_t lds) {
    const KfaFftArgs& A = const_args<KfaFftArgs>(uniform64(args));
    mixgen_tile<T, N, 4096 / N, false, U>(
        A, (uint64_t)__builtin_amdgcn_readfirstlane(tile) * (4096 / N),
        lds_at<cx<T>>(__builtin_amdgcn_readfirstlane(lds)), threadIdx.x);
}

// Real-input rebuild, KFA_RAG_POST_PAIRS (instance, bin pair)s per task (gx = h/2 + 1
// pairs per instance): each thread's pairs are read together, four at a time.
template <typename T>
__device__ __forceinline__ void rag_real_post(const RealPostArgs& p, uint32_t gx, uint32_t tile,
                                              uint32_t tid) {
    constexpr int CH = 4;
    for (uint32_t o = tid; o < KFA_RAG_POST_PAIRS; o += CH * KFA_RAG_THREADS) {
        uint32_t kk[CH];
        uint64_t bb[CH];
        RealPair<T> r[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i) {
            const uint64_t idx = (uint64_t)tile * KFA_RAG_POST_PAIRS + o + i * KFA_RAG_THREADS;
            const uint64_t b = idx / gx;
            kk[i] = (uint32_t)(idx - b * gx);
            bb[i] = b;
            // (past the batch: the first pair, read and not written)
            r[i] = real_post_read<T>(p, b < p.batch ? kk[i] : 0u, b < p.batch ? b : 0u);
        }
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (bb[i] < p.batch)
                real_post_write<T>(p, kk[i], r[i]);
    }
}

// A task's latency (ticket, dependency wait, HBM load, LDS stages, store)
// is hidden only by other resident workgroups: registers are held to what
// three (FP32) or two (FP64) workgroups per CU need, which the LDS budget of
// the plans also allows.
template <typename T>
__global__ void __launch_bounds__(KFA_RAG_THREADS)
    __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 3 : 2))) k_ragged(const RagArgs R) {
    extern __shared__ __align__(16) unsigned char kfa_smem[];
    typedef __attribute__((address_space(3))) unsigned char* LP;
    const uint32_t lds = (uint32_t)(uintptr_t)(LP)kfa_smem;
    // (two slots in turn: the next ticket is written while slow waves may still
    // read the current one)
    __shared__ uint32_t sh_ticket[2];

    const uint32_t q = xcc_id() % R.nq;
    const uint32_t t0 = R.tq_off[q], nt = R.tq_off[q + 1] - t0;
    uint32_t* tick = R.ctr + 16 * q;
    uint32_t* done = R.ctr + 16 * R.nq;
    uint32_t* err = done + R.nrec;
    if (threadIdx.x == 0)
        sh_ticket[0] = __hip_atomic_fetch_add(tick, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();

    for (uint32_t it = 0;; ++it) {
        // (opaque per task, so that no tile's index arithmetic is hoisted out of the
        // ticket loop)
        uint32_t tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const uint32_t t = __builtin_amdgcn_readfirstlane(sh_ticket[it & 1]);
        if (t >= nt)
            break;
        const RagTicket& k = const_args<RagTicket>((uint64_t)(R.tq + t0 + t));
        const uint64_t a = (uint64_t)(R.blob + k.args);
        {
            // every line of the arguments requested at once: a tile reads them
            // field by field, each line's first use being a miss to memory
            static_assert((sizeof(KfaFftArgs) + 63) / 64 * 64 <= KFA_RAG_BLOB_PAD,
                          "the lines past the last record's arguments are in the blob");
            uint32_t x = 0;
#pragma unroll
            for (uint32_t i = 0; i < (sizeof(KfaFftArgs) + 63) / 64; ++i)
                x ^= const_args<uint32_t>(a + 64 * i);
            asm volatile("" ::"s"(x));
        }
        if (k.dep >= 0) {
            if (tid == 0)
                wait_geq(done + k.dep, k.dep_tiles, R.spin_limit, err);
            __syncthreads();
            acquire_agent();
        }
        const uint32_t tile = k.tile;
        switch (k.type & 255u) {
        case KFA_REC_FFT: {
            rag_fft<T>(a, tile, lds);
            break;
        }
        case KFA_REC_MIX: {
            // the shaped tile of a power-of-two pass: 4096 / L instances fill
            // the workgroup's 256 threads exactly (L / 16 threads each)
            switch (k.type >> 8) {
#define KFA_RAG_MIX(LG, U)                                                                         \
    case (U) | (LG) << 8:                                                                          \
        rag_mix<T, 1 << (LG), U>(a, tile, lds);                                                    \
        break;
                KFA_RAG_MIXES(KFA_RAG_MIX)
#undef KFA_RAG_MIX
            default:
                break;
            }
            break;
        }
        case KFA_REC_GATHER: {
            const GatherArgs& g = const_args<GatherArgs>(a);
            const uint64_t b = (uint64_t)tile * KFA_RAG_THREADS + tid;
            if (b < g.batch)
                gather_first_one<T>(g, b);
            break;
        }
        case KFA_REC_DC: {
            const DcArgs& d = const_args<DcArgs>(a);
            const uint64_t b = (uint64_t)tile * KFA_RAG_THREADS + tid;
            if (b < d.batch)
                rader_dc_one<T>(d, b);
            break;
        }
        case KFA_REC_REAL_POST: {
            rag_real_post<T>(const_args<RealPostArgs>(a), k.gx, tile, tid);
            break;
        }
        default:
            break;
        }
        signal_done_next(done + k.rec, tick, &sh_ticket[(it + 1) & 1]);
    }
}

// Writes the caller's base pointers into the argument blob: entry i sets the
// 64-bit word at byte offset off[i] to (which[i] ? out : in) + delta[i].
__global__ void k_ragged_patch(unsigned char* blob, const uint64_t* off, const uint32_t* which,
                               const int64_t* delta, uint32_t n, uint64_t in, uint64_t out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        *reinterpret_cast<uint64_t*>(blob + off[i]) = (which[i] ? out : in) + (uint64_t)delta[i];
}

template <typename T>
static hipError_t ragged_prepare_t(uint32_t lds, int* occupancy) {
    static uint32_t set_lds = 0; // largest dynamic LDS size allowed so far
    if (lds > set_lds) {
        hipError_t e = hipFuncSetAttribute((const void*)k_ragged<T>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) {
            (void)hipGetLastError(); // do not leave the error for the next launch
            return e;
        }
        set_lds = lds;
    }
    int blocks = 0;
    hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, k_ragged<T>,
                                                                KFA_RAG_THREADS, lds);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        return e;
    }
    *occupancy = blocks;
    return hipSuccess;
}

hipError_t ragged_prepare(int prec, uint32_t lds, int* occupancy) {
    if (lds > 160 * 1024 - 64)
        return hipErrorInvalidValue;
    return prec == 8 ? ragged_prepare_t<double>(lds, occupancy)
                     : ragged_prepare_t<float>(lds, occupancy);
}

hipError_t launch_ragged(int prec, const RagArgs& r, uint32_t groups, uint32_t lds, hipStream_t s) {
    if (prec == 8)
        hipLaunchKernelGGL(k_ragged<double>, dim3(groups), dim3(KFA_RAG_THREADS), lds, s, r);
    else
        hipLaunchKernelGGL(k_ragged<float>, dim3(groups), dim3(KFA_RAG_THREADS), lds, s, r);
    return hipGetLastError();
}

hipError_t launch_ragged_patch(void* blob, const uint64_t* off, const uint32_t* which,
                               const int64_t* delta, uint32_t n, const void* in, void* out,
                               hipStream_t s) {
    if (!n)
        return hipSuccess;
    hipLaunchKernelGGL(k_ragged_patch, dim3((n + 255) / 256), dim3(256), 0, s,
                       (unsigned char*)blob, off, which, delta, n, (uint64_t)in, (uint64_t)out);
    return hipGetLastError();
}

} // namespace kfa
