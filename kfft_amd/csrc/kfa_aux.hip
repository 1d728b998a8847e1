// Auxiliary gfx950 kernels of the transform engine: exact twiddle tables,
// Bluestein/Rader precompute, real-FFT pre/post passes, tiled transposes,
// pointwise products and copies; plus the host launchers.
#include <cstring>

#include "kfa_aux_dev.h"
#include "kfa_kernels.h"

namespace kfa {

// ---------------------------------------------------------------------------
// exact-argument twiddles in double: angle = -2*pi*m/M with the octant found
// from integers and sincospi on the reduced remainder
// ---------------------------------------------------------------------------
__device__ __forceinline__ cx<double> twiddle_d(uint64_t m, uint64_t M) {
    m %= M;
    const uint64_t u = 8 * m; // angle = (pi/4) * u / M
    const uint64_t o = u / M, rem = u - o * M;
    uint64_t quad;
    double phi; // in units of pi
    int sg;
    if ((o & 1) == 0) {
        quad = o / 2;
        phi = 0.25 * (double)rem / (double)M;
        sg = 1;
    } else {
        quad = (o + 1) / 2;
        phi = 0.25 * (double)(M - rem) / (double)M;
        sg = -1;
    }
    double sp, cp;
    sincospi(phi, &sp, &cp);
    double ca = 0, sa = 0;
    switch (quad & 3) {
    case 0: ca = 1; break;
    case 1: sa = 1; break;
    case 2: ca = -1; break;
    default: sa = -1; break;
    }
    const double c = ca * cp - sa * sg * sp, s = sa * cp + ca * sg * sp;
    return {c, -s}; // exp(-i angle)
}

template <typename T>
__global__ void k_stage_twiddles(cx<T>* tw, KfaFftArgs A) {
    // A.st[s].tw_off / ns / radix describe the table layout; entries L-1 max
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    for (uint32_t s = 1; s < A.nstages; ++s) {
        const uint32_t R = A.st[s].radix, ns = A.st[s].ns, off = A.st[s].tw_off;
        const uint32_t cnt = ns * (R - 1);
        if (i >= off && i < off + cnt) {
            const uint32_t j = i - off, k = j / (R - 1), r = j % (R - 1) + 1;
            const cx<double> w = twiddle_d((uint64_t)r * k, (uint64_t)ns * R);
            tw[i] = {(T)w.re, (T)w.im};
        }
    }
}

__global__ void k_twiddle_table(cx<double>* out, uint64_t count, uint64_t step, uint64_t M) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count)
        out[i] = twiddle_d(i * step, M);
}

// tab[k * cols + c] = exp(-2 pi i * (k c) / M): the four-step twiddles laid out so
// that consecutive columns c are adjacent
__global__ void k_twiddle_2d(cx<double>* out, uint64_t rows, uint64_t cols, uint64_t M) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < rows * cols) {
        const uint64_t k = i / cols, c = i - k * cols;
        out[i] = twiddle_d(k * c, M);
    }
}

// tab[i] = exp(-2 pi i * idx[i] / M)  (Rader b vector)
__global__ void k_twiddle_indexed(cx<double>* out, const uint32_t* idx, uint64_t count,
                                  uint64_t M, int conjugate) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) {
        cx<double> w = twiddle_d(idx[i], M);
        if (conjugate)
            w.im = -w.im;
        out[i] = w;
    }
}

// Bluestein chirp c[n] = exp(-i pi n^2 / N) for n < N and its kernel
// h[m] = conj(c[m]), h[M-m] = conj(c[m]) (1 <= m < N), zero elsewhere.
__global__ void k_bluestein_tables(cx<double>* chirp, cx<double>* h, uint64_t N, uint64_t M) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < N) {
        const uint64_t sq = (i * i) % (2 * N);
        const cx<double> c = twiddle_d(sq, 2 * N);
        chirp[i] = c;
        h[i] = conj(c);
        if (i > 0)
            h[M - i] = conj(c);
    } else if (i < M - N + 1) {
        h[i] = {0.0, 0.0};
    }
}

template <typename T>
__global__ void k_convert_from_f64(cx<T>* dst, const cx<double>* src, uint64_t n, double scale) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        dst[i] = {(T)(src[i].re * scale), (T)(src[i].im * scale)};
}

// Real-output pre-processing (even n = 2h): Z[k] from the half spectrum X[0..h]
// (the reference's rebuild_inverse, which yields 2*Z).  General strided input.
template <typename T>
__global__ void k_real_pre(const cx<T>* X, int64_t x_dist_hi, int64_t x_dist_lo, int64_t x_stride,
                           uint32_t C, cx<T>* Z, int64_t z_dist, uint32_t h, uint64_t batch,
                           const cx<T>* st, const cx<T>* pw, int blk) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t b = blockIdx.y + (uint64_t)gridDim.y * blockIdx.z;
    if (b >= batch || k > h / 2)
        return;
    const uint64_t bh = b / C, bl = b - bh * C;
    const int64_t xb = (int64_t)bh * x_dist_hi + (int64_t)bl * x_dist_lo;
    cx<T>* z = Z + (int64_t)b * z_dist;
    // the spectrum, times pw (same layout) where a convolution fuses its product here
    auto get = [&](uint32_t i) {
        const int64_t a = xb + (blk ? (int64_t)(i >> 2) * x_stride + (i & 3u)
                                    : (int64_t)i * x_stride);
        return pw ? cmul(X[a], pw[a]) : X[a];
    };
    if (k == 0) {
        const cx<T> x0 = get(0), xh = get(h);
        z[0] = {x0.re + xh.re, x0.re - xh.re};
        return;
    }
    const cx<T> fk = get(k), fr = get(h - k);
    const cx<T> fnkc = {fr.re, -fr.im};
    const cx<T> fek = fk + fnkc, tmp = fk - fnkc;
    const cx<T> fok = cmul(tmp, st[k - 1]);
    z[k] = fek + fok;
    const cx<T> w = fek - fok;
    z[h - k] = {w.re, -w.im};
}

// out[i*y + j] = in[j*x + i]  (the reference's transpose, kfft_math.c:60-78),
// through 32x32 LDS tiles; batched over z.
template <typename T>
__global__ void k_transpose(const T* in, T* out, uint32_t x, uint32_t y, uint64_t mat) {
    __shared__ T tile[32][33];
    const uint64_t zb = (uint64_t)blockIdx.z * mat;
    const uint32_t i0 = blockIdx.x * 32, j0 = blockIdx.y * 32;
    for (uint32_t r = threadIdx.y; r < 32; r += blockDim.y) {
        const uint32_t j = j0 + r, i = i0 + threadIdx.x;
        if (i < x && j < y)
            tile[r][threadIdx.x] = in[zb + (uint64_t)j * x + i];
    }
    __syncthreads();
    for (uint32_t r = threadIdx.y; r < 32; r += blockDim.y) {
        const uint32_t i = i0 + r, j = j0 + threadIdx.x;
        if (i < x && j < y)
            out[zb + (uint64_t)i * y + j] = tile[threadIdx.x][r];
    }
}

template <typename T>
__global__ void k_hadamard(cx<T>* acc, const cx<T>* other, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        acc[i] = cmul(acc[i], other[i]);
}

template <typename T>
__global__ void k_hadamard_real(T* acc, const T* other, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        acc[i] *= other[i];
}

// generic strided complex copy with optional conjugation and scaling
template <typename T>
__global__ void k_copy(const cx<T>* in, cx<T>* out, uint64_t n, int conj_, double scale) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        cx<T> v = in[i];
        if (conj_)
            v.im = -v.im;
        out[i] = {(T)(v.re * (T)scale), (T)(v.im * (T)scale)};
    }
}

// Refinement of the precision form (FP32 data, FP64 residual):
//   z = widen(y0);  z = T^-1(z) in FP64;  r = x - z (rounded once);  y = y0 + T(r)
__global__ void k_widen(const cx<float>* in, cx<double>* out, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        out[i] = {(double)in[i].re, (double)in[i].im};
}

__global__ void k_residual(const cx<float>* x, const cx<double>* z, cx<float>* r, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        r[i] = {(float)((double)x[i].re - z[i].re), (float)((double)x[i].im - z[i].im)};
}

__global__ void k_accumulate(cx<float>* y, const cx<float>* d, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const cx<float> a = y[i], b = d[i];
        y[i] = {a.re + b.re, a.im + b.im};
    }
}

// one thread per (instance, bin pair): idx = b * (h/2 + 1) + kk
template <typename T>
__global__ void k_real_post(const RealPostArgs a) {
    const uint64_t idx = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t per = a.h / 2 + 1;
    const uint64_t b = idx / per;
    if (b < a.batch)
        real_post_one<T>(a, (uint32_t)(idx - b * per), b);
}

template <typename T>
__global__ void k_gather_first(const GatherArgs a) {
    const uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b < a.batch)
        gather_first_one<T>(a, b);
}

template <typename T>
__global__ void k_rader_dc(const DcArgs a) {
    const uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (b < a.batch)
        rader_dc_one<T>(a, b);
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
static inline unsigned blocks_for(uint64_t n, unsigned bs) { return (unsigned)((n + bs - 1) / bs); }

hipError_t launch_fft(int prec, int maxe, const KfaFftArgs& a, uint32_t lds_bytes, hipStream_t s,
                      uint32_t dft) {
    if (Recorder* r = recorder())
        return r->add(KFA_REC_FFT, prec, maxe, lds_bytes, 0, 0, &a, sizeof(a));
    const int dk = (dft & KFA_FAST_MFMA_F16) ? 1 : (dft & KFA_FAST_MFMA_BF16) ? 2 : 0;
    return prec == 8 ? launch_fft_f64(maxe, a, lds_bytes, s)
                     : launch_fft_f32(maxe, a, lds_bytes, s, dk);
}

hipError_t launch_stage_twiddles(int prec, void* tw, const KfaFftArgs& a, hipStream_t s) {
    if (a.L < 2 || a.nstages < 2)
        return hipSuccess;
    const unsigned bs = 256;
    if (prec == 8)
        hipLaunchKernelGGL(k_stage_twiddles<double>, dim3(blocks_for(a.L, bs)), dim3(bs), 0, s,
                           (cx<double>*)tw, a);
    else
        hipLaunchKernelGGL(k_stage_twiddles<float>, dim3(blocks_for(a.L, bs)), dim3(bs), 0, s,
                           (cx<float>*)tw, a);
    return hipGetLastError();
}

hipError_t launch_twiddle_table(void* out_d, uint64_t count, uint64_t step, uint64_t M,
                                hipStream_t s) {
    if (!count)
        return hipSuccess;
    hipLaunchKernelGGL(k_twiddle_table, dim3(blocks_for(count, 256)), dim3(256), 0, s,
                       (cx<double>*)out_d, count, step, M);
    return hipGetLastError();
}

hipError_t launch_twiddle_2d(void* out_d, uint64_t rows, uint64_t cols, uint64_t M,
                             hipStream_t s) {
    const uint64_t n = rows * cols;
    if (!n)
        return hipSuccess;
    hipLaunchKernelGGL(k_twiddle_2d, dim3(blocks_for(n, 256)), dim3(256), 0, s,
                       (cx<double>*)out_d, rows, cols, M);
    return hipGetLastError();
}

hipError_t launch_twiddle_indexed(void* out_d, const uint32_t* idx, uint64_t count, uint64_t M,
                                  int conjugate, hipStream_t s) {
    if (!count)
        return hipSuccess;
    hipLaunchKernelGGL(k_twiddle_indexed, dim3(blocks_for(count, 256)), dim3(256), 0, s,
                       (cx<double>*)out_d, idx, count, M, conjugate);
    return hipGetLastError();
}

hipError_t launch_bluestein_tables(void* chirp_d, void* h_d, uint64_t N, uint64_t M,
                                   hipStream_t s) {
    const uint64_t cnt = (M - N + 1 > N) ? (M - N + 1) : N;
    hipLaunchKernelGGL(k_bluestein_tables, dim3(blocks_for(cnt, 256)), dim3(256), 0, s,
                       (cx<double>*)chirp_d, (cx<double>*)h_d, N, M);
    return hipGetLastError();
}

hipError_t launch_convert_from_f64(int prec, void* dst, const void* src_d, uint64_t n,
                                   double scale, hipStream_t s) {
    if (!n)
        return hipSuccess;
    if (prec == 8)
        hipLaunchKernelGGL(k_convert_from_f64<double>, dim3(blocks_for(n, 256)), dim3(256), 0, s,
                           (cx<double>*)dst, (const cx<double>*)src_d, n, scale);
    else
        hipLaunchKernelGGL(k_convert_from_f64<float>, dim3(blocks_for(n, 256)), dim3(256), 0, s,
                           (cx<float>*)dst, (const cx<double>*)src_d, n, scale);
    return hipGetLastError();
}

static dim3 batch_grid(uint32_t gx, uint64_t batch) {
    const uint64_t y = batch < 65535 ? batch : 65535;
    const uint64_t z = (batch + y - 1) / y;
    return dim3(gx, (unsigned)y, (unsigned)z);
}

hipError_t launch_real_post(int prec, const void* Z, int64_t z_dist, void* X, int64_t xdh,
                            int64_t xdl, int64_t xs, uint32_t C, uint32_t h, uint64_t batch,
                            const void* st, int expand, int conj_out, hipStream_t s,
                            const int64_t* ztbl, const int64_t* xtbl) {
    if (!batch)
        return hipSuccess;
    RealPostArgs a;
    memset(&a, 0, sizeof(a));
    a.Z = (uint64_t)Z;
    a.X = (uint64_t)X;
    a.st = (uint64_t)st;
    a.ztbl = (uint64_t)ztbl;
    a.xtbl = (uint64_t)xtbl;
    a.z_dist = z_dist;
    a.xdh = xdh;
    a.xdl = xdl;
    a.xs = xs;
    a.batch = batch;
    a.C = C;
    a.h = h;
    a.expand = (uint32_t)expand;
    a.conj_out = (uint32_t)conj_out;
    const unsigned bs = 256;
    const uint64_t pairs = (uint64_t)(h / 2 + 1) * batch; // one thread per bin pair
    if (Recorder* r = recorder())
        return r->add(KFA_REC_REAL_POST, prec, 0, 0, (pairs + KFA_RAG_POST_PAIRS - 1) / KFA_RAG_POST_PAIRS, h / 2 + 1, &a,
                      sizeof(a));
    const uint64_t blocks = (pairs + bs - 1) / bs;
    if (blocks > 0x7fffffffull)
        return hipErrorInvalidValue;
    const dim3 g((unsigned)blocks);
    if (prec == 8)
        hipLaunchKernelGGL(k_real_post<double>, g, dim3(bs), 0, s, a);
    else
        hipLaunchKernelGGL(k_real_post<float>, g, dim3(bs), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_real_pre(int prec, const void* X, int64_t xdh, int64_t xdl, int64_t xs,
                           uint32_t C, void* Z, int64_t z_dist, uint32_t h, uint64_t batch,
                           const void* st, const void* pw, hipStream_t s, int blk) {
    if (!batch)
        return hipSuccess;
    const unsigned bs = 128;
    const dim3 g = batch_grid(blocks_for(h / 2 + 1, bs), batch);
    if (prec == 8)
        hipLaunchKernelGGL(k_real_pre<double>, g, dim3(bs), 0, s, (const cx<double>*)X, xdh, xdl,
                           xs, C, (cx<double>*)Z, z_dist, h, batch, (const cx<double>*)st,
                           (const cx<double>*)pw, blk);
    else
        hipLaunchKernelGGL(k_real_pre<float>, g, dim3(bs), 0, s, (const cx<float>*)X, xdh, xdl, xs,
                           C, (cx<float>*)Z, z_dist, h, batch, (const cx<float>*)st,
                           (const cx<float>*)pw, blk);
    return hipGetLastError();
}

template <typename T>
__global__ void k_bluestein_pre(const T* x, int64_t stride, int real_in, int conj_in,
                                const cx<T>* c, cx<T>* y, uint32_t n, uint32_t M) {
    const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= M)
        return;
    cx<T> v = {T(0), T(0)};
    if (j < n) {
        if (real_in)
            v.re = x[(int64_t)j * stride];
        else
            v = ((const cx<T>*)x)[(int64_t)j * stride];
        if (conj_in)
            v.im = -v.im;
        v = cmul(v, c[j]);
    }
    y[j] = v;
}

template <typename T>
__global__ void k_mul_conj(cx<T>* y, const cx<T>* h, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        cx<T> v = cmul(y[i], h[i]);
        v.im = -v.im;
        y[i] = v;
    }
}

template <typename T>
__global__ void k_bluestein_post(const cx<T>* y, const cx<T>* c, T* out, int64_t stride,
                                 int real_out, int conj_out, T scale, uint32_t n) {
    const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n)
        return;
    cx<T> v = y[k];
    v.im = -v.im;
    v = cmul(v, c[k]);
    v.re *= scale;
    v.im *= scale;
    if (conj_out)
        v.im = -v.im;
    if (real_out)
        out[(int64_t)k * stride] = v.re;
    else
        ((cx<T>*)out)[(int64_t)k * stride] = v;
}

hipError_t launch_bluestein_pre(int prec, const void* x, int64_t stride, bool real_in, bool conj_in,
                                const void* chirp, void* y, uint32_t n, uint32_t M, hipStream_t s) {
    const unsigned bs = 256;
    const dim3 g((unsigned)blocks_for(M, bs));
    if (prec == 8)
        hipLaunchKernelGGL(k_bluestein_pre<double>, g, dim3(bs), 0, s, (const double*)x, stride,
                           real_in ? 1 : 0, conj_in ? 1 : 0, (const cx<double>*)chirp,
                           (cx<double>*)y, n, M);
    else
        hipLaunchKernelGGL(k_bluestein_pre<float>, g, dim3(bs), 0, s, (const float*)x, stride,
                           real_in ? 1 : 0, conj_in ? 1 : 0, (const cx<float>*)chirp,
                           (cx<float>*)y, n, M);
    return hipGetLastError();
}

hipError_t launch_mul_conj(int prec, void* y, const void* h, uint64_t n, hipStream_t s) {
    const unsigned bs = 256;
    const dim3 g((unsigned)blocks_for(n, bs));
    if (prec == 8)
        hipLaunchKernelGGL(k_mul_conj<double>, g, dim3(bs), 0, s, (cx<double>*)y,
                           (const cx<double>*)h, n);
    else
        hipLaunchKernelGGL(k_mul_conj<float>, g, dim3(bs), 0, s, (cx<float>*)y,
                           (const cx<float>*)h, n);
    return hipGetLastError();
}

hipError_t launch_bluestein_post(int prec, const void* y, const void* chirp, void* out,
                                 int64_t stride, bool real_out, bool conj_out, double scale,
                                 uint32_t n, hipStream_t s) {
    const unsigned bs = 256;
    const dim3 g((unsigned)blocks_for(n, bs));
    if (prec == 8)
        hipLaunchKernelGGL(k_bluestein_post<double>, g, dim3(bs), 0, s, (const cx<double>*)y,
                           (const cx<double>*)chirp, (double*)out, stride, real_out ? 1 : 0,
                           conj_out ? 1 : 0, scale, n);
    else
        hipLaunchKernelGGL(k_bluestein_post<float>, g, dim3(bs), 0, s, (const cx<float>*)y,
                           (const cx<float>*)chirp, (float*)out, stride, real_out ? 1 : 0,
                           conj_out ? 1 : 0, (float)scale, n);
    return hipGetLastError();
}

hipError_t launch_transpose(int elem_bytes, const void* in, void* out, uint32_t x, uint32_t y,
                            uint32_t nmat, hipStream_t s) {
    const dim3 g((x + 31) / 32, (y + 31) / 32, nmat), b(32, 8);
    const uint64_t mat = (uint64_t)x * y;
    switch (elem_bytes) {
    case 4:
        hipLaunchKernelGGL(k_transpose<float>, g, b, 0, s, (const float*)in, (float*)out, x, y,
                           mat);
        break;
    case 8:
        hipLaunchKernelGGL(k_transpose<double>, g, b, 0, s, (const double*)in, (double*)out, x, y,
                           mat);
        break;
    default:
        hipLaunchKernelGGL(k_transpose<cx<double>>, g, b, 0, s, (const cx<double>*)in,
                           (cx<double>*)out, x, y, mat);
        break;
    }
    return hipGetLastError();
}

// fftshift of a y x x row-major matrix (one row when y = 1, kfft_shift.c:4-61,
// ext/2d/kfft_cpx2.c:188-240) as a 2D roll by (rx, ry):
//   out[r][c] = in[(r - ry) mod y][(c - rx) mod x]
template <typename E>
__global__ void k_shift_gather(const E* src, E* dst, uint32_t x, uint32_t y, uint32_t rx,
                               uint32_t ry) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (uint64_t)x * y)
        return;
    const uint32_t r = (uint32_t)(i / x), c = (uint32_t)(i - (uint64_t)r * x);
    const uint32_t sr = r >= ry ? r - ry : r + y - ry;
    const uint32_t sc = c >= rx ? c - rx : c + x - rx;
    dst[i] = src[(uint64_t)sr * x + sc];
}

// The same roll in place when every dimension is even or 1: a roll by half of
// each even dimension pairs element i with p(i) (an involution); the thread of
// the smaller index swaps the pair.
template <typename E>
__global__ void k_shift_swap(E* buf, uint32_t x, uint32_t y) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (uint64_t)x * y)
        return;
    const uint32_t hx = (x % 2 == 0) ? x / 2 : 0, hy = (y % 2 == 0) ? y / 2 : 0;
    const uint32_t r = (uint32_t)(i / x), c = (uint32_t)(i - (uint64_t)r * x);
    const uint32_t pr = r + hy < y ? r + hy : r + hy - y;
    const uint32_t pc = c + hx < x ? c + hx : c + hx - x;
    const uint64_t p = (uint64_t)pr * x + pc;
    if (i < p) {
        const E a = buf[i];
        buf[i] = buf[p];
        buf[p] = a;
    }
}

template <typename E>
static void shift_launch_t(void* buf, void* tmp, uint32_t x, uint32_t y, uint32_t rx, uint32_t ry,
                           bool swap, hipStream_t s) {
    const uint64_t n = (uint64_t)x * y;
    const dim3 g((unsigned)((n + 255) / 256)), b(256);
    if (swap)
        hipLaunchKernelGGL(k_shift_swap<E>, g, b, 0, s, (E*)buf, x, y);
    else
        hipLaunchKernelGGL(k_shift_gather<E>, g, b, 0, s, (const E*)buf, (E*)tmp, x, y, rx, ry);
}

bool shift_in_place(uint32_t x, uint32_t y) {
    return (x % 2 == 0 || x == 1) && (y % 2 == 0 || y == 1);
}

hipError_t launch_shift(int elem_bytes, void* buf, void* tmp, uint32_t x, uint32_t y, bool inverse,
                        hipStream_t s) {
    const uint64_t n = (uint64_t)x * y;
    if (n < 2)
        return hipSuccess;
    if ((n + 255) / 256 > 0x7fffffffull)
        return hipErrorInvalidValue;
    // forward rolls by floor(d/2), inverse by ceil(d/2) (equal for even d)
    const uint32_t rx = inverse ? x - x / 2 : x / 2, ry = inverse ? y - y / 2 : y / 2;
    const bool swap = shift_in_place(x, y);
    if (!swap && !tmp)
        return hipErrorInvalidValue;
    switch (elem_bytes) {
    case 4:
        shift_launch_t<uint32_t>(buf, tmp, x, y, rx % x, ry % y, swap, s);
        break;
    case 8:
        shift_launch_t<uint64_t>(buf, tmp, x, y, rx % x, ry % y, swap, s);
        break;
    case 16:
        shift_launch_t<cx<double>>(buf, tmp, x, y, rx % x, ry % y, swap, s);
        break;
    default:
        return hipErrorInvalidValue;
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && !swap)
        e = hipMemcpyAsync(buf, tmp, n * (uint64_t)elem_bytes, hipMemcpyDeviceToDevice, s);
    return e;
}

// |z| = sqrt(re^2 + im^2) (kfft_math.c:123-138 with a correctly rounded root)
template <typename T>
__global__ void k_magnitude(const cx<T>* in, T* out, uint64_t n) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const cx<T> v = in[i];
        out[i] = sqrt(v.re * v.re + v.im * v.im);
    }
}

hipError_t launch_magnitude(int prec, const void* in, void* out, uint64_t n, hipStream_t s) {
    if (!n)
        return hipSuccess;
    const dim3 g(blocks_for(n, 256)), b(256);
    if (prec == 8)
        hipLaunchKernelGGL(k_magnitude<double>, g, b, 0, s, (const cx<double>*)in, (double*)out, n);
    else
        hipLaunchKernelGGL(k_magnitude<float>, g, b, 0, s, (const cx<float>*)in, (float*)out, n);
    return hipGetLastError();
}

// Partial sums in FP64: block k sums elements k*256 + t, stepping by the grid,
// in a fixed order (deterministic), into partial[k].
template <typename T>
__global__ void __launch_bounds__(256) k_partial_sum(const T* in, uint64_t n, double* partial) {
    __shared__ double red[256];
    double acc = 0.0;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * 256)
        acc += (double)in[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (unsigned w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w)
            red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0)
        partial[blockIdx.x] = red[0];
}

hipError_t launch_partial_sum(int prec, const void* in, uint64_t n, double* partial, uint32_t blocks,
                              hipStream_t s) {
    if (prec == 8)
        hipLaunchKernelGGL(k_partial_sum<double>, dim3(blocks), dim3(256), 0, s, (const double*)in,
                           n, partial);
    else
        hipLaunchKernelGGL(k_partial_sum<float>, dim3(blocks), dim3(256), 0, s, (const float*)in, n,
                           partial);
    return hipGetLastError();
}

hipError_t launch_hadamard(int prec, void* acc, const void* other, uint64_t n, hipStream_t s) {
    if (!n)
        return hipSuccess;
    if (prec == 8)
        hipLaunchKernelGGL(k_hadamard<double>, dim3(blocks_for(n, 256)), dim3(256), 0, s,
                           (cx<double>*)acc, (const cx<double>*)other, n);
    else
        hipLaunchKernelGGL(k_hadamard<float>, dim3(blocks_for(n, 256)), dim3(256), 0, s,
                           (cx<float>*)acc, (const cx<float>*)other, n);
    return hipGetLastError();
}

hipError_t launch_hadamard_real(int prec, void* acc, const void* other, uint64_t n,
                                hipStream_t s) {
    if (!n)
        return hipSuccess;
    if (prec == 8)
        hipLaunchKernelGGL(k_hadamard_real<double>, dim3(blocks_for(n, 256)), dim3(256), 0, s,
                           (double*)acc, (const double*)other, n);
    else
        hipLaunchKernelGGL(k_hadamard_real<float>, dim3(blocks_for(n, 256)), dim3(256), 0, s,
                           (float*)acc, (const float*)other, n);
    return hipGetLastError();
}

hipError_t launch_copy(int prec, const void* in, void* out, uint64_t n, int conj_, double scale,
                       hipStream_t s) {
    if (!n)
        return hipSuccess;
    if (prec == 8)
        hipLaunchKernelGGL(k_copy<double>, dim3(blocks_for(n, 256)), dim3(256), 0, s,
                           (const cx<double>*)in, (cx<double>*)out, n, conj_, scale);
    else
        hipLaunchKernelGGL(k_copy<float>, dim3(blocks_for(n, 256)), dim3(256), 0, s,
                           (const cx<float>*)in, (cx<float>*)out, n, conj_, scale);
    return hipGetLastError();
}

hipError_t launch_widen(const void* in, void* out, uint64_t n, hipStream_t s) {
    if (!n)
        return hipSuccess;
    hipLaunchKernelGGL(k_widen, dim3(blocks_for(n, 256)), dim3(256), 0, s, (const cx<float>*)in,
                       (cx<double>*)out, n);
    return hipGetLastError();
}

hipError_t launch_residual(const void* x, const void* z, void* r, uint64_t n, hipStream_t s) {
    if (!n)
        return hipSuccess;
    hipLaunchKernelGGL(k_residual, dim3(blocks_for(n, 256)), dim3(256), 0, s, (const cx<float>*)x,
                       (const cx<double>*)z, (cx<float>*)r, n);
    return hipGetLastError();
}

hipError_t launch_accumulate(void* y, const void* d, uint64_t n, hipStream_t s) {
    if (!n)
        return hipSuccess;
    hipLaunchKernelGGL(k_accumulate, dim3(blocks_for(n, 256)), dim3(256), 0, s, (cx<float>*)y,
                       (const cx<float>*)d, n);
    return hipGetLastError();
}

hipError_t launch_gather_first(int prec, int real_in, const void* in, int64_t dist_hi,
                               int64_t dist_lo, uint32_t C, void* out, uint64_t batch,
                               hipStream_t s, const int64_t* tbl) {
    if (!batch)
        return hipSuccess;
    GatherArgs a;
    memset(&a, 0, sizeof(a));
    a.in = (uint64_t)in;
    a.out = (uint64_t)out;
    a.tbl = (uint64_t)tbl;
    a.dist_hi = dist_hi;
    a.dist_lo = dist_lo;
    a.batch = batch;
    a.C = C;
    a.comps = real_in ? 1 : 2;
    if (Recorder* r = recorder())
        return r->add(KFA_REC_GATHER, prec, 0, 0, blocks_for(batch, KFA_RAG_THREADS), 0, &a,
                      sizeof(a));
    if (prec == 8)
        hipLaunchKernelGGL(k_gather_first<double>, dim3(blocks_for(batch, 256)), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL(k_gather_first<float>, dim3(blocks_for(batch, 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_rader_dc(int prec, const void* x0, int x0_real, const void* A, uint32_t L,
                           void* out, int64_t dh, int64_t dl, uint32_t C, int real_out, int conj_,
                           double scale, uint64_t batch, hipStream_t s, const int64_t* tbl) {
    if (!batch)
        return hipSuccess;
    DcArgs a;
    memset(&a, 0, sizeof(a));
    a.x0 = (uint64_t)x0;
    a.A = (uint64_t)A;
    a.out = (uint64_t)out;
    a.tbl = (uint64_t)tbl;
    a.dh = dh;
    a.dl = dl;
    a.scale = scale;
    a.batch = batch;
    a.L = L;
    a.C = C;
    a.x0_real = (uint32_t)x0_real;
    a.real_out = (uint32_t)real_out;
    a.conj_ = (uint32_t)conj_;
    if (Recorder* r = recorder())
        return r->add(KFA_REC_DC, prec, 0, 0, blocks_for(batch, KFA_RAG_THREADS), 0, &a, sizeof(a));
    if (prec == 8)
        hipLaunchKernelGGL(k_rader_dc<double>, dim3(blocks_for(batch, 256)), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL(k_rader_dc<float>, dim3(blocks_for(batch, 256)), dim3(256), 0, s, a);
    return hipGetLastError();
}

} // namespace kfa
