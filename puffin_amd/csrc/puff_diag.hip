// Diagnostics (power, slice bunching) and layout conversion kernels.
//
//   power    gPowerP / fPower_3D / fPower_1D, io/av_write.f90:39-202
//   bunching getSliceTwiss, io/av_write.f90:405-773 (harmonic sums 562-650,
//            magnitudes 725-729)
//   slice moments  getSliceTwiss's per-slice sums (av_write.f90:505-536)
//   current  getCurr's linear binning of the charge (av_write.f90:297-368)
#include "puff_common.hpp"
#include "puff_kernels.hpp"

namespace puff {

// Power of one z2 plane: trapezoidal integral of |A|^2 over x then y
// (m_trapz2D, av_write.f90:217-238) on a uniform axis; |A|^2 in 1-D.
// Accumulated in FP64 (the reference's m_trapz is a default-real function).
template <typename R>
__global__ __launch_bounds__(256) void k_power(const cplx<R>* a, int nx, int ny, double dx,
                                               double dy, double* out) {
    const int iz = blockIdx.x;
    const int64_t ntr = (int64_t)nx * ny;
    const cplx<R>* p = a + (int64_t)iz * ntr;
    __shared__ double red[4];
    double s = 0.0;
    if (nx == 1 && ny == 1) {
        if (threadIdx.x == 0) {
            const double r = (double)p[0].x, i = (double)p[0].y;
            out[iz] = r * r + i * i;
        }
        return;
    }
    for (int64_t t = threadIdx.x; t < ntr; t += blockDim.x) {
        const int ix = (int)(t % nx), iy = (int)(t / nx);
        const double r = (double)p[t].x, i = (double)p[t].y;
        double w = 1.0;
        if (ix == 0 || ix == nx - 1) w *= 0.5;
        if (iy == 0 || iy == ny - 1) w *= 0.5;
        s += w * (r * r + i * i);
    }
    s = wave_sum(s);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) out[iz] = (red[0] + red[1] + red[2] + red[3]) * dx * dy;
}

// ---- binned sums over the macroparticles ----------------------------------------
// The slots are sorted by cell, so the 64 macroparticles of a wavefront lie in
// one bin, or a few.  An LDS atomic per macroparticle and sum then piles 64
// lanes onto one word: the 13 slice sums took 1.08 ms for 2^24 sorted
// macroparticles (0.21 ms of reads at the streaming rate), one harmonic of the
// bunching 0.43 ms.  Here a wavefront walks a contiguous stretch of the slots
// and keeps NV sums per lane in registers for the bin it is in (RunSums),
// adding the wavefront's total to LDS only when the bin changes: 0.16 and
// 0.14 ms (the current: 0.17 to 0.15).  Lanes of
// other bins than the run's and the next one, and wavefronts whose lanes lie
// in many bins (macroparticles not sorted: a change of bin, 12 cross-lane
// moves per sum, would serve fewer than RUN_MIN lanes), add with an LDS
// atomic per lane and sum.
// A wavefront keeps runs at all only if its stretch is longer than `turns` turns
// of 64 and its first slots are in order (RUN_ORDERED neighbours in one bin);
// else every lane adds by itself throughout.  Calls with runs and without, in
// us: slice sums of 20011 sorted slots (one turn) 40 and 35, of 2^19 (two) 46
// and 67; of 2^22 slots in no order 100 and 89; the current of 2^20 sorted slots
// (four turns, one sum: little to gain) 41 and 37, of 2^22 (sixteen) 63 and 78.
constexpr int BIN_THREADS = 256;
constexpr int RUN_MIN = 16;
constexpr int RUN_ORDERED = 48;

// Slots of a wavefront's stretch.
__device__ __forceinline__ int64_t wave_stretch(int64_t n) {
    const int64_t nw = (int64_t)gridDim.x * (BIN_THREADS / 64);
    return (n + nw * 64 - 1) / (nw * 64) * 64;
}

// All wavefront-uniform but the values.
template <int NV>
struct RunSums {
    double v[NV] = {};
    int bin = -1;   // -1: none yet
    bool on;        // keeps runs
    bool first;     // of the stretch
    __device__ __forceinline__ RunSums(int64_t n, int turns) : on(wave_stretch(n) > 64 * turns), first(true) {}
};

// acc[k * stride + bin] += the wavefront's sums, and start anew.
template <int NV>
__device__ __forceinline__ void run_flush(RunSums<NV>& r, double* sh, int stride) {
    if (r.bin < 0) return;
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        const double t = wave_sum(r.v[k]);
        if (lane == 0 && t != 0.0) atomicAdd(&sh[k * stride + r.bin], t);
        r.v[k] = 0.0;
    }
}

// Adds the lanes' values x (bin < 0: none) to their bins.  All lanes call.
template <int NV>
__device__ __forceinline__ void run_add(RunSums<NV>& r, int bin, const double (&x)[NV], double* sh, int stride) {
    const int lane = threadIdx.x & 63;
    bool alone = bin >= 0;
    if (r.on && r.first) r.on = __builtin_popcountll(__ballot(bin == __shfl_up(bin, 1, 64))) >= RUN_ORDERED;
    r.first = false;
    if (r.on) {
        unsigned long long left = __ballot(bin >= 0);
        for (int peel = 0; left && peel < 2; ++peel) {
            // the lanes of the current bin first, then those of the first other one
            unsigned long long same = __ballot(bin == r.bin) & left;
            if (!same) {
                const int next = __builtin_amdgcn_readlane(bin, __builtin_ctzll(left));
                same = __ballot(bin == next) & left;
                if (__builtin_popcountll(same) < RUN_MIN) break;
                run_flush<NV>(r, sh, stride);
                r.bin = next;
            }
            if ((same >> lane) & 1ull) {
#pragma unroll
                for (int k = 0; k < NV; ++k) r.v[k] += x[k];
            }
            left &= ~same;
        }
        alone = (left >> lane) & 1ull;
    }
    if (alone) {
#pragma unroll
        for (int k = 0; k < NV; ++k) atomicAdd(&sh[k * stride + bin], x[k]);
    }
}

// Calls f(i) for every slot of this wavefront's stretch, with i = -1 on lanes
// past the end: all lanes take every turn.
template <typename F>
__device__ __forceinline__ void for_wave_slots(int64_t n, F f) {
    const int64_t per = wave_stretch(n);
    const int64_t w = (int64_t)blockIdx.x * (BIN_THREADS / 64) + (threadIdx.x >> 6);
    const int64_t end = min(n, (w + 1) * per);
    for (int64_t b = w * per; b < end; b += 64) {
        const int64_t i = b + (threadIdx.x & 63);
        f(i < end ? i : (int64_t)-1);
    }
}

// Slice of getSliceTwiss (ceil(z2 / slice), 1-based; the reference's periodic
// wrap, av_write.f90:505-518), or 0 outside the slices.
__device__ __forceinline__ int slice_of(double z, double slice, int nslices, int periodic) {
    int is = (int)ceil(z / slice);
    if (periodic) {
        if (is >= nslices) is = is - ((int)floor((double)is / (double)nslices) * nslices) + 1;
        return is < 1 ? 0 : is;
    }
    return (is > nslices || is < 1) ? 0 : is;
}

// Per-slice sums sum chi cos(h z2 / 2 rho) w, sum chi sin(...) w and the
// slice charge, with the linear split between slices is and is+1 on a
// temporal mesh (av_write.f90:505-530, 562-572).  acc = [br | bi | sdata].
template <typename R>
__global__ __launch_bounds__(BIN_THREADS) void k_bunching(const double* z2, const R* chi, int64_t n,
                                                          double rho, int harmonic, int nslices,
                                                          double slice, int periodic, double* acc) {
    extern __shared__ double sh[];
    for (int t = threadIdx.x; t < 3 * nslices; t += blockDim.x) sh[t] = 0.0;
    __syncthreads();
    RunSums<3> r(n, 1);    // slice is
    RunSums<2> up(n, 1);   // slice is + 1
    for_wave_slots(n, [&](int64_t i) {
        double x[3] = {0, 0, 0}, x2[2] = {0, 0};
        int bin = -1, bin2 = -1;
        if (i >= 0) {
            const double z = z2[i];
            const int is = slice_of(z, slice, nslices, periodic);
            if (is > 0) {
                const double c = (double)chi[i];
                double sn, cs;
                sincos((double)harmonic * z / (2.0 * rho), &sn, &cs);
                const double w1 = ((is * slice - z) / slice);
                bin = is - 1;
                x[0] = c * cs * w1;
                x[1] = c * sn * w1;
                x[2] = c;
                if (!periodic && is < nslices) {
                    const double w2 = (-((is - 1) * slice - z) / slice);
                    bin2 = is;
                    x2[0] = c * cs * w2;
                    x2[1] = c * sn * w2;
                }
            }
        }
        run_add<3>(r, bin, x, sh, nslices);
        run_add<2>(up, bin2, x2, sh, nslices);
    });
    run_flush<3>(r, sh, nslices);
    run_flush<2>(up, sh, nslices);
    __syncthreads();
    for (int t = threadIdx.x; t < 3 * nslices; t += blockDim.x)
        if (sh[t] != 0.0) atomicAdd(&acc[t], sh[t]);
}

// Per-slice sums of getSliceTwiss for the slices [s0, s0 + nch) of nslices
// (av_write.f90:505-536), in LDS then one global atomic per slice and sum:
// acc[k * nslices + slice] for the NSLICE_SUMS sums, in the order
// chi, chi x, chi y, chi px, -chi py, chi Gamma, chi x^2, chi x px,
// chi px^2, chi py^2, -chi y py, chi y^2, chi Gamma^2 (py is stored as -py,
// hence the signs).  Slice index and periodic wrap as k_bunching.
template <typename R>
__global__ __launch_bounds__(BIN_THREADS) void k_slice_moments(PartPtrs<R> y, const R* chi, int64_t n, int nslices,
                                                               double slice, int periodic, int s0, int nch,
                                                               double* acc) {
    extern __shared__ double sh[];
    for (int t = threadIdx.x; t < NSLICE_SUMS * nch; t += blockDim.x) sh[t] = 0.0;
    __syncthreads();
    RunSums<NSLICE_SUMS> r(n, 1);
    for_wave_slots(n, [&](int64_t i) {
        double v[NSLICE_SUMS];
#pragma unroll
        for (int k = 0; k < NSLICE_SUMS; ++k) v[k] = 0.0;
        int bin = -1;
        if (i >= 0) {
            const int l = slice_of(y.z2[i], slice, nslices, periodic) - 1 - s0;
            if (l >= 0 && l < nch) {
                bin = l;
                const double c = (double)chi[i], x = (double)y.x[i], yy = (double)y.y[i];
                const double px = (double)y.pr[i], py = (double)y.pi[i], g = y.g[i];
                v[0] = c;
                v[1] = c * x;
                v[2] = c * yy;
                v[3] = c * px;
                v[4] = -(c * py);
                v[5] = c * g;
                v[6] = c * x * x;
                v[7] = c * x * px;
                v[8] = c * px * px;
                v[9] = c * py * py;
                v[10] = -(c * yy * py);
                v[11] = c * yy * yy;
                v[12] = c * g * g;
            }
        }
        run_add<NSLICE_SUMS>(r, bin, v, sh, nch);
    });
    run_flush<NSLICE_SUMS>(r, sh, nch);
    __syncthreads();
    for (int t = threadIdx.x; t < NSLICE_SUMS * nch; t += blockDim.x)
        if (sh[t] != 0.0) atomicAdd(&acc[(t / nch) * nslices + s0 + (t % nch)], sh[t]);
}

// Charge binned linearly onto npts nodes spaced sam apart (getCurr,
// av_write.f90:297-368): nodes [p0, p0 + nch) of this launch, in LDS.  A
// macroparticle outside the nodes (the reference STOPs) adds 1 to
// acc[npts].
template <typename R>
__global__ __launch_bounds__(BIN_THREADS) void k_current(const double* z2, const R* chi, int64_t n, int npts,
                                                         double sam, int periodic, int p0, int nch, double* acc) {
    extern __shared__ double sh[];
    for (int t = threadIdx.x; t < nch; t += blockDim.x) sh[t] = 0.0;
    __syncthreads();
    double bad = 0.0;
    RunSums<1> rl(n, 8), ru(n, 8);   // lower and upper node
    for_wave_slots(n, [&](int64_t i) {
        int lo = 0, hi = 0;
        double x1[1] = {0.0}, x2[1] = {0.0};
        if (i >= 0) {
            const double z = z2[i];
            const int inl = (int)ceil(z / sam);
            const int inu = inl + 1;
            lo = inl;
            hi = inu;
            bool out = inl <= 0;
            if (periodic) {
                if (inu >= npts) hi = inu - (int)floor((double)inu / (double)npts) * npts + 1;
                if (inl >= npts) lo = inl - (int)floor((double)inl / (double)npts) * npts + 1;
            } else {
                out = out || inu > npts;
            }
            if (out) {
                bad += 1.0;
                lo = hi = 0;
            } else {
                const double li2 = (z - (double)(inl - 1) * sam) / sam;
                const double c = (double)chi[i];
                x1[0] = (1.0 - li2) * c;
                x2[0] = li2 * c;
            }
        }
        const int bl = lo - 1 - p0, bu = hi - 1 - p0;
        run_add<1>(rl, (lo > 0 && bl >= 0 && bl < nch) ? bl : -1, x1, sh, nch);
        run_add<1>(ru, (hi > 0 && bu >= 0 && bu < nch) ? bu : -1, x2, sh, nch);
    });
    run_flush<1>(rl, sh, nch);
    run_flush<1>(ru, sh, nch);
    __syncthreads();
    for (int t = threadIdx.x; t < nch; t += blockDim.x)
        if (sh[t] != 0.0) atomicAdd(&acc[p0 + t], sh[t]);
    bad = wave_sum(bad);
    if (p0 == 0 && (threadIdx.x & 63) == 0 && bad > 0.0) atomicAdd(&acc[npts], bad);
}

// Split FP64 arrays of the caller to the mesh's interleaved field and back:
// both ways bound by their own bytes (32 per node in the FP64 form).
template <typename R>
__global__ __launch_bounds__(256) void k_pack(const double* ar, const double* ai, cplx<R>* a, int64_t n,
                                              int64_t alias_from) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const int64_t j = i < alias_from ? i : i - alias_from;
        a[i] = {(R)ar[j], (R)ai[j]};
    }
}

template <typename R>
__global__ __launch_bounds__(256) void k_unpack(const cplx<R>* a, double* ar, double* ai, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const cplx<R> v = a[i];
        if (ar) ar[i] = (double)v.x;
        if (ai) ai[i] = (double)v.y;
    }
}

template <typename R>
__global__ void k_convert(const double* s, R* d, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = (R)s[i];
}

template <typename R>
__global__ void k_convert_back(const R* s, double* d, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = (double)s[i];
}

__global__ void k_fill_zero(double* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

static dim3 grid_for(int64_t n) { return dim3((unsigned)((n + 255) / 256 > 0 ? (n + 255) / 256 : 1)); }

__global__ void k_store_words(uint32_t* dst, Words64 src, int n) {
    const int t = threadIdx.x;
    if (t < n) dst[t] = src.w[t];
}

__global__ __launch_bounds__(256) void k_copy_sections(CopySections c) {
    const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nth = (int64_t)gridDim.x * blockDim.x;
    for (int s = 0; s < c.n; ++s) {
        const int64_t n16 = c.bytes[s] / 16;
        const uint4* sp = reinterpret_cast<const uint4*>(c.src[s]);
        uint4* dp = reinterpret_cast<uint4*>(c.dst[s]);
        for (int64_t i = tid; i < n16; i += nth) dp[i] = sp[i];
        const int64_t rem = (c.bytes[s] - n16 * 16) / 4;
        const uint32_t* s4 = reinterpret_cast<const uint32_t*>(c.src[s] + n16 * 16);
        uint32_t* d4 = reinterpret_cast<uint32_t*>(c.dst[s] + n16 * 16);
        for (int64_t i = tid; i < rem; i += nth) d4[i] = s4[i];
    }
}

void launch_copy_sections(const CopySections& c, hipStream_t s) {
    int64_t total = 0;
    for (int k = 0; k < c.n; ++k) total += c.bytes[k] / 16;
    int64_t blocks = (total + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_copy_sections, dim3((unsigned)blocks), dim3(256), 0, s, c);
}

void launch_store_words(uint32_t* dst, const Words64& src, int nwords, hipStream_t s) {
    hipLaunchKernelGGL(k_store_words, dim3(1), dim3(64), 0, s, dst, src, nwords);
}

void launch_fill_zero(double* p, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_fill_zero, grid_for(n), dim3(256), 0, s, p, n);
}

template <typename R>
void launch_power(const cplx<R>* a, int nx, int ny, int nz2, double dx, double dy, double* out,
                  hipStream_t s) {
    hipLaunchKernelGGL((k_power<R>), dim3(nz2), dim3(256), 0, s, a, nx, ny, dx, dy, out);
}

template <typename R>
void launch_bunching(const double* z2, const R* chi, int64_t n, double rho, int harmonic,
                     int nslices, double slice, int periodic, double* acc, hipStream_t s) {
    int64_t blocks = (n + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL((k_bunching<R>), dim3((unsigned)blocks), dim3(256),
                       3 * (size_t)nslices * sizeof(double), s, z2, chi, n, rho, harmonic, nslices,
                       slice, periodic, acc);
}

template <typename R>
void launch_slice_moments(PartPtrs<R> y, const R* chi, int64_t n, int nslices, double slice, int periodic,
                          double* acc, hipStream_t s) {
    int64_t blocks = (n + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    if (blocks < 1) blocks = 1;
    for (int s0 = 0; s0 < nslices; s0 += SLICE_CHUNK) {
        const int nch = nslices - s0 < SLICE_CHUNK ? nslices - s0 : SLICE_CHUNK;
        hipLaunchKernelGGL((k_slice_moments<R>), dim3((unsigned)blocks), dim3(256),
                           (size_t)NSLICE_SUMS * nch * sizeof(double), s, y, chi, n, nslices, slice, periodic,
                           s0, nch, acc);
    }
}

template <typename R>
void launch_current(const double* z2, const R* chi, int64_t n, int npts, double sam, int periodic,
                    double* acc, hipStream_t s) {
    int64_t blocks = (n + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    if (blocks < 1) blocks = 1;
    for (int p0 = 0; p0 < npts; p0 += CURRENT_CHUNK) {
        const int nch = npts - p0 < CURRENT_CHUNK ? npts - p0 : CURRENT_CHUNK;
        hipLaunchKernelGGL((k_current<R>), dim3((unsigned)blocks), dim3(256), (size_t)nch * sizeof(double), s,
                           z2, chi, n, npts, sam, periodic, p0, nch, acc);
    }
}

template <typename R>
void launch_pack_field(const double* ar, const double* ai, cplx<R>* a, int64_t n, int64_t alias_from, hipStream_t s) {
    hipLaunchKernelGGL((k_pack<R>), grid_for(n), dim3(256), 0, s, ar, ai, a, n, alias_from);
}
template <typename R>
void launch_unpack_field(const cplx<R>* a, double* ar, double* ai, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL((k_unpack<R>), grid_for(n), dim3(256), 0, s, a, ar, ai, n);
}
template <typename R>
void launch_convert(const double* src, R* dst, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL((k_convert<R>), grid_for(n), dim3(256), 0, s, src, dst, n);
}
template <typename R>
void launch_convert_back(const R* src, double* dst, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL((k_convert_back<R>), grid_for(n), dim3(256), 0, s, src, dst, n);
}

#define PUFF_INST(R)                                                                              \
    template void launch_power<R>(const cplx<R>*, int, int, int, double, double, double*,          \
                                  hipStream_t);                                                   \
    template void launch_bunching<R>(const double*, const R*, int64_t, double, int, int, double,  \
                                     int, double*, hipStream_t);                                  \
    template void launch_slice_moments<R>(PartPtrs<R>, const R*, int64_t, int, double, int,       \
                                          double*, hipStream_t);                                  \
    template void launch_current<R>(const double*, const R*, int64_t, int, double, int, double*,  \
                                    hipStream_t);                                                 \
    template void launch_pack_field<R>(const double*, const double*, cplx<R>*, int64_t, int64_t,  \
                                       hipStream_t);                                              \
    template void launch_unpack_field<R>(const cplx<R>*, double*, double*, int64_t, hipStream_t); \
    template void launch_convert<R>(const double*, R*, int64_t, hipStream_t);                     \
    template void launch_convert_back<R>(const R*, double*, int64_t, hipStream_t);
PUFF_INST(double)
PUFF_INST(float)
#undef PUFF_INST

}  // namespace puff
