// Batched mixed-radix complex FFT along one axis of the field mesh, and the
// diffraction step built from it.
//
// Convention of the reference's FFTW plans (transforms.f90:186-211, 423):
// sign -1 forward, +1 backward, unnormalised; the backward result is divided
// by ffact = NX NY NZ2' afterwards (diffraction.f90:310, 513).
//
// Routes by line length: z2 lines of a power of two from 128 to 4096 in
// registers (k_fft_zreg); transverse lines of 257 points by Rader's algorithm in
// registers (k_rader_x, k_rader_y); all others as whole lines in LDS, a
// workgroup B of them, in Stockham passes (natural order in and out), one LDS
// round trip each: compiled plans for 33 and 129 points, and runtime plans of
// passes of 2 to 16 points, a large prime on the matrix cores, or direct sums
// for what is larger still (line_plan).
//
// DiffractionStep (diffraction.f90:209-348) becomes nine line passes:
//   x fwd | y fwd | z fwd . multiplyexp . z inv | y inv |
//   x inv . /ffact . mask split . x fwd | y fwd | z fwd . damping . z inv |
//   y inv | x inv . /ffact . + interior
#include "puff_common.hpp"
#include "puff_kernels.hpp"

namespace puff {

// Threads per z2 workgroup.  512 and 1024 (more loads in flight per line
// at the same LDS) measured 6 % and 30 % slower on the C1 mesh in FP64;
// 512 gained 2 % on the C4 mesh.
#ifndef PUFF_Z_THREADS
#define PUFF_Z_THREADS 256
#endif
// LDS index of element j of line b.  Interleaved layout (b fastest) keeps
// the strided y / z2 loads conflict free; line-major suits contiguous x lines.
template <bool IL>
__device__ __forceinline__ int lidx(int b, int j, int B, int N) {
    return lpad<IL>(IL ? j * B + b : b * N + j);
}

// Line staging between global memory and LDS with U loads (or stores) per
// thread issued back to back.  A plain element loop (U = 1) writes each
// loaded value to LDS before it issues the next load, so every thread has
// one load in flight and pays the memory latency once per element.  U = 8
// took C4's x and y passes from 4.69 and 3.37 ms to 4.25 and 2.66 ms, and
// (with the XCD-grouped z2 workgroups) C1's FP64 event from 2.47 to 2.40 ms
// through its z2 passes.
constexpr int STAGE_UNROLL = 8;
#ifndef PUFF_Z_UNROLL
#define PUFF_Z_UNROLL 8
#endif

// dst[lpad<IL>(w)] = get(w) for 0 <= w < n.
template <bool IL, int U, typename R, typename F>
__device__ __forceinline__ void lds_fill(cplx<R>* dst, int n, F get) {
    for (int w0 = threadIdx.x; w0 < n; w0 += U * (int)blockDim.x) {
        cplx<R> v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int w = w0 + u * (int)blockDim.x;
            v[u] = (w < n) ? get(w) : cplx<R>{0, 0};
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int w = w0 + u * (int)blockDim.x;
            if (w < n) dst[lpad<IL>(w)] = v[u];
        }
    }
}

// put(w, src[lpad<IL>(w)]) for 0 <= w < n.  The LDS reads are unconditional
// (element 0 stands in past n), so that v stays in registers: with
// conditional reads the compiler kept v in scratch memory (144 bytes per
// lane in FP64).
template <bool IL, int U, typename R, typename F>
__device__ __forceinline__ void lds_drain(const cplx<R>* src, int n, F put) {
    for (int w0 = threadIdx.x; w0 < n; w0 += U * (int)blockDim.x) {
        cplx<R> v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int w = w0 + u * (int)blockDim.x;
            v[u] = src[lpad<IL>(w < n ? w : 0)];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int w = w0 + u * (int)blockDim.x;
            if (w < n) put(w, v[u]);
        }
    }
}

// threadIdx.x through an empty asm statement: index arithmetic built on it is
// not merged with the same arithmetic of another call site, so it is
// recomputed where it is used instead of held in registers between the
// passes of a kernel (with two in-place Rader transforms per line, 181
// VGPRs without it).
__device__ __forceinline__ int opaque_tid() {
    int t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

template <typename R>
__device__ __forceinline__ cplx<R> tw_get(const cplx<R>* tw, int e, int sign) {
    cplx<R> w = tw[e];
    if (sign > 0) w.y = -w.y;
    return w;
}

// Index of X_k in dft16's output.
__host__ __device__ constexpr int dft16_at(int k) { return 4 * (k & 3) + (k >> 2); }
template <typename R>
__device__ __forceinline__ void dft16(cplx<R>* v, R sg);

// ---- DFTs of up to 16 points in registers ---------------------------------------
// In place, natural order in; on return X_q stands at at(q).  The sign enters as
// the factor sg = -1 or +1 of the sines, in FMAs that round the same value.
template <int RR>
struct OddTable;   // cos and sin of 2 pi m / RR, m = 1 .. (RR - 1) / 2
template <>
struct OddTable<3> {
    static constexpr double c[] = {-0.5};
    static constexpr double s[] = {0.86602540378443864676};
};
template <>
struct OddTable<5> {
    static constexpr double c[] = {0.3090169943749474241, -0.8090169943749474241};
    static constexpr double s[] = {0.95105651629515357212, 0.58778525229247312917};
};
template <>
struct OddTable<7> {
    static constexpr double c[] = {0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624};
    static constexpr double s[] = {0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048};
};
template <>
struct OddTable<11> {
    static constexpr double c[] = {0.84125353283118116886, 0.41541501300188642553, -0.14231483827328514044, -0.65486073394528506406, -0.95949297361449738989};
    static constexpr double s[] = {0.54064081745559758211, 0.90963199535451837141, 0.98982144188093273238, 0.75574957435425828377, 0.28173255684142969771};
};
template <>
struct OddTable<13> {
    static constexpr double c[] = {0.8854560256532098959, 0.56806474673115580251, 0.12053668025532305335, -0.35460488704253562597, -0.74851074817110109863, -0.97094181742605202716};
    static constexpr double s[] = {0.46472317204376854566, 0.82298386589365639458, 0.9927088740980539928, 0.93501624268541482344, 0.66312265824079520238, 0.23931566428755776715};
};

template <typename R>
__device__ __forceinline__ cplx<R> plus_i(const cplx<R>& a, const cplx<R>& b, R sg) {   // a + i sg b
    return {fma(-sg, b.y, a.x), fma(sg, b.x, a.y)};
}

// An odd prime, folded as in direct_pass.
template <typename R, int RR>
__device__ __forceinline__ void dft_odd(cplx<R>* v, R sg) {
    constexpr int h = (RR - 1) / 2;
    cplx<R> u[h + 1], d[h + 1];
#pragma unroll
    for (int j = 1; j <= h; ++j) {
        u[j] = cadd(v[j], v[RR - j]);
        d[j] = csub(v[j], v[RR - j]);
    }
    const cplx<R> y0 = v[0];
    cplx<R> sum = y0;
#pragma unroll
    for (int j = 1; j <= h; ++j) sum = cadd(sum, u[j]);
    v[0] = sum;
#pragma unroll
    for (int q = 1; q <= h; ++q) {
        cplx<R> c = y0, t = {0, 0};
#pragma unroll
        for (int j = 1; j <= h; ++j) {
            const int m = (j * q) % RR;
            const R cc = (R)OddTable<RR>::c[(m <= h ? m : RR - m) - 1];
            const R ss = (R)(m <= h ? OddTable<RR>::s[m - 1] : -OddTable<RR>::s[RR - m - 1]);
            c = {fma(u[j].x, cc, c.x), fma(u[j].y, cc, c.y)};
            t = {fma(d[j].x, ss, t.x), fma(d[j].y, ss, t.y)};
        }
        v[q] = plus_i(c, t, sg);
        v[RR - q] = plus_i(c, t, -sg);
    }
}

template <typename R, int RR>
struct SmallDft {
    static constexpr int at(int q) { return q; }
    static __device__ __forceinline__ void run(cplx<R>* v, R sg) { dft_odd<R, RR>(v, sg); }
};
template <typename R>
struct SmallDft<R, 2> {
    static constexpr int at(int q) { return q; }
    static __device__ __forceinline__ void run(cplx<R>* v, R) {
        const cplx<R> t = v[0];
        v[0] = cadd(t, v[1]);
        v[1] = csub(t, v[1]);
    }
};
template <typename R>
struct SmallDft<R, 4> {
    static constexpr int at(int q) { return q; }
    static __device__ __forceinline__ void run(cplx<R>* v, R sg) {
        const cplx<R> a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]);
        const cplx<R> b0 = cadd(v[1], v[3]), b1 = csub(v[1], v[3]);
        v[0] = cadd(a0, b0);
        v[1] = plus_i(a1, b1, sg);
        v[2] = csub(a0, b0);
        v[3] = plus_i(a1, b1, -sg);
    }
};
// N1 N2 points with a rotation between the steps: n = N2 n1 + n2, X at
// q = q1 + N1 q2.
template <typename R>
struct SmallDft<R, 8> {
    static constexpr int at(int q) { return q; }
    static __device__ __forceinline__ void run(cplx<R>* v, R sg) {
        const R h = (R)0.70710678118654752440;
        cplx<R> e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
        SmallDft<R, 4>::run(e, sg);
        SmallDft<R, 4>::run(o, sg);
        const cplx<R> z = {0, 0};
        o[1] = cmul(o[1], cplx<R>{h, sg * h});
        o[2] = plus_i(z, o[2], sg);
        o[3] = cmul(o[3], cplx<R>{-h, sg * h});
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = cadd(e[k], o[k]);
            v[4 + k] = csub(e[k], o[k]);
        }
    }
};
template <typename R>
struct SmallDft<R, 9> {
    static constexpr int at(int q) { return q; }
    static __device__ __forceinline__ void run(cplx<R>* v, R sg) {
        cplx<R> t[3][3];
#pragma unroll
        for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
            for (int n1 = 0; n1 < 3; ++n1) t[n2][n1] = v[3 * n1 + n2];
            dft_odd<R, 3>(t[n2], sg);
        }
        const cplx<R> w1 = {(R)0.7660444431189780352, sg * (R)0.64278760968653932632}, w2 = {(R)0.17364817766693034885, sg * (R)0.98480775301220805937};
        const cplx<R> w4 = {(R)-0.93969262078590838405, sg * (R)0.34202014332566873304};
        t[1][1] = cmul(t[1][1], w1);
        t[1][2] = cmul(t[1][2], w2);
        t[2][1] = cmul(t[2][1], w2);
        t[2][2] = cmul(t[2][2], w4);
#pragma unroll
        for (int q1 = 0; q1 < 3; ++q1) {
            cplx<R> x[3] = {t[0][q1], t[1][q1], t[2][q1]};
            dft_odd<R, 3>(x, sg);
#pragma unroll
            for (int q2 = 0; q2 < 3; ++q2) v[q1 + 3 * q2] = x[q2];
        }
    }
};
template <typename R>
struct SmallDft<R, 16> {
    static constexpr int at(int q) { return dft16_at(q); }
    static __device__ __forceinline__ void run(cplx<R>* v, R sg) { dft16(v, sg); }
};
// N1 N2 points, coprime: n = N2 n1 + N1 n2 and the Chinese remainders q1, q2 of
// q need no rotations.
template <typename R, int N1, int N2>
struct CoprimeDft {
    static constexpr int at(int q) { return q; }
    static __device__ __forceinline__ void run(cplx<R>* v, R sg) {
        constexpr int N = N1 * N2;
        cplx<R> t[N2][N1];
#pragma unroll
        for (int n2 = 0; n2 < N2; ++n2) {
#pragma unroll
            for (int n1 = 0; n1 < N1; ++n1) t[n2][n1] = v[(N2 * n1 + N1 * n2) % N];
            SmallDft<R, N1>::run(t[n2], sg);
        }
#pragma unroll
        for (int q1 = 0; q1 < N1; ++q1) {
            cplx<R> x[N2];
#pragma unroll
            for (int n2 = 0; n2 < N2; ++n2) x[n2] = t[n2][q1];
            SmallDft<R, N2>::run(x, sg);
#pragma unroll
            for (int q = 0; q < N; ++q)
                if (q % N1 == q1) v[q] = x[q % N2];
        }
    }
};
template <typename R>
struct SmallDft<R, 6> : CoprimeDft<R, 2, 3> {};
template <typename R>
struct SmallDft<R, 10> : CoprimeDft<R, 2, 5> {};
template <typename R>
struct SmallDft<R, 12> : CoprimeDft<R, 4, 3> {};
template <typename R>
struct SmallDft<R, 14> : CoprimeDft<R, 2, 7> {};
template <typename R>
struct SmallDft<R, 15> : CoprimeDft<R, 3, 5> {};

// 4-point DFT in place (x_k = sum_n x_n W4^(nk), W4 = exp(sg 2 pi i / 4)).
template <typename R>
__device__ __forceinline__ void dft4(cplx<R>& x0, cplx<R>& x1, cplx<R>& x2, cplx<R>& x3, R sg) {
    cplx<R> v[4] = {x0, x1, x2, x3};
    SmallDft<R, 4>::run(v, sg);
    x0 = v[0];
    x1 = v[1];
    x2 = v[2];
    x3 = v[3];
}

// 16-point DFT in registers as 4 x 4 (Cooley-Tukey): with j = 4 j1 + j0 and
// q = q0 + 4 q1, X_q = sum_j0 W4^(j0 q1) [w^(j0 q0) sum_j1 v_(4 j1 + j0) W4^(j1 q0)],
// w = exp(sg 2 pi i / 16).  On return v[4 q0 + q1] = X_(q0 + 4 q1).
template <typename R>
__device__ __forceinline__ void dft16(cplx<R>* v, R sg) {
    const R c1 = (R)0.92387953251128675613, s1 = (R)0.38268343236508977173;   // cos, sin of pi/8
    const R c2 = (R)0.70710678118654752440;                                    // cos pi/4
#pragma unroll
    for (int j0 = 0; j0 < 4; ++j0) dft4(v[j0], v[4 + j0], v[8 + j0], v[12 + j0], sg);
    // v[4 q0 + j0] = Y[j0][q0]; twiddle by w^(j0 q0): m = 1, 2, 3 | 2, 4, 6 | 3, 6, 9
    const cplx<R> w1 = {c1, sg * s1}, w2 = {c2, sg * c2}, w3 = {s1, sg * c1};
    const cplx<R> w6 = {-c2, sg * c2}, w9 = {-c1, -sg * s1};
    v[5] = cmul(v[5], w1);
    v[9] = cmul(v[9], w2);
    v[13] = cmul(v[13], w3);
    v[6] = cmul(v[6], w2);
    v[10] = {-sg * v[10].y, sg * v[10].x};   // w^4 = W4
    v[14] = cmul(v[14], w6);
    v[7] = cmul(v[7], w3);
    v[11] = cmul(v[11], w6);
    v[15] = cmul(v[15], w9);
#pragma unroll
    for (int q0 = 0; q0 < 4; ++q0) dft4(v[4 * q0], v[4 * q0 + 1], v[4 * q0 + 2], v[4 * q0 + 3], sg);
}

// ---- compile-time line plans --------------------------------------------------
// The transverse lengths of the workloads get kernels with their length, radix
// passes (factorize()'s order) and lines per workgroup as constants: every
// index division and modulo by B, T, p and N then becomes a multiply and
// shift, and the pass loops unroll.  Other lengths take a runtime plan
// (NC = 0).  A diffraction step with them and by the runtime plans (129 with
// its 43 on the matrix cores): 129 x 129 x 1024 1642 and 1815 us (FP64), 950
// and 1033 us (mixed); 33 x 33 x 256 82 and 115 us, 81 and 99 us.
template <int N>
struct CtPlan {
    static constexpr int np = 0;
    static constexpr int r[1] = {0};
};
#define PUFF_CT_PLAN(N_, ...)                                 \
    template <>                                               \
    struct CtPlan<N_> {                                       \
        static constexpr int r[] = {__VA_ARGS__};             \
        static constexpr int np = sizeof(r) / sizeof(int);    \
    };
PUFF_CT_PLAN(33, 11, 3)
PUFF_CT_PLAN(129, 43, 3)
#undef PUFF_CT_PLAN

// Quotients of 0 <= a < 2^16 by 1 <= d < 2^13: the high word of a ceil(2^32 / d).
struct Div {
    uint32_t m;   // 0: d = 1
};
__device__ __forceinline__ Div div_by(int d) { return {d > 1 ? 0xffffffffu / (uint32_t)d + 1 : 0}; }
__device__ __forceinline__ int over(int a, Div d) { return d.m ? (int)__umulhi((uint32_t)a, d.m) : a; }

// Line b and butterfly i (of T) of work item w: b fastest in interleaved buffers.
template <bool IL>
__device__ __forceinline__ void pass_item(int w, int B, Div by_b, int T, Div by_t, int& b, int& i) {
    if (IL) {
        i = over(w, by_b);
        b = w - i * B;
    } else {
        b = over(w, by_t);
        i = w - b * T;
    }
}

// Direct DFT pass for an odd prime r (a radix pass of lds_pass), folded:
// with the pre-twiddled inputs y_j = x_j W^(j k twst), u_j = y_j + y_(r-j),
// v_j = y_j - y_(r-j) (j = 1 .. (r-1)/2) and w^(jq) = c + i s
// (w^((r-j)q) = c - i s),
//   X_q     = y_0 + sum u_j c + i sum v_j s
//   X_(r-q) = y_0 + sum u_j c - i sum v_j s,
// four FMAs per input pair for both outputs.  Each work item forms the
// outputs of NQ consecutive values of q (with their mirrors r - q), sharing
// the input loads, the folding and the loop bookkeeping: per input pair it
// reads 2 inputs and NQ rotations from LDS for 4 NQ FMAs.  The pass is bound
// by LDS reads; q >= (r + 1) / 2 slots of the last item read a valid table
// entry (q = 0) and store nothing.
#ifndef PUFF_DFT_WIDE
#define PUFF_DFT_WIDE 4
#endif
#ifndef PUFF_DFT_WIDE_MIN
#define PUFF_DFT_WIDE_MIN 23
#endif
template <typename R, bool IL, int NQ>
__device__ __forceinline__ void direct_pass(const cplx<R>* src, cplx<R>* dst, int B, int LD, int N, int r,
                                            int p, const cplx<R>* tw, int sign) {
    const int T = N / r;
    const int twst = N / (p * r);
    const int nr = N / r;
    const int hq = (r + 1) / 2;
    const int nqq = (hq + NQ - 1) / NQ;
    const Div by_b = div_by(B), by_t = div_by(T), by_tq = div_by(T * nqq), by_p = div_by(p);
    for (int w = threadIdx.x; w < B * T * nqq; w += blockDim.x) {
        int b, t;
        pass_item<IL>(w, B, by_b, T * nqq, by_tq, b, t);
        const int qq = over(t, by_t);
        const int q0 = NQ * qq;
        const int i = t - qq * T;
        const int k = i - over(i, by_p) * p;
        const int dk = k * twst;
        int dq[NQ], f[NQ];
#pragma unroll
        for (int m = 0; m < NQ; ++m) {
            dq[m] = (q0 + m < hq) ? (q0 + m) * nr : 0;   // 0: a valid table index, result unused
            f[m] = dq[m];
        }
        const cplx<R> y0 = src[lidx<IL>(b, i, B, LD)];
        int e1 = dk, e2 = (r - 1) * dk;   // e1, e2 < N throughout
        R sr[NQ], si[NQ], tr[NQ], ti[NQ];
#pragma unroll
        for (int m = 0; m < NQ; ++m) sr[m] = si[m] = tr[m] = ti[m] = (R)0;
        constexpr int UJ = NQ >= 4 ? 2 : 4;
#pragma unroll UJ
        for (int j = 1; j < hq; ++j) {
            cplx<R> xa = src[lidx<IL>(b, i + j * T, B, LD)];
            cplx<R> xb = src[lidx<IL>(b, i + (r - j) * T, B, LD)];
            if (dk) {
                xa = cmul(xa, tw_get(tw, e1, sign));
                xb = cmul(xb, tw_get(tw, e2, sign));
            }
            const R ux = xa.x + xb.x, uy = xa.y + xb.y;
            const R vx = xa.x - xb.x, vy = xa.y - xb.y;
#pragma unroll
            for (int m = 0; m < NQ; ++m) {
                const cplx<R> o = tw_get(tw, f[m], sign);
                sr[m] = fma(ux, o.x, sr[m]);
                si[m] = fma(uy, o.x, si[m]);
                tr[m] = fma(vx, o.y, tr[m]);
                ti[m] = fma(vy, o.y, ti[m]);
                f[m] += dq[m];
                if (f[m] >= N) f[m] -= N;
            }
            e1 += dk;
            e2 -= dk;
        }
        const int ob = (i - k) * r + k;
#pragma unroll
        for (int m = 0; m < NQ; ++m) {
            const int q = q0 + m;
            if (q < hq) {
                dst[lidx<IL>(b, ob + q * p, B, LD)] = {y0.x + sr[m] - ti[m], y0.y + si[m] + tr[m]};
                if (q > 0) dst[lidx<IL>(b, ob + (r - q) * p, B, LD)] = {y0.x + sr[m] + ti[m], y0.y + si[m] - tr[m]};
            }
        }
    }
}

// LDS read of a complex value at a byte offset from base, as one 2-vector
// whose alignment is its size: one ds_read_b128 (FP64) or ds_read_b64
// (FP32) whose 16-bit offset field takes the compile-time part of the
// address.  A cplx<double> read (8-byte aligned) becomes ds_read2_b64,
// whose offsets reach only 2040 bytes.
template <typename R>
struct Vec2;
template <>
struct Vec2<double> {
    typedef double __attribute__((ext_vector_type(2))) T;
};
template <>
struct Vec2<float> {
    typedef float __attribute__((ext_vector_type(2))) T;
};
template <typename R>
__device__ __forceinline__ cplx<R> lds_at(const cplx<R>* base, uint32_t byte_off) {
    const typename Vec2<R>::T v =
        *reinterpret_cast<const typename Vec2<R>::T*>(reinterpret_cast<const char*>(base) + byte_off);
    return {v.x, v.y};
}

// direct_pass for a compile-time radix RR of a compile-time line length N,
// after passes whose radices multiply to P (same arithmetic, bit for bit):
// - the j loop has a compile-time trip count and unrolls in groups;
// - the rotations w^(jq) are read from the forward table and the sign
//   applied to the s sums at the end (X_q takes +-i sum v s; negation is
//   exact and commutes with the FMA rounding), instead of a conditional
//   negate per rotation;
// - each rotation's table offset is kept in bytes and advanced by q nr with
//   one unsigned min for the wrap at N (a + d and a + d - N: the one below N
//   is the smaller as unsigned), instead of add, compare, select and an
//   address computation.
template <typename R, bool IL, int NQ, int N, int RR, int P>
__device__ __forceinline__ void direct_pass_ct(const cplx<R>* src, cplx<R>* dst, int B, const cplx<R>* tw,
                                               int sign) {
    constexpr int T = N / RR;
    constexpr int twst = N / (P * RR);
    constexpr int nr = N / RR;
    constexpr int hq = (RR + 1) / 2;
    constexpr int nqq = (hq + NQ - 1) / NQ;
    constexpr uint32_t ES = sizeof(cplx<R>);
    constexpr uint32_t WRAP = (uint32_t)N * ES;
    for (int w = threadIdx.x; w < B * T * nqq; w += blockDim.x) {
        int b, t;
        if (IL) { b = w % B; t = w / B; } else { t = w % (T * nqq); b = w / (T * nqq); }
        const int q0 = NQ * (t / T);
        const int i = t % T;
        const int k = i % P;
        const int dk = k * twst;
        uint32_t ofs[NQ], stp[NQ], stw[NQ];
#pragma unroll
        for (int m = 0; m < NQ; ++m) {
            // q >= hq: offset 0 throughout (a valid table entry, result unused)
            stp[m] = (q0 + m < hq) ? (uint32_t)((q0 + m) * nr) * ES : 0u;
            stw[m] = stp[m] - WRAP;
            ofs[m] = stp[m];
        }
        const uint32_t la = (uint32_t)lidx<IL>(b, i, B, N) * ES;
        const cplx<R> y0 = lds_at(src, la);
        R sr[NQ], si[NQ], tr[NQ], ti[NQ];
#pragma unroll
        for (int m = 0; m < NQ; ++m) sr[m] = si[m] = tr[m] = ti[m] = (R)0;
        // unrolled in groups (a full unroll hoists every LDS read and takes
        // ~490 VGPRs); the groups' reads take their offsets from the
        // instruction
        constexpr int UJ = (hq - 1) <= 6 ? (hq - 1) : ((hq - 1) % 3 == 0 ? 3 : 2);
#pragma unroll UJ
        for (int j = 1; j < hq; ++j) {
            cplx<R> o[NQ];
#pragma unroll
            for (int m = 0; m < NQ; ++m) {
                o[m] = lds_at(tw, ofs[m]);
                ofs[m] = min(ofs[m] + stp[m], ofs[m] + stw[m]);
            }
            // interleaved lines: element i + j T of line b sits j T B
            // elements after element i
            cplx<R> xa = IL ? lds_at(src, la + (uint32_t)(j * T * B) * ES)
                            : lds_at(src, (uint32_t)lidx<IL>(b, i + j * T, B, N) * ES);
            cplx<R> xb = IL ? lds_at(src, la + (uint32_t)((RR - j) * T * B) * ES)
                            : lds_at(src, (uint32_t)lidx<IL>(b, i + (RR - j) * T, B, N) * ES);
            if constexpr (P > 1) {
                if (dk) {   // exponents j dk, (RR - j) dk < N
                    xa = cmul(xa, tw_get(tw, j * dk, sign));
                    xb = cmul(xb, tw_get(tw, (RR - j) * dk, sign));
                }
            }
            const R ux = xa.x + xb.x, uy = xa.y + xb.y;
            const R vx = xa.x - xb.x, vy = xa.y - xb.y;
#pragma unroll
            for (int m = 0; m < NQ; ++m) {
                sr[m] = fma(ux, o[m].x, sr[m]);
                si[m] = fma(uy, o[m].x, si[m]);
                tr[m] = fma(vx, o[m].y, tr[m]);
                ti[m] = fma(vy, o[m].y, ti[m]);
            }
        }
        const int ob = (i / P) * P * RR + k;
#pragma unroll
        for (int m = 0; m < NQ; ++m) {
            if (sign > 0) {
                tr[m] = -tr[m];
                ti[m] = -ti[m];
            }
            const int q = q0 + m;
            if (q < hq) {
                dst[lidx<IL>(b, ob + q * P, B, N)] = {y0.x + sr[m] - ti[m], y0.y + si[m] + tr[m]};
                if (q > 0) dst[lidx<IL>(b, ob + (RR - q) * P, B, N)] = {y0.x + sr[m] + ti[m], y0.y + si[m] - tr[m]};
            }
        }
    }
}

// One pass of radix RR <= 16 (after passes whose radices multiply to p) of an
// in-LDS mixed-radix transform of length N over elements 0..N-1 of B lines
// laid out with line length LD (N <= LD; elements N..LD-1 are left alone).
// TWO buffers: src to dst, any number of butterflies.  Otherwise in place
// (src = dst): a thread reads its 16 / RR butterflies or fewer into registers,
// the workgroup passes a barrier, and the outputs overwrite the buffer; half
// the LDS, hence more workgroups per CU; B N / RR <= 16 / RR blockDim (checked
// on the host).
template <typename R, bool IL, int RR, bool TWO>
__device__ __forceinline__ void radix_pass(const cplx<R>* src, cplx<R>* dst, int B, int LD, int N, int p,
                                           const cplx<R>* tw, int sign) {
    constexpr int KB = TWO ? 1 : 16 / RR;
    const int T = N / RR;
    const int twst = T / p;   // twiddle exponents j k twst (j < RR, k < p) stay below N: no reduction
    const R sg = (R)sign;
    const Div by_b = div_by(B), by_t = div_by(T), by_p = div_by(p);
    const int tid = opaque_tid();
    for (int w0 = tid; !TWO || w0 < B * T; w0 += (int)blockDim.x) {
        cplx<R> v[KB][RR];
        int b[KB], ob[KB];
#pragma unroll
        for (int it = 0; it < KB; ++it) {
            const int w = w0 + it * (int)blockDim.x;
            int i;
            pass_item<IL>(w < B * T ? w : 0, B, by_b, T, by_t, b[it], i);
            const int k = i - over(i, by_p) * p;
            ob[it] = (i - k) * RR + k;
#pragma unroll
            for (int j = 0; j < RR; ++j) v[it][j] = src[lidx<IL>(b[it], i + j * T, B, LD)];
            if (p > 1) {
#pragma unroll
                for (int j = 1; j < RR; ++j) v[it][j] = cmul(v[it][j], tw_get(tw, j * k * twst, sign));
            }
            SmallDft<R, RR>::run(v[it], sg);
        }
        if (!TWO) __syncthreads();
#pragma unroll
        for (int it = 0; it < KB; ++it) {
            if (!TWO && w0 + it * (int)blockDim.x >= B * T) continue;
#pragma unroll
            for (int q = 0; q < RR; ++q) dst[lidx<IL>(b[it], ob[it] + q * p, B, LD)] = v[it][SmallDft<R, RR>::at(q)];
        }
        if (!TWO) break;
    }
}

// A pass of runtime radix.
template <typename R, bool IL, bool TWO>
__device__ __forceinline__ void lds_pass(const cplx<R>* src, cplx<R>* dst, int B, int LD, int N, int r, int p,
                                         const cplx<R>* tw, int sign) {
    switch (r) {
#define PUFF_RADIX(RR) \
    case RR: return radix_pass<R, IL, RR, TWO>(src, dst, B, LD, N, p, tw, sign);
        PUFF_RADIX(2)
        PUFF_RADIX(3)
        PUFF_RADIX(4)
        PUFF_RADIX(5)
        PUFF_RADIX(6)
        PUFF_RADIX(7)
        PUFF_RADIX(8)
        PUFF_RADIX(9)
        PUFF_RADIX(10)
        PUFF_RADIX(11)
        PUFF_RADIX(12)
        PUFF_RADIX(13)
        PUFF_RADIX(14)
        PUFF_RADIX(15)
        PUFF_RADIX(16)
#undef PUFF_RADIX
        default: break;
    }
    if constexpr (TWO) {
        if (r >= PUFF_DFT_WIDE_MIN) direct_pass<R, IL, PUFF_DFT_WIDE>(src, dst, B, LD, N, r, p, tw, sign);
        else direct_pass<R, IL, 2>(src, dst, B, LD, N, r, p, tw, sign);
    }
}

// ---- the first pass for a large prime, on the matrix cores ------------------------
// direct_pass's folded sums for p = 1 (no input rotations) as two products
//   C = [cos 2 pi j q / r] U,  S = [sin] V,  q = 0 .. h, j = 1 .. h = (r - 1) / 2,
// with one real column per line, butterfly and component: tiles of 16 q by 16
// columns (8 butterflies), four j per MFMA.  Each operand is read once per
// 1024 FMAs instead of once per 4 (direct_pass reads 6 LDS words of 16 bytes
// for 16 FMAs per lane and is bound by that).  In place: the tiles stay in
// accumulators until every input is read; the wavefronts deal the tiles out,
// at most MFMA_TILES each (checked on the host).  A spectral pass over 61 x 47
// lines of 389 points, FP64: 200 -> 124 us (bound by LDS latency at two
// workgroups a CU).
//   Operands: lane l holds A[row l % 16][k = l / 16] and B[k = l / 16][column l % 16];
//   results: column l % 16, row l / 16 + 4 v (FP64) or 4 (l / 16) + v (FP32), v < 4.
template <typename R>
struct Mfma;
template <>
struct Mfma<double> {
    typedef double T __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ T fma(double a, double b, T c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int v) { return (l >> 4) + 4 * v; }
};
template <>
struct Mfma<float> {
    typedef float T __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ T fma(float a, float b, T c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int l, int v) { return 4 * (l >> 4) + v; }
};

template <typename R, bool IL>
__device__ __forceinline__ void mfma_pass(cplx<R>* buf, int B, int N, int r, const cplx<R>* tp, int sign) {
    using M = Mfma<R>;
    const int T = N / r, cols = B * T, h = (r - 1) / 2, qt = (h + 16) / 16;
    const int units = (cols + 7) / 8 * qt;
    const int l = opaque_tid() & 63, k = l >> 4, n = l & 15, part = n & 1;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const Div by_b = div_by(B), by_t = div_by(T), by_q = div_by(qt), by_r = div_by(r);
    const R* in = reinterpret_cast<const R*>(buf);
    typename M::T C[MFMA_TILES], S[MFMA_TILES];
    R y0[MFMA_TILES];
#pragma unroll
    for (int m = 0; m < MFMA_TILES; ++m) {
        C[m] = S[m] = typename M::T{0, 0, 0, 0};
        y0[m] = 0;
        const int unit = wave + 4 * m;
        if (unit < units) {
            const int ct = over(unit, by_q), q = 16 * (unit - ct * qt) + n;
            const int item = 8 * ct + (n >> 1);
            int b, i;
            pass_item<IL>(item < cols ? item : 0, B, by_b, T, by_t, b, i);
            auto at = [&](int j) { return in[2 * lidx<IL>(b, i + j * T, B, N) + part]; };
            y0[m] = at(0);
            const int d0 = (q <= h ? q : 0) * (k + 1), d4 = 4 * (q <= h ? q : 0);
            int e = d0 - over(d0, by_r) * r;
            const int d = d4 - over(d4, by_r) * r;
            for (int j0 = 1; j0 <= h; j0 += 4) {
                const int j = j0 + k, jj = j <= h ? j : 1;
                const R xa = at(jj), xb = at(r - jj);
                const cplx<R> w = tp[e];
                C[m] = M::fma(w.x, j <= h ? xa + xb : (R)0, C[m]);
                S[m] = M::fma(w.y, j <= h ? xa - xb : (R)0, S[m]);
                e += d;
                e = (int)min((uint32_t)e, (uint32_t)(e - r));
            }
        }
    }
    __syncthreads();
    // i S: the other component of the same column, one lane away.  The table
    // is the forward one (sin negated), the sign turns S.
    const R sg = (R)((sign < 0) == (part == 0) ? -1 : 1);
    R* out = reinterpret_cast<R*>(buf);
#pragma unroll
    for (int m = 0; m < MFMA_TILES; ++m) {
        const int unit = wave + 4 * m;
        if (unit < units) {
            const int ct = over(unit, by_q);
            const int item = 8 * ct + (n >> 1);
            int b, i;
            pass_item<IL>(item < cols ? item : 0, B, by_b, T, by_t, b, i);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int q = 16 * (unit - ct * qt) + M::row(l, v);
                const R other = __shfl_xor(S[m][v], 1, 64);
                const R a = y0[m] + C[m][v], t = sg * other;
                if (item < cols && q <= h) {
                    out[2 * lidx<IL>(b, i * r + q, B, N) + part] = a + t;
                    if (q > 0) out[2 * lidx<IL>(b, i * r + r - q, B, N) + part] = a - t;
                }
            }
        }
    }
}

// The rotations of the matrix pass, every N / r-th of the table, side by side in
// LDS: the lanes read them at random, and N / r apart a power of two of them
// would share banks.
template <typename R>
__device__ __forceinline__ const cplx<R>* prime_table(cplx<R>* tp, const cplx<R>* tw, const FftAxis& ax) {
    const int r = ax.radix[0], T = ax.n / r;
    for (int e = threadIdx.x; e < r; e += blockDim.x) tp[e] = tw[e * T];
    return tp;
}

// The passes of a runtime plan.  src holds the input; returns the buffer
// holding the output (src or dst; in place: src).
template <typename R, bool IL, int KIND>
__device__ __forceinline__ cplx<R>* lds_passes(cplx<R>* src, cplx<R>* dst, int B, int LD, int N, int npass,
                                               const int* radix, const cplx<R>* tw, const cplx<R>* tp, int sign) {
    constexpr bool TWO = KIND == LINE_TWO;
    int p = 1, ps = 0;
    if constexpr (KIND == LINE_PRIME) {
        mfma_pass<R, IL>(src, B, N, radix[0], tp, sign);
        __syncthreads();
        p = radix[ps++];
    }
    for (; ps < npass; ++ps) {
        const int r = radix[ps];
        lds_pass<R, IL, TWO>(src, TWO ? dst : src, B, LD, N, r, p, tw, sign);
        __syncthreads();
        if (TWO) {
            cplx<R>* t = src;
            src = dst;
            dst = t;
        }
        p *= r;
    }
    return src;
}

// The passes K.. of CtPlan<NC> (P: product of the earlier radices), with
// the radix and its offsets as constants.
template <typename R, bool IL, int NC, int K = 0, int P = 1>
__device__ __forceinline__ cplx<R>* ct_passes(cplx<R>* src, cplx<R>* dst, int B, int LD, int N,
                                              const cplx<R>* tw, int sign) {
    if constexpr (K == CtPlan<NC>::np) {
        return src;
    } else {
        constexpr int r = CtPlan<NC>::r[K];
        if constexpr (r > 3) {
            constexpr int nq = r >= PUFF_DFT_WIDE_MIN ? PUFF_DFT_WIDE : 2;
            direct_pass_ct<R, IL, nq, NC, r, P>(src, dst, B, tw, sign);
        } else {
            radix_pass<R, IL, r, true>(src, dst, B, LD, N, P, tw, sign);
        }
        __syncthreads();
        return ct_passes<R, IL, NC, K + 1, P * r>(dst, src, B, LD, N, tw, sign);
    }
}

// Rader's algorithm for a prime N with N - 1 = M a power of two (FftAxis):
// a_j = x[g^j], A = DFT_M(a), C = A . rb_s, c = IDFT_M(C) (unnormalised; rb
// carries the 1/M), X[g^-q] = x_0 + c_q, X_0 = x_0 + A_0.  Element M of each
// line buffer is outside the M-point transforms: it keeps x_0 in dst and
// X_0 in src until the final permutation.
template <typename R, bool IL>
__device__ __forceinline__ cplx<R>* lds_rader(cplx<R>* src, cplx<R>* dst, int B, const FftAxis& ax,
                                              const cplx<R>* tw, int sign) {
    const int N = ax.n, M = N - 1;
    const cplx<R>* rb = reinterpret_cast<const cplx<R>*>(ax.rb) + (sign > 0 ? M : 0);
    cplx<R>* P = dst;   // element M: x_0
    cplx<R>* Q = src;   // element M: X_0
    for (int w = threadIdx.x; w < B * N; w += blockDim.x) {
        int b, j;
        if (IL) { b = w % B; j = w / B; } else { j = w % N; b = w / N; }
        P[lidx<IL>(b, j, B, N)] = src[lidx<IL>(b, j < M ? ax.rperm[j] : 0, B, N)];
    }
    __syncthreads();
    cplx<R>* res = lds_passes<R, IL, LINE_TWO>(P, Q, B, N, M, ax.npass, ax.radix, tw, tw, -1);
    for (int w = threadIdx.x; w < B * M; w += blockDim.x) {
        int b, k;
        if (IL) { b = w % B; k = w / B; } else { k = w % M; b = w / M; }
        const cplx<R> v = res[lidx<IL>(b, k, B, N)];
        if (k == 0) {
            const cplx<R> x0 = P[lidx<IL>(b, M, B, N)];
            Q[lidx<IL>(b, M, B, N)] = cadd(x0, v);
        }
        res[lidx<IL>(b, k, B, N)] = cmul(v, rb[k]);
    }
    __syncthreads();
    cplx<R>* other = (res == P) ? Q : P;
    res = lds_passes<R, IL, LINE_TWO>(res, other, B, N, M, ax.npass, ax.radix, tw, tw, +1);
    cplx<R>* out = (res == P) ? Q : P;
    // every output element except element M (which holds x_0 or X_0 in out)
    const int qm = M / 2;   // g^-(M/2) = -1 = M (mod N)
    for (int w = threadIdx.x; w < B * M; w += blockDim.x) {
        int b, q;
        if (IL) { b = w % B; q = w / B; } else { q = w % M; b = w / M; }
        const cplx<R> x0 = P[lidx<IL>(b, M, B, N)];
        if (q == qm) {
            out[lidx<IL>(b, 0, B, N)] = Q[lidx<IL>(b, M, B, N)];
        } else {
            out[lidx<IL>(b, ax.riperm[q], B, N)] = cadd(x0, res[lidx<IL>(b, q, B, N)]);
        }
    }
    __syncthreads();
    for (int b = threadIdx.x; b < B; b += blockDim.x) {
        const cplx<R> x0 = P[lidx<IL>(b, M, B, N)];
        out[lidx<IL>(b, M, B, N)] = cadd(x0, res[lidx<IL>(b, qm, B, N)]);
    }
    __syncthreads();
    return out;
}

// In-LDS transform of B lines of length ax.n.  src holds the input; returns
// the buffer holding the output (src or dst; one buffer: src).
template <typename R, bool IL, int NC, int KIND>
__device__ __forceinline__ cplx<R>* lds_fft(cplx<R>* src, cplx<R>* dst, int B, const FftAxis& ax,
                                            const cplx<R>* tw, const cplx<R>* tp, int sign) {
    if constexpr (NC > 0) {
        return ct_passes<R, IL, NC>(src, dst, B, NC, NC, tw, sign);
    } else {
        if constexpr (KIND == LINE_TWO) {
            if (ax.rader) return lds_rader<R, IL>(src, dst, B, ax, tw, sign);
        }
        return lds_passes<R, IL, KIND>(src, dst, B, ax.n, ax.n, ax.npass, ax.radix, tw, tp, sign);
    }
}

// ---- Rader passes of 257-point transverse lines ------------------------------
// The n-point DFT of a prime n as a cyclic convolution of M = n - 1 = 256
// points: a_k = x[g^k], A = DFT_M(a), C = A . rb_s, c = IDFT_M(C) (rb carries
// the 1/M), X[g^-k] = x_0 + c_k, X_0 = x_0 + A_0.
//
// Sixteen threads hold a line, thread u its elements u + 16 j (j = 0 .. 15) in
// registers, and a workgroup holds BL lines.  With M = 16 x 16,
//   A[q + 16 p] = sum_u W256^(u q) W16^(u p) sum_j a[u + 16 j] W16^(j q),
// the transform is a 16-point DFT per thread, one exchange through LDS, and a
// second one that leaves thread q with A[q + 16 p]; the product with rb and
// the inverse's first 16-point DFT stay in the thread, and a second exchange
// brings c[u + 16 j] back to thread u.  Two LDS round trips and three barriers
// per transform, every thread busy, and the y pass moves its rows between
// memory and registers directly (the permutation moves whole rows of BL
// x-columns).  The x passes turn their lines through LDS in natural order, so
// that memory sees contiguous lines, and apply masks, scalings and the kept
// copies there.
//
// On 257 x 257 x 4096 (FP32) the y pass takes 0.99 ms and the x passes (forward,
// split, recombination) 0.80, 2.25 and 1.33 ms; moving the field once takes
// 0.89 ms at the rate of a large copy.  With the lines in LDS throughout (eight
// per workgroup, half the threads idle in the 16-point passes, seven LDS round
// trips per transform) they took 1.55 and 1.54, 3.31 and 1.80 ms.
constexpr int RAD_N = 257, RAD_M = 256;
constexpr int RAD_LD = 272;   // LDS elements of a line: 256 + 256 / 16, see rad_at

// Lines per workgroup: 35 KiB of LDS in either form, four workgroups per CU.
template <typename R>
constexpr int rad_lines() { return sizeof(R) == 8 ? 8 : 16; }

constexpr int rad_pow(int b, int e) {
    int r = 1;
    for (; e > 0; --e) r = r * b % RAD_N;
    return r;
}
// g^(16 j) for j < 16; inverse powers with b = g^-1
template <int B>
struct RadPowers {
    int v[16];
    constexpr RadPowers() : v() {
        for (int j = 0; j < 16; ++j) v[j] = rad_pow(B, 16 * j);
    }
};
constexpr int RAD_G = 3;                                 // the host's generator of 257 (make_axis)
constexpr int RAD_GI = rad_pow(RAD_G, RAD_M - 1);        // its inverse
static_assert(rad_pow(RAD_G, RAD_M / 2) == RAD_N - 1 && RAD_G * RAD_GI % RAD_N == 1, "primitive root of 257");

// x mod 257 for 0 <= x <= 65536: 256 = -1, so the low byte less the rest, and
// the wrapped one of r and r + 257 is the larger as unsigned.
__device__ __forceinline__ int rad_mod(int x) {
    const unsigned r = (unsigned)(x & 255) - (unsigned)(x >> 8);
    return (int)min(r, r + 257u);
}

// b^u mod 257 for u < 16.
template <int B>
__device__ __forceinline__ int rad_pow16(int u) {
    constexpr int b2 = rad_pow(B, 2), b4 = rad_pow(B, 4), b8 = rad_pow(B, 8);
    int r = (u & 1) ? B : 1;
    r = rad_mod(r * ((u & 2) ? b2 : 1));
    r = rad_mod(r * ((u & 4) ? b4 : 1));
    return rad_mod(r * ((u & 8) ? b8 : 1));
}

// LDS element e of line b.  XL (x lines: the 16 threads of a line
// consecutive): line-major, a spare element after every 16, so that a wave's
// writes (16 consecutive elements of four lines) and reads (elements 16
// apart) each touch every bank once.  Otherwise (y: the BL columns of an
// element consecutive) rows of BL with a spare row after every 16.
template <int BL, bool XL>
__device__ __forceinline__ int rad_at(int b, int e) {
    return XL ? b * RAD_LD + e + (e >> 4) : (e + (e >> 4)) * BL + b;
}

// v[j] = a[u + 16 j] -> v[j] = c[u + 16 j]; returns A_0 (in thread u = 0).
// rb: the table of the transform's sign (global memory, L2).  The buffer may
// be in use when called; every thread has passed a barrier after its last
// read of it, except of its own elements u + 16 j, on return.
template <typename R, int BL, bool XL>
__device__ __forceinline__ cplx<R> rader_core(cplx<R> (&v)[16], int b, int u, cplx<R>* buf, const cplx<R>* tw,
                                              const cplx<R>* rb) {
    dft16(v, (R)-1);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; ++q) {
        const cplx<R> y = q ? cmul(v[dft16_at(q)], tw[u * q]) : v[0];
        buf[rad_at<BL, XL>(b, q * 16 + u)] = y;
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 16; ++t) v[t] = buf[rad_at<BL, XL>(b, u * 16 + t)];
    dft16(v, (R)-1);
    const cplx<R> a0 = v[0];
    cplx<R> c[16];
#pragma unroll
    for (int p = 0; p < 16; ++p) c[p] = cmul(v[dft16_at(p)], rb[u + 16 * p]);
    dft16(c, (R)+1);
    // back to the elements this thread read: no barrier before the writes
#pragma unroll
    for (int t = 0; t < 16; ++t) {
        const cplx<R> y = t ? cmul(c[dft16_at(t)], tw_get(tw, u * t, +1)) : c[0];
        buf[rad_at<BL, XL>(b, u * 16 + t)] = y;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; ++q) c[q] = buf[rad_at<BL, XL>(b, q * 16 + u)];
    dft16(c, (R)+1);
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = c[dft16_at(j)];
    return a0;
}

template <typename R>
__global__ __launch_bounds__(16 * rad_lines<R>()) void k_rader_y(DiffArgs<R> a, int sign) {
    constexpr int BL = rad_lines<R>();
    __shared__ cplx<R> buf[RAD_LD * BL];
    __shared__ cplx<R> tw[RAD_M];
    const int b = (int)threadIdx.x % BL, u = (int)threadIdx.x / BL;
    // blocks of BL x-columns, x fastest; neighbouring blocks share the cache
    // lines at their edges, so they go to one XCD
    const int nxb = (a.nx + BL - 1) / BL;
    const int64_t blk = xcd_block((int64_t)nxb * a.nzp);
    if (blk >= (int64_t)nxb * a.nzp) return;
    const int x = (int)(blk % nxb) * BL + b;
    const bool in = x < a.nx;
    cplx<R>* col = a.a + (blk / nxb) * (int64_t)a.nx * RAD_N + x;
    const cplx<R>* twg = reinterpret_cast<const cplx<R>*>(a.ay.tw);
    const cplx<R>* rb = reinterpret_cast<const cplx<R>*>(a.ay.rb) + (sign > 0 ? RAD_M : 0);
    constexpr RadPowers<RAD_G> GP;
    constexpr RadPowers<RAD_GI> GI;
    cplx<R> v[16];
    const int gu = rad_pow16<RAD_G>(u);
#pragma unroll
    for (int j = 0; j < 16; ++j)
        v[j] = in ? col[rad_mod(gu * GP.v[j]) * a.nx] : cplx<R>{0, 0};
    const cplx<R> x0 = in ? col[0] : cplx<R>{0, 0};
    for (int w = threadIdx.x; w < RAD_M; w += 16 * BL) tw[w] = twg[w];
    const cplx<R> a0 = rader_core<R, BL, false>(v, b, u, buf, tw, rb);
    if (!in) return;
    const int hu = rad_pow16<RAD_GI>(u);
#pragma unroll
    for (int j = 0; j < 16; ++j) col[rad_mod(hu * GI.v[j]) * a.nx] = cadd(x0, v[j]);
    if (u == 0) col[0] = cadd(x0, a0);
}

// The DFT of the BL lines held in natural order in buf (element x of line b at
// b * RAD_LD + x), back in natural order.  Starts and ends with a barrier.
template <typename R, int BL>
__device__ __forceinline__ void rader_natural(int b, int u, cplx<R>* buf, const cplx<R>* tw, const cplx<R>* rb) {
    constexpr RadPowers<RAD_G> GP;
    constexpr RadPowers<RAD_GI> GI;
    cplx<R>* line = buf + b * RAD_LD;
    __syncthreads();
    cplx<R> v[16];
    const int gu = rad_pow16<RAD_G>(u);
#pragma unroll
    for (int j = 0; j < 16; ++j) v[j] = line[rad_mod(gu * GP.v[j])];
    const cplx<R> x0 = line[0];
    const cplx<R> a0 = rader_core<R, BL, true>(v, b, u, buf, tw, rb);
    __syncthreads();
    const int hu = rad_pow16<RAD_GI>(u);
#pragma unroll
    for (int j = 0; j < 16; ++j) line[rad_mod(hu * GI.v[j])] = cadd(x0, v[j]);
    if (u == 0) line[0] = cadd(x0, a0);
    __syncthreads();
}

// x lines of 257 points, OP an XOP_ value as in k_fft_x.
template <typename R, int OP>
__global__ __launch_bounds__(16 * rad_lines<R>()) void k_rader_x(DiffArgs<R> a, int sign) {
    constexpr int BL = rad_lines<R>();
    constexpr int T = 16 * BL;
    constexpr int KE = 17;   // elements per thread: 16, and one more for the first BL threads
    __shared__ cplx<R> buf[RAD_LD * BL];
    __shared__ cplx<R> tw[RAD_M];
    const int b = (int)threadIdx.x / 16, u = (int)threadIdx.x % 16;
    const int64_t L0 = (int64_t)blockIdx.x * BL;
    const int nb = (int)min<int64_t>(BL, (int64_t)a.ny * a.nzp - L0);
    cplx<R>* base = a.a + L0 * RAD_N;
    cplx<R>* keep = a.anb + L0 * RAD_N;
    const cplx<R>* twg = reinterpret_cast<const cplx<R>*>(a.ax.tw);
    const cplx<R>* rbg = reinterpret_cast<const cplx<R>*>(a.ax.rb);
    const int64_t alias = (int64_t)(a.nz2 - 1) * a.nx * a.ny;   // the last plane of a periodic mesh
    const double rff = 1.0 / a.ffact;
    // the backward transform's 1/ffact: a divide in FP64 (the reference's
    // arithmetic), a reciprocal multiply in the mixed form
    auto unscale = [&](R s) -> double {
        if constexpr (sizeof(R) == 8) return (double)s / a.ffact;
        else return (double)s * rff;
    };
    // f(k, w, lb, x) for the thread's elements w = x + 257 lb of the block's lines
    auto each = [&](auto f) {
#pragma unroll
        for (int k = 0; k < KE; ++k) {
            const int w = (int)threadIdx.x + k * T;
            const int lb = w / RAD_N;
            if (w < nb * RAD_N) f(k, w, lb, w - lb * RAD_N);
        }
    };
    // mask of element x of line lb
    const int iy0 = (int)(L0 % a.ny), iz0 = (int)(L0 / a.ny);
    auto mask = [&](int lb, int x) {
        const int l = iy0 + lb;
        const double mxy = a.mxy[(int64_t)(l % a.ny) * a.nx + x];
        return mxy + (a.mz[iz0 + l / a.ny] * (1.0 - mxy));
    };
    cplx<R> in[KE];
#pragma unroll
    for (int k = 0; k < KE; ++k) in[k] = cplx<R>{0, 0};
    each([&](int k, int w, int, int) { in[k] = base[w]; });
    for (int w = threadIdx.x; w < RAD_M; w += T) tw[w] = twg[w];
    if constexpr (OP == XOP_ADJ_FOLD_SAVE_FWD) {
        each([&](int k, int w, int lb, int x) {
            const int64_t L = L0 + lb;
            if (a.periodic && L < a.ny) {
                // the output's aliased plane copies plane 1: fold its cotangent
                cplx<R>* al = a.a + alias + L * RAD_N + x;
                in[k] = cadd(in[k], *al);
                *al = cplx<R>{0, 0};
            }
            keep[w] = in[k];
        });
    }
#pragma unroll
    for (int k = 0; k < KE; ++k) {   // zeros on lines past the end
        const int w = (int)threadIdx.x + k * T;
        if (w < BL * RAD_N) buf[(w / RAD_N) * RAD_LD + w % RAD_N] = in[k];
    }
    const int s1 = OP == XOP_FORWARD ? sign : (OP == XOP_ADJ_FOLD_SAVE_FWD ? -1 : +1);
    rader_natural<R, BL>(b, u, buf, tw, rbg + (s1 > 0 ? RAD_M : 0));
    // the kept copy, all loads before the first use (held across the
    // transform it cost 40 to 90 registers, one to two waves per SIMD)
    cplx<R> kept[OP == XOP_INV_RECOMBINE || OP == XOP_ADJ_INV_MIX_FWD ? KE : 1];
    if constexpr (OP == XOP_INV_RECOMBINE || OP == XOP_ADJ_INV_MIX_FWD)
        each([&](int k, int w, int, int) { kept[k] = keep[w]; });
    if constexpr (OP == XOP_INV_SPLIT_FWD || OP == XOP_ADJ_INV_MIX_FWD) {
        each([&](int k, int w, int lb, int x) {
            cplx<R>* e = buf + lb * RAD_LD + x;
            const double m = mask(lb, x);
            const double vr = unscale(e->x), vi = unscale(e->y);
            if constexpr (OP == XOP_INV_SPLIT_FWD) {
                // /ffact then AbsorptionStep's split (diffraction.f90:310, 454-470)
                keep[w] = {(R)((1.0 - m) * vr), (R)((1.0 - m) * vi)};
                *e = {(R)(m * vr), (R)(m * vi)};
            } else {
                // adjoint of the split: (1 - m) cotangent + m W^H G W cotangent / ffact
                *e = {(R)((1.0 - m) * (double)kept[k].x + m * vr), (R)((1.0 - m) * (double)kept[k].y + m * vi)};
            }
        });
        rader_natural<R, BL>(b, u, buf, tw, rbg);
    }
    each([&](int k, int w, int lb, int x) {
        cplx<R> v = buf[lb * RAD_LD + x];
        if constexpr (OP == XOP_INV_RECOMBINE) {
            // /ffact + interior (diffraction.f90:513-517)
            if constexpr (sizeof(R) == 8) v = {unscale(v.x) + kept[k].x, unscale(v.y) + kept[k].y};
            else v = {(R)unscale(v.x) + kept[k].x, (R)unscale(v.y) + kept[k].y};
            // keep the aliased plane NZ2 equal to plane 1 (para_field.f90:3197-3244)
            const int64_t L = L0 + lb;
            if (a.periodic && L < a.ny) a.a[alias + L * RAD_N + x] = v;
        } else if constexpr (OP == XOP_ADJ_INV_SCALE) {
            v = {(R)unscale(v.x), (R)unscale(v.y)};
        }
        base[w] = v;
    });
}

// ---- x lines (contiguous) --------------------------------------------------
// OP (an XOP_ value) is a template parameter: each fused operation gets its
// own register allocation.  Four wavefronts a SIMD for the plans in place (433 ->
// 376 us for 61 x 47 x 389); the direct sums of two buffers keep their rotations
// in 150 registers instead: 26 x 26 x 521 (FP64) 457 -> 412 us.
template <typename R, int NC, int BC, int KIND, int OP>
__global__ __launch_bounds__(256, KIND == LINE_TWO ? 1 : 4) void k_fft_x(DiffArgs<R> a, int Bp, int sign) {
    constexpr int op = OP;
    constexpr bool TWO = KIND == LINE_TWO;
    extern __shared__ unsigned char smem_raw[];
    const int N = NC ? NC : a.nx;
    const int B = BC ? BC : Bp;
    const FftAxis& ax = a.ax;
    cplx<R>* s0 = reinterpret_cast<cplx<R>*>(smem_raw);
    cplx<R>* s1 = s0 + lpad<false>(B * N);
    const int64_t nlines = (int64_t)a.ny * a.nzp;
    const int64_t L0 = (int64_t)blockIdx.x * B;
    const int nb = (int)min<int64_t>(B, nlines - L0);
    const cplx<R>* twg = reinterpret_cast<const cplx<R>*>(ax.tw);
    cplx<R>* tw = TWO ? s1 + lpad<false>(B * N) : s1;   // twiddle table staged in LDS
    for (int w = threadIdx.x; w < N; w += blockDim.x) tw[w] = twg[w];
    const cplx<R>* tp = KIND == LINE_PRIME ? prime_table(tw + N, twg, ax) : tw;
    cplx<R>* base = a.a + L0 * N;
    const int64_t ntr = (int64_t)a.nx * a.ny;
    // plane and row of the block's first line; line L0 + b is row iy0 + b
    // counted on from there (b < B)
    const int iy0 = (int)(L0 % a.ny), iz0 = (int)(L0 / a.ny);
    const double rff = 1.0 / a.ffact;
    const Div by_n = div_by(N);
    if (op == XOP_ADJ_FOLD_SAVE_FWD) {
        for (int w = threadIdx.x; w < B * N; w += blockDim.x) {
            const int b = over(w, by_n);
            cplx<R> v = (b < nb) ? base[w] : cplx<R>{0, 0};
            if (b < nb) {
                const int64_t L = L0 + b;
                if (a.periodic && L < a.ny) {
                    // the output's aliased plane copies plane 1: fold its cotangent
                    cplx<R>* al = a.a + (int64_t)(a.nz2 - 1) * ntr + L * N + (w - b * N);
                    const cplx<R> t = *al;
                    v.x += t.x;
                    v.y += t.y;
                    *al = cplx<R>{0, 0};
                }
                a.anb[L0 * N + w] = v;
            }
            s0[lpad<false>(w)] = v;
        }
    } else {
        const int nv = nb * N;
        lds_fill<false, STAGE_UNROLL>(s0, B * N, [&](int w) { return w < nv ? base[w] : cplx<R>{0, 0}; });
    }
    __syncthreads();
    const int first_sign = (op == XOP_FORWARD) ? sign : (op == XOP_ADJ_FOLD_SAVE_FWD ? -1 : +1);
    // the backward transform's 1/ffact: a divide in FP64 (the reference's
    // arithmetic), a reciprocal multiply (rff) in the mixed form
    auto unscale = [&](R v) -> double {
        if constexpr (sizeof(R) == 8) return (double)v / a.ffact;
        else return (double)v * rff;
    };
    cplx<R>* res = lds_fft<R, false, NC, KIND>(s0, s1, B, ax, tw, tp, first_sign);
    if (op == XOP_ADJ_INV_MIX_FWD) {
        // adjoint of the absorption split: (1 - m) cotangent + m W^H G W cotangent / ffact
        const cplx<R>* lam = a.anb + L0 * N;
        for (int w = threadIdx.x; w < nb * N; w += blockDim.x) {
            const int b = over(w, by_n), j = w - b * N;
            const int lb = iy0 + b;   // (iy, iz) of line L0 + b
            const int iy = lb % a.ny, iz = iz0 + lb / a.ny;
            const double mxy = a.mxy[(int64_t)iy * a.nx + j];
            const double m = mxy + (a.mz[iz] * (1.0 - mxy));
            const cplx<R> v = res[lpad<false>(w)];
            const cplx<R> l = lam[w];
            res[lpad<false>(w)] = {(R)((1.0 - m) * (double)l.x + m * unscale(v.x)),
                            (R)((1.0 - m) * (double)l.y + m * unscale(v.y))};
        }
        __syncthreads();
        cplx<R>* other = (TWO && res == s0) ? s1 : s0;
        res = lds_fft<R, false, NC, KIND>(res, other, B, ax, tw, tp, -1);
    } else if (op == XOP_ADJ_INV_SCALE) {
        for (int w = threadIdx.x; w < nb * N; w += blockDim.x) {
            const cplx<R> v = res[lpad<false>(w)];
            res[lpad<false>(w)] = {(R)unscale(v.x), (R)unscale(v.y)};
        }
        __syncthreads();
    } else if (op == XOP_INV_SPLIT_FWD) {
        // /ffact then AbsorptionStep's split (diffraction.f90:310, 454-470)
        cplx<R>* anb = a.anb + L0 * N;
        for (int w = threadIdx.x; w < nb * N; w += blockDim.x) {
            const int b = over(w, by_n), j = w - b * N;
            const int lb = iy0 + b;   // (iy, iz) of line L0 + b
            const int iy = lb % a.ny, iz = iz0 + lb / a.ny;
            const double mxy = a.mxy[(int64_t)iy * a.nx + j];
            const double m = mxy + (a.mz[iz] * (1.0 - mxy));
            cplx<R> v = res[lpad<false>(w)];
            const double vr = unscale(v.x), vi = unscale(v.y);
            anb[w] = {(R)((1.0 - m) * vr), (R)((1.0 - m) * vi)};
            res[lpad<false>(w)] = {(R)(m * vr), (R)(m * vi)};
        }
        __syncthreads();
        cplx<R>* other = (TWO && res == s0) ? s1 : s0;
        res = lds_fft<R, false, NC, KIND>(res, other, B, ax, tw, tp, -1);
    } else if (op == XOP_INV_RECOMBINE) {
        // /ffact + interior (diffraction.f90:513-517)
        const cplx<R>* anb = a.anb + L0 * N;
        for (int w = threadIdx.x; w < nb * N; w += blockDim.x) {
            const cplx<R> v = res[lpad<false>(w)];
            const cplx<R> q = anb[w];
            if (sizeof(R) == 8) {
                res[lpad<false>(w)] = {(R)(unscale(v.x) + (double)q.x), (R)(unscale(v.y) + (double)q.y)};
            } else {
                res[lpad<false>(w)] = {(R)unscale(v.x) + q.x, (R)unscale(v.y) + q.y};
            }
        }
        __syncthreads();
    }
    lds_drain<false, STAGE_UNROLL>(res, nb * N, [&](int w, const cplx<R>& v) { base[w] = v; });
    if (op == XOP_INV_RECOMBINE && a.periodic) {
        // keep the aliased plane NZ2 equal to plane 1 (para_field.f90:3197-3244)
        for (int w = threadIdx.x; w < nb * N; w += blockDim.x) {
            const int b = over(w, by_n);
            const int64_t L = L0 + b;
            if (L < a.ny) a.a[(int64_t)(a.nz2 - 1) * ntr + L * N + (w - b * N)] = res[lpad<false>(w)];
        }
    }
}

// ---- y lines (stride nx), B consecutive x per block -------------------------
template <typename R, int NC, int BC, int KIND>
__global__ __launch_bounds__(256, KIND == LINE_TWO ? 1 : 4) void k_fft_y(DiffArgs<R> a, int Bp, int sign) {
    constexpr bool TWO = KIND == LINE_TWO;
    extern __shared__ unsigned char smem_raw[];
    const int N = NC ? NC : a.ny;
    const int B = BC ? BC : Bp;
    const FftAxis& ay = a.ay;
    cplx<R>* s0 = reinterpret_cast<cplx<R>*>(smem_raw);
    cplx<R>* s1 = s0 + lpad<true>(B * N);
    // blocks of B x-columns, x fastest; neighbouring blocks share the cache
    // lines at their edges, so they go to one XCD
    const int nxb = (a.nx + B - 1) / B;
    const int64_t blk = xcd_block((int64_t)nxb * a.nzp);
    if (blk >= (int64_t)nxb * a.nzp) return;
    const int x0 = (int)(blk % nxb) * B;
    const int iz = (int)(blk / nxb);
    const int nb = min(B, a.nx - x0);
    const cplx<R>* twg = reinterpret_cast<const cplx<R>*>(ay.tw);
    cplx<R>* tw = TWO ? s1 + lpad<true>(B * N) : s1;   // twiddle table staged in LDS
    for (int w = threadIdx.x; w < N; w += blockDim.x) tw[w] = twg[w];
    const cplx<R>* tp = KIND == LINE_PRIME ? prime_table(tw + N, twg, ay) : tw;
    const Div by_b = div_by(B);
    cplx<R>* base = a.a + (int64_t)iz * a.nx * a.ny + x0;
    lds_fill<true, STAGE_UNROLL>(s0, B * N, [&](int w) {
        const int j = over(w, by_b), b = w - j * B;
        return (b < nb) ? base[(int64_t)j * a.nx + b] : cplx<R>{0, 0};
    });
    __syncthreads();
    cplx<R>* res = lds_fft<R, true, NC, KIND>(s0, s1, B, ay, tw, tp, sign);
    lds_drain<true, STAGE_UNROLL>(res, B * N, [&](int w, const cplx<R>& v) {
        const int j = over(w, by_b), b = w - j * B;
        if (b < nb) base[(int64_t)j * a.nx + b] = v;
    });
}

// The spectral factor between the forward and inverse z2 transforms, at
// wavenumbers (kx, ky, kz): multiplyexp's propagator (with its filter) or
// AbsorptionStep's damping.  FP64 form: in FP64, rounded once.  Mixed form
// (an FP32 field): the propagator phase is formed and reduced in FP64; the
// damping exponent is formed in FP64 and exponentiated in FP32.  The mixed
// form also takes rz, 1/(2 kz) (propagator) or 1/sqrt|2 kz| (damping), from a
// per-wavenumber table (kzr) instead of an FP64 divide and square root per
// node; the FP64 form ignores it.  SMALL: the phases are below PHASE_LIMIT.
template <typename R, bool SMALL>
__device__ __forceinline__ cplx<R> spectral_op(const DiffArgs<R>& a, int op, double kx, double ky, double kz,
                                               double rz, cplx<R> v) {
    if (op == SPEC_PROPAGATE) {
        // multiplyexp (diffraction.f90:150-168)
        if ((kz > a.cutoff) || (kz < -a.cutoff)) {
            if (kz != 0.0) {
                const double th = sizeof(R) == 4 ? a.h * (kx * kx + ky * ky) * rz : a.h * (kx * kx + ky * ky) / (2.0 * kz);
                SinCos<R> t;
                if constexpr (SMALL) {
                    t = sincos_phase<R>(th);
                } else {
                    double sn, cs;
                    sincos(th, &sn, &cs);
                    t = {(R)sn, (R)cs};
                }
                v = {t.c * v.x - t.s * v.y, t.s * v.x + t.c * v.y};
            }
        } else if (a.filter) {
            v = {(R)0, (R)0};
        }
    } else if (kz != 0.0) {
        // AbsorptionStep damping (diffraction.f90:484-497)
        if constexpr (sizeof(R) == 4) {
            const float f = expf((float)(-a.h * a.beta * (fabs(kx) + fabs(ky)) * rz));
            v = {f * v.x, f * v.y};
        } else {
            const double f = exp(-a.h * a.beta * (fabs(kx) + fabs(ky)) / (sqrt(fabs(2.0 * kz))));
            v = {f * v.x, f * v.y};
        }
    }
    return v;
}

// ---- z2 lines (stride nx ny), B consecutive x per block ----------------------
// op < 0: plain transform with `sign`; else forward, spectral op, inverse.
template <typename R, int KIND>
__global__ __launch_bounds__(PUFF_Z_THREADS, KIND == LINE_TWO ? 1 : 4) void k_fft_z(DiffArgs<R> a, int B, int op, int sign) {
    constexpr bool TWO = KIND == LINE_TWO;
    extern __shared__ unsigned char smem_raw[];
    const int N = a.nzp;
    const FftAxis& az = a.az;
    cplx<R>* s0 = reinterpret_cast<cplx<R>*>(smem_raw);
    cplx<R>* s1 = TWO ? s0 + lpad<true>(B * N) : s0;
    // blocks of B x-columns, x fastest; neighbouring blocks share the cache
    // lines of every z2 plane, so they go to one XCD
    const int nxb = (a.nx + B - 1) / B;
    const int64_t blk = xcd_block((int64_t)nxb * a.ny);
    if (blk >= (int64_t)nxb * a.ny) return;
    const int x0 = (int)(blk % nxb) * B;
    const int iy = (int)(blk / nxb);
    const int nb = min(B, a.nx - x0);
    const int64_t ntr = (int64_t)a.nx * a.ny;
    // few lines per workgroup here: the twiddles stay in global memory (L2)
    const cplx<R>* tw = reinterpret_cast<const cplx<R>*>(az.tw);
    const cplx<R>* tp = KIND == LINE_PRIME ? prime_table(s0 + lpad<true>(B * N), tw, az) : tw;
    cplx<R>* base = a.a + (int64_t)iy * a.nx + x0;
    const Div by_b = div_by(B);
    lds_fill<true, PUFF_Z_UNROLL>(s0, B * N, [&](int w) {
        const int j = over(w, by_b), b = w - j * B;
        return (b < nb) ? base[(int64_t)j * ntr + b] : cplx<R>{0, 0};
    });
    __syncthreads();
    cplx<R>* res;
    if (op < 0) {
        res = lds_fft<R, true, 0, KIND>(s0, s1, B, az, tw, tp, sign);
    } else {
        res = lds_fft<R, true, 0, KIND>(s0, s1, B, az, tw, tp, -1);
        const double ky = a.ky[iy];
        const bool small_phase = a.phase_max < PHASE_LIMIT;
        for (int w = threadIdx.x; w < B * N; w += blockDim.x) {
            const int q = over(w, by_b), b = w - q * B;
            if (b >= nb) continue;
            const double rz = sizeof(R) == 4 ? a.kzr[2 * q + (op == SPEC_ABSORB ? 1 : 0)] : 0.0;
            const cplx<R> v = res[lpad<true>(w)];
            res[lpad<true>(w)] = small_phase ? spectral_op<R, true>(a, op, a.kx[x0 + b], ky, a.kz[q], rz, v)
                                             : spectral_op<R, false>(a, op, a.kx[x0 + b], ky, a.kz[q], rz, v);
        }
        __syncthreads();
        cplx<R>* other = (TWO && res == s0) ? s1 : s0;
        res = lds_fft<R, true, 0, KIND>(res, other, B, az, tw, tp, +1);
    }
    lds_drain<true, PUFF_Z_UNROLL>(res, B * N, [&](int w, const cplx<R>& v) {
        const int j = over(w, by_b), b = w - j * B;
        if (b < nb) base[(int64_t)j * ntr + b] = v;
    });
}

// ---- z2 lines of a power of two, in registers ---------------------------------
// A thread holds 16 points of one column (FP64) or of two neighbouring columns
// (FP32) of the mesh, 16 bytes per point either way; N / 16 threads share a
// column group and a workgroup takes BG groups, rows of 16 BG bytes (64 to 512)
// of every plane.  With N = 16 M, M = 16 L (M = L up to 256 points):
//   X[q + 16 (q2 + 16 p)] = sum_v W_L^(v p) W_M^(v q2) sum_j W16^(j q2) W_N^(u q) sum_i W16^(i q) x[u + M i],
// u = v + L j: a 16-point DFT per thread, an exchange, a second one, an
// exchange, and 16 / L DFTs of L points; after them a thread holds its
// wavenumbers, applies the spectral factor to them, and the inverse retraces
// the steps.  Nothing is brought into natural order.  An exchange moves the
// real parts through LDS and then the imaginary parts, in words of 8 bytes, so
// that a workgroup's LDS is half of what it holds in registers: two workgroups
// a CU at 1024 points, one at 4096.
//   layout 1, of (q, u): q-major, a spare row of BG words after every q;
//   layout 2, of (v, q, q2): v-major, a spare row after every v.
// Both spread the lanes of a write and of a read over all banks.
// A spectral pass over 129 x 129 lines of 1024 points (FP64; 112 us at the rate
// of a large copy) took 269 us with two lines a workgroup in LDS; a diffraction
// step, two such passes of nine, went from 1895 to 1797 us.  257 x 257 lines of
// 4096 (FP32): three passes of memory became one, 19.4 -> 16.7 ms.
template <int N>
struct ZReg {
    static constexpr int M = N / 16;                                  // threads per column group
    static constexpr int L = M > 16 ? M / 16 : M;                     // points of the last DFT
    static constexpr bool TWO = M > 16;                               // two exchanges
    static constexpr int BG = N >= 2048 ? 4 : (N >= 512 ? 8 : 4096 / N);
    static constexpr int THREADS = M * BG;
    static constexpr int ROW1 = M * BG + BG;
    static constexpr int ROW2 = 256 * BG + BG;
    static constexpr int WORDS = TWO ? (16 * ROW1 > L * ROW2 ? 16 * ROW1 : L * ROW2) : 16 * ROW1;
    static_assert(L >= 2 && L <= 16 && WORDS * 8 <= LDS_BYTES, "128 to 4096 points");
};

// One component (8 bytes) and one point (16 bytes) of a thread's columns.
template <typename R>
struct ZWord;
template <>
struct ZWord<double> {
    static constexpr int C = 1;   // columns
    using type = double;
    static __device__ __forceinline__ double pack(double a, double) { return a; }
    static __device__ __forceinline__ double get(double w, int) { return w; }
};
template <>
struct ZWord<float> {
    static constexpr int C = 2;
    struct alignas(8) type {   // (not a vector type: see zreg_exchange)
        float x, y;
    };
    static __device__ __forceinline__ type pack(float a, float b) { return type{a, b}; }
    static __device__ __forceinline__ float get(type w, int c) { return c ? w.y : w.x; }
};

struct alignas(8) ZPair {
    float x, y, z, w;
};

// The columns' element wr(i) of the thread that writes word wa(i) to element i
// of the thread that reads that word as ra(i).  Starts and ends with the buffer
// free.  (The words of two columns are structs and the columns arrays of their
// own: of vectors built from array elements, and of rows of one array, the
// compiler makes vector loads of the array, which then stays in memory.)
template <typename R, typename WA, typename WR, typename RA>
__device__ __forceinline__ void zreg_exchange(cplx<R> (&v)[16], cplx<R> (&w)[16], typename ZWord<R>::type* buf, WA wa,
                                              WR wr, RA ra) {
    cplx<R> tv[16], tw[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) buf[wa(i)] = ZWord<R>::pack(v[wr(i)].x, w[wr(i)].x);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const auto e = buf[ra(i)];
        tv[i].x = ZWord<R>::get(e, 0);
        tw[i].x = ZWord<R>::get(e, 1);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) buf[wa(i)] = ZWord<R>::pack(v[wr(i)].y, w[wr(i)].y);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const auto e = buf[ra(i)];
        v[i] = {tv[i].x, ZWord<R>::get(e, 0)};
        w[i] = {tw[i].x, ZWord<R>::get(e, 1)};
    }
    __syncthreads();
}

// The 16 / L DFTs of L points of v (group g: v[g L ..], natural order in and out).
template <typename R, int L>
__device__ __forceinline__ void zreg_last(cplx<R> (&v)[16], R sg) {
#pragma unroll
    for (int g = 0; g < 16 / L; ++g) {
        cplx<R> x[L];
#pragma unroll
        for (int k = 0; k < L; ++k) x[k] = v[g * L + k];
        SmallDft<R, L>::run(x, sg);
#pragma unroll
        for (int k = 0; k < L; ++k) v[g * L + k] = x[SmallDft<R, L>::at(k)];
    }
}

// OP < 0: plain transform with `sign`; else forward, spectral factor (phases
// below PHASE_LIMIT), inverse.
template <typename R, int N, int OP>
__global__ __launch_bounds__(ZReg<N>::THREADS, 4) void k_fft_zreg(DiffArgs<R> a, int sign) {
    using Z = ZReg<N>;
    constexpr int C = ZWord<R>::C, M = Z::M, L = Z::L, BG = Z::BG;
    extern __shared__ unsigned char smem_raw[];
    auto* buf = reinterpret_cast<typename ZWord<R>::type*>(smem_raw);
    // columns counted over x, then y; neighbouring blocks share the cache
    // lines of every plane, so they go to one XCD
    const int64_t ntr = (int64_t)a.nx * a.ny;
    const int64_t nblk = (ntr + BG * C - 1) / (BG * C);
    const int64_t blk = xcd_block(nblk);
    if (blk >= nblk) return;
    int b = (int)threadIdx.x % BG, t = (int)threadIdx.x / BG;
    // the thread's columns, moved back to the mesh's last ones past its end; of
    // those only the columns that no other thread holds are stored
    const int64_t col0 = (blk * BG + b) * C;
    const int64_t col = min(col0, ntr - C);
    const cplx<R>* tw = reinterpret_cast<const cplx<R>*>(a.az.tw);
    int q1 = t / L, v1 = t % L;   // (q, v) of the middle step
    uint32_t off = (uint32_t)((t * ntr + col) * (int64_t)sizeof(cplx<R>));
    // addresses are formed again after it, not held
    auto refresh = [&]() { asm volatile("" : "+v"(b), "+v"(t), "+v"(q1), "+v"(v1), "+v"(off)); };

    cplx<R> v[16], w[16];   // the two columns (w: FP32 only)
    // planes t + M i: a scalar row of planes and the thread's 32-bit offset
    auto place = [&](int i) { return reinterpret_cast<cplx<R>*>(reinterpret_cast<char*>(a.a + (int64_t)(M * i) * ntr) + off); };
    auto put = [&](cplx<R>* p, int i) {
        if constexpr (C == 1) *p = v[i];
        else *reinterpret_cast<ZPair*>(p) = ZPair{v[i].x, v[i].y, w[i].x, w[i].y};
    };
    // element at(i) of the thread to p(i)
    auto store = [&](auto p, auto at) {
        if (col0 == col) {
#pragma unroll
            for (int i = 0; i < 16; ++i) put(p(i), at(i));
        } else if (C > 1 && col0 == ntr - 1) {
#pragma unroll
            for (int i = 0; i < 16; ++i) p(i)[C - 1] = w[at(i)];
        }
    };
    // four rotations in flight: all fifteen, loaded at once, spill
    auto twiddle = [&](int k, int i, int e, int sg) {
        if (k % 4 == 0) __builtin_amdgcn_sched_barrier(0);
        const cplx<R> r = tw_get(tw, e, sg);
        v[i] = cmul(v[i], r);
        if constexpr (C > 1) w[i] = cmul(w[i], r);
    };
    auto dft = [&](int sg) {
        dft16(v, (R)sg);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (C > 1) {
            dft16(w, (R)sg);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto last = [&](int sg) {
        zreg_last<R, L>(v, (R)sg);
        if constexpr (C > 1) zreg_last<R, L>(w, (R)sg);
    };
    // words of (q, u), of (v, q 16 + q2), and of the last step's (group, point)
    auto w1 = [&](int q, int u) { return q * Z::ROW1 + u * BG + b; };
    auto w2 = [&](int vv, int c) { return vv * Z::ROW2 + c * BG + b; };
    auto w3 = [&](int i) {
        const int g = i / L, p = i % L;
        return Z::TWO ? w2(p, t + M * g) : w1(t + M * g, p);
    };
    auto same = [](int i) { return i; };
    // wavenumber of element i after the last step
    auto wave = [&](int i) {
        const int c = t + M * (i / L), p = i % L;
        return Z::TWO ? (c >> 4) + 16 * (c & 15) + 256 * p : c + 16 * p;
    };

#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const cplx<R>* p = place(i);
        if constexpr (C == 1) {
            v[i] = *p;
        } else {   // 16 bytes at once, aligned to the 8 of a node
            const ZPair e = *reinterpret_cast<const ZPair*>(p);
            v[i] = {e.x, e.y};
            w[i] = {e.z, e.w};
        }
    }
    // the plain transform of sign +1 is the conjugate of the conjugate's
    const bool mirror = OP < 0 && sign > 0;
    auto conjugate = [&]() {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            v[i].y = -v[i].y;
            if constexpr (C > 1) w[i].y = -w[i].y;
        }
    };
    if (mirror) conjugate();
    dft(-1);
#pragma unroll
    for (int q = 1; q < 16; ++q) twiddle(q, dft16_at(q), t * q, -1);
    if constexpr (Z::TWO) {
        refresh();
        zreg_exchange<R>(v, w, buf, [&](int q) { return w1(q, t); }, dft16_at, [&](int j) { return w1(q1, v1 + L * j); });
        dft(-1);
        refresh();
#pragma unroll
        for (int q = 1; q < 16; ++q) twiddle(q, dft16_at(q), 16 * v1 * q, -1);
        refresh();
        zreg_exchange<R>(v, w, buf, [&](int q) { return w2(v1, 16 * q1 + q); }, dft16_at, w3);
    } else {
        refresh();
        zreg_exchange<R>(v, w, buf, [&](int q) { return w1(q, t); }, dft16_at, w3);
    }
    refresh();
    last(-1);

    if constexpr (OP < 0) {
        if (mirror) conjugate();
        // every thread of the columns has read them: two barriers back at least
        store([&](int i) { return a.a + wave(i) * ntr + col; }, same);
        return;
    }

    double kx[C], ky[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        kx[c] = a.kx[(col + c) % a.nx];
        ky[c] = a.ky[(col + c) / a.nx];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        refresh();
        const int k = wave(i);
        const double kz = a.kz[k];
        const double rz = sizeof(R) == 4 ? a.kzr[2 * k + (OP == SPEC_ABSORB ? 1 : 0)] : 0.0;
        v[i] = spectral_op<R, true>(a, OP, kx[0], ky[0], kz, rz, v[i]);
        asm volatile("" : "+v"(v[i].x), "+v"(v[i].y));   // one after the other
        if constexpr (C > 1) {
            w[i] = spectral_op<R, true>(a, OP, kx[C - 1], ky[C - 1], kz, rz, w[i]);
            asm volatile("" : "+v"(w[i].x), "+v"(w[i].y));
        }
    }

    refresh();
    last(+1);
    if constexpr (Z::TWO) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (i % L) twiddle(i, i, 16 * (i % L) * ((t + M * (i / L)) & 15), +1);
        refresh();
        zreg_exchange<R>(v, w, buf, w3, same, [&](int q) { return w2(v1, 16 * q1 + q); });
        dft(+1);
        refresh();
#pragma unroll
        for (int j = 0; j < 16; ++j) twiddle(j, dft16_at(j), (v1 + L * j) * q1, +1);
        refresh();
        zreg_exchange<R>(v, w, buf, [&](int j) { return w1(q1, v1 + L * j); }, dft16_at, [&](int q) { return w1(q, t); });
    } else {
#pragma unroll
        for (int i = 0; i < 16; ++i)
            if (i % L) twiddle(i, i, (i % L) * (t + M * (i / L)), +1);
        refresh();
        zreg_exchange<R>(v, w, buf, w3, same, [&](int q) { return w1(q, t); });
    }
    dft(+1);
    refresh();
    store(place, dft16_at);
}

// ---- host side -----------------------------------------------------------------

// Dynamic LDS above 64 KiB needs the kernel's opt-in (up to 160 KiB).
static void lds_opt_in(const void* kernel, size_t bytes) {
    if (bytes > 64 * 1024)
        (void)hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, LDS_BYTES);
}

template <typename R, int NC>
static constexpr int ct_lines_x() {
    return lines_per_block(NC, sizeof(cplx<R>), 64, PUFF_XY_LDS_BUDGET, false, true, NC);
}
template <typename R, int NC>
static constexpr int ct_lines_y() {
    return lines_per_block(NC, sizeof(cplx<R>), 16, PUFF_Y_LDS_BUDGET, true, true, NC);
}
template <typename R, int NC, int BC, int KIND, int OP>
static void launch_x_op(const DiffArgs<R>& a, int B, int sign, hipStream_t s) {
    const int64_t nlines = (int64_t)a.ny * a.nzp;
    const size_t sh = line_lds(a.ax, B, KIND, sizeof(cplx<R>), 0);
    lds_opt_in(reinterpret_cast<const void*>(&k_fft_x<R, NC, BC, KIND, OP>), sh);
    hipLaunchKernelGGL((k_fft_x<R, NC, BC, KIND, OP>), dim3((unsigned)((nlines + B - 1) / B)), dim3(256), sh, s, a, B,
                       sign);
}

template <typename R, int OP>
static void launch_rader_x(const DiffArgs<R>& a, int sign, hipStream_t s) {
    constexpr int BL = rad_lines<R>();
    const int64_t nlines = (int64_t)a.ny * a.nzp;
    hipLaunchKernelGGL((k_rader_x<R, OP>), dim3((unsigned)((nlines + BL - 1) / BL)), dim3(16 * BL), 0, s, a, sign);
}

template <typename R>
static void run_rader_x(const DiffArgs<R>& a, int op, int sign, hipStream_t s) {
    switch (op) {
        case XOP_FORWARD: return launch_rader_x<R, XOP_FORWARD>(a, sign, s);
        case XOP_INV_SPLIT_FWD: return launch_rader_x<R, XOP_INV_SPLIT_FWD>(a, sign, s);
        case XOP_INV_RECOMBINE: return launch_rader_x<R, XOP_INV_RECOMBINE>(a, sign, s);
        case XOP_ADJ_FOLD_SAVE_FWD: return launch_rader_x<R, XOP_ADJ_FOLD_SAVE_FWD>(a, sign, s);
        case XOP_ADJ_INV_MIX_FWD: return launch_rader_x<R, XOP_ADJ_INV_MIX_FWD>(a, sign, s);
        default: return launch_rader_x<R, XOP_ADJ_INV_SCALE>(a, sign, s);
    }
}

template <typename R, int NC, int BC, int KIND>
static void launch_x(const DiffArgs<R>& a, int B, int op, int sign, hipStream_t s) {
    if (BC) B = BC;   // compile-time plans fix their lines per workgroup
    switch (op) {
        case XOP_FORWARD: return launch_x_op<R, NC, BC, KIND, XOP_FORWARD>(a, B, sign, s);
        case XOP_INV_SPLIT_FWD: return launch_x_op<R, NC, BC, KIND, XOP_INV_SPLIT_FWD>(a, B, sign, s);
        case XOP_INV_RECOMBINE: return launch_x_op<R, NC, BC, KIND, XOP_INV_RECOMBINE>(a, B, sign, s);
        case XOP_ADJ_FOLD_SAVE_FWD: return launch_x_op<R, NC, BC, KIND, XOP_ADJ_FOLD_SAVE_FWD>(a, B, sign, s);
        case XOP_ADJ_INV_MIX_FWD: return launch_x_op<R, NC, BC, KIND, XOP_ADJ_INV_MIX_FWD>(a, B, sign, s);
        default: return launch_x_op<R, NC, BC, KIND, XOP_ADJ_INV_SCALE>(a, B, sign, s);
    }
}

template <typename R>
static void run_x(const DiffArgs<R>& a, int op, int sign, hipStream_t s) {
    if (a.nx == RAD_N) return run_rader_x(a, op, sign, s);
    if (a.nx == 129) return launch_x<R, 129, ct_lines_x<R, 129>(), LINE_TWO>(a, 0, op, sign, s);
    if (a.nx == 33) return launch_x<R, 33, ct_lines_x<R, 33>(), LINE_TWO>(a, 0, op, sign, s);
    const LinePlan lp = axis_plan(a.ax, sizeof(cplx<R>), 0, (int64_t)a.ny * a.nzp, 1);
    switch (lp.kind) {
        case LINE_SMALL: return launch_x<R, 0, 0, LINE_SMALL>(a, lp.B, op, sign, s);
        case LINE_PRIME: return launch_x<R, 0, 0, LINE_PRIME>(a, lp.B, op, sign, s);
        default: return launch_x<R, 0, 0, LINE_TWO>(a, lp.B, op, sign, s);
    }
}

template <typename R, int NC, int BC, int KIND>
static void launch_y(const DiffArgs<R>& a, int B, int sign, hipStream_t s) {
    if (BC) B = BC;   // compile-time plans fix their lines per workgroup
    const size_t sh = line_lds(a.ay, B, KIND, sizeof(cplx<R>), 1);
    lds_opt_in(reinterpret_cast<const void*>(&k_fft_y<R, NC, BC, KIND>), sh);
    hipLaunchKernelGGL((k_fft_y<R, NC, BC, KIND>), dim3((unsigned)xcd_grid((int64_t)((a.nx + B - 1) / B) * a.nzp)),
                       dim3(256), sh, s, a, B, sign);
}

template <typename R>
static void run_y(const DiffArgs<R>& a, int sign, hipStream_t s) {
    if (a.ny == RAD_N) {
        constexpr int BL = rad_lines<R>();
        const int64_t blocks = xcd_grid((int64_t)((a.nx + BL - 1) / BL) * a.nzp);
        hipLaunchKernelGGL((k_rader_y<R>), dim3((unsigned)blocks), dim3(16 * BL), 0, s, a, sign);
        return;
    }
    if (a.ny == 129) return launch_y<R, 129, ct_lines_y<R, 129>(), LINE_TWO>(a, 0, sign, s);
    if (a.ny == 33) return launch_y<R, 33, ct_lines_y<R, 33>(), LINE_TWO>(a, 0, sign, s);
    const LinePlan lp = axis_plan(a.ay, sizeof(cplx<R>), 1, a.nx, a.nzp);
    switch (lp.kind) {
        case LINE_SMALL: return launch_y<R, 0, 0, LINE_SMALL>(a, lp.B, sign, s);
        case LINE_PRIME: return launch_y<R, 0, 0, LINE_PRIME>(a, lp.B, sign, s);
        default: return launch_y<R, 0, 0, LINE_TWO>(a, lp.B, sign, s);
    }
}

template <typename R, int KIND>
static void launch_z(const DiffArgs<R>& a, int B, int op, int sign, hipStream_t s) {
    const size_t sh = line_lds(a.az, B, KIND, sizeof(cplx<R>), 2);
    const int64_t blocks = xcd_grid((int64_t)((a.nx + B - 1) / B) * a.ny);
    lds_opt_in(reinterpret_cast<const void*>(&k_fft_z<R, KIND>), sh);
    hipLaunchKernelGGL((k_fft_z<R, KIND>), dim3((unsigned)blocks), dim3(PUFF_Z_THREADS), sh, s, a, B, op,
                       sign);
}

// Powers of two from 128 to 4096 points run in registers (k_fft_zreg), other
// lengths through LDS.
template <typename R, int N>
static bool launch_zreg(const DiffArgs<R>& a, int op, int sign, hipStream_t s) {
    const int64_t ntr = (int64_t)a.nx * a.ny;
    if (a.nzp != N || ntr < ZWord<R>::C || ntr * (N / 16) * (int64_t)sizeof(cplx<R>) >= ((int64_t)1 << 32) || (op == SPEC_PROPAGATE && !(a.phase_max < PHASE_LIMIT))) return false;
    using Z = ZReg<N>;
    constexpr int cols = Z::BG * ZWord<R>::C;
    const int64_t blocks = xcd_grid((ntr + cols - 1) / cols);
    auto launch = [&](auto kernel) {
        lds_opt_in(reinterpret_cast<const void*>(kernel), Z::WORDS * 8);
        hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(Z::THREADS), Z::WORDS * 8, s, a, sign);
    };
    if (op < 0) launch(&k_fft_zreg<R, N, -1>);
    else if (op == SPEC_ABSORB) launch(&k_fft_zreg<R, N, SPEC_ABSORB>);
    else launch(&k_fft_zreg<R, N, SPEC_PROPAGATE>);
    return true;
}

template <typename R>
static void run_z(const DiffArgs<R>& a, int op, int sign, hipStream_t s) {
    if (launch_zreg<R, 128>(a, op, sign, s) || launch_zreg<R, 256>(a, op, sign, s) ||
        launch_zreg<R, 512>(a, op, sign, s) || launch_zreg<R, 1024>(a, op, sign, s) ||
        launch_zreg<R, 2048>(a, op, sign, s) || launch_zreg<R, 4096>(a, op, sign, s))
        return;
    const LinePlan lp = axis_plan(a.az, sizeof(cplx<R>), 2, a.nx, a.ny);
    switch (lp.kind) {
        case LINE_SMALL: return launch_z<R, LINE_SMALL>(a, lp.B, op, sign, s);
        case LINE_PRIME: return launch_z<R, LINE_PRIME>(a, lp.B, op, sign, s);
        default: return launch_z<R, LINE_TWO>(a, lp.B, op, sign, s);
    }
}

template <typename R>
void launch_diffraction(const DiffArgs<R>& a, hipStream_t s) {
    run_x(a, XOP_FORWARD, -1, s);
    run_y(a, -1, s);
    run_z(a, SPEC_PROPAGATE, 0, s);
    run_y(a, +1, s);
    run_x(a, XOP_INV_SPLIT_FWD, 0, s);
    run_y(a, -1, s);
    run_z(a, SPEC_ABSORB, 0, s);
    run_y(a, +1, s);
    run_x(a, XOP_INV_RECOMBINE, 0, s);
}

// Adjoint of launch_diffraction.  With W the unnormalised forward transform,
// E the multiplyexp factor (with its filter), G the real damping and M the
// real mask, the forward step is D = Q P with P = W^H E W / ffact and
// Q = (1 - M) + W^H G W M / ffact, so D^H = P^H Q^H with
// Q^H = (1 - M) + M W^H G W / ffact and P^H = W^H conj(E) W / ffact:
//   x fwd (fold alias, keep copy) | y fwd | z fwd . damping . z inv | y inv |
//   x inv . /ffact . mix with copy . x fwd | y fwd | z fwd . conj(E) . z inv |
//   y inv | x inv . /ffact
template <typename R>
void launch_diffraction_adjoint(const DiffArgs<R>& a, hipStream_t s) {
    DiffArgs<R> c = a;
    run_x(c, XOP_ADJ_FOLD_SAVE_FWD, 0, s);
    run_y(c, -1, s);
    run_z(c, SPEC_ABSORB, 0, s);
    run_y(c, +1, s);
    run_x(c, XOP_ADJ_INV_MIX_FWD, 0, s);
    run_y(c, -1, s);
    c.h = -a.h;   // conj(E): the propagator phase with -h (the filter is real)
    run_z(c, SPEC_PROPAGATE, 0, s);
    c.h = a.h;
    run_y(c, +1, s);
    run_x(c, XOP_ADJ_INV_SCALE, 0, s);
}

template <typename R>
void launch_fft3d(cplx<R>* data, int nx, int ny, int nz, const FftAxis& ax, const FftAxis& ay, const FftAxis& az,
                  int sign, hipStream_t s) {
    DiffArgs<R> a{};
    a.a = data;
    a.nx = nx;
    a.ny = ny;
    a.nz2 = nz;
    a.nzp = nz;
    a.ax = ax;
    a.ay = ay;
    a.az = az;
    run_x(a, XOP_FORWARD, sign, s);
    run_y(a, sign, s);
    run_z(a, -1, sign, s);
}

template void launch_diffraction<double>(const DiffArgs<double>&, hipStream_t);
template void launch_diffraction<float>(const DiffArgs<float>&, hipStream_t);
template void launch_diffraction_adjoint<double>(const DiffArgs<double>&, hipStream_t);
template void launch_diffraction_adjoint<float>(const DiffArgs<float>&, hipStream_t);
template void launch_fft3d<double>(cplx<double>*, int, int, int, const FftAxis&, const FftAxis&, const FftAxis&, int,
                                   hipStream_t);
template void launch_fft3d<float>(cplx<float>*, int, int, int, const FftAxis&, const FftAxis&, const FftAxis&, int,
                                  hipStream_t);

}  // namespace puff
