// Counting sort of the macroparticles by mesh cell, so that the lanes of a
// wavefront gather from and deposit to the same few cache lines.  The
// reference keeps its particles in generation order; the permutation is kept
// (orig[j] = reference index of slot j) and undone on download.
#include "puff_common.hpp"
#include "puff_kernels.hpp"

namespace puff {

// Bin of a particle's cell in the slot order (bricks of cells, see
// sort_bins); particles outside the mesh go to the last bin.
template <typename R>
__device__ __forceinline__ int cell_key(const MeshGeom& m, int ncell, R x, R y, double z2) {
    int k = ncell;
    const double zq = floor(z2 * m.inv_dz2);
    int iz = -1;
    if (m.periodic) {
        if (fabs(zq) < 1.0e9) {
            long long r = (long long)zq % m.nzp;
            if (r < 0) r += m.nzp;
            iz = (int)r;
        }
    } else if (zq >= 0.0 && zq <= (double)(m.nzp - 2)) {
        iz = (int)zq;
    }
    if (iz >= 0) {
        if (m.one_d) {
            k = iz;
        } else {
            const R xq = floor((x + (R)m.halfx) * (R)m.inv_dx);
            const R yq = floor((y + (R)m.halfy) * (R)m.inv_dy);
            if (xq >= (R)0 && xq <= (R)(m.nx - 2) && yq >= (R)0 && yq <= (R)(m.ny - 2)) {
                const int ix = (int)xq, iy = (int)yq;
                const int nbx = (m.nx - 1 + BRICK_X - 1) / BRICK_X;
                const int nby = (m.ny - 1 + BRICK_Y - 1) / BRICK_Y;
                // bricks: planes along z2, rows of bricks snaking, so that
                // consecutive bricks are neighbours
                const int bz = iz / BRICK_Z;
                int by = iy / BRICK_Y, bx = ix / BRICK_X;
                if (bz & 1) by = nby - 1 - by;
                const int brow = bz * nby + by;
                if (brow & 1) bx = nbx - 1 - bx;
                int lx = ix % BRICK_X, ly = iy % BRICK_Y, lz = iz % BRICK_Z;
                int cell;
                if (BRICK_XFAST) {
                    // cells of a brick: rows along x in planes, snaking
                    if (lz & 1) ly = BRICK_Y - 1 - ly;
                    const int row = lz * BRICK_Y + ly;
                    if (row & 1) lx = BRICK_X - 1 - lx;
                    cell = row * BRICK_X + lx;
                } else {
                    // cells of a brick: columns along z2, snaking
                    if (ly & 1) lx = BRICK_X - 1 - lx;
                    const int col = ly * BRICK_X + lx;
                    if (col & 1) lz = BRICK_Z - 1 - lz;
                    cell = col * BRICK_Z + lz;
                }
                k = (int)(((int64_t)brow * nbx + bx) * BRICK_CELLS + cell);
            }
        }
    }
    return k;
}

__global__ void k_fill_int(int* p, int64_t n, int v) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ void k_iota(int* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = (int)i;
}

// Runs of equal keys within a wavefront (the input is in the previous sorted
// order, so equal cells are mostly adjacent): the run's first lane does one
// atomic for the whole run.
struct Run {
    int head_lane;
    int len;
    bool head;
};

__device__ __forceinline__ Run run_of(int k, bool valid) {
    const int lane = threadIdx.x & 63;
    const int kk = valid ? k : -1 - lane;
    const int prev = __shfl_up(kk, 1, 64);
    const bool head = (lane == 0) || (prev != kk);
    const unsigned long long heads = __ballot(head);
    const unsigned long long le = (lane == 63) ? heads : (heads & ((2ull << lane) - 1ull));
    const unsigned long long after = (lane == 63) ? 0ull : (heads >> (lane + 1));
    Run r;
    r.head = head;
    r.head_lane = 63 - __builtin_clzll(le);
    const int seg_end = after ? lane + __builtin_ctzll(after) : 63;
    r.len = seg_end - lane + 1;   // meaningful on the head lane
    return r;
}

// Key of every particle, and the histogram of the keys (counts zeroed
// before): one atomic per run of equal keys in a wavefront.
template <typename R>
__global__ __launch_bounds__(256) void k_keys_histogram(const R* x, const R* y, const double* z2,
                                                        int64_t n, MeshGeom m, int ncell, int* key,
                                                        int* counts) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    const int k = valid ? cell_key<R>(m, ncell, x[i], y[i], z2[i]) : 0;
    if (valid) key[i] = k;
    const Run r = run_of(k, valid);
    if (valid && r.head) atomicAdd(&counts[k], r.len);
}

// Exclusive scan in three passes over tiles of SCAN_TILE elements.
constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 16;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;

__device__ __forceinline__ int block_exclusive_scan(int v, int* sh, int* total) {
    // inclusive scan within the wavefront
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    int s = v;
    for (int o = 1; o < 64; o <<= 1) {
        const int t = __shfl_up(s, o, 64);
        if (lane >= o) s += t;
    }
    if (lane == 63) sh[wv] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        int acc = 0;
        for (int k = 0; k < SCAN_THREADS / 64; ++k) {
            const int t = sh[k];
            sh[k] = acc;
            acc += t;
        }
        sh[SCAN_THREADS / 64] = acc;
    }
    __syncthreads();
    const int excl = s - v + sh[wv];
    *total = sh[SCAN_THREADS / 64];
    __syncthreads();
    return excl;
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_tiles(const int* in, int64_t n, int* tile_sums) {
    __shared__ int sh[SCAN_THREADS / 64 + 1];
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int s = 0;
    for (int k = 0; k < SCAN_ITEMS; ++k)
        if (base + k < n) s += in[base + k];
    int total;
    block_exclusive_scan(s, sh, &total);
    if (threadIdx.x == 0) tile_sums[blockIdx.x] = total;
}

// Single block: exclusive scan of the tile sums in place.
__global__ __launch_bounds__(SCAN_THREADS) void k_scan_sums(int* sums, int64_t n) {
    __shared__ int sh[SCAN_THREADS / 64 + 1];
    int carry = 0;
    for (int64_t off = 0; off < n; off += SCAN_TILE) {
        const int64_t base = off + (int64_t)threadIdx.x * SCAN_ITEMS;
        int v[SCAN_ITEMS];
        int s = 0;
        for (int k = 0; k < SCAN_ITEMS; ++k) {
            v[k] = (base + k < n) ? sums[base + k] : 0;
            s += v[k];
        }
        int total;
        int e = block_exclusive_scan(s, sh, &total) + carry;
        for (int k = 0; k < SCAN_ITEMS; ++k) {
            if (base + k < n) sums[base + k] = e;
            e += v[k];
        }
        carry += total;
        __syncthreads();
    }
}

__global__ __launch_bounds__(SCAN_THREADS) void k_scan_apply(const int* in, int64_t n, const int* tile_sums,
                                                             int* out) {
    __shared__ int sh[SCAN_THREADS / 64 + 1];
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    int v[SCAN_ITEMS];
    int s = 0;
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        v[k] = (base + k < n) ? in[base + k] : 0;
        s += v[k];
    }
    int total;
    int e = block_exclusive_scan(s, sh, &total) + tile_sums[blockIdx.x];
    for (int k = 0; k < SCAN_ITEMS; ++k) {
        if (base + k < n) out[base + k] = e;
        e += v[k];
    }
}

__global__ __launch_bounds__(256) void k_scatter_perm(const int* key, int64_t n, int* cursor, int* perm) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    const int k = valid ? key[i] : 0;
    const Run r = run_of(k, valid);
    int base = 0;
    if (valid && r.head) base = atomicAdd(&cursor[k], r.len);
    base = __shfl(base, r.head_lane, 64);
    const int lane = threadIdx.x & 63;
    if (valid) perm[base + (lane - r.head_lane)] = (int)i;
}

// Every per-particle array into slot order: dst[j] = src[perm[j]].
template <typename R>
__global__ __launch_bounds__(256) void k_gather_all(PartPtrs<R> y, const R* chi, const int* orig,
                                                    const int* perm, int64_t n, PartPtrs<R> t,
                                                    R* chi_out, int* orig_out) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const int p = perm[j];
    t.x[j] = y.x[p];
    t.y[j] = y.y[p];
    t.z2[j] = y.z2[p];
    t.pr[j] = y.pr[p];
    t.pi[j] = y.pi[p];
    t.g[j] = y.g[p];
    chi_out[j] = chi[p];
    orig_out[j] = orig[p];
}

// ---- records ------------------------------------------------------------------
// A wavefront moves 64 records of Q quads between its lanes' registers and
// memory through LDS, so that each instruction covers whole records (64 / Q of
// them) instead of one quad of each of 64.  The LDS rows are Q + 1 quads
// apart: with Q apart, the lanes' rows would share banks.

// rec[to] = q on every lane with to >= 0.  All lanes must call.
template <int Q>
__device__ __forceinline__ void wave_store_records(uint4* sh, const uint4 (&q)[Q], int64_t to, uint4* rec) {
    const int lane = threadIdx.x & 63;
    uint4* w = sh + (threadIdx.x >> 6) * 64 * (Q + 1);
#pragma unroll
    for (int k = 0; k < Q; ++k) w[lane * (Q + 1) + k] = q[k];
    __syncthreads();
    const int lo = (int)(to & 0xffffffffll), hi = (int)(to >> 32);
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        const int r = k * (64 / Q) + lane / Q, part = lane % Q;
        const int64_t t = ((int64_t)__shfl(hi, r, 64) << 32) | (uint32_t)__shfl(lo, r, 64);
        const uint4 v = w[r * (Q + 1) + part];
        if (t >= 0) rec[t * Q + part] = v;
    }
}

// q = rec[from] on every lane with from >= 0.  All lanes must call.
template <int Q>
__device__ __forceinline__ void wave_load_records(uint4* sh, uint4 (&q)[Q], int64_t from, const uint4* rec) {
    const int lane = threadIdx.x & 63;
    uint4* w = sh + (threadIdx.x >> 6) * 64 * (Q + 1);
    const int lo = (int)(from & 0xffffffffll), hi = (int)(from >> 32);
    uint4 v[Q];
#pragma unroll
    for (int k = 0; k < Q; ++k) {
        const int r = k * (64 / Q) + lane / Q, part = lane % Q;
        const int64_t f = ((int64_t)__shfl(hi, r, 64) << 32) | (uint32_t)__shfl(lo, r, 64);
        v[k] = f >= 0 ? rec[f * Q + part] : uint4{0, 0, 0, 0};
    }
#pragma unroll
    for (int k = 0; k < Q; ++k) w[(k * (64 / Q) + lane / Q) * (Q + 1) + lane % Q] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < Q; ++k) q[k] = w[lane * (Q + 1) + k];
}

__device__ __forceinline__ uint4 quad(double a, double b) {
    return {(uint32_t)__double2loint(a), (uint32_t)__double2hiint(a), (uint32_t)__double2loint(b),
            (uint32_t)__double2hiint(b)};
}
__device__ __forceinline__ uint4 quad(float a, float b, float c, float d) {
    return {__float_as_uint(a), __float_as_uint(b), __float_as_uint(c), __float_as_uint(d)};
}
__device__ __forceinline__ double first(const uint4& q) { return __hiloint2double((int)q.y, (int)q.x); }
__device__ __forceinline__ double second(const uint4& q) { return __hiloint2double((int)q.w, (int)q.z); }

template <typename R>
struct OneState {
    R x, y, pr, pi;
    double z2, g;
};

template <typename R>
__device__ __forceinline__ OneState<R> read_state(const PartPtrs<R>& y, int64_t i) {
    return {y.x[i], y.y[i], y.pr[i], y.pi[i], y.z2[i], y.g[i]};
}
template <typename R>
__device__ __forceinline__ void write_state(const PartPtrs<R>& y, int64_t i, const OneState<R>& v) {
    y.x[i] = v.x;
    y.y[i] = v.y;
    y.z2[i] = v.z2;
    y.pr[i] = v.pr;
    y.pi[i] = v.pi;
    y.g[i] = v.g;
}

// The state's quads: FP64 (x, y) (z2, pr) (pi, Gamma); mixed (z2, Gamma)
// (x, y, pr, pi).
template <typename R, int Q>
__device__ __forceinline__ void pack_state(const OneState<R>& v, uint4 (&q)[Q]) {
    if constexpr (sizeof(R) == 8) {
        q[0] = quad(v.x, v.y);
        q[1] = quad(v.z2, v.pr);
        q[2] = quad(v.pi, v.g);
    } else {
        q[0] = quad(v.z2, v.g);
        q[1] = quad(v.x, v.y, v.pr, v.pi);
    }
}
template <typename R, int Q>
__device__ __forceinline__ OneState<R> unpack_state(const uint4 (&q)[Q]) {
    OneState<R> v;
    if constexpr (sizeof(R) == 8) {
        v.x = first(q[0]);
        v.y = second(q[0]);
        v.z2 = first(q[1]);
        v.pr = second(q[1]);
        v.pi = first(q[2]);
        v.g = second(q[2]);
    } else {
        v.z2 = first(q[0]);
        v.g = second(q[0]);
        v.x = __uint_as_float(q[1].x);
        v.y = __uint_as_float(q[1].y);
        v.pr = __uint_as_float(q[1].z);
        v.pi = __uint_as_float(q[1].w);
    }
    return v;
}

// Sort out of the reference order: each macroparticle's record straight to
// its slot (cursor: the scanned bins).  The slots are as scattered as the
// macroparticles came, whatever moves them; here each is one 64-byte write.
template <typename R>
__global__ __launch_bounds__(256) void k_scatter_records(PartPtrs<R> y, const R* chi, const int* key, int64_t n,
                                                         int* cursor, uint4* rec) {
    constexpr int Q = RECORD_QUADS;
    __shared__ uint4 sh[4 * 64 * (Q + 1)];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < n;
    const int k = valid ? key[i] : 0;
    uint4 q[Q] = {};
    if (valid) {
        pack_state<R, Q>(read_state(y, i), q);
        if constexpr (sizeof(R) == 8) q[3] = {(uint32_t)__double2loint(chi[i]), (uint32_t)__double2hiint(chi[i]), (uint32_t)i, 0};
        else q[2] = {__float_as_uint(chi[i]), (uint32_t)i, 0, 0};
    }
    const Run r = run_of(k, valid);
    int base = 0;
    if (valid && r.head) base = atomicAdd(&cursor[k], r.len);
    base = __shfl(base, r.head_lane, 64);
    const int lane = threadIdx.x & 63;
    wave_store_records<Q>(sh, q, valid ? (int64_t)(base + (lane - r.head_lane)) : -1, rec);
}

template <typename R>
__global__ __launch_bounds__(256) void k_slots_from_records(const uint4* rec, int64_t n, PartPtrs<R> y, R* chi,
                                                            int* orig) {
    constexpr int Q = RECORD_QUADS;
    __shared__ uint4 sh[4 * 64 * (Q + 1)];
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint4 q[Q];
    wave_load_records<Q>(sh, q, j < n ? j : -1, rec);
    if (j >= n) return;
    write_state(y, j, unpack_state<R, Q>(q));
    if constexpr (sizeof(R) == 8) {
        chi[j] = first(q[3]);
        orig[j] = (int)q[3].z;
    } else {
        chi[j] = __uint_as_float(q[2].x);
        orig[j] = (int)q[2].y;
    }
}

template <typename R>
__global__ __launch_bounds__(256) void k_records_scatter(PartPtrs<R> y, const int* to, int64_t n, uint4* rec) {
    constexpr int Q = RECORD_QUADS;
    __shared__ uint4 sh[4 * 64 * (Q + 1)];
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint4 q[Q] = {};
    if (j < n) pack_state<R, Q>(read_state(y, j), q);
    wave_store_records<Q>(sh, q, j < n ? (int64_t)to[j] : -1, rec);
}

template <typename R>
__global__ __launch_bounds__(256) void k_records_gather(const uint4* rec, const int* from, int64_t n, PartPtrs<R> y) {
    constexpr int Q = RECORD_QUADS;
    __shared__ uint4 sh[4 * 64 * (Q + 1)];
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint4 q[Q];
    wave_load_records<Q>(sh, q, j < n ? (int64_t)from[j] : -1, rec);
    if (j < n) write_state(y, j, unpack_state<R, Q>(q));
}

struct StateOut {
    double* p[6];
};
template <typename R>
__global__ __launch_bounds__(256) void k_records_unpack(const uint4* rec, int64_t n, StateOut out) {
    constexpr int Q = RECORD_QUADS;
    __shared__ uint4 sh[4 * 64 * (Q + 1)];
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    uint4 q[Q];
    wave_load_records<Q>(sh, q, i < n ? i : -1, rec);
    if (i >= n) return;
    const OneState<R> v = unpack_state<R, Q>(q);
    out.p[0][i] = (double)v.x;
    out.p[1][i] = (double)v.y;
    out.p[2][i] = v.z2;
    out.p[3][i] = (double)v.pr;
    out.p[4][i] = (double)v.pi;
    out.p[5][i] = v.g;
}

struct StateIn {
    const double* p[7];
};
template <typename R>
__global__ __launch_bounds__(256) void k_load_state(StateIn in, int64_t n, PartPtrs<R> y, R* chi) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    write_state<R>(y, i, {(R)in.p[0][i], (R)in.p[1][i], (R)in.p[3][i], (R)in.p[4][i], in.p[2][i], in.p[5][i]});
    chi[i] = (R)in.p[6][i];
}

// dst[orig[j]] = (double) src[j]: slot order back to the reference order.
template <typename T>
__global__ __launch_bounds__(256) void k_unpermute(const T* src, const int* orig, int64_t n, double* dst) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) dst[orig[j]] = (double)src[j];
}

// dst[j] = (T) src[orig[j]]: reference order into slot order.
template <typename T>
__global__ __launch_bounds__(256) void k_permute_in(const double* src, const int* orig, int64_t n, T* dst) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n) dst[j] = (T)src[orig[j]];
}

static dim3 g1(int64_t n) { return dim3((unsigned)(n > 0 ? (n + 255) / 256 : 1)); }

template <typename R>
void launch_sort(const SortArgs<R>& a, hipStream_t s) {
    const int64_t n = a.n;
    const int64_t nb = (int64_t)a.ncell + 1;
    hipLaunchKernelGGL(k_fill_int, g1(nb), dim3(256), 0, s, a.counts, nb, 0);
    hipLaunchKernelGGL((k_keys_histogram<R>), g1(n), dim3(256), 0, s, a.y.x, a.y.y, a.y.z2, n, a.mesh,
                       a.ncell, a.key, a.counts);
    const int64_t ntiles = (nb + SCAN_TILE - 1) / SCAN_TILE;
    hipLaunchKernelGGL(k_scan_tiles, dim3((unsigned)ntiles), dim3(SCAN_THREADS), 0, s, a.counts, nb, a.tile_sums);
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SCAN_THREADS), 0, s, a.tile_sums, ntiles);
    hipLaunchKernelGGL(k_scan_apply, dim3((unsigned)ntiles), dim3(SCAN_THREADS), 0, s, a.counts, nb,
                       a.tile_sums, a.cursor);
    if (a.rec) {
        hipLaunchKernelGGL((k_scatter_records<R>), g1(n), dim3(256), 0, s, a.y, a.chi, a.key, n, a.cursor, a.rec);
        hipLaunchKernelGGL((k_slots_from_records<R>), g1(n), dim3(256), 0, s, a.rec, n, a.y, a.chi, a.orig);
        return;
    }
    hipLaunchKernelGGL(k_scatter_perm, g1(n), dim3(256), 0, s, a.key, n, a.cursor, a.perm);
    // permute every coordinate into the spare arrays
    hipLaunchKernelGGL((k_gather_all<R>), g1(n), dim3(256), 0, s, a.y, a.chi, a.orig, a.perm, n, a.spare,
                       a.chi_spare, a.orig_spare);
}

template <typename R>
void launch_records_scatter(const PartPtrs<R>& y, const int* to, int64_t n, uint4* rec, hipStream_t s) {
    hipLaunchKernelGGL((k_records_scatter<R>), g1(n), dim3(256), 0, s, y, to, n, rec);
}

template <typename R>
void launch_records_gather(const uint4* rec, const int* from, int64_t n, const PartPtrs<R>& y, hipStream_t s) {
    hipLaunchKernelGGL((k_records_gather<R>), g1(n), dim3(256), 0, s, rec, from, n, y);
}

template <typename R>
void launch_records_unpack(const uint4* rec, int64_t n, double* const out[6], hipStream_t s) {
    StateOut o;
    for (int k = 0; k < 6; ++k) o.p[k] = out[k];
    hipLaunchKernelGGL((k_records_unpack<R>), g1(n), dim3(256), 0, s, rec, n, o);
}

template <typename R>
void launch_load_state(const double* const in[7], int64_t n, const PartPtrs<R>& y, R* chi, hipStream_t s) {
    StateIn i;
    for (int k = 0; k < 7; ++k) i.p[k] = in[k];
    hipLaunchKernelGGL((k_load_state<R>), g1(n), dim3(256), 0, s, i, n, y, chi);
}

void launch_iota(int* p, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_iota, g1(n), dim3(256), 0, s, p, n);
}

template <typename T>
void launch_unpermute(const T* src, const int* orig, int64_t n, double* dst, hipStream_t s) {
    hipLaunchKernelGGL((k_unpermute<T>), g1(n), dim3(256), 0, s, src, orig, n, dst);
}

template <typename T>
void launch_permute_in(const double* src, const int* orig, int64_t n, T* dst, hipStream_t s) {
    hipLaunchKernelGGL((k_permute_in<T>), g1(n), dim3(256), 0, s, src, orig, n, dst);
}

#define PUFF_INST(R)                                                                                     \
    template void launch_sort<R>(const SortArgs<R>&, hipStream_t);                                       \
    template void launch_records_scatter<R>(const PartPtrs<R>&, const int*, int64_t, uint4*, hipStream_t); \
    template void launch_records_gather<R>(const uint4*, const int*, int64_t, const PartPtrs<R>&, hipStream_t); \
    template void launch_records_unpack<R>(const uint4*, int64_t, double* const[6], hipStream_t);        \
    template void launch_load_state<R>(const double* const[7], int64_t, const PartPtrs<R>&, R*, hipStream_t);
PUFF_INST(double)
PUFF_INST(float)
#undef PUFF_INST
template void launch_unpermute<double>(const double*, const int*, int64_t, double*, hipStream_t);
template void launch_unpermute<float>(const float*, const int*, int64_t, double*, hipStream_t);
template void launch_permute_in<double>(const double*, const int*, int64_t, double*, hipStream_t);
template void launch_permute_in<float>(const double*, const int*, int64_t, float*, hipStream_t);

}  // namespace puff
