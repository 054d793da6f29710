// BLAS-1 of the Krylov drivers on device vectors of double or complex<double>, with fused forms
// (axpy + dot, axpy + norm, dot_many / axpy_many for Gram-Schmidt). Every reduction is
// deterministic: a fixed grid for a given n, a fixed xor-butterfly inside the wavefront, fixed
// slots across wavefronts and blocks, and a final tree over the block partials in a fixed order.
// The result stays in device memory; the host reads it when it needs it.
#include "dev_common.h"
#include "launch.h"

namespace qsa::dev {

namespace {

constexpr int kThreads = 256;
constexpr int kMaxBlocks = 1024;
constexpr int kWaves = kThreads / 64;

inline unsigned grid_for(std::size_t n) {
    const std::size_t b = (n + kThreads * 4 - 1) / (kThreads * 4);
    return static_cast<unsigned>(b < 1 ? 1 : (b > kMaxBlocks ? kMaxBlocks : b));
}

__device__ __forceinline__ double wave_sum(double x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, 64);
    return x;
}

/// Block sum of (a, b): every thread returns the block total (wave sums, then the waves in order).
__device__ __forceinline__ void block_sum2(double& a, double& b) {
    __shared__ double sa[kWaves], sb[kWaves];
    a = wave_sum(a);
    b = wave_sum(b);
    const int w = threadIdx.x >> 6;
    __syncthreads();
    if ((threadIdx.x & 63) == 0) {
        sa[w] = a;
        sb[w] = b;
    }
    __syncthreads();
    a = 0.0;
    b = 0.0;
    for (int i = 0; i < kWaves; ++i) {
        a += sa[i];
        b += sb[i];
    }
}

template <bool C> struct V;
template <> struct V<false> {
    static __device__ __forceinline__ Zd load(const void* p, std::size_t i) { return Zd{static_cast<const double*>(p)[i], 0.0}; }
    static __device__ __forceinline__ void store(void* p, std::size_t i, Zd z) { static_cast<double*>(p)[i] = z.re; }
};
template <> struct V<true> {
    static __device__ __forceinline__ Zd load(const void* p, std::size_t i) { return static_cast<const Zd*>(p)[i]; }
    static __device__ __forceinline__ void store(void* p, std::size_t i, Zd z) { static_cast<Zd*>(p)[i] = z; }
};

__device__ __forceinline__ Zd cmul(Zd a, Zd b) { return Zd{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ Zd cadd(Zd a, Zd b) { return Zd{a.re + b.re, a.im + b.im}; }
/// conj(a) b
__device__ __forceinline__ Zd cdot(Zd a, Zd b) { return Zd{a.re * b.re + a.im * b.im, a.re * b.im - a.im * b.re}; }

template <bool C> __global__ void k_fill_zero(void* x, std::size_t n) {
    for (std::size_t i = blockIdx.x * static_cast<std::size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<std::size_t>(gridDim.x) * blockDim.x)
        V<C>::store(x, i, Zd{0.0, 0.0});
}

// Entry i of a Gaussian test vector: two uniforms from splitmix64 of (seed, i), Box-Muller.
__device__ __forceinline__ u64 mix64(u64 z) {
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}
template <bool C> __global__ void k_fill_gauss(void* x, std::size_t n, u64 seed) {
    for (std::size_t i = blockIdx.x * static_cast<std::size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<std::size_t>(gridDim.x) * blockDim.x) {
        const u64 a = mix64(seed ^ (2 * i)), b = mix64(seed ^ (2 * i + 1));
        const double u1 = (static_cast<double>(a >> 11) + 0.5) * 0x1.0p-53;
        const double u2 = static_cast<double>(b >> 11) * 0x1.0p-53;
        const double r = sqrt(-2.0 * log(u1));
        const double t = 6.283185307179586 * u2;
        V<C>::store(x, i, Zd{r * cos(t), r * sin(t)});
    }
}

/// A coefficient's value (Coef): given by the host, or read on the device.
__device__ __forceinline__ Zd coef_value(const Coef& c) {
    if (c.kind == 1) return Zd{-c.p[0], 0.0};
    if (c.kind == 2) {
        const Zd v{c.p[0], c.p[1]};
        return sqrt(v.re * v.re + v.im * v.im) > c.threshold ? Zd{-v.re, -v.im} : Zd{0.0, 0.0};
    }
    return c.a;
}

template <bool C> __global__ void k_axpby(Coef ca, const void* x, Zd b, void* y, std::size_t n, int mode) {
    // mode 0: y += a x; 1: y *= a; 2: y = a x + b y
    const Zd a = coef_value(ca);
    for (std::size_t i = blockIdx.x * static_cast<std::size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<std::size_t>(gridDim.x) * blockDim.x) {
        if (mode == 1) {
            V<C>::store(y, i, C ? cmul(a, V<C>::load(y, i)) : Zd{a.re * V<C>::load(y, i).re, 0.0});
        } else if (mode == 0) {
            const Zd xv = V<C>::load(x, i), yv = V<C>::load(y, i);
            V<C>::store(y, i, C ? cadd(yv, cmul(a, xv)) : Zd{yv.re + a.re * xv.re, 0.0});
        } else {
            const Zd xv = V<C>::load(x, i), yv = V<C>::load(y, i);
            V<C>::store(y, i, C ? cadd(cmul(a, xv), cmul(b, yv)) : Zd{a.re * xv.re + b.re * yv.re, 0.0});
        }
    }
}

// out = w / *norm (out may be w).
template <bool C> __global__ void k_scale_by(const void* w, const double* norm, void* out, std::size_t n) {
    const double f = 1.0 / *norm;
    for (std::size_t i = blockIdx.x * static_cast<std::size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<std::size_t>(gridDim.x) * blockDim.x) {
        const Zd v = V<C>::load(w, i);
        V<C>::store(out, i, Zd{v.re * f, v.im * f});
    }
}

// Reduction kinds: 0 dot z^H y; 1 sum |y|^2; both optionally after y += a x (fuse != 0; a zero
// coefficient read on the device adds nothing).
template <bool C, int KIND>
__global__ __launch_bounds__(kThreads) void k_reduce(Coef ca, const void* x, void* y, const void* z, std::size_t n,
                                                     int fuse, double* partial) {
    const Zd a = coef_value(ca);
    if (ca.kind == 2 && a.re == 0.0 && a.im == 0.0) fuse = 0;
    double s0 = 0.0, s1 = 0.0;
    for (std::size_t i = blockIdx.x * static_cast<std::size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<std::size_t>(gridDim.x) * blockDim.x) {
        Zd yv = V<C>::load(y, i);
        if (fuse) {
            const Zd xv = V<C>::load(x, i);
            yv = C ? cadd(yv, cmul(a, xv)) : Zd{yv.re + a.re * xv.re, 0.0};
            V<C>::store(y, i, yv);
        }
        if constexpr (KIND == 0) {
            const Zd zv = V<C>::load(z, i);
            if constexpr (C) {
                const Zd d = cdot(zv, yv);
                s0 += d.re;
                s1 += d.im;
            } else {
                s0 += zv.re * yv.re;
            }
        } else {
            s0 += yv.re * yv.re;
            if constexpr (C) s0 += yv.im * yv.im;
        }
    }
    block_sum2(s0, s1);
    if (threadIdx.x == 0) {
        partial[2 * blockIdx.x] = s0;
        partial[2 * blockIdx.x + 1] = s1;
    }
}

/// Sum of nb partial pairs (stride 2) by one block: thread t takes t, t + 256, ... in order, then
/// the block sum. out_kind 0: Zd, 1: sqrt of the first part (a norm), 2: the first part.
__device__ void finish_pairs(const double* partial, int nb, int out_kind, void* out) {
    double a = 0.0, b = 0.0;
    for (int i = threadIdx.x; i < nb; i += blockDim.x) {
        a += partial[2 * i];
        b += partial[2 * i + 1];
    }
    block_sum2(a, b);
    if (threadIdx.x == 0) {
        if (out_kind == 0) *static_cast<Zd*>(out) = Zd{a, b};
        else if (out_kind == 1) *static_cast<double*>(out) = sqrt(a);
        else *static_cast<double*>(out) = a;
    }
}

__global__ __launch_bounds__(kThreads) void k_finish(const double* partial, int nb, int out_kind, void* out,
                                                     const int* gate) {
    if (gate && !*gate) return;
    finish_pairs(partial, nb, out_kind, out);
}

// The DGKS gate of a Gram-Schmidt pass: it is repeated when the norm it left is below kappa of the norm
// it found.
__global__ void k_cgs_gate(const double* before2, const double* after2, double kappa, int* again) {
    *again = sqrt(*after2) < kappa * sqrt(*before2) ? 1 : 0;
}

__global__ void k_add_pair(const Zd* a, const Zd* b, Zd* out) { *out = Zd{a->re + b->re, a->im + b->im}; }

// The columns of a Gram-Schmidt block: column j at base + j stride (bytes), or table[j] when a
// table of device pointers is given (the reference's array-of-vectors form).
struct Cols {
    const char* base;
    std::size_t stride;
    const void* const* table;
    __device__ __forceinline__ const void* at(int j) const {
        return table ? table[j] : static_cast<const void*>(base + static_cast<std::size_t>(j) * stride);
    }
};

// dot_many: block (b, g) owns a row range and a group of `per` columns; the rows come in tiles of kTile
// staged in LDS (the w tile), wavefront v owns the columns j = v, v + 4, ... of the group: its lanes read
// 64 consecutive rows of column j per load (coalesced), sum, and the wave total accumulates into the
// column's LDS slot (one owner: no race). Partials are written column-major [j][b] so the finish
// reads them contiguously. Few rows leave the card idle with every block taking every column (n = 9252:
// 10 blocks of 100 columns took 50 us): there the columns go to several blocks (dot_columns, 7 us;
// 112,632 complex rows and 25 columns 22 -> 13 us). Four loads in flight per lane: eight are slower where
// HBM bounds it (2.6M rows and 50 columns 224 us for 200).
constexpr int kManyCols = 256;   // columns per launch
constexpr int kTile = 1024;      // rows per LDS tile

template <bool C>
__global__ __launch_bounds__(kThreads) void k_dot_many(Cols Vb, int m, int per, const void* w,
                                                       std::size_t n, std::size_t rows_per_block, double* partial,
                                                       int nb, int want_norm, const int* gate) {
    if (gate && !*gate) return;
    __shared__ Zd sw[kTile];
    __shared__ Zd acc[kManyCols + 1];
    const std::size_t r0 = blockIdx.x * rows_per_block;
    const std::size_t r1 = (r0 + rows_per_block < n) ? r0 + rows_per_block : n;
    const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
    const int j0 = static_cast<int>(blockIdx.y) * per, j1 = j0 + per < m ? j0 + per : m;
    const bool norm = want_norm && blockIdx.y == 0;
    for (int j = j0 + static_cast<int>(threadIdx.x); j < j1; j += blockDim.x) acc[j] = Zd{0.0, 0.0};
    double nrm = 0.0;
    __syncthreads();
    for (std::size_t t0 = r0; t0 < r1; t0 += kTile) {
        const int cnt = static_cast<int>((t0 + kTile < r1) ? kTile : (r1 - t0));
        for (int i = threadIdx.x; i < cnt; i += blockDim.x) {
            const Zd v = V<C>::load(w, t0 + i);
            sw[i] = v;
            if (norm) nrm += v.re * v.re + (C ? v.im * v.im : 0.0);
        }
        __syncthreads();
        for (int j = j0 + wv; j < j1; j += kWaves) {
            const void* cj = Vb.at(j);
            double pr = 0.0, pi = 0.0;
#pragma unroll 4
            for (int i = ln; i < cnt; i += 64) {
                const Zd vj = V<C>::load(cj, t0 + i);
                if constexpr (C) {
                    const Zd d = cdot(vj, sw[i]);
                    pr += d.re;
                    pi += d.im;
                } else {
                    pr += vj.re * sw[i].re;
                }
            }
            pr = wave_sum(pr);
            if constexpr (C) pi = wave_sum(pi);
            if (ln == 0) acc[j] = Zd{acc[j].re + pr, acc[j].im + pi};
        }
        __syncthreads();
    }
    if (norm) {
        double dummy = 0.0;
        block_sum2(nrm, dummy);
        if (threadIdx.x == 0) {
            partial[(static_cast<std::size_t>(m) * nb + blockIdx.x) * 2] = nrm;
            partial[(static_cast<std::size_t>(m) * nb + blockIdx.x) * 2 + 1] = 0.0;
        }
    }
    for (int j = j0 + static_cast<int>(threadIdx.x); j < j1; j += blockDim.x) {
        partial[(static_cast<std::size_t>(j) * nb + blockIdx.x) * 2] = acc[j].re;
        partial[(static_cast<std::size_t>(j) * nb + blockIdx.x) * 2 + 1] = acc[j].im;
    }
}

/// Columns per block of dot_many: all of them when the row blocks alone fill the card, else as few (four,
/// one per wavefront, or more) as make about three blocks per compute unit.
inline int dot_columns(int m, std::size_t row_blocks) {
    const int most = (m + kWaves - 1) / kWaves;
    const int groups = static_cast<int>(std::min<std::size_t>(static_cast<std::size_t>(most), (768 + row_blocks - 1) / row_blocks));
    if (groups <= 1) return m;
    return ((m + groups - 1) / groups + kWaves - 1) / kWaves * kWaves;
}

// One block per column: the sum of its nb block partials (contiguous) in a fixed order.
__global__ __launch_bounds__(kThreads) void k_dot_many_finish(const double* partial, int nb, int m, Zd* coeffs,
                                                              double* wnorm2, const int* gate) {
    if (gate && !*gate) return;
    const int j = blockIdx.x;
    if (j < m) finish_pairs(partial + static_cast<std::size_t>(j) * nb * 2, nb, 0, coeffs + j);
    else if (wnorm2) finish_pairs(partial + static_cast<std::size_t>(j) * nb * 2, nb, 2, wnorm2);
}

// w += sign sum_j c_j V_j over grid-strided rows, four columns per step; the partial of ||w||^2 after.
template <bool C>
__global__ __launch_bounds__(kThreads) void k_axpy_many(const Zd* coeffs, Cols Vb, int m,
                                                        void* w, std::size_t n, double* partial, int want_norm,
                                                        double sign, const int* gate) {
    if (gate && !*gate) return;
    __shared__ Zd sc[kManyCols];
    for (int j = threadIdx.x; j < m; j += blockDim.x) sc[j] = Zd{sign * coeffs[j].re, sign * coeffs[j].im};
    __syncthreads();
    double s0 = 0.0, s1 = 0.0;
    for (std::size_t i = blockIdx.x * static_cast<std::size_t>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<std::size_t>(gridDim.x) * blockDim.x) {
        Zd acc = V<C>::load(w, i);
        int j = 0;
        for (; j + 4 <= m; j += 4) {
            const Zd v0 = V<C>::load(Vb.at(j), i);
            const Zd v1 = V<C>::load(Vb.at(j + 1), i);
            const Zd v2 = V<C>::load(Vb.at(j + 2), i);
            const Zd v3 = V<C>::load(Vb.at(j + 3), i);
            if constexpr (C) {
                acc = cadd(acc, cmul(sc[j], v0));
                acc = cadd(acc, cmul(sc[j + 1], v1));
                acc = cadd(acc, cmul(sc[j + 2], v2));
                acc = cadd(acc, cmul(sc[j + 3], v3));
            } else {
                acc.re += sc[j].re * v0.re;
                acc.re += sc[j + 1].re * v1.re;
                acc.re += sc[j + 2].re * v2.re;
                acc.re += sc[j + 3].re * v3.re;
            }
        }
        for (; j < m; ++j) {
            const Zd vj = V<C>::load(Vb.at(j), i);
            acc = C ? cadd(acc, cmul(sc[j], vj)) : Zd{acc.re + sc[j].re * vj.re, 0.0};
        }
        V<C>::store(w, i, acc);
        if (want_norm) s0 += acc.re * acc.re + (C ? acc.im * acc.im : 0.0);
    }
    if (want_norm) {
        block_sum2(s0, s1);
        if (threadIdx.x == 0) {
            partial[2 * blockIdx.x] = s0;
            partial[2 * blockIdx.x + 1] = 0.0;
        }
    }
}

// axpy_many below kSplitRows rows: a thread takes one row and all columns, sixteen loads in flight (then
// four, then one), added in column order as above (the same bits). One thread per four rows with four
// loads in flight left the card idle: 44 us for 9252 rows and 100 columns. Workgroups of one wavefront up
// to 2^16 rows, so that these spread over the compute units, of four above, a row a thread up to
// kSplitRows: at most 2048 of them (400,000 rows, a call with its 40 us of host work: 20 real columns 60
// us and 100 complex 167; 61 and 163 by the kernel above, 69 and 176 with 1024 workgroups of one wavefront
// at most and the last columns one at a time).
// From 2^19 rows on the threads of the kernel above keep enough loads in flight.
constexpr std::size_t kSplitRows = std::size_t{1} << 19;
inline int split_threads(std::size_t n) { return n <= (std::size_t{1} << 16) ? 64 : 256; }

template <bool C, int U>
__device__ __forceinline__ void add_columns(const Cols& Vb, const Zd* sc, int m, std::size_t i, int& j, Zd& acc) {
    for (; j + U <= m; j += U) {
        Zd v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = V<C>::load(Vb.at(j + u), i);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if constexpr (C) acc = cadd(acc, cmul(sc[j + u], v[u]));
            else acc.re += sc[j + u].re * v[u].re;
        }
    }
}

template <bool C>
__global__ __launch_bounds__(kThreads) void k_axpy_many_split(const Zd* coeffs, Cols Vb, int m, void* w,
                                                              std::size_t n, double* partial, int want_norm,
                                                              double sign, const int* gate) {
    if (gate && !*gate) return;
    __shared__ Zd sc[kManyCols];
    __shared__ double wave[kWaves];
    for (int j = threadIdx.x; j < m; j += blockDim.x) sc[j] = Zd{sign * coeffs[j].re, sign * coeffs[j].im};
    __syncthreads();
    double s0 = 0.0;
    const std::size_t i = blockIdx.x * static_cast<std::size_t>(blockDim.x) + threadIdx.x;
    if (i < n) {
        Zd acc = V<C>::load(w, i);
        int j = 0;
        add_columns<C, 16>(Vb, sc, m, i, j, acc);
        add_columns<C, 4>(Vb, sc, m, i, j, acc);
        add_columns<C, 1>(Vb, sc, m, i, j, acc);
        V<C>::store(w, i, acc);
        s0 = acc.re * acc.re + (C ? acc.im * acc.im : 0.0);
    }
    if (want_norm) {   // the wavefronts' sums in order
        s0 = wave_sum(s0);
        if ((threadIdx.x & 63u) == 0) wave[threadIdx.x >> 6] = s0;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (unsigned q = 1; q < blockDim.x / 64; ++q) s0 += wave[q];
            partial[2 * blockIdx.x] = s0;
            partial[2 * blockIdx.x + 1] = 0.0;
        }
    }
}

constexpr int kRotCols = 16;
template <bool C>
__global__ __launch_bounds__(256) void k_block_rotate(const void* Vb, std::size_t ld, int mm, const double* S, int c0,
                                                      int nc, void* out, std::size_t n) {
    const std::size_t i = blockIdx.x * static_cast<std::size_t>(blockDim.x) + threadIdx.x;
    if (i >= n) return;
    Zd acc[kRotCols];
#pragma unroll
    for (int c = 0; c < kRotCols; ++c) acc[c] = Zd{0.0, 0.0};
    for (int r = 0; r < mm; ++r) {
        const Zd v = V<C>::load(Vb, r * ld + i);
#pragma unroll
        for (int c = 0; c < kRotCols; ++c)
            if (c < nc) {
                const double s = S[static_cast<std::size_t>(c0 + c) * mm + r];
                acc[c].re += v.re * s;
                if constexpr (C) acc[c].im += v.im * s;
            }
    }
#pragma unroll
    for (int c = 0; c < kRotCols; ++c)
        if (c < nc) V<C>::store(out, static_cast<std::size_t>(c0 + c) * n + i, acc[c]);
}

}  // namespace

std::size_t blas_scratch_bytes(std::size_t max_cols) {
    (void)max_cols;
    const std::size_t red = 2 * std::max<std::size_t>(kMaxBlocks, kSplitRows / 256) * sizeof(double);
    const std::size_t many = static_cast<std::size_t>(kMaxBlocks) * (kManyCols + 1) * 2 * sizeof(double);
    return red > many ? red : many;
}

void fill_zero(bool c, void* x, std::size_t n, hipStream_t st) {
    if (!n) return;
    const unsigned g = grid_for(n);
    if (c) hipLaunchKernelGGL(k_fill_zero<true>, dim3(g), dim3(kThreads), 0, st, x, n);
    else hipLaunchKernelGGL(k_fill_zero<false>, dim3(g), dim3(kThreads), 0, st, x, n);
}

void fill_gaussian(bool c, void* x, std::size_t n, u64 seed, hipStream_t st) {
    if (!n) return;
    const unsigned g = grid_for(n);
    if (c) hipLaunchKernelGGL(k_fill_gauss<true>, dim3(g), dim3(kThreads), 0, st, x, n, seed);
    else hipLaunchKernelGGL(k_fill_gauss<false>, dim3(g), dim3(kThreads), 0, st, x, n, seed);
}

static void launch_axpby(bool c, Coef a, const void* x, Zd b, void* y, std::size_t n, int mode, hipStream_t st) {
    if (!n) return;
    const unsigned g = grid_for(n);
    if (c) hipLaunchKernelGGL(k_axpby<true>, dim3(g), dim3(kThreads), 0, st, a, x, b, y, n, mode);
    else hipLaunchKernelGGL(k_axpby<false>, dim3(g), dim3(kThreads), 0, st, a, x, b, y, n, mode);
}

void axpy(bool c, Zd a, const void* x, void* y, std::size_t n, hipStream_t st) { launch_axpby(c, Coef{a}, x, Zd{0, 0}, y, n, 0, st); }
void axpy(bool c, Coef a, const void* x, void* y, std::size_t n, hipStream_t st) { launch_axpby(c, a, x, Zd{0, 0}, y, n, 0, st); }
void scale(bool c, Zd a, void* x, std::size_t n, hipStream_t st) { launch_axpby(c, Coef{a}, nullptr, Zd{0, 0}, x, n, 1, st); }
void axpby(bool c, Zd a, const void* x, Zd b, void* y, std::size_t n, hipStream_t st) {
    launch_axpby(c, Coef{a}, x, b, y, n, 2, st);
}

void scale_by(bool c, const void* w, const double* norm, void* out, std::size_t n, hipStream_t st) {
    if (!n) return;
    const unsigned g = grid_for(n);
    if (c) hipLaunchKernelGGL(k_scale_by<true>, dim3(g), dim3(kThreads), 0, st, w, norm, out, n);
    else hipLaunchKernelGGL(k_scale_by<false>, dim3(g), dim3(kThreads), 0, st, w, norm, out, n);
}

void cgs_gate(const double* before2, const double* after2, double kappa, int* again, hipStream_t st) {
    hipLaunchKernelGGL(k_cgs_gate, dim3(1), dim3(1), 0, st, before2, after2, kappa, again);
}

void add_pair(const Zd* a, const Zd* b, Zd* out, hipStream_t st) {
    hipLaunchKernelGGL(k_add_pair, dim3(1), dim3(1), 0, st, a, b, out);
}

static void reduce(bool c, int kind, Coef a, const void* x, void* y, const void* z, std::size_t n, int fuse,
                   void* scratch, int out_kind, void* out, hipStream_t st) {
    const unsigned g = grid_for(n);
    double* part = static_cast<double*>(scratch);
    if (c) {
        if (kind == 0) hipLaunchKernelGGL((k_reduce<true, 0>), dim3(g), dim3(kThreads), 0, st, a, x, y, z, n, fuse, part);
        else hipLaunchKernelGGL((k_reduce<true, 1>), dim3(g), dim3(kThreads), 0, st, a, x, y, z, n, fuse, part);
    } else {
        if (kind == 0) hipLaunchKernelGGL((k_reduce<false, 0>), dim3(g), dim3(kThreads), 0, st, a, x, y, z, n, fuse, part);
        else hipLaunchKernelGGL((k_reduce<false, 1>), dim3(g), dim3(kThreads), 0, st, a, x, y, z, n, fuse, part);
    }
    hipLaunchKernelGGL(k_finish, dim3(1), dim3(kThreads), 0, st, part, static_cast<int>(g), out_kind, out, static_cast<const int*>(nullptr));
}

void dot(bool c, const void* x, const void* y, std::size_t n, void* scratch, Zd* result, hipStream_t st) {
    reduce(c, 0, Coef{}, nullptr, const_cast<void*>(y), x, n, 0, scratch, 0, result, st);
}
void nrm2(bool c, const void* x, std::size_t n, void* scratch, double* result, hipStream_t st) {
    reduce(c, 1, Coef{}, nullptr, const_cast<void*>(x), nullptr, n, 0, scratch, 1, result, st);
}
void axpy_dot(bool c, Zd a, const void* x, void* y, const void* z, std::size_t n, void* scratch, Zd* result,
              hipStream_t st) {
    reduce(c, 0, Coef{a}, x, y, z, n, 1, scratch, 0, result, st);
}
void axpy_dot(bool c, Coef a, const void* x, void* y, const void* z, std::size_t n, void* scratch, Zd* result,
              hipStream_t st) {
    reduce(c, 0, a, x, y, z, n, 1, scratch, 0, result, st);
}
void axpy_nrm2(bool c, Zd a, const void* x, void* y, std::size_t n, void* scratch, double* result, hipStream_t st) {
    reduce(c, 1, Coef{a}, x, y, nullptr, n, 1, scratch, 1, result, st);
}
void axpy_nrm2(bool c, Coef a, const void* x, void* y, std::size_t n, void* scratch, double* result, hipStream_t st) {
    reduce(c, 1, a, x, y, nullptr, n, 1, scratch, 1, result, st);
}

static void dot_many_cols(bool c, const void* V, std::size_t ld, const void* const* table, std::size_t m,
                          const void* w, std::size_t n, void* scratch, Zd* coeffs, double* wnorm2, hipStream_t st,
                          const int* gate) {
    double* part = static_cast<double*>(scratch);
    const std::size_t elem = c ? sizeof(Zd) : sizeof(double);
    std::size_t done = 0;
    bool first = true;
    std::size_t nb = (n + kTile - 1) / kTile;
    if (nb > static_cast<std::size_t>(kMaxBlocks)) nb = kMaxBlocks;
    if (nb < 1) nb = 1;
    const std::size_t rpb = (n + nb - 1) / nb;
    do {
        const int mc = static_cast<int>((m - done) < static_cast<std::size_t>(kManyCols) ? (m - done) : kManyCols);
        const Cols Vc{table ? nullptr : static_cast<const char*>(V) + done * ld * elem, ld * elem,
                      table ? table + done : nullptr};
        const int want = (first && wnorm2) ? 1 : 0;
        const int per = dot_columns(mc, nb);
        const dim3 grid(static_cast<unsigned>(nb), static_cast<unsigned>(mc > 0 ? (mc + per - 1) / per : 1));
        if (c)
            hipLaunchKernelGGL(k_dot_many<true>, grid, dim3(kThreads), 0, st, Vc, mc, per, w, n, rpb, part,
                               static_cast<int>(nb), want, gate);
        else
            hipLaunchKernelGGL(k_dot_many<false>, grid, dim3(kThreads), 0, st, Vc, mc, per, w, n, rpb, part,
                               static_cast<int>(nb), want, gate);
        hipLaunchKernelGGL(k_dot_many_finish, dim3(static_cast<unsigned>(mc + want)), dim3(kThreads), 0, st, part,
                           static_cast<int>(nb), mc, coeffs + done, want ? wnorm2 : nullptr, gate);
        done += static_cast<std::size_t>(mc);
        first = false;
    } while (done < m);
}

void dot_many(bool c, const void* V, std::size_t ld, std::size_t m, const void* w, std::size_t n, void* scratch,
              Zd* coeffs, double* wnorm2, hipStream_t st, const int* gate) {
    dot_many_cols(c, V, ld, nullptr, m, w, n, scratch, coeffs, wnorm2, st, gate);
}
void dot_many_table(bool c, const void* const* table, std::size_t m, const void* w, std::size_t n, void* scratch,
                    Zd* coeffs, hipStream_t st) {
    if (m) dot_many_cols(c, nullptr, 0, table, m, w, n, scratch, coeffs, nullptr, st, nullptr);
}

static void axpy_many_cols(bool c, const Zd* coeffs, const void* V, std::size_t ld, const void* const* table,
                           std::size_t m, void* w, std::size_t n, void* scratch, double* wnorm2, hipStream_t st,
                           double sign, const int* gate, bool root) {
    double* part = static_cast<double*>(scratch);
    const std::size_t elem = c ? sizeof(Zd) : sizeof(double);
    const bool split = n < kSplitRows;
    const std::size_t threads = split ? static_cast<std::size_t>(split_threads(n)) : kThreads;
    const unsigned g = split ? static_cast<unsigned>(std::max<std::size_t>((n + threads - 1) / threads, 1)) : grid_for(n);
    std::size_t done = 0;
    do {
        const int mc = static_cast<int>((m - done) < static_cast<std::size_t>(kManyCols) ? (m - done) : kManyCols);
        const bool last = done + static_cast<std::size_t>(mc) >= m;
        const int want = (last && wnorm2) ? 1 : 0;
        const Cols Vc{table ? nullptr : static_cast<const char*>(V) + done * ld * elem, ld * elem,
                      table ? table + done : nullptr};
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(g), dim3(static_cast<unsigned>(threads)), 0, st, coeffs + done, Vc, mc, w, n, part,
                               want, sign, gate);
        };
        if (split && c) go(k_axpy_many_split<true>);
        else if (split) go(k_axpy_many_split<false>);
        else if (c) go(k_axpy_many<true>);
        else go(k_axpy_many<false>);
        if (want) hipLaunchKernelGGL(k_finish, dim3(1), dim3(kThreads), 0, st, part, static_cast<int>(g), root ? 1 : 2,
                                     wnorm2, gate);
        done += static_cast<std::size_t>(mc);
    } while (done < m);
}

void axpy_many(bool c, const Zd* coeffs, const void* V, std::size_t ld, std::size_t m, void* w, std::size_t n,
               void* scratch, double* wnorm2, hipStream_t st, double sign, const int* gate, bool root) {
    axpy_many_cols(c, coeffs, V, ld, nullptr, m, w, n, scratch, wnorm2, st, sign, gate, root);
}
void axpy_many_table(bool c, const Zd* coeffs, const void* const* table, std::size_t m, void* w, std::size_t n,
                     hipStream_t st) {
    if (m) axpy_many_cols(c, coeffs, nullptr, 0, table, m, w, n, nullptr, nullptr, st, 1.0, nullptr, false);
}

void block_rotate(bool c, const void* Vm, std::size_t ld, std::size_t mm, const double* S, std::size_t cols, void* out,
                  std::size_t n, hipStream_t st) {
    const dim3 grid(static_cast<unsigned>((n + 255) / 256)), block(256);
    for (std::size_t c0 = 0; c0 < cols; c0 += kRotCols) {
        const int nc = static_cast<int>(std::min<std::size_t>(kRotCols, cols - c0));
        if (c)
            hipLaunchKernelGGL(k_block_rotate<true>, grid, block, 0, st, Vm, ld, static_cast<int>(mm), S,
                               static_cast<int>(c0), nc, out, n);
        else
            hipLaunchKernelGGL(k_block_rotate<false>, grid, block, 0, st, Vm, ld, static_cast<int>(mm), S,
                               static_cast<int>(c0), nc, out, n);
    }
}

}  // namespace qsa::dev
