// Reduced-CSR SpMV for the symmetry-sector operator, real or complex, one to eight vectors.
//
// L lanes of a wavefront share a row: lane l takes entries e0 + l, e0 + l + L, ... (coalesced
// column / id streams), and the L partial sums meet through a fixed xor-butterfly, so the result
// is deterministic and a k-vector apply equals k single applies bit for bit (the contract of the
// reference's csr_spmv, src/gpu/rep_matvec.cu:1003-1036). Values come from a dictionary by u8 or
// u16 id (the reference's reduced_csr.h layout) or are stored in full.
#include <hipcub/hipcub.hpp>

#include "dev_common.h"
#include "launch.h"

namespace qsa::dev {

namespace {

template <int NV> struct Ptrs {
    const void* in[NV];
    void* out[NV];
};

// The dictionary an entry's value id points into. LD: in LDS (staged at kernel start, a complex value
// as one 16-byte word), else in global memory. A lookup is a gather over a handful of lines, and the
// vector cache serves one line per clock to lanes that do not share theirs with a neighbour, so a
// dictionary in global memory costs as much as the gather of x itself (twice that for a complex value,
// whose parts lie apart). With u16 ids read from global memory, then from LDS: a 9.4M-row real sector
// (609 values) 1.236 -> 1.105 ms an apply, four interleaved vectors on a 1.43M-row complex one (405
// values) 0.399 -> 0.367 ms.
template <bool LD> struct Dict {
    const double* re;
    const double* im;
};

extern __shared__ __align__(16) double lds_dict[];

/// LDS bytes a launch with the dictionary staged needs.
inline std::size_t dict_lds_bytes(const CsrView& A) {
    return A.width == 0 ? 0 : static_cast<std::size_t>(A.dict_n) * (A.values_real ? 8 : 16);
}
/// The largest staged dictionary: with the kernels' own arrays (256 bytes in k_sell_lanczos) within 64 KB
/// a workgroup.
constexpr std::size_t kLdsDictMax = 64 * 1024 - 512;
inline bool dict_in_lds(const CsrView& A) { return A.lds_dict && dict_lds_bytes(A) <= kLdsDictMax; }

template <int WIDTH, bool VREAL, bool LD> __device__ __forceinline__ Dict<LD> stage_dict(const CsrView& A) {
    if constexpr (LD && WIDTH != 0) {
        for (int i = threadIdx.x; i < A.dict_n; i += blockDim.x) {
            if constexpr (VREAL) {
                lds_dict[i] = A.dict_re[i];
            } else {
                lds_dict[2 * i] = A.dict_re[i];
                lds_dict[2 * i + 1] = A.dict_im[i];
            }
        }
        __syncthreads();
    }
    return Dict<LD>{A.dict_re, A.dict_im};
}

template <bool VREAL, bool LD> __device__ __forceinline__ void dict_value(const Dict<LD>& d, u32 id, double& vr, double& vi) {
    if constexpr (LD) {
        if constexpr (VREAL) {
            vr = lds_dict[id];
        } else {
            const Zd z = reinterpret_cast<const Zd*>(lds_dict)[id];
            vr = z.re;
            vi = z.im;
        }
    } else {
        vr = d.re[id];
        if constexpr (!VREAL) vi = d.im[id];
    }
}

template <int WIDTH, bool VREAL, bool LD>
__device__ __forceinline__ void value_at(const CsrView& A, const Dict<LD>& d, u64 e, double& vr, double& vi) {
    if constexpr (WIDTH == 1) {
        const u32 id = A.nt ? __builtin_nontemporal_load(static_cast<const u8*>(A.vals) + e) : static_cast<const u8*>(A.vals)[e];
        dict_value<VREAL, LD>(d, id, vr, vi);
    } else if constexpr (WIDTH == 2) {
        const u32 id = A.nt ? __builtin_nontemporal_load(static_cast<const u16*>(A.vals) + e) : static_cast<const u16*>(A.vals)[e];
        dict_value<VREAL, LD>(d, id, vr, vi);
    } else {
        if constexpr (VREAL) {
            vr = static_cast<const double*>(A.vals)[e];
        } else {
            const Zd z = static_cast<const Zd*>(A.vals)[e];
            vr = z.re;
            vi = z.im;
        }
    }
}

// The workgroup's place in the row order. With A.xcd the grid is a multiple of 8 and the
// workgroups the dispatcher sends to one XCD (blockIdx = x mod 8, round robin) take one contiguous
// eighth of the rows, so each XCD's L2 sees the columns of neighbouring rows together.
__device__ __forceinline__ i64 row_block(const CsrView& A) {
    if (!A.xcd) return blockIdx.x;
    const u32 per = gridDim.x >> 3;
    return static_cast<i64>(blockIdx.x & 7u) * per + (blockIdx.x >> 3);
}

/// Threads per workgroup; 1024 where smaller workgroups' copies of the dictionary would leave a compute
/// unit short of waves.
inline unsigned block_threads(const CsrView& A) {
    if (dict_in_lds(A) && dict_lds_bytes(A) > 16 * 1024) return 1024;
    return (A.wg == 512 || A.wg == 1024) ? A.wg : 256;
}

/// A as a launch of `vectors` with `lanes` threads per row reads it: more than 256 values (u16 ids) are
/// staged only where a workgroup looks up enough of them to pay for its copy: 7/10 of the dictionary's
/// size below 2^18 rows (a few workgroups per compute unit, bound by the chain of loads); from there on,
/// where the loads themselves bound it, its size, and 9/4 of it for one vector of a real operator (one
/// load a lookup saved, not two). us an apply from global memory / staged, lookups over values: 32,066
/// rows, 3637 real 7.7 / 6.7 at 0.8; 32,065, 3841 complex 10.3 / 7.6 at 0.8; 9252, 1890 real 4.3 / 3.9 at
/// 0.7; 3432, 1730 real, four vectors 4.1 / 4.3 at 0.6; 112,720, 7683 real 23.0 / 23.7 at 0.4, four vectors
/// 55 / 59; 5.17 million, 996 real 707 / 773 at 1.0, 719 / 727 at 2.1, four vectors 2170 / 2070 at 1.0; 1.43
/// million, 804 real 169 / 162 at 2.4, 892 complex 222 / 208 at 1.1.
inline CsrView staged(const CsrView& A, unsigned lanes, int vectors) {
    CsrView B = A;
    if (A.dict_n > 256 && dict_in_lds(A)) {
        const double rows = std::min<double>(static_cast<double>(A.rows), block_threads(A) / lanes);
        const double least = A.rows < (i64{1} << 18) ? 0.7 : A.values_real && vectors == 1 ? 2.25 : 1.0;
        if (rows * A.mean_row < least * A.dict_n) B.lds_dict = 0;
    }
    return B;
}

inline unsigned grid_blocks(const CsrView& A, u64 threads) {
    const u64 t = block_threads(A);
    u64 b = (threads + t - 1) / t;
    if (A.xcd) b = (b + 7) / 8 * 8;
    return static_cast<unsigned>(b);
}

// Column and value of entry e. WIDTH 3: the u8 id packed in the top byte of the column word
// (columns below 2^24), one 4-byte load per entry.
template <int WIDTH, bool VREAL, bool LD>
__device__ __forceinline__ void load_entry(const CsrView& A, const Dict<LD>& d, u64 e, u32& c, double& vr, double& vi) {
    if constexpr (WIDTH == 3) {
        const u32 w = A.nt ? __builtin_nontemporal_load(A.col + e) : A.col[e];
        c = w & 0xFFFFFFu;
        dict_value<VREAL, LD>(d, w >> 24, vr, vi);
    } else {
        c = A.nt ? __builtin_nontemporal_load(A.col + e) : A.col[e];
        value_at<WIDTH, VREAL, LD>(A, d, e, vr, vi);
    }
}

template <int WIDTH, bool VREAL, bool REAL, bool LD, int L, int NV, int U>
__global__ __launch_bounds__(1024) void k_spmv(CsrView A, Ptrs<NV> v) {
    const Dict<LD> d = stage_dict<WIDTH, VREAL, LD>(A);
    const i64 gid = row_block(A) * blockDim.x + threadIdx.x;
    const i64 row = gid / L;
    const int lane = static_cast<int>(gid % L);
    double ar[NV], ai[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) ar[k] = ai[k] = 0.0;
    auto accumulate = [&](u32 c, double vr, double vi) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            if constexpr (REAL) {
                ar[k] += vr * static_cast<const double*>(v.in[k])[c];
            } else {
                const Zd x = static_cast<const Zd*>(v.in[k])[c];
                ar[k] += vr * x.re - vi * x.im;
                ai[k] += vr * x.im + vi * x.re;
            }
        }
    };
    if (row < A.rows) {
        const u64 e0 = A.row_ptr[row], e1 = A.row_ptr[row + 1];
        u64 e = e0 + lane;
        if constexpr (U > 1) {
            // U of the lane's entries per round: their columns and values first, then the U gathers
            // issued together; the sums are taken in entry order, as in the one-at-a-time loop
            for (; e + static_cast<u64>(U - 1) * L < e1; e += static_cast<u64>(U) * L) {
                u32 c[U];
                double vr[U], vi[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    vi[u] = 0.0;
                    load_entry<WIDTH, VREAL, LD>(A, d, e + u * L, c[u], vr[u], vi[u]);
                }
                if constexpr (REAL && NV == 1) {
                    double x[U];
#pragma unroll
                    for (int u = 0; u < U; ++u) x[u] = static_cast<const double*>(v.in[0])[c[u]];
#pragma unroll
                    for (int u = 0; u < U; ++u) ar[0] += vr[u] * x[u];
                } else {
#pragma unroll
                    for (int u = 0; u < U; ++u) accumulate(c[u], vr[u], vi[u]);
                }
            }
        }
        for (; e < e1; e += L) {
            u32 c;
            double vr, vi = 0.0;
            load_entry<WIDTH, VREAL, LD>(A, d, e, c, vr, vi);
            accumulate(c, vr, vi);
        }
    }
#pragma unroll
    for (int off = L / 2; off > 0; off >>= 1) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            ar[k] += __shfl_xor(ar[k], off, L);
            if constexpr (!REAL) ai[k] += __shfl_xor(ai[k], off, L);
        }
    }
    if (row < A.rows && lane == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            if constexpr (REAL) static_cast<double*>(v.out[k])[row] = ar[k];
            else static_cast<Zd*>(v.out[k])[row] = Zd{ar[k], ai[k]};
        }
    }
}

// Block-interleaved vectors: X[row * NV + k].
template <int WIDTH, bool VREAL, bool REAL, bool LD, int L, int NV>
__global__ __launch_bounds__(256) void k_spmv_block(CsrView A, const void* X, void* Y) {
    const Dict<LD> d = stage_dict<WIDTH, VREAL, LD>(A);
    const i64 gid = row_block(A) * blockDim.x + threadIdx.x;
    const i64 row = gid / L;
    const int lane = static_cast<int>(gid % L);
    double ar[NV], ai[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) ar[k] = ai[k] = 0.0;
    if (row < A.rows) {
        const u64 e0 = A.row_ptr[row], e1 = A.row_ptr[row + 1];
        for (u64 e = e0 + lane; e < e1; e += L) {
            u32 c32;
            double vr, vi = 0.0;
            load_entry<WIDTH, VREAL, LD>(A, d, e, c32, vr, vi);
            const u64 c = c32;
#pragma unroll
            for (int k = 0; k < NV; ++k) {
                if constexpr (REAL) {
                    ar[k] += vr * static_cast<const double*>(X)[c * NV + k];
                } else {
                    const Zd x = static_cast<const Zd*>(X)[c * NV + k];
                    ar[k] += vr * x.re - vi * x.im;
                    ai[k] += vr * x.im + vi * x.re;
                }
            }
        }
    }
#pragma unroll
    for (int off = L / 2; off > 0; off >>= 1) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            ar[k] += __shfl_xor(ar[k], off, L);
            if constexpr (!REAL) ai[k] += __shfl_xor(ai[k], off, L);
        }
    }
    if (row < A.rows && lane == 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            if constexpr (REAL) static_cast<double*>(Y)[row * NV + k] = ar[k];
            else static_cast<Zd*>(Y)[row * NV + k] = Zd{ar[k], ai[k]};
        }
    }
}

// ---- SELL-64 ------------------------------------------------------------------------------------
// Slice s holds rows 64 s .. 64 s + 63 in groups of four entries: entry k of row 64 s + j sits at
// sell_ptr[s] + 256 (k / 4) + 4 j + k % 4, so one 16-byte load gives a lane four consecutive
// entries of its row and the group loads of a wavefront's 64 rows are one contiguous kilobyte. A
// slice is padded to its longest row, rounded up to whole groups; a row's last group is filled up with
// zeros, what the slice holds past it is not written, and no entry beyond a row's length is used. One lane owns a row and sums its entries in CSR order: the sum
// depends neither on the workgroup size nor on how many gathers are in flight, and a k-vector
// apply equals k single applies bit for bit. U entries per round: their groups first, then the U
// gathers together, then the sums in entry order.
// ACC partial sums per row and vector: entry k goes to sum k mod ACC (k in the row's order), and
// the sums meet in a fixed tree, (s0 + s2) + (s1 + s3) for ACC = 4 -- the order a 4-lane butterfly
// gives, so the block kernel's 4 lanes per row produce the same bits.
__device__ __forceinline__ u64 sell_at(u64 slice, u32 j, u32 k) {
    return slice + static_cast<u64>(k >> 2) * 256 + static_cast<u64>(j) * 4 + (k & 3u);
}

typedef u32 u32x4 __attribute__((ext_vector_type(4)));
typedef u16 u16x4 __attribute__((ext_vector_type(4)));
typedef u8 u8x4 __attribute__((ext_vector_type(4)));

template <class V> __device__ __forceinline__ V load_vec(const CsrView& A, const void* p) {
    return A.nt ? __builtin_nontemporal_load(static_cast<const V*>(p)) : *static_cast<const V*>(p);
}

// The four entries of the group at e (a multiple of four): columns and values.
template <int WIDTH, bool VREAL, bool LD>
__device__ __forceinline__ void load_quad(const CsrView& A, const Dict<LD>& d, u64 e, u32* c, double* vr, double* vi) {
    const u32x4 w = load_vec<u32x4>(A, A.col + e);
    if constexpr (WIDTH == 3) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            c[u] = w[u] & 0xFFFFFFu;
            dict_value<VREAL, LD>(d, w[u] >> 24, vr[u], vi[u]);
        }
    } else {
#pragma unroll
        for (int u = 0; u < 4; ++u) c[u] = w[u];
        if constexpr (WIDTH == 1) {
            const u8x4 id = load_vec<u8x4>(A, static_cast<const u8*>(A.vals) + e);
#pragma unroll
            for (int u = 0; u < 4; ++u) dict_value<VREAL, LD>(d, id[u], vr[u], vi[u]);
        } else if constexpr (WIDTH == 2) {
            const u16x4 id = load_vec<u16x4>(A, static_cast<const u16*>(A.vals) + e);
#pragma unroll
            for (int u = 0; u < 4; ++u) dict_value<VREAL, LD>(d, id[u], vr[u], vi[u]);
        } else {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if constexpr (VREAL) {
                    vr[u] = static_cast<const double*>(A.vals)[e + u];
                } else {
                    const Zd z = static_cast<const Zd*>(A.vals)[e + u];
                    vr[u] = z.re;
                    vi[u] = z.im;
                }
            }
        }
    }
}

template <int ACC> __device__ __forceinline__ double tree(const double* s) {
    if constexpr (ACC == 4) return (s[0] + s[2]) + (s[1] + s[3]);
    else return s[0];
}

/// Row `row` of the SELL layout applied to the NV vectors: ACC partial sums per vector, entries in
/// groups of four, U per round.
template <int WIDTH, bool VREAL, bool REAL, bool LD, int NV, int U, int ACC>
__device__ __forceinline__ void sell_row_sums(const CsrView& A, const Dict<LD>& d, i64 row, const Ptrs<NV>& v,
                                              double (&ar)[NV][ACC], double (&ai)[NV][ACC]) {
    static_assert(U % 4 == 0, "whole groups of four entries per round");
    const u32 n = A.nt ? __builtin_nontemporal_load(A.sell_len + row) : A.sell_len[row];
    const u64 first = A.sell_ptr[row >> 6] + static_cast<u64>(row & 63) * 4;   // group g at first + 256 g
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
        for (int j = 0; j < ACC; ++j) ar[k][j] = ai[k][j] = 0.0;
    auto accumulate = [&](int j, u32 c, double vr, double vi) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            if constexpr (REAL) {
                ar[k][j] += vr * static_cast<const double*>(v.in[k])[c];
            } else {
                const Zd x = static_cast<const Zd*>(v.in[k])[c];
                ar[k][j] += vr * x.re - vi * x.im;
                ai[k][j] += vr * x.im + vi * x.re;
            }
        }
    };
    u32 k = 0;
    for (; k + U <= n; k += U) {
        u32 c[U];
        double vr[U], vi[U];
#pragma unroll
        for (int u = 0; u < U; ++u) vi[u] = 0.0;
#pragma unroll
        for (int g = 0; g < U / 4; ++g)
            load_quad<WIDTH, VREAL, LD>(A, d, first + static_cast<u64>(k / 4 + g) * 256, c + 4 * g, vr + 4 * g, vi + 4 * g);
        if constexpr (REAL && NV == 1) {
            double x[U];
#pragma unroll
            for (int u = 0; u < U; ++u) x[u] = static_cast<const double*>(v.in[0])[c[u]];
#pragma unroll
            for (int u = 0; u < U; ++u) ar[0][u % ACC] += vr[u] * x[u];
        } else {
#pragma unroll
            for (int u = 0; u < U; ++u) accumulate(u % ACC, c[u], vr[u], vi[u]);
        }
    }
    for (; k < n; k += 4) {   // the last groups, entries below n (k stays a multiple of four)
        u32 c[4];
        double vr[4], vi[4] = {0.0, 0.0, 0.0, 0.0};
        load_quad<WIDTH, VREAL, LD>(A, d, first + static_cast<u64>(k / 4) * 256, c, vr, vi);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (k + static_cast<u32>(u) < n) accumulate(u % ACC, c[u], vr[u], vi[u]);
    }
}

template <int WIDTH, bool VREAL, bool REAL, bool LD, int NV, int U, int ACC>
__global__ __launch_bounds__(1024) void k_sell(CsrView A, Ptrs<NV> v) {
    const Dict<LD> d = stage_dict<WIDTH, VREAL, LD>(A);
    const i64 row = row_block(A) * blockDim.x + threadIdx.x;
    if (row >= A.rows) return;
    double ar[NV][ACC], ai[NV][ACC];
    sell_row_sums<WIDTH, VREAL, REAL, LD, NV, U, ACC>(A, d, row, v, ar, ai);
#pragma unroll
    for (int q = 0; q < NV; ++q) {
        if constexpr (REAL) static_cast<double*>(v.out[q])[row] = tree<ACC>(ar[q]);
        else static_cast<Zd*>(v.out[q])[row] = Zd{tree<ACC>(ar[q]), tree<ACC>(ai[q])};
    }
}

// The Lanczos step's first pass in the SpMV's epilogue: w = H v - beta v_prev (v_prev null at the
// first step) written, and the partial of <v, w> of each kLanczosPart rows (the wavefronts' xor trees,
// then the wavefronts in order) into partial -- the apply followed by axpy_dot, without writing and
// reading w in between. k_lanczos_finish sums the partials in row order, so alpha's bits do not depend on
// the workgroup size that the tuner picked.
constexpr int kLanczosPart = 256;
template <int WIDTH, bool VREAL, bool REAL, bool LD, int U, int ACC>
__global__ __launch_bounds__(1024) void k_sell_lanczos(CsrView A, Ptrs<1> v, const void* vprev,
                                                       const double* betap, double* partial) {
    __shared__ double wr[16], wi[16];
    const Dict<LD> d = stage_dict<WIDTH, VREAL, LD>(A);
    const i64 row0 = row_block(A) * blockDim.x, row = row0 + threadIdx.x;
    const double beta = vprev ? *betap : 0.0;
    double pr = 0.0, pi = 0.0;
    if (row < A.rows) {
        double ar[1][ACC], ai[1][ACC];
        sell_row_sums<WIDTH, VREAL, REAL, LD, 1, U, ACC>(A, d, row, v, ar, ai);
        if constexpr (REAL) {
            double w = tree<ACC>(ar[0]);
            if (vprev) w = w - beta * static_cast<const double*>(vprev)[row];
            static_cast<double*>(v.out[0])[row] = w;
            pr = static_cast<const double*>(v.in[0])[row] * w;
        } else {
            Zd w{tree<ACC>(ar[0]), tree<ACC>(ai[0])};
            if (vprev) {
                const Zd p = static_cast<const Zd*>(vprev)[row];
                w = Zd{w.re - beta * p.re, w.im - beta * p.im};
            }
            static_cast<Zd*>(v.out[0])[row] = w;
            const Zd x = static_cast<const Zd*>(v.in[0])[row];   // conj(x) w
            pr = x.re * w.re + x.im * w.im;
            pi = x.re * w.im - x.im * w.re;
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        pr += __shfl_xor(pr, off, 64);
        pi += __shfl_xor(pi, off, 64);
    }
    const int wave = static_cast<int>(threadIdx.x >> 6);
    if ((threadIdx.x & 63) == 0) {
        wr[wave] = pr;
        wi[wave] = pi;
    }
    __syncthreads();
    constexpr int kWaves = kLanczosPart / 64;
    const i64 first = row0 + static_cast<i64>(threadIdx.x) * kLanczosPart;   // thread t sums the workgroup's part t
    if (threadIdx.x < blockDim.x / kLanczosPart && first < A.rows) {
        double a = 0.0, b = 0.0;
        for (int q = 0; q < kWaves; ++q) {
            a += wr[static_cast<int>(threadIdx.x) * kWaves + q];
            b += wi[static_cast<int>(threadIdx.x) * kWaves + q];
        }
        partial[2 * (first / kLanczosPart)] = a;
        partial[2 * (first / kLanczosPart) + 1] = b;
    }
}

// (One workgroup sums all pairs: 1024 threads take 5 us for 10,106 of them, 256 took 16.)
constexpr int kFinishThreads = 1024;
__global__ __launch_bounds__(kFinishThreads) void k_lanczos_finish(const double* partial, int nb, Zd* alpha) {
    __shared__ double sr[kFinishThreads], si[kFinishThreads];
    double a = 0.0, b = 0.0;
#pragma unroll 4
    for (int i = static_cast<int>(threadIdx.x); i < nb; i += kFinishThreads) {
        a += partial[2 * i];
        b += partial[2 * i + 1];
    }
    sr[threadIdx.x] = a;
    si[threadIdx.x] = b;
    __syncthreads();
    for (int h = kFinishThreads / 2; h > 0; h >>= 1) {
        if (static_cast<int>(threadIdx.x) < h) {
            sr[threadIdx.x] += sr[threadIdx.x + h];
            si[threadIdx.x] += si[threadIdx.x + h];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) *alpha = Zd{sr[0], si[0]};
}

// Block-interleaved vectors X[row * NV + k] on the SELL layout: LR lanes share a row, each holding 16
// bytes of its vectors (one complex or two real) in the single-vector kernel's ACC partial sums and
// tree, so the same bits as single applies. What bounds a gather is the vector cache's one line a
// clock among adjacent lanes, so lanes side by side read the two to eight pieces of one row of X
// rather than each lane all pieces of its own row; the row's entries are read by its lanes from the
// same addresses. us a launch, each lane all pieces / so: 1.43 million rows, 4 complex 367 / 335 (19
// million L2 misses at 7.2 TB/s of 128-byte lines); 400,023 rows, complex 2, 4, 8: 37 / 36, 57 / 53,
// 118 / 79; 2.7 million, real 8: 293 / 245. (4 complex at 1.43 million rows:
// eight entries a round 352, the next group's entries prefetched 357, a row's sums on twice the lanes
// 373: more registers or rows further apart in flight.)
struct alignas(8) Two {
    double a, b;
};

template <int WIDTH, bool VREAL, bool REAL, bool LD, int LR, int ACC>
__global__ __launch_bounds__(1024) void k_sell_block(CsrView A, const Two* X, Two* Y) {
    const Dict<LD> d = stage_dict<WIDTH, VREAL, LD>(A);
    const i64 gid = row_block(A) * blockDim.x + threadIdx.x;
    const i64 row = gid / LR;
    const u32 lane = static_cast<u32>(gid % LR);
    if (row >= A.rows) return;
    const u32 n = A.nt ? __builtin_nontemporal_load(A.sell_len + row) : A.sell_len[row];
    const u64 first = A.sell_ptr[row >> 6] + static_cast<u64>(row & 63) * 4;
    double s0[ACC], s1[ACC];
#pragma unroll
    for (int j = 0; j < ACC; ++j) s0[j] = s1[j] = 0.0;
    auto accumulate = [&](int j, const Two& x, double vr, double vi) {
        if constexpr (REAL) {
            s0[j] += vr * x.a;
            s1[j] += vr * x.b;
        } else {
            s0[j] += vr * x.a - vi * x.b;
            s1[j] += vr * x.b + vi * x.a;
        }
    };
    u32 k = 0;
    for (; k + 4 <= n; k += 4) {
        u32 c[4];
        double vr[4], vi[4] = {0.0, 0.0, 0.0, 0.0};
        Two x[4];
        load_quad<WIDTH, VREAL, LD>(A, d, first + static_cast<u64>(k / 4) * 256, c, vr, vi);
#pragma unroll
        for (int u = 0; u < 4; ++u) x[u] = X[static_cast<u64>(c[u]) * LR + lane];
#pragma unroll
        for (int u = 0; u < 4; ++u) accumulate(u % ACC, x[u], vr[u], vi[u]);
    }
    if (k < n) {   // the last group, entries below n
        u32 c[4];
        double vr[4], vi[4] = {0.0, 0.0, 0.0, 0.0};
        load_quad<WIDTH, VREAL, LD>(A, d, first + static_cast<u64>(k / 4) * 256, c, vr, vi);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (k + static_cast<u32>(u) < n) accumulate(u % ACC, X[static_cast<u64>(c[u]) * LR + lane], vr[u], vi[u]);
    }
    Y[static_cast<u64>(row) * LR + lane] = Two{tree<ACC>(s0), tree<ACC>(s1)};
}

// The same for 2 and 4 real vectors: ACC lanes share a row, lane l taking entries l, l + ACC, ..., their
// sums combined by the xor butterfly in the tree's order. With 16 or 32 bytes a row of X, fewer rows in
// flight weigh more than the cache's lines where a sector's columns scatter (1.43 million rows of a
// momentum sector, 2 and 4 vectors: 103 and 143 us, one lane or two per row 113 and 150; 400,023 rows,
// 4 vectors: 36 and 37), though not without a lattice symmetry (705,432 rows: 31 and 41, there 24 and 35).
template <int WIDTH, bool LD, int NV, int ACC>
__global__ __launch_bounds__(256) void k_sell_block_rows(CsrView A, const double* X, double* Y) {
    const Dict<LD> d = stage_dict<WIDTH, true, LD>(A);
    const i64 gid = row_block(A) * blockDim.x + threadIdx.x;
    const i64 row = gid / ACC;
    const int lane = static_cast<int>(gid % ACC);
    double ar[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q) ar[q] = 0.0;
    if (row < A.rows) {
        const u32 n = A.sell_len[row];
        const u64 slice = A.sell_ptr[row >> 6];
        const u32 j = static_cast<u32>(row & 63);
        for (u32 k = static_cast<u32>(lane); k < n; k += ACC) {
            u32 c32;
            double vr, vi = 0.0;
            load_entry<WIDTH, true, LD>(A, d, sell_at(slice, j, k), c32, vr, vi);
            const double* x = X + static_cast<u64>(c32) * NV;
#pragma unroll
            for (int q = 0; q < NV; ++q) ar[q] += vr * x[q];
        }
    }
#pragma unroll
    for (int off = ACC / 2; off > 0; off >>= 1) {
#pragma unroll
        for (int q = 0; q < NV; ++q) ar[q] += __shfl_xor(ar[q], off, ACC);
    }
    if (row < A.rows && lane == 0) {
#pragma unroll
        for (int q = 0; q < NV; ++q) Y[row * NV + q] = ar[q];
    }
}

/// Launch with the dictionary in LDS when it fits there (dict_in_lds), else from global memory: tag
/// is std::true_type / std::false_type, lds the dynamic LDS bytes.
template <int WIDTH, class F> void by_dict(const CsrView& A, F&& f) {
    if constexpr (WIDTH == 0) {
        f(std::false_type{}, std::size_t{0});
    } else {
        if (dict_in_lds(A)) f(std::true_type{}, dict_lds_bytes(A));
        else f(std::false_type{}, std::size_t{0});
    }
}

/// The vectors of the set in launches of 8, 4, 2 and 1: go(std::integral_constant<int, NV>, Ptrs<NV>).
template <class F> void by_vectors(const VecSet& v, F&& go) {
    int done = 0;
    auto next = [&](auto tag) {
        constexpr int NV = decltype(tag)::value;
        Ptrs<NV> p;
        for (int k = 0; k < NV; ++k) {
            p.in[k] = v.in[done + k];
            p.out[k] = v.out[done + k];
        }
        go(tag, p);
        done += NV;
    };
    while (done < v.k) {
        const int rest = v.k - done;
        if (rest >= 8) next(std::integral_constant<int, 8>{});
        else if (rest >= 4) next(std::integral_constant<int, 4>{});
        else if (rest >= 2) next(std::integral_constant<int, 2>{});
        else next(std::integral_constant<int, 1>{});
    }
}

template <int WIDTH, bool VREAL, bool REAL> void launch_sell_set(const CsrView& V, const VecSet& v, hipStream_t st) {
    const CsrView A = staged(V, 1, v.k);
    const dim3 grid(grid_blocks(A, static_cast<u64>(A.rows))), block(block_threads(A));
    by_dict<WIDTH>(A, [&](auto in_lds, std::size_t lds) {
        constexpr bool LD = decltype(in_lds)::value;
        by_vectors(v, [&](auto tag, const auto& p) {
            constexpr int NV = decltype(tag)::value;
#define QSA_SELL(U, ACC) hipLaunchKernelGGL((k_sell<WIDTH, VREAL, REAL, LD, NV, U, ACC>), grid, block, lds, st, A, p)
            if (A.sell_acc == 4) {
                if (NV == 1 && A.unroll >= 16) QSA_SELL((NV == 1 ? 16 : 4), 4);
                else if (NV == 1 && A.unroll >= 8) QSA_SELL((NV == 1 ? 8 : 4), 4);
                else QSA_SELL(4, 4);
            } else {
                if (NV == 1 && A.unroll >= 16) QSA_SELL((NV == 1 ? 16 : 4), 1);
                else if (NV == 1 && A.unroll >= 8) QSA_SELL((NV == 1 ? 8 : 4), 1);
                else QSA_SELL(4, 1);
            }
#undef QSA_SELL
        });
    });
}

/// The block kernels' workgroup and whether a dictionary of u16 ids is staged (one of u8 ids always is).
/// A row's entries are looked up once for all its vectors, so the more vectors the less a copy in LDS
/// saves. On the SELL layout complex vectors stage it, in workgroups of 1024 where it is over 2 KB
/// (4 of 1.43 million rows: 399 us from global memory, 367 so); on the CSR layout 2 vectors do, in
/// workgroups of 256 (32,065 rows: 6.2 and 5.4 us), while 8 in 1024 threads took 16.1 against 9.4 us
/// on 9225 rows and 73 against 58 on 112,640. Of those that stage it, a launch with too few lookups for
/// its copy does not (staged).
inline CsrView block_view(const CsrView& A, bool stage_u16, bool large, unsigned lanes, int nv) {
    CsrView B = A;
    if (A.dict_n > 256 && !stage_u16) B.lds_dict = 0;
    B.wg = large && dict_in_lds(B) && dict_lds_bytes(A) > 2048 ? 1024 : 256;
    B = staged(B, lanes, nv);
    if (!dict_in_lds(B)) B.wg = 256;
    return B;
}

template <int WIDTH, bool VREAL, bool REAL, int ACC>
void launch_sell_block_acc(const CsrView& A, int nv, const void* X, void* Y, hipStream_t st) {
    if constexpr (REAL) {
        if (nv <= 4) {
            const CsrView B = block_view(A, false, false, ACC, nv);
            const dim3 grid(grid_blocks(B, static_cast<u64>(A.rows) * ACC)), block(block_threads(B));
            by_dict<WIDTH>(B, [&](auto in_lds, std::size_t lds) {
                constexpr bool LD = decltype(in_lds)::value;
                const double* x = static_cast<const double*>(X);
                double* y = static_cast<double*>(Y);
                if (nv == 2) hipLaunchKernelGGL((k_sell_block_rows<WIDTH, LD, 2, ACC>), grid, block, lds, st, B, x, y);
                else hipLaunchKernelGGL((k_sell_block_rows<WIDTH, LD, 4, ACC>), grid, block, lds, st, B, x, y);
            });
            return;
        }
    }
    const int lanes = REAL ? nv / 2 : nv;   // 16 bytes each
    const CsrView B = block_view(A, true, true, static_cast<unsigned>(lanes), nv);
    const dim3 grid(grid_blocks(B, static_cast<u64>(A.rows) * static_cast<u64>(lanes))), block(block_threads(B));
    by_dict<WIDTH>(B, [&](auto in_lds, std::size_t lds) {
        constexpr bool LD = decltype(in_lds)::value;
#define QSA_SELL_BLOCK(LR)                                                                                     \
    hipLaunchKernelGGL((k_sell_block<WIDTH, VREAL, REAL, LD, LR, ACC>), grid, block, lds, st, B,               \
                       static_cast<const Two*>(X), static_cast<Two*>(Y))
        switch (lanes) {
        case 2:
            if constexpr (!REAL) QSA_SELL_BLOCK(2);
            break;
        case 4: QSA_SELL_BLOCK(4); break;
        case 8:
            if constexpr (!REAL) QSA_SELL_BLOCK(8);
            break;
        default: break;
        }
#undef QSA_SELL_BLOCK
    });
}
template <int WIDTH, bool VREAL, bool REAL>
void launch_sell_block(const CsrView& A, int nv, const void* X, void* Y, hipStream_t st) {
    if (nv == 1) {   // one vector: the single apply
        VecSet v;
        v.k = 1;
        v.in[0] = X;
        v.out[0] = Y;
        launch_sell_set<WIDTH, VREAL, REAL>(A, v, st);
    } else if (A.sell_acc == 4) launch_sell_block_acc<WIDTH, VREAL, REAL, 4>(A, nv, X, Y, st);
    else launch_sell_block_acc<WIDTH, VREAL, REAL, 1>(A, nv, X, Y, st);
}

template <int WIDTH, bool VREAL, bool REAL, int L> void launch_set(const CsrView& V, const VecSet& v, hipStream_t st) {
    const CsrView A = staged(V, L, v.k);
    const dim3 grid(grid_blocks(A, static_cast<u64>(A.rows) * L)), block(block_threads(A));
    by_dict<WIDTH>(A, [&](auto in_lds, std::size_t lds) {
        constexpr bool LD = decltype(in_lds)::value;
        by_vectors(v, [&](auto tag, const auto& p) {
            constexpr int NV = decltype(tag)::value;
#define QSA_SPMV(U) hipLaunchKernelGGL((k_spmv<WIDTH, VREAL, REAL, LD, L, NV, U>), grid, block, lds, st, A, p)
            if (NV == 1 && A.unroll >= 8) QSA_SPMV((NV == 1 ? 8 : 1));
            else if (NV == 1 && A.unroll >= 4) QSA_SPMV((NV == 1 ? 4 : 1));
            else if (NV == 1 && A.unroll > 1) QSA_SPMV((NV == 1 ? 2 : 1));
            else QSA_SPMV(1);
#undef QSA_SPMV
        });
    });
}

template <int WIDTH, bool VREAL, bool REAL> void pick_lanes(const CsrView& A, const VecSet& v, hipStream_t st) {
    switch (A.lanes) {
    case 4: launch_set<WIDTH, VREAL, REAL, 4>(A, v, st); break;
    case 8: launch_set<WIDTH, VREAL, REAL, 8>(A, v, st); break;
    case 32: launch_set<WIDTH, VREAL, REAL, 32>(A, v, st); break;
    case 64: launch_set<WIDTH, VREAL, REAL, 64>(A, v, st); break;
    default: launch_set<WIDTH, VREAL, REAL, 16>(A, v, st); break;
    }
}

template <int WIDTH, bool VREAL, bool REAL, int L>
void launch_block(const CsrView& A, int nv, const void* X, void* Y, hipStream_t st) {
    const CsrView B = block_view(A, nv <= 2 && dict_lds_bytes(A) <= 16 * 1024, false, L, nv);
    const dim3 grid(grid_blocks(B, static_cast<u64>(A.rows) * L)), block(block_threads(B));
    by_dict<WIDTH>(B, [&](auto in_lds, std::size_t lds) {
        constexpr bool LD = decltype(in_lds)::value;
#define QSA_SPMV_BLOCK(NV) hipLaunchKernelGGL((k_spmv_block<WIDTH, VREAL, REAL, LD, L, NV>), grid, block, lds, st, B, X, Y)
        switch (nv) {
        case 1: QSA_SPMV_BLOCK(1); break;
        case 2: QSA_SPMV_BLOCK(2); break;
        case 4: QSA_SPMV_BLOCK(4); break;
        case 8: QSA_SPMV_BLOCK(8); break;
        default: break;
        }
#undef QSA_SPMV_BLOCK
    });
}

template <int WIDTH, bool VREAL, bool REAL> void pick_lanes_block(const CsrView& A, int nv, const void* X, void* Y, hipStream_t st) {
    switch (A.lanes) {
    case 4: launch_block<WIDTH, VREAL, REAL, 4>(A, nv, X, Y, st); break;
    case 8: launch_block<WIDTH, VREAL, REAL, 8>(A, nv, X, Y, st); break;
    case 32: launch_block<WIDTH, VREAL, REAL, 32>(A, nv, X, Y, st); break;
    case 64: launch_block<WIDTH, VREAL, REAL, 64>(A, nv, X, Y, st); break;
    default: launch_block<WIDTH, VREAL, REAL, 16>(A, nv, X, Y, st); break;
    }
}

template <bool BLOCK>
void dispatch(const CsrView& A, bool vreal, bool real, const VecSet* v, int nv, const void* X, void* Y, hipStream_t st) {
    // real vectors need real values; complex vectors take either
    auto go = [&](auto w, auto vr, auto xr) {
        constexpr int W = decltype(w)::value;
        constexpr bool VR = decltype(vr)::value, XR = decltype(xr)::value;
        if (A.sell_ptr) {
            if constexpr (BLOCK) launch_sell_block<W, VR, XR>(A, nv, X, Y, st);
            else launch_sell_set<W, VR, XR>(A, *v, st);
        } else {
            if constexpr (BLOCK) pick_lanes_block<W, VR, XR>(A, nv, X, Y, st);
            else pick_lanes<W, VR, XR>(A, *v, st);
        }
    };
    using T = std::true_type;
    using F = std::false_type;
    auto by_width = [&](auto vr, auto xr) {
        if (A.width == 1) go(std::integral_constant<int, 1>{}, vr, xr);
        else if (A.width == 2) go(std::integral_constant<int, 2>{}, vr, xr);
        else if (A.width == 3) go(std::integral_constant<int, 3>{}, vr, xr);
        else go(std::integral_constant<int, 0>{}, vr, xr);
    };
    if (real) by_width(T{}, T{});
    else if (vreal) by_width(T{}, F{});
    else by_width(F{}, F{});
}

__global__ void k_pack_col_ids(u32* col, const u8* id, u64 nnz) {
    for (u64 e = blockIdx.x * static_cast<u64>(blockDim.x) + threadIdx.x; e < nnz; e += static_cast<u64>(gridDim.x) * blockDim.x)
        col[e] |= static_cast<u32>(id[e]) << 24;
}

// One thread per row; a wavefront is one slice (the grid's blocks are multiples of 64 threads).
__global__ __launch_bounds__(256) void k_sell_lengths(const u64* row_ptr, i64 rows, u16* sell_len, u64* slice_words,
                                                      u32* too_long) {
    const i64 r = static_cast<i64>(blockIdx.x) * blockDim.x + threadIdx.x;
    u32 n = 0;
    if (r < rows) {
        const u64 len = row_ptr[r + 1] - row_ptr[r];
        if (len > 0xFFFFu) atomicOr(too_long, 1u);
        n = len > 0xFFFFu ? 0xFFFFu : static_cast<u32>(len);
        sell_len[r] = static_cast<u16>(n);
    }
    u32 m = n;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const u32 o = static_cast<u32>(__shfl_xor(static_cast<int>(m), off, 64));
        m = o > m ? o : m;
    }
    if ((threadIdx.x & 63) == 0 && r < rows) slice_words[r >> 6] = static_cast<u64>((m + 3u) & ~3u) * 64;
}

// diag_first (a square operator): a row's diagonal entry, when it has one, moves to its first slot,
// the others keeping their order -- the k = 0 loads of a wavefront then read x[row] for 64
// consecutive rows, one coalesced line instead of 64 gathers.
// A lane gathers four entries of its row and writes the group whole, zeros past the row's end: a
// wavefront's stores are 1 KB of consecutive words (716,000 rows, 20.7 million entries: 626 us an entry at a time
// into cleared memory, 182 so). What the slice holds past a row's last group is never read.
template <class T, int V> struct alignas(sizeof(T) * V) Group {
    T v[V];
};

template <class T, class G>
__device__ __forceinline__ void sell_group(const void* vals, void* sell_vals, u64 dst, const G& source) {
    constexpr int V = sizeof(T) >= 8 ? 16 / sizeof(T) : 4;   // 16 bytes a store at most
#pragma unroll
    for (int h = 0; h < 4 / V; ++h) {
        Group<T, V> w;
#pragma unroll
        for (int u = 0; u < V; ++u) {
            const u64 from = source(h * V + u);
            w.v[u] = from == ~u64{0} ? T{} : static_cast<const T*>(vals)[from];
        }
        *reinterpret_cast<Group<T, V>*>(static_cast<T*>(sell_vals) + dst + h * V) = w;
    }
}

__global__ __launch_bounds__(256) void k_sell_fill(const u64* row_ptr, const u32* col, const void* vals, int vb,
                                                   i64 rows, const u64* sell_ptr, u32* sell_col, void* sell_vals,
                                                   int diag_first, int packed) {
    const i64 r = static_cast<i64>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (r >= rows) return;
    const u64 e0 = row_ptr[r], n = row_ptr[r + 1] - e0;
    const u64 slice = sell_ptr[r >> 6];
    const u32 j = static_cast<u32>(r & 63);
    u64 diag = n;   // the diagonal entry's position in the row (n: none)
    if (diag_first)
        for (u64 k = 0; k < n && diag == n; ++k)
            if ((packed ? (col[e0 + k] & 0xFFFFFFu) : col[e0 + k]) == static_cast<u32>(r)) diag = k;
    for (u64 k0 = 0; k0 < n; k0 += 4) {
        // slot k takes the diagonal first, then the row's other entries in order
        auto source = [&](int u) -> u64 {
            const u64 k = k0 + static_cast<u64>(u);
            if (k >= n) return ~u64{0};
            return e0 + (diag == n ? k : (k == 0 ? diag : (k <= diag ? k - 1 : k)));
        };
        const u64 dst = sell_at(slice, j, static_cast<u32>(k0));
        sell_group<u32>(col, sell_col, dst, source);
        if (vb == 1) sell_group<u8>(vals, sell_vals, dst, source);
        else if (vb == 2) sell_group<u16>(vals, sell_vals, dst, source);
        else if (vb == 8) sell_group<double>(vals, sell_vals, dst, source);
        else if (vb == 16) sell_group<Zd>(vals, sell_vals, dst, source);
    }
}

}  // namespace

void sell_lengths(const u64* row_ptr, i64 rows, u16* sell_len, u64* slice_words, u32* too_long, hipStream_t st) {
    if (rows <= 0) return;
    const u64 g = (static_cast<u64>(rows) + 255) / 256;
    hipLaunchKernelGGL(k_sell_lengths, dim3(static_cast<unsigned>(g)), dim3(256), 0, st, row_ptr, rows, sell_len,
                       slice_words, too_long);
}

std::size_t sell_scan_temp_bytes(i64 n_slices) {
    std::size_t bytes = 0;
    (void)hipcub::DeviceScan::ExclusiveSum(nullptr, bytes, static_cast<const u64*>(nullptr), static_cast<u64*>(nullptr),
                                           static_cast<int>(n_slices + 1));
    return bytes;
}

hipError_t sell_scan(const u64* slice_words, i64 n_slices, u64* sell_ptr, void* temp, std::size_t temp_bytes,
                     hipStream_t st) {
    if (n_slices < 0 || n_slices >= (i64{1} << 31) - 1) return hipErrorInvalidValue;   // (counted in 32 bits)
    return hipcub::DeviceScan::ExclusiveSum(temp, temp_bytes, slice_words, sell_ptr, static_cast<int>(n_slices + 1), st);
}

void sell_fill(const u64* row_ptr, const u32* col, const void* vals, int value_bytes, i64 rows, const u64* sell_ptr,
               u32* sell_col, void* sell_vals, bool diag_first, bool packed, hipStream_t st) {
    if (rows <= 0) return;
    const u64 g = (static_cast<u64>(rows) + 255) / 256;
    hipLaunchKernelGGL(k_sell_fill, dim3(static_cast<unsigned>(g)), dim3(256), 0, st, row_ptr, col, vals, value_bytes,
                       rows, sell_ptr, sell_col, sell_vals, diag_first ? 1 : 0, packed ? 1 : 0);
}

void pack_col_ids(u32* col, const u8* id, u64 nnz, hipStream_t st) {
    if (!nnz) return;
    u64 g = (nnz + 255) / 256;
    if (g > 65536) g = 65536;
    hipLaunchKernelGGL(k_pack_col_ids, dim3(static_cast<unsigned>(g)), dim3(256), 0, st, col, id, nnz);
}

void csr_spmv(const CsrView& A, bool real, const VecSet& v, hipStream_t st) {
    if (A.rows == 0 || v.k == 0) return;
    dispatch<false>(A, A.values_real, real, &v, 0, nullptr, nullptr, st);
}

void csr_spmv_block(const CsrView& A, bool real, int nv, const void* X, void* Y, hipStream_t st) {
    if (A.rows == 0) return;
    dispatch<true>(A, A.values_real, real, nullptr, nv, X, Y, st);
}

bool spmv_workgroup_fixed(const CsrView& A) {
    const CsrView B = staged(A, A.sell_ptr ? 1u : static_cast<unsigned>(A.lanes), 1);
    return dict_in_lds(B) && dict_lds_bytes(B) > 16 * 1024;
}

unsigned sell_lanczos_parts(const CsrView& A) { return static_cast<unsigned>((A.rows + kLanczosPart - 1) / kLanczosPart); }

bool sell_lanczos(const CsrView& V, bool real, const void* v, const void* vprev, const double* beta, void* w,
                  double* partial, Zd* alpha, hipStream_t st) {
    if (!V.sell_ptr || V.rows == 0 || (real && !V.values_real)) return false;
    const CsrView A = staged(V, 1, 1);
    const dim3 grid(grid_blocks(A, static_cast<u64>(A.rows))), block(block_threads(A));
    Ptrs<1> p;
    p.in[0] = v;
    p.out[0] = w;
    auto go = [&](auto wd, auto vr, auto xr) {
        constexpr int W = decltype(wd)::value;
        constexpr bool VR = decltype(vr)::value, XR = decltype(xr)::value;
        by_dict<W>(A, [&](auto in_lds, std::size_t lds) {
            constexpr bool LD = decltype(in_lds)::value;
#define QSA_SELL_LANCZOS(U, ACC) \
    hipLaunchKernelGGL((k_sell_lanczos<W, VR, XR, LD, U, ACC>), grid, block, lds, st, A, p, vprev, beta, partial)
            if (A.sell_acc == 4) {
                if (A.unroll >= 16) QSA_SELL_LANCZOS(16, 4);
                else if (A.unroll >= 8) QSA_SELL_LANCZOS(8, 4);
                else QSA_SELL_LANCZOS(4, 4);
            } else {
                if (A.unroll >= 16) QSA_SELL_LANCZOS(16, 1);
                else if (A.unroll >= 8) QSA_SELL_LANCZOS(8, 1);
                else QSA_SELL_LANCZOS(4, 1);
            }
#undef QSA_SELL_LANCZOS
        });
    };
    using T = std::true_type;
    using F = std::false_type;
    auto by_width = [&](auto vr, auto xr) {
        if (A.width == 1) go(std::integral_constant<int, 1>{}, vr, xr);
        else if (A.width == 2) go(std::integral_constant<int, 2>{}, vr, xr);
        else if (A.width == 3) go(std::integral_constant<int, 3>{}, vr, xr);
        else go(std::integral_constant<int, 0>{}, vr, xr);
    };
    if (real) by_width(T{}, T{});
    else if (A.values_real) by_width(T{}, F{});
    else by_width(F{}, F{});
    hipLaunchKernelGGL(k_lanczos_finish, dim3(1), dim3(kFinishThreads), 0, st, partial, static_cast<int>(sell_lanczos_parts(A)), alpha);
    return true;
}

}  // namespace qsa::dev
