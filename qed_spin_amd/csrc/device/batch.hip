// The batched Krylov engine: many symmetry blocks of uneven dimension and R vectors per block
// advance one Lanczos step together.
//
// Layout: the blocks' CSRs are packed into one block-diagonal CSR (rows and columns offset by the
// block's first row; values as 16-bit ids into the blocks' dictionaries laid end to end when every
// block has one and they hold at most 65536 values together, else in full); a batch vector holds R
// entries per row, X[row R + s], so the R vectors of a row are one contiguous line. Rows are cut into
// tiles of at most kBatchTileRows rows of one block, one workgroup per tile (256 threads; the SpMV of
// R > 1 has 512).
//
// Vector kernels: thread t of a tile is (slot t / R, vector t % R); the 256 / R slots take the
// tile's rows in turn, so consecutive threads touch consecutive entries whatever R is. A
// per-(block, vector) reduction is each thread's sum over its rows, then the slots' sums in slot
// order (LDS), then the block's tile sums by a fixed tree: deterministic, and independent of which
// other blocks share the batch.
//
// SpMV: for R > 1 a group of 2, 4 or 8 threads per row, one vector each, that share the row's columns
// and value ids; above 8 vectors a work item is a tile and a run of eight of its vectors. For R = 1
// one thread per row of a slice layout (OneView); without room for that, the kernel of R > 1.
//
// The order of a block's rows is the engine's own: blocks whose vectors (eight of them at most) do not
// fit an XCD's L2 are stored by breadth-first level of their matrix's graph, the blocks' states'
// order within a level. A row's columns then lie in its own and the two neighbouring levels, so with
// the tiles of a block run in order on one XCD each entry of X comes from memory once.
//
// The Lanczos scalars alpha, beta, the local-reorthogonalisation overlap, the active flags and the
// step counter live on the device; a step needs no host synchronisation, so it is captured once
// as a hipGraph and replayed.
#include <hipcub/hipcub.hpp>

#include "dev_common.h"
#include "launch.h"

namespace qsa::dev {

namespace {

constexpr int kThreads = 256;

typedef u32 u32x4 __attribute__((ext_vector_type(4)));
typedef u16 u16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ Zd cmul(Zd a, Zd b) { return Zd{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ Zd cdot(Zd a, Zd b) { return Zd{a.re * b.re + a.im * b.im, a.re * b.im - a.im * b.re}; }

/// The SpMV work of a workgroup: a tile and a run of at most eight vectors (`chunk`), by the schedule's
/// entry (tile * chunks + chunk, ~0: none) or, without one, in order. An item's work and partial sums
/// are the same whichever workgroup runs it.
struct Work {
    u32 tile;
    int chunk;
    bool any;
};
__device__ __forceinline__ Work work_item(const BatchView& B, int chunks) {
    const u32 id = B.sched ? B.sched[blockIdx.x] : blockIdx.x;
    if (id == ~0u) return Work{0, 0, false};
    if (chunks == 1) return Work{id, 0, true};
    return Work{id / static_cast<u32>(chunks), static_cast<int>(id % static_cast<u32>(chunks)), true};
}

__device__ __forceinline__ bool pair_live(const BatchView& B, u32 block, int s) {
    return !B.active || B.active[static_cast<u64>(block) * B.R + s] != 0;
}

__device__ __forceinline__ Zd entry_value(const BatchView& B, u64 e) {
    if (B.vid) {
        const u32 id = B.vid[e];
        return Zd{B.dict_re[id], B.dict_im[id]};
    }
    return B.val[e];
}

/// A stored entry times its pair's factor.
__device__ __forceinline__ Zd scaled(Zd v, double f) { return Zd{v.re * f, v.im * f}; }

// R > 1: a row's group of RP = 2, 4 or 8 lanes, lane s holding vector s of the item's run. The lanes
// load the row's columns and value ids together, eight entries a round (each pair or quad of lanes
// reads consecutive entries once), and pass them on by DPP; every lane then gathers its vector's entry,
// a group's lanes one contiguous line, eight gathers in flight. The block's dictionary is in LDS. Each
// lane keeps two partial sums.
//
// What bounds it: with every lane of a row reading every column, id, and both halves of the value from
// global memory, the vector cache's address rate (one line per clock for lanes that do not share one
// with a neighbour); so it took 2.83 ms a step at N = 24, R = 4 (9.07M rows, 2.2e8 entries), and
// 1.68 ms (the first recurrence pass included) with the group's lanes sharing their loads and the L2
// missing on 77M lines a step: X fetched again and again, 870 bytes a row of 64. In level order the
// misses are 27M (what the matrix and the vectors are) and the step 1.59 ms: the L1 fetches, a line
// for almost every entry at 2.5 clocks, are left. At R = 40 a row's 640 bytes times the rows of the
// tiles in flight fit an L2 in no order, hence the runs of eight vectors (a line): N = 22 (2.29M rows)
// 3.54 -> 1.99 ms a step, 6.6 GB of memory traffic at 3.3 TB/s.
constexpr int kBatchDictMax = 1024;   // LDS dictionary entries of a tile's block (16 KB)

/// The value of lane J of the caller's pair (Q = 2) or quad (Q = 4) of lanes.
template <int Q, int J> __device__ __forceinline__ u32 group_lane(u32 v) {
    constexpr int ctrl = Q == 2 ? (J == 0 ? 0xA0 : 0xF5) : J * 0x55;   // quad_perm
    return static_cast<u32>(__builtin_amdgcn_mov_dpp(static_cast<int>(v), ctrl, 0xF, 0xF, true));
}
template <int Q, int J> __device__ __forceinline__ double group_lane(double v) {
    const u64 b = static_cast<u64>(__double_as_longlong(v));
    const u64 lo = group_lane<Q, J>(static_cast<u32>(b)), hi = group_lane<Q, J>(static_cast<u32>(b >> 32));
    return __longlong_as_double(static_cast<long long>(lo | (hi << 32)));
}

/// The dictionary of the tile's block into LDS, a zero after its last value (every thread of the
/// workgroup calls it; the caller synchronises): the block's first id, and the zero's.
struct BlockDict {
    u32 first, zero;
};
__device__ __forceinline__ BlockDict stage_block_dict(const BatchView& B, u32 block, Zd* dict) {
    const u32 d0 = B.dict_begin[block], n = B.dict_begin[block + 1] - d0;
    for (u32 i = threadIdx.x; i < n; i += blockDim.x) dict[i] = Zd{B.dict_re[d0 + i], B.dict_im[d0 + i]};
    if (threadIdx.x == 0) dict[n] = Zd{0.0, 0.0};
    return BlockDict{d0, n};
}

extern __shared__ __align__(16) Zd batch_dict[];

// Entry e of one block's own CSR: its column, its dictionary id (width 1 / 2 / 3), its value.
__device__ __forceinline__ u32 entry_column(const CsrView& A, u64 e) {
    const u32 w = A.col[e];
    return A.width == 3 ? (w & 0xFFFFFFu) : w;
}
__device__ __forceinline__ u32 entry_id(const CsrView& A, u64 e) {
    if (A.width == 3) return A.col[e] >> 24;
    return A.width == 1 ? static_cast<u32>(static_cast<const u8*>(A.vals)[e])
                        : static_cast<u32>(static_cast<const u16*>(A.vals)[e]);
}
__device__ __forceinline__ Zd csr_value(const CsrView& A, u64 e) {
    if (A.width != 0) {
        const u32 id = entry_id(A, e);
        return Zd{A.dict_re[id], A.values_real ? 0.0 : A.dict_im[id]};
    }
    if (A.values_real) return Zd{static_cast<const double*>(A.vals)[e], 0.0};
    return static_cast<const Zd*>(A.vals)[e];
}

// ar + i ai += v x, by fused multiply-adds.
__device__ __forceinline__ void zfma(Zd v, Zd x, double& ar, double& ai) {
    ar = __builtin_fma(v.re, x.re, ar);
    ai = __builtin_fma(v.re, x.im, ai);
    ar = __builtin_fma(-v.im, x.im, ar);
    ai = __builtin_fma(v.im, x.re, ai);
}

/// Four entries of the caller's row: their columns and value ids (values), one to each lane of a quad
/// (RP = 2: two to each lane of a pair). Past the row's end, its last entry with value zero.
template <int RP, bool LD> struct Quad {
    static constexpr int Q = RP == 2 ? 2 : 4, NL = 4 / Q;
    u32 c[NL], id[NL];
    Zd v[NL];
    __device__ __forceinline__ void load(const BatchView& B, u64 first, u32 d0, u32 zero, u32 e, u32 b1) {
        const u32 p = threadIdx.x & (Q - 1);
#pragma unroll
        for (int q = 0; q < NL; ++q) {
            const u32 k = e + static_cast<u32>(q * Q) + p;
            const u64 at = first + (k < b1 ? k : b1 - 1);
            c[q] = B.col[at];
            if constexpr (LD) {
                const u32 i = B.vid[at] - d0;
                id[q] = k < b1 ? i : zero;
            } else {
                const Zd w = entry_value(B, at);
                v[q] = k < b1 ? w : Zd{0.0, 0.0};
            }
        }
    }
    template <int J> __device__ __forceinline__ Zd gather(const char* X, u32 stride) const {
        return *reinterpret_cast<const Zd*>(X + static_cast<u64>(group_lane<Q, J % Q>(c[J / Q])) * stride);
    }
    template <int J> __device__ __forceinline__ Zd value() const {
        if constexpr (LD) return batch_dict[group_lane<Q, J % Q>(id[J / Q])];
        else return Zd{group_lane<Q, J % Q>(v[J / Q].re), group_lane<Q, J % Q>(v[J / Q].im)};
    }
};

/// One row of the SpMV for the caller's vector: entries [b0, b1) past `first`; X at the vector's first
/// entry, `stride` bytes between rows, `zero` the dictionary's zero. Eight gathers in flight, the next
/// eight entries' columns and ids loaded behind them. Two partial sums (entries 0 to 3 and 4 to 7 of
/// each round).
template <int RP, bool LD>
__device__ __forceinline__ Zd group_row(const BatchView& B, const char* X, u32 stride, u64 first, u32 d0, u32 zero, u32 b0,
                                        u32 b1) {
    double ar = 0.0, ai = 0.0, br = 0.0, bi = 0.0;
    if (b0 >= b1) return Zd{0.0, 0.0};   // one answer, and one trip count below, for all lanes of the row
    Quad<RP, LD> lo, hi;
    lo.load(B, first, d0, zero, b0, b1);
    hi.load(B, first, d0, zero, b0 + 4, b1);
    for (u32 e = b0;;) {
        const Zd x0 = lo.template gather<0>(X, stride), x1 = lo.template gather<1>(X, stride),
                 x2 = lo.template gather<2>(X, stride), x3 = lo.template gather<3>(X, stride);
        Zd x4{0.0, 0.0}, x5{0.0, 0.0}, x6{0.0, 0.0}, x7{0.0, 0.0};
        const Quad<RP, LD> a = lo, b = hi;
        if (e + 4 < b1) {
            x4 = b.template gather<0>(X, stride);
            x5 = b.template gather<1>(X, stride);
            x6 = b.template gather<2>(X, stride);
            x7 = b.template gather<3>(X, stride);
        }
        e += 8;
        const bool more = e < b1;
        if (more) {
            lo.load(B, first, d0, zero, e, b1);
            hi.load(B, first, d0, zero, e + 4, b1);
        }
        zfma(a.template value<0>(), x0, ar, ai);
        zfma(a.template value<1>(), x1, ar, ai);
        zfma(a.template value<2>(), x2, ar, ai);
        zfma(a.template value<3>(), x3, ar, ai);
        zfma(b.template value<0>(), x4, br, bi);
        zfma(b.template value<1>(), x5, br, bi);
        zfma(b.template value<2>(), x6, br, bi);
        zfma(b.template value<3>(), x7, br, bi);
        if (!more) break;
    }
    return Zd{ar + br, ai + bi};
}

/// Threads of the grouped SpMV: more rows per pass in fewer workgroups keep the rows in flight on an XCD
/// (resident workgroups times a tile) close together.
constexpr int kGroupThreads = 512;

/// Y = A X, or (FUSED) the first recurrence pass with it: W = H V_cur - beta V_prev (beta of this step;
/// skipped at step 0) and the partial of <V_cur, W> (a group's lanes' rows in order, the wave's groups
/// by an xor tree, then the waves in order).
///
/// With sprev / scur the stored vectors are the unnormalised ones and V = U f with the pair's factor
/// f (1 / beta of the step that made it), applied to the row's sum and to V_prev: no separate scaling
/// pass over the vectors.
template <int RP, bool LD, bool FUSED>
__global__ __launch_bounds__(kGroupThreads) void k_batch_spmv_group(BatchView B, int chunks, const Zd* Vprev,
                                                                    const Zd* X, Zd* Y, const double* beta,
                                                                    double* partial, const double* sprev,
                                                                    const double* scur) {
    __shared__ u32 rp[kBatchTileRows + 1];
    __shared__ double sr[FUSED ? kGroupThreads / 64 * RP : 1], si[FUSED ? kGroupThreads / 64 * RP : 1];
    const Work w = work_item(B, chunks);
    if (!w.any) return;   // the whole workgroup
    const Tile t = B.tiles[w.tile];
    const u64 first = B.row_ptr[t.row_begin];
    const u32 n = static_cast<u32>(t.row_end - t.row_begin);
    for (u32 i = threadIdx.x; i <= n; i += kGroupThreads) rp[i] = static_cast<u32>(B.row_ptr[t.row_begin + i] - first);
    BlockDict dict{0, 0};
    if constexpr (LD) dict = stage_block_dict(B, t.block, batch_dict);
    __syncthreads();
    const int R = B.R, lane = static_cast<int>(threadIdx.x % RP), s = w.chunk * 8 + lane;
    const bool live = s < R && pair_live(B, t.block, s);
    const int sv = s < R ? s : R - 1;   // idle lanes gather what a neighbour does
    const u64 bs = static_cast<u64>(t.block) * R + sv;
    const double fc = scur ? scur[bs] : 1.0;
    const bool sub = FUSED && *B.step > 0;
    const double b = sub ? beta[bs] * (sprev ? sprev[bs] : 1.0) : 0.0;
    const u32 stride = static_cast<u32>(R) * 16u;
    const char* Xs = reinterpret_cast<const char*>(X + sv);
    double pr = 0.0, pi = 0.0;
    for (u32 r = threadIdx.x / RP; r < n; r += kGroupThreads / RP) {
        const u64 i = (t.row_begin + r) * R + sv;
        Zd p{0.0, 0.0}, x{0.0, 0.0};
        if constexpr (FUSED) {
            if (sub) p = Vprev[i];
            x = X[i];
        }
        Zd y = scaled(group_row<RP, LD>(B, Xs, stride, first, dict.first, dict.zero, rp[r], rp[r + 1]), fc);
        if (!live) continue;
        if constexpr (FUSED) {
            y = Zd{y.re - b * p.re, y.im - b * p.im};
            const Zd d = cdot(scaled(x, fc), y);
            pr += d.re;
            pi += d.im;
        }
        Y[i] = y;
    }
    if constexpr (FUSED) {
#pragma unroll
        for (int off = 32; off >= RP; off >>= 1) {
            pr += __shfl_xor(pr, off, 64);
            pi += __shfl_xor(pi, off, 64);
        }
        const u32 wave = threadIdx.x >> 6;
        if ((threadIdx.x & 63u) < static_cast<u32>(RP)) {
            sr[wave * RP + lane] = pr;
            si[wave * RP + lane] = pi;
        }
        __syncthreads();
        if (threadIdx.x < static_cast<u32>(RP) && s < R) {
            double a = 0.0, c = 0.0;
            for (int q = 0; q < kGroupThreads / 64; ++q) {
                a += sr[q * RP + lane];
                c += si[q * RP + lane];
            }
            partial[(static_cast<u64>(w.tile) * 64 + s) * 2] = a;
            partial[(static_cast<u64>(w.tile) * 64 + s) * 2 + 1] = c;
        }
    }
}

// The fused pass for R = 1 (the continued fractions: one vector per block), on slices of 64 rows of a
// tile: one lane per row, its entries in groups of four (OneView), eight gathers in flight and two
// partial sums. With eight lanes per row on the packed CSR, the value's two halves read from a
// dictionary in global memory and one entry in flight, the step at N = 26 (10.4M rows, 1.5e8 entries)
// took 0.906 ms; with the dictionary in LDS and four entries in flight 0.785 ms, in level order
// (L2 misses 26.7M -> 10.7M lines) 0.769 ms: latency, every row being a chain of loads for a couple of
// entries per lane. So: 0.626 ms.
//
// Where an entry's value comes from: kOneFull in full; kOneLds ids, every block's dictionary staged;
// kOneMixed ids, a dictionary above kBatchDictMax values read from global memory and the others staged,
// so that one large dictionary costs the other blocks nothing and no block 20 bytes an entry for 6.
enum OneValues { kOneFull, kOneLds, kOneMixed };

template <OneValues MODE>
__global__ __launch_bounds__(kThreads) void k_batch_spmv_one_fused(BatchView B, const Zd* Vprev,
                                                                   const Zd* Vcur, Zd* W, const double* beta,
                                                                   double* partial, const double* sprev,
                                                                   const double* scur) {
    static_assert(kThreads == kBatchTileRows, "a thread per row of a tile");
    __shared__ double sr[kThreads / 64], si[kThreads / 64];
    const OneView& S = B.one;
    const Work w = work_item(B, 1);
    if (!w.any) return;   // the whole workgroup
    const Tile t = B.tiles[w.tile];
    const u64 r = t.row_begin + threadIdx.x;
    const bool on = r < t.row_end && pair_live(B, t.block, 0);
    const u32 n = on ? S.len[r] : 0u;
    const u64 at = S.ptr[static_cast<u64>(w.tile) * (kBatchTileRows / 64) + (threadIdx.x >> 6)] + (threadIdx.x & 63u) * 4u;
    bool lds = MODE == kOneLds;   // the same for the whole workgroup
    u32 d0 = 0;
    if constexpr (MODE == kOneMixed) {
        d0 = B.dict_begin[t.block];
        lds = B.dict_begin[t.block + 1] - d0 <= static_cast<u32>(kBatchDictMax);
    }
    if (lds) {
        (void)stage_block_dict(B, t.block, batch_dict);
        __syncthreads();
    }
    double ar = 0.0, ai = 0.0, br = 0.0, bi = 0.0;
    for (u32 k = 0; k < n; k += 8) {
        u32x4 c[2];
        u16x4 id[2];
        Zd v[8], x[8];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const u64 e = at + static_cast<u64>(k / 4 + static_cast<u32>(g)) * 256;
            c[g] = *reinterpret_cast<const u32x4*>(S.col + e);
            if constexpr (MODE != kOneFull) {
                id[g] = *reinterpret_cast<const u16x4*>(S.vid + e);
            } else {
#pragma unroll
                for (int u = 0; u < 4; ++u) v[4 * g + u] = S.val[e + static_cast<u64>(u)];
            }
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) x[u] = Vcur[c[u / 4][u % 4]];
        if constexpr (MODE == kOneMixed) {
            if (!lds) {
#pragma unroll
                for (int u = 0; u < 8; ++u) {   // (past the row's end: id 0, counted as zero)
                    const u32 i = d0 + id[u / 4][u % 4];
                    const Zd q{B.dict_re[i], B.dict_im[i]};
                    v[u] = k + static_cast<u32>(u) < n ? q : Zd{0.0, 0.0};
                }
            }
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if constexpr (MODE == kOneLds) v[u] = batch_dict[id[u / 4][u % 4]];
            if constexpr (MODE == kOneMixed) {
                if (lds) v[u] = batch_dict[id[u / 4][u % 4]];
            }
            if (u < 4) zfma(v[u], x[u], ar, ai);
            else zfma(v[u], x[u], br, bi);
        }
    }
    double pr = 0.0, pi = 0.0;
    if (on) {
        const double fc = scur ? scur[t.block] : 1.0;
        Zd y = scaled(Zd{ar + br, ai + bi}, fc);
        if (*B.step > 0) {
            const double b = beta[t.block] * (sprev ? sprev[t.block] : 1.0);
            const Zd p = Vprev[r];
            y = Zd{y.re - b * p.re, y.im - b * p.im};
        }
        W[r] = y;
        const Zd d = cdot(scaled(Vcur[r], fc), y);
        pr = d.re;
        pi = d.im;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        pr += __shfl_xor(pr, off, 64);
        pi += __shfl_xor(pi, off, 64);
    }
    if ((threadIdx.x & 63u) == 0) {
        sr[threadIdx.x >> 6] = pr;
        si[threadIdx.x >> 6] = pi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double a = 0.0, c = 0.0;
        for (int q = 0; q < kThreads / 64; ++q) {
            a += sr[q];
            c += si[q];
        }
        partial[static_cast<u64>(w.tile) * 64 * 2] = a;
        partial[static_cast<u64>(w.tile) * 64 * 2 + 1] = c;
    }
}

// The slices of the R = 1 layout: entries of each slice (64 lanes times its longest row in whole groups
// of eight), the rows' lengths, then the entries; past a row's end its own row with value zero.
__global__ __launch_bounds__(kThreads) void k_one_lengths(BatchView B, u32* len, u64* slice) {
    const Tile t = B.tiles[blockIdx.x];
    const u64 r = t.row_begin + threadIdx.x;
    u32 n = 0;
    if (r < t.row_end) {
        n = static_cast<u32>(B.row_ptr[r + 1] - B.row_ptr[r]);
        len[r] = n;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const u32 o = static_cast<u32>(__shfl_xor(static_cast<int>(n), off, 64));
        n = o > n ? o : n;
    }
    if ((threadIdx.x & 63u) == 0)
        slice[static_cast<u64>(blockIdx.x) * (kBatchTileRows / 64) + (threadIdx.x >> 6)] = static_cast<u64>((n + 7u) & ~7u) * 64;
}

// One block's entries into the slices, from its own CSR: its tile blockIdx.x (the packed tile tile0 +
// blockIdx.x), packed row p holding row order[p] (null: p) and column c at place[c]; ids count from the
// block's first.
__global__ __launch_bounds__(kThreads) void k_one_fill(CsrView A, u64 row0, u32 tile0, const u32* order, const u32* place,
                                                       const u64* slice, u32* col, u16* vid, Zd* val, u32 zero) {
    const u64 q = blockIdx.x * static_cast<u64>(kBatchTileRows) + threadIdx.x;
    if (q >= static_cast<u64>(A.rows)) return;
    const u64 p = row0 + q, r = order ? order[p] - row0 : q;
    const u64 from = A.row_ptr[r];
    const u32 n = static_cast<u32>(A.row_ptr[r + 1] - from), end = (n + 7u) & ~7u;
    const u64 at = slice[static_cast<u64>(tile0 + blockIdx.x) * (kBatchTileRows / 64) + (threadIdx.x >> 6)] + (threadIdx.x & 63u) * 4u;
    for (u32 k = 0; k < end; k += 4) {
        u32x4 c;
        u16x4 id;
        Zd v[4];
#pragma unroll
        for (u32 u = 0; u < 4; ++u) {
            const bool in = k + u < n;
            const u64 e = from + (in ? k + u : 0u);
            const u64 to = row0 + entry_column(A, e);
            c[u] = in ? (place ? place[to] : static_cast<u32>(to)) : static_cast<u32>(p);
            if (vid) id[u] = static_cast<u16>(in ? entry_id(A, e) : zero);
            else v[u] = in ? csr_value(A, e) : Zd{0.0, 0.0};
        }
        const u64 e = at + static_cast<u64>(k / 4) * 256;
        *reinterpret_cast<u32x4*>(col + e) = c;
        if (vid) {
            *reinterpret_cast<u16x4*>(vid + e) = id;
        } else {
            for (u32 u = 0; u < 4; ++u) val[e + u] = v[u];
        }
    }
}

// The slots' sums of each vector in slot order into partial[tile][s] (re, im); with only, just the
// vectors whose flag is set. Every thread of the workgroup calls it.
__device__ __forceinline__ void tile_partial(const BatchView& B, double pr, double pi, double* partial,
                                             const int* only = nullptr) {
    __shared__ double sr[kThreads], si[kThreads];
    const int R = B.R, slots = kThreads / R;
    sr[threadIdx.x] = pr;
    si[threadIdx.x] = pi;
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < R &&
        (!only || only[static_cast<u64>(B.tiles[blockIdx.x].block) * R + threadIdx.x])) {
        double a = 0.0, b = 0.0;
        for (int q = 0; q < slots; ++q) {
            a += sr[q * R + threadIdx.x];
            b += si[q * R + threadIdx.x];
        }
        partial[(static_cast<u64>(blockIdx.x) * 64 + threadIdx.x) * 2] = a;
        partial[(static_cast<u64>(blockIdx.x) * 64 + threadIdx.x) * 2 + 1] = b;
    }
}

// mode 1: W -= alpha V_cur, then partial of <V_cur, W> (the local overlap);
// mode 5: mode 1, and the partial of ||W||^2 into partial2 as well (what mode 2 sums when it does
//         not correct W);
// mode 4: W -= alpha V_cur, then partial of ||W||^2 (no reorthogonalisation);
// mode 2: W -= ov V_cur when |ov| > threshold (from step 1 on), then partial of ||W||^2; with
//         B.fix (after mode 5) only the pairs flagged there, their norms into partial2;
// mode 3: W *= 1 / beta_next (the next basis vector).
// Pairs no longer running are left alone.
__global__ __launch_bounds__(kThreads) void k_batch_vec(BatchView B, int mode, const Zd* Vcur, Zd* W,
                                                        const double* coef, const Zd* zcoef, double threshold,
                                                        double* partial, double* partial2, const double* vscale) {
    const Tile t = B.tiles[blockIdx.x];
    const int R = B.R, slots = kThreads / R;
    const int slot = threadIdx.x / R, s = threadIdx.x % R;
    const u64 bs = static_cast<u64>(t.block) * R + s;
    if (mode == 2 && B.fix) {
        // nothing to correct in this tile's block: the whole workgroup leaves (the usual case)
        bool any = false;
        for (int q = 0; q < R; ++q) any = any || B.fix[static_cast<u64>(t.block) * R + q] != 0;
        if (!any) return;
    }
    const bool live = slot < slots && pair_live(B, t.block, s) && !(mode == 2 && B.fix && !B.fix[bs]);
    double pr = 0.0, pi = 0.0, pn = 0.0;
    if (live) {
        const int step = *B.step;
        const double fc = vscale ? vscale[bs] : 1.0;   // V_cur = stored V_cur times fc
        for (u64 r = t.row_begin + slot; r < t.row_end; r += slots) {
            const u64 i = r * R + s;
            Zd w = W[i];
            if (mode == 1 || mode == 4 || mode == 5) {
                const double a = coef[bs];
                const Zd v = scaled(Vcur[i], fc);
                w = Zd{w.re - a * v.re, w.im - a * v.im};
                W[i] = w;
                if (mode != 4) {
                    const Zd d = cdot(v, w);
                    pr += d.re;
                    pi += d.im;
                    if (mode == 5) pn += w.re * w.re + w.im * w.im;
                } else {
                    pr += w.re * w.re + w.im * w.im;
                }
            } else if (mode == 2) {
                const Zd ov = zcoef[bs];
                if (step > 0 && sqrt(ov.re * ov.re + ov.im * ov.im) > threshold) {
                    const Zd m = cmul(ov, scaled(Vcur[i], fc));
                    w = Zd{w.re - m.re, w.im - m.im};
                    W[i] = w;
                }
                pr += w.re * w.re + w.im * w.im;
            } else {
                const double inv = coef[bs];
                W[i] = Zd{w.re * inv, w.im * inv};
            }
        }
    }
    if (mode == 5) {
        tile_partial(B, pr, pi, partial);
        __syncthreads();   // the LDS of the first sums is read before the second overwrites it
        tile_partial(B, pn, 0.0, partial2);
    } else if (mode == 2 && B.fix) {
        tile_partial(B, pr, pi, partial2, B.fix);
    } else if (mode != 3) {
        tile_partial(B, pr, pi, partial);
    }
}

// The sum over block b's tiles of partial[tile][s] (re, im), one workgroup of 256 threads per
// (block, vector): thread t takes tiles t, t + 256, ... in order, then a fixed pairwise tree in LDS.
// Thread 0 returns the sums. Every thread of the workgroup calls it.
__device__ __forceinline__ void block_sum(const BatchView& B, int b, int s, const double* partial, double& a,
                                          double& c) {
    __shared__ double ra[kThreads], rc[kThreads];
    double x = 0.0, y = 0.0;
    for (u32 t = B.tile_begin[b] + threadIdx.x; t < B.tile_begin[b + 1]; t += kThreads) {
        x += partial[(static_cast<u64>(t) * 64 + s) * 2];
        y += partial[(static_cast<u64>(t) * 64 + s) * 2 + 1];
    }
    ra[threadIdx.x] = x;
    rc[threadIdx.x] = y;
    __syncthreads();
    for (int off = kThreads / 2; off > 0; off >>= 1) {
        if (static_cast<int>(threadIdx.x) < off) {
            ra[threadIdx.x] += ra[threadIdx.x + off];
            rc[threadIdx.x] += rc[threadIdx.x + off];
        }
        __syncthreads();
    }
    a = ra[0];
    c = rc[0];
}

// The DGKS gate of the second Gram-Schmidt pass, one workgroup per (block, vector): the pass is
// repeated when the first one left less than kappa of the norm it found.
__global__ __launch_bounds__(kThreads) void k_batch_dgks_gate(BatchView B, const double* before, const double* after,
                                                              const int* full, double kappa, int* on) {
    const u32 b = blockIdx.x / static_cast<u32>(B.R);
    const int s = static_cast<int>(blockIdx.x % static_cast<u32>(B.R));
    double n0 = 0.0, n1 = 0.0, unused = 0.0;
    block_sum(B, static_cast<int>(b), s, before, n0, unused);
    __syncthreads();   // every thread has read the first sum before the LDS is reused
    block_sum(B, static_cast<int>(b), s, after, n1, unused);
    if (threadIdx.x == 0)
        on[blockIdx.x] = (full[b] && pair_live(B, b, s) && sqrt(n1) < kappa * sqrt(n0)) ? 1 : 0;
}

// One workgroup per (block, vector). kind 0: alpha (real part) -> alpha_hist[step]; kind 1: the
// overlap (complex) -> ov; kind 2: beta = sqrt -> beta_hist[step], 1 / beta -> inv_beta; breakdown
// (beta < tol) or the block's Krylov cap ends the pair's run.
__global__ __launch_bounds__(kThreads) void k_batch_finish(BatchView B, int kind, const double* partial,
                                                           double* alpha_hist, double* beta_hist, Zd* ov,
                                                           double* cur_alpha, double* cur_beta, double* inv_beta,
                                                           const double* breakdown_tol, double threshold) {
    const int R = B.R;
    const u64 bs = blockIdx.x;
    const int b = static_cast<int>(bs / R), s = static_cast<int>(bs % R);
    if (!B.active[bs]) return;   // the whole workgroup
    double a, c;
    block_sum(B, b, s, partial, a, c);
    if (threadIdx.x != 0) return;
    const int step = *B.step;
    const u64 hist = static_cast<u64>(step) * B.n_blocks * R + bs;
    if (kind == 0) {
        alpha_hist[hist] = a;
        cur_alpha[bs] = a;
    } else if (kind == 1) {
        ov[bs] = Zd{a, c};
        if (B.fix) B.fix[bs] = (step > 0 && sqrt(a * a + c * c) > threshold) ? 1 : 0;
    } else {
        const double beta = sqrt(a);
        beta_hist[hist] = beta;
        cur_beta[bs] = beta;
        B.steps[bs] = step + 1;
        if (!(beta >= breakdown_tol[b]) || step + 1 >= B.cap[b]) {
            B.active[bs] = 0;   // the pair's run ends here (breakdown, or the block's Krylov space is full)
            inv_beta[bs] = 0.0;
        } else {
            inv_beta[bs] = 1.0 / beta;
        }
    }
}

// ||V||^2 per pair, then V scaled by 1 / ||V||: the normalisation of the start vectors.
__global__ __launch_bounds__(kThreads) void k_batch_norm_partial(BatchView B, const Zd* V, double* partial) {
    const Tile t = B.tiles[blockIdx.x];
    const int R = B.R, slots = kThreads / R;
    const int slot = threadIdx.x / R, s = threadIdx.x % R;
    double p = 0.0;
    if (slot < slots)
        for (u64 r = t.row_begin + slot; r < t.row_end; r += slots) {
            const Zd v = V[r * R + s];
            p += v.re * v.re + v.im * v.im;
        }
    tile_partial(B, p, 0.0, partial);
}

__global__ __launch_bounds__(kThreads) void k_batch_norm_finish(BatchView B, const double* partial, double* inv,
                                                                double* norm2) {
    const u64 bs = blockIdx.x;
    const int b = static_cast<int>(bs / B.R), s = static_cast<int>(bs % B.R);
    double a, c;
    block_sum(B, b, s, partial, a, c);
    if (threadIdx.x != 0) return;
    inv[bs] = a > 0.0 ? 1.0 / sqrt(a) : 0.0;
    if (norm2) norm2[bs] = a;
}

__global__ __launch_bounds__(kThreads) void k_batch_scale(BatchView B, Zd* V, const double* inv) {
    const Tile t = B.tiles[blockIdx.x];
    const int R = B.R, slots = kThreads / R;
    const int slot = threadIdx.x / R, s = threadIdx.x % R;
    if (slot >= slots) return;
    const double f = inv[static_cast<u64>(t.block) * R + s];
    for (u64 r = t.row_begin + slot; r < t.row_end; r += slots) {
        const Zd v = V[r * R + s];
        V[r * R + s] = Zd{v.re * f, v.im * f};
    }
}

// One vector placed into the batch layout: state i of the block at packed row row0 + i, or, with the
// engine's row order, place[row0 + i].
__global__ void k_batch_place(Zd* V, int R, u64 row0, int s, const Zd* src, u64 n, const u32* place) {
    for (u64 i = blockIdx.x * static_cast<u64>(blockDim.x) + threadIdx.x; i < n; i += static_cast<u64>(gridDim.x) * blockDim.x) {
        const u64 r = place ? place[row0 + i] : row0 + i;
        V[r * R + s] = src[i];
    }
}

// The whole batch vector from the states' order into the engine's: out[place[r] R + s] = in[r R + s].
__global__ void k_batch_reorder(const Zd* in, u64 rows, int R, const u32* place, Zd* out) {
    const u64 n = rows * static_cast<u64>(R);
    for (u64 i = blockIdx.x * static_cast<u64>(blockDim.x) + threadIdx.x; i < n; i += static_cast<u64>(gridDim.x) * blockDim.x)
        out[place[i / R] * static_cast<u64>(R) + i % R] = in[i];
}

// ---- the engine's row order ---------------------------------------------------------------------
// Breadth-first levels of the blocks flagged in `reorder`, from each block's first row: a sweep takes the
// rows of level l and marks their unmarked columns l + 1 (several rows may mark one, with the same
// value; the matrix is Hermitian, so its pattern is symmetric). 255: not reached.
constexpr u32 kLevelNone = 255;

__global__ __launch_bounds__(kThreads) void k_level_init(BatchView B, const u8* reorder, u8* level) {
    const Tile t = B.tiles[blockIdx.x];
    const bool on = reorder[t.block] != 0;
    const u64 first = B.tiles[B.tile_begin[t.block]].row_begin;
    for (u64 r = t.row_begin + threadIdx.x; r < t.row_end; r += kThreads)
        level[r] = static_cast<u8>(on && r != first ? kLevelNone : 0u);
}

__global__ __launch_bounds__(kThreads) void k_level_sweep(BatchView B, const u8* reorder, u32 l, u8* level, u32* marked) {
    const Tile t = B.tiles[blockIdx.x];
    if (!reorder[t.block]) return;
    const u64 n = t.row_end - t.row_begin;
    bool any = false;
    for (u64 r = threadIdx.x >> 3; r < n; r += kThreads / 8) {
        if (level[t.row_begin + r] != l) continue;
        const u64 e1 = B.row_ptr[t.row_begin + r + 1];
        for (u64 e = B.row_ptr[t.row_begin + r] + (threadIdx.x & 7u); e < e1; e += 8) {
            const u32 c = B.col[e];
            if (level[c] == kLevelNone) {
                level[c] = static_cast<u8>(l + 1);
                any = true;
            }
        }
    }
    if (any) marked[l] = 1u;
}

__global__ __launch_bounds__(kThreads) void k_level_keys(BatchView B, const u8* level, u32* key, u32* row) {
    const Tile t = B.tiles[blockIdx.x];
    for (u64 r = t.row_begin + threadIdx.x; r < t.row_end; r += kThreads) {
        key[r] = (t.block << 8) | level[r];
        row[r] = static_cast<u32>(r);
    }
}

__global__ void k_order_invert(const u32* order, u64 n, u32* place) {
    for (u64 i = blockIdx.x * static_cast<u64>(blockDim.x) + threadIdx.x; i < n; i += static_cast<u64>(gridDim.x) * blockDim.x)
        place[order[i]] = static_cast<u32>(i);
}

__global__ void k_order_lengths(const u64* row_ptr, const u32* order, u64 n, u32* len) {
    for (u64 i = blockIdx.x * static_cast<u64>(blockDim.x) + threadIdx.x; i < n; i += static_cast<u64>(gridDim.x) * blockDim.x) {
        const u64 r = order[i];
        len[i] = static_cast<u32>(row_ptr[r + 1] - row_ptr[r]);
    }
}

__global__ void k_batch_advance(BatchView B) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *B.step += 1;
}

__global__ void k_fill_zd(Zd* x, u64 n) {
    for (u64 i = blockIdx.x * static_cast<u64>(blockDim.x) + threadIdx.x; i < n; i += static_cast<u64>(gridDim.x) * blockDim.x)
        x[i] = Zd{0.0, 0.0};
}

// Entry e of a sector CSR: its column and its value (dictionary ids of width 1 / 2 / 3, or in full).
__device__ __forceinline__ void decode_entry(const CsrView& A, u64 e, u32& c, Zd& v) {
    const u32 w = A.col[e];
    c = A.width == 3 ? (w & 0xFFFFFFu) : w;
    if (A.width == 3) {
        const u32 id = w >> 24;
        v = Zd{A.dict_re[id], A.values_real ? 0.0 : A.dict_im[id]};
    } else if (A.width == 1) {
        const u32 id = static_cast<const u8*>(A.vals)[e];
        v = Zd{A.dict_re[id], A.values_real ? 0.0 : A.dict_im[id]};
    } else if (A.width == 2) {
        const u32 id = static_cast<const u16*>(A.vals)[e];
        v = Zd{A.dict_re[id], A.values_real ? 0.0 : A.dict_im[id]};
    } else if (A.values_real) {
        v = Zd{static_cast<const double*>(A.vals)[e], 0.0};
    } else {
        v = static_cast<const Zd*>(A.vals)[e];
    }
}

// A square sector CSR as a dense column-major matrix (out zeroed first): out[c n + r] = H[r, c], one
// thread per row (a merged row holds each column once).
__global__ void k_csr_to_dense(CsrView A, Zd* out) {
    const u64 r = blockIdx.x * static_cast<u64>(blockDim.x) + threadIdx.x;
    const u64 n = static_cast<u64>(A.rows);
    if (r >= n) return;
    for (u64 e = A.row_ptr[r]; e < A.row_ptr[r + 1]; ++e) {
        u32 c;
        Zd v;
        decode_entry(A, e, c, v);
        out[static_cast<u64>(c) * n + r] = v;
    }
}

// One block's CSR into the packed one, eight lanes per row, each row's entries in their order. Rows: at
// row_off + r and nnz_off, the row pointers written here, or (row_place set) at row_place[row_off + r],
// whose first entry row_ptr already holds. Columns (col null: the row pointers alone): col_off + c, or
// col_place[col_off + c]. Values: in full into val, or the ids offset by the block's first entry in the
// packed dictionary into vid (the caller checked that the block has ids and the offset ids fit 16 bits),
// or neither.
__global__ __launch_bounds__(kThreads) void k_pack_csr(CsrView A, u64 row_off, const u32* row_place, u64 col_off,
                                                       const u32* col_place, u64 nnz_off, u64* row_ptr, u32* col, Zd* val,
                                                       u16* vid, u32 dict_off) {
    const u64 rows = static_cast<u64>(A.rows), stride = static_cast<u64>(gridDim.x) * (kThreads / 8);
    const u32 lane = threadIdx.x & 7u;
    for (u64 r = blockIdx.x * static_cast<u64>(kThreads / 8) + (threadIdx.x >> 3); r < rows; r += stride) {
        const u64 from = A.row_ptr[r], end = A.row_ptr[r + 1];
        u64 to = nnz_off + from;
        if (row_place) {
            to = row_ptr[row_place[row_off + r]];
        } else if (lane == 0) {
            row_ptr[row_off + r] = to;
            if (r + 1 == rows) row_ptr[row_off + rows] = nnz_off + end;
        }
        if (!col) continue;
        for (u64 k = lane; k < end - from; k += 8) {
            const u64 c = col_off + entry_column(A, from + k);
            col[to + k] = col_place ? col_place[c] : static_cast<u32>(c);
            if (vid) vid[to + k] = static_cast<u16>(dict_off + entry_id(A, from + k));
            else if (val) val[to + k] = csr_value(A, from + k);
        }
    }
}

// The row lengths of one block at its rows' places.
__global__ void k_place_lengths(CsrView A, u64 row_off, const u32* place, u32* len) {
    const u64 r = blockIdx.x * static_cast<u64>(blockDim.x) + threadIdx.x;
    if (r < static_cast<u64>(A.rows)) len[place[row_off + r]] = static_cast<u32>(A.row_ptr[r + 1] - A.row_ptr[r]);
}

// Whether block b takes a Gram-Schmidt pass: it is fully reorthogonalised and, with per-pair flags,
// at least one of its pairs is flagged.
__device__ __forceinline__ bool gs_block(const BatchView& B, u32 b, const int* full, const int* on) {
    if (!full[b]) return false;
    if (!on) return true;
    bool any = false;
    for (int q = 0; q < B.R; ++q) any = any || on[static_cast<u64>(b) * B.R + q] != 0;
    return any;
}

// Full Gram-Schmidt against kept basis layers (layer k at basis + k * layer, the batch layout), for
// the blocks flagged in full (and, with on, the pairs flagged there). Coefficients: one workgroup
// per (block, k); thread (slot, s) sums <V_k, W> over the block's rows r = first + slot, first +
// slot + slots, ..., then the slots' sums in slot order: coef[(b * kmax + k) * R + s].
// Deterministic, independent of the other blocks.
__global__ __launch_bounds__(kThreads) void k_batch_gs_coef(BatchView B, const Zd* basis, u64 layer, int K, int kmax,
                                                            const Zd* W, const int* full, const int* on, Zd* coef) {
    const u32 b = blockIdx.x / static_cast<u32>(K);
    const int k = static_cast<int>(blockIdx.x % static_cast<u32>(K));
    if (!gs_block(B, b, full, on)) return;   // the whole workgroup
    const int R = B.R, slots = kThreads / R;
    const int slot = threadIdx.x / R, s = threadIdx.x % R;
    const u64 first = B.tiles[B.tile_begin[b]].row_begin, last = B.tiles[B.tile_begin[b + 1] - 1].row_end;
    double pr = 0.0, pi = 0.0;
    if (slot < slots && pair_live(B, b, s) && (!on || on[static_cast<u64>(b) * R + s])) {
        const Zd* V = basis + static_cast<u64>(k) * layer;
        for (u64 r = first + slot; r < last; r += slots) {
            const u64 i = r * R + s;
            const Zd d = cdot(V[i], W[i]);
            pr += d.re;
            pi += d.im;
        }
    }
    __shared__ double sr[kThreads], si[kThreads];
    sr[threadIdx.x] = pr;
    si[threadIdx.x] = pi;
    __syncthreads();
    if (static_cast<int>(threadIdx.x) < R) {
        double a = 0.0, c = 0.0;
        for (int q = 0; q < slots; ++q) {
            a += sr[q * R + threadIdx.x];
            c += si[q * R + threadIdx.x];
        }
        coef[(static_cast<u64>(b) * kmax + k) * R + threadIdx.x] = Zd{a, c};
    }
}

// W -= sum_{k < K} coef_k V_k on the tiles of the flagged blocks, k ascending.
__global__ __launch_bounds__(kThreads) void k_batch_gs_update(BatchView B, const Zd* basis, u64 layer, int K, int kmax,
                                                              Zd* W, const int* full, const int* on, const Zd* coef) {
    const Tile t = B.tiles[blockIdx.x];
    if (!gs_block(B, t.block, full, on)) return;
    const int R = B.R, slots = kThreads / R;
    const int slot = threadIdx.x / R, s = threadIdx.x % R;
    if (slot >= slots || !pair_live(B, t.block, s) || (on && !on[static_cast<u64>(t.block) * R + s])) return;
    const Zd* c = coef + static_cast<u64>(t.block) * kmax * R + s;
    for (u64 r = t.row_begin + slot; r < t.row_end; r += slots) {
        const u64 i = r * R + s;
        Zd w = W[i];
        for (int k = 0; k < K; ++k) {
            const Zd m = cmul(c[static_cast<u64>(k) * R], basis[static_cast<u64>(k) * layer + i]);
            w = Zd{w.re - m.re, w.im - m.im};
        }
        W[i] = w;
    }
}

// Layers [K][rows][R] to [R][K][rows]: each pair's vectors contiguous, layer after layer (the
// column-major panels a library GEMM reads).
__global__ void k_batch_layers_transpose(const Zd* in, u64 rows, int R, int K, Zd* out) {
    const u64 n = rows * static_cast<u64>(R) * static_cast<u64>(K);
    for (u64 i = blockIdx.x * static_cast<u64>(blockDim.x) + threadIdx.x; i < n; i += static_cast<u64>(gridDim.x) * blockDim.x) {
        const u64 s = i % static_cast<u64>(R), kr = i / static_cast<u64>(R);
        const u64 r = kr % rows, k = kr / rows;
        out[(s * static_cast<u64>(K) + k) * rows + r] = in[i];
    }
}

// Kept-basis overlaps X^H Y per chunk of rows on the FP64 matrix cores. A workgroup owns a 64 x 64
// tile of one chunk's (a, b) product; its four waves own 32 x 32 quarters, each four 16 x 16 MFMA
// tiles with a real and an imaginary accumulator (re += xr yr + xi yi, im += xr yi - xi yr: four
// v_mfma_f64_16x16x4 per tile and four rows). 16-row slices of the tile's 64 X and 64 Y vectors are
// staged in LDS with the vector index fastest. Operand layout of v_mfma_f64_16x16x4 (wave64): lane l
// holds A[l % 16][l / 16] and B[l / 16][l % 16]; accumulator entry v of lane l is
// D[4 v + l / 16][l % 16]. A wave skips its 16 x 16 tiles that lie outside the pair's ma x mb product.
// The grid is one-dimensional: workgroup g runs on XCD g % 8, and the tiles of a chunk are
// consecutive on one XCD, so the chunk's vectors, read by every tile of it, stay in that XCD's L2.
typedef double mf_acc __attribute__((ext_vector_type(4)));
constexpr int kOvTile = 64, kOvRows = 16, kXcds = 8;
__global__ __launch_bounds__(256) void k_overlap_mfma(const Zd* X, u64 ldx, const Zd* Y, u64 ldy,
                                                      const OverlapChunk* chunks, u32 n_chunks, int tiles,
                                                      const int* ma, const int* mb, int kmax, Zd* partial) {
    __shared__ Zd xs[kOvRows][kOvTile + 1], ys[kOvRows][kOvTile + 1];   // padded: the column stores spread over banks
    const u32 g = blockIdx.x, xcd = g % kXcds, slot = g / kXcds;
    const u32 per_chunk = static_cast<u32>(tiles * tiles);
    const u32 q = (slot / per_chunk) * kXcds + xcd;   // the chunk
    if (q >= n_chunks) return;
    const u32 tile = slot % per_chunk;
    const OverlapChunk ch = chunks[q];
    const int a0 = static_cast<int>(tile / static_cast<u32>(tiles)) * kOvTile;
    const int b0 = static_cast<int>(tile % static_cast<u32>(tiles)) * kOvTile;
    const int na = ma[ch.pair], nb = mb[ch.pair];
    if (a0 >= na || b0 >= nb) return;   // the whole workgroup: tile outside this pair's product
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wa = (wave & 1) * 32, wb = (wave >> 1) * 32;
    const int li = lane & 15, lk = lane >> 4;
    bool on[2][2];
    mf_acc cr[2][2], ci[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            on[i][j] = a0 + wa + 16 * i < na && b0 + wb + 16 * j < nb;   // uniform over the wave
            cr[i][j] = mf_acc{0.0, 0.0, 0.0, 0.0};
            ci[i][j] = mf_acc{0.0, 0.0, 0.0, 0.0};
        }
    for (u32 r0 = 0; r0 < ch.rows; r0 += kOvRows) {
        for (int idx = threadIdx.x; idx < kOvTile * kOvRows; idx += 256) {
            const int k = idx / kOvRows, rr = idx % kOvRows;   // consecutive threads: consecutive rows
            const u32 row = r0 + static_cast<u32>(rr);
            const bool in_row = row < ch.rows;
            xs[rr][k] = (in_row && a0 + k < na) ? X[ch.x_base + static_cast<u64>(a0 + k) * ldx + row] : Zd{0.0, 0.0};
            ys[rr][k] = (in_row && b0 + k < nb) ? Y[ch.y_base + static_cast<u64>(b0 + k) * ldy + row] : Zd{0.0, 0.0};
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kOvRows / 4; ++kk) {
            const int rr = kk * 4 + lk;
            Zd xv[2], yv[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) xv[i] = xs[rr][wa + 16 * i + li];
#pragma unroll
            for (int j = 0; j < 2; ++j) yv[j] = ys[rr][wb + 16 * j + li];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    if (on[i][j]) {
                        cr[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(xv[i].re, yv[j].re, cr[i][j], 0, 0, 0);
                        ci[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(xv[i].re, yv[j].im, ci[i][j], 0, 0, 0);
                    }
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    if (on[i][j]) {
                        cr[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(xv[i].im, yv[j].im, cr[i][j], 0, 0, 0);
                        ci[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(-xv[i].im, yv[j].re, ci[i][j], 0, 0, 0);
                    }
        }
        __syncthreads();
    }
    Zd* out = partial + static_cast<u64>(q) * kmax * kmax;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int a = a0 + wa + 16 * i + 4 * v + lk, b = b0 + wb + 16 * j + li;
                if (a < na && b < nb) out[static_cast<u64>(b) * na + a] = Zd{cr[i][j][v], ci[i][j][v]};
            }
}

// omega[p](a, b) = the sum of the pair's chunk partials in chunk order; one thread per (pair, a, b).
__global__ void k_overlap_reduce(const Zd* partial, const u32* chunk_begin, const int* ma, const int* mb, u32 n_pairs,
                                 int kmax, Zd* omega) {
    const u64 per = static_cast<u64>(kmax) * kmax;
    for (u64 i = blockIdx.x * static_cast<u64>(blockDim.x) + threadIdx.x; i < n_pairs * per;
         i += static_cast<u64>(gridDim.x) * blockDim.x) {
        const u32 p = static_cast<u32>(i / per);
        const u64 e = i % per;
        if (e >= static_cast<u64>(ma[p]) * mb[p]) continue;
        double re = 0.0, im = 0.0;
        for (u32 q = chunk_begin[p]; q < chunk_begin[p + 1]; ++q) {
            const Zd v = partial[static_cast<u64>(q) * per + e];
            re += v.re;
            im += v.im;
        }
        omega[static_cast<u64>(p) * per + e] = Zd{re, im};
    }
}

unsigned grid_for(u64 n) {
    u64 g = (n + 255) / 256;
    if (g > 65536) g = 65536;
    return static_cast<unsigned>(g ? g : 1);
}

}  // namespace

namespace {
/// Whether every block's dictionary fits the SpMV's LDS.
bool batch_dict_in_lds(const BatchView& B) {
    return B.dict_begin && B.dict_max > 0 && B.dict_max <= static_cast<u32>(kBatchDictMax);
}

template <bool FUSED>
void launch_group(const BatchView& B, const Zd* Vprev, const Zd* X, Zd* Y, const double* beta, double* partial,
                  const double* sprev, const double* scur, hipStream_t st) {
    const int chunks = batch_chunks(B.R);
    const dim3 grid(B.sched ? B.n_sched : B.n_tiles * static_cast<u32>(chunks)), block(kGroupThreads);
    auto go = [&](auto in_lds, std::size_t lds) {
        constexpr bool LD = decltype(in_lds)::value;
#define QSA_GROUP(RP)                                                                                                  \
    hipLaunchKernelGGL((k_batch_spmv_group<RP, LD, FUSED>), grid, block, lds, st, B, chunks, Vprev, X, Y, beta, partial, \
                       sprev, scur)
        if (B.R <= 2) QSA_GROUP(2);
        else if (B.R <= 4) QSA_GROUP(4);
        else QSA_GROUP(8);
#undef QSA_GROUP
    };
    if (B.vid && batch_dict_in_lds(B)) go(std::true_type{}, (static_cast<std::size_t>(B.dict_max) + 1) * sizeof(Zd));
    else go(std::false_type{}, std::size_t{0});
}
}  // namespace

void batch_spmv(const BatchView& B, const Zd* X, Zd* Y, hipStream_t st) {
    if (B.n_tiles) launch_group<false>(B, nullptr, X, Y, nullptr, nullptr, nullptr, nullptr, st);
}

void batch_spmv_fused(const BatchView& B, const Zd* Vprev, const Zd* Vcur, Zd* W, const double* beta, double* partial,
                      hipStream_t st, const double* sprev, const double* scur) {
    if (!B.n_tiles) return;
    if (!B.one.ptr) {
        launch_group<true>(B, Vprev, Vcur, W, beta, partial, sprev, scur, st);
        return;
    }
    const dim3 grid(B.sched ? B.n_sched : B.n_tiles), block(kThreads);
    const std::size_t lds = (std::min<std::size_t>(B.dict_max, kBatchDictMax) + 1) * sizeof(Zd);
#define QSA_ONE(MODE, LDS)                                                                                            \
    hipLaunchKernelGGL((k_batch_spmv_one_fused<MODE>), grid, block, LDS, st, B, Vprev, Vcur, W, beta, partial, sprev, \
                       scur)
    if (!B.one.vid) QSA_ONE(kOneFull, 0);
    else if (batch_dict_in_lds(B)) QSA_ONE(kOneLds, lds);
    else QSA_ONE(kOneMixed, lds);
#undef QSA_ONE
}

void one_lengths(const BatchView& B, u32* len, u64* slice, hipStream_t st) {
    if (B.n_tiles) hipLaunchKernelGGL(k_one_lengths, dim3(B.n_tiles), dim3(kThreads), 0, st, B, len, slice);
}

void one_fill(const CsrView& A, u64 row0, u32 tile0, const u32* order, const u32* place, const u64* slice, u32* col,
              u16* vid, Zd* val, hipStream_t st) {
    static_assert(kThreads == kBatchTileRows, "a thread per row of a tile");
    if (!A.rows) return;
    // the zero after a staged dictionary's last value; a dictionary in global memory counts the padding out
    const u32 zero = A.dict_n <= kBatchDictMax ? static_cast<u32>(A.dict_n) : 0u;
    hipLaunchKernelGGL(k_one_fill, dim3(static_cast<unsigned>((static_cast<u64>(A.rows) + kThreads - 1) / kThreads)),
                       dim3(kThreads), 0, st, A, row0, tile0, order, place, slice, col, vid, val, zero);
}

void batch_vec(const BatchView& B, int mode, const Zd* Vcur, Zd* W, const double* coef, const Zd* zcoef,
               double threshold, double* partial, hipStream_t st, double* partial2, const double* vscale) {
    if (!B.n_tiles) return;
    hipLaunchKernelGGL(k_batch_vec, dim3(B.n_tiles), dim3(kThreads), 0, st, B, mode, Vcur, W, coef, zcoef, threshold,
                       partial, partial2, vscale);
}

void batch_finish(const BatchView& B, int kind, const double* partial, double* alpha_hist, double* beta_hist, Zd* ov,
                  double* cur_alpha, double* cur_beta, double* inv_beta, const double* breakdown_tol, hipStream_t st,
                  double threshold) {
    hipLaunchKernelGGL(k_batch_finish, dim3(B.n_blocks * static_cast<u32>(B.R)), dim3(kThreads), 0, st, B, kind, partial,
                       alpha_hist, beta_hist, ov, cur_alpha, cur_beta, inv_beta, breakdown_tol, threshold);
}

void batch_normalize(const BatchView& B, Zd* V, double* partial, double* inv, double* norm2, hipStream_t st) {
    if (!B.n_tiles) return;
    hipLaunchKernelGGL(k_batch_norm_partial, dim3(B.n_tiles), dim3(kThreads), 0, st, B, V, partial);
    hipLaunchKernelGGL(k_batch_norm_finish, dim3(B.n_blocks * static_cast<u32>(B.R)), dim3(kThreads), 0, st, B, partial,
                       inv, norm2);
    hipLaunchKernelGGL(k_batch_scale, dim3(B.n_tiles), dim3(kThreads), 0, st, B, V, inv);
}

void batch_place(Zd* V, int R, u64 row0, int s, const Zd* src, u64 n, const u32* place, hipStream_t st) {
    if (!n) return;
    hipLaunchKernelGGL(k_batch_place, dim3(grid_for(n)), dim3(256), 0, st, V, R, row0, s, src, n, place);
}

void batch_reorder(const Zd* in, u64 rows, int R, const u32* place, Zd* out, hipStream_t st) {
    if (!rows) return;
    hipLaunchKernelGGL(k_batch_reorder, dim3(grid_for(rows * static_cast<u64>(R))), dim3(256), 0, st, in, rows, R, place, out);
}

void level_init(const BatchView& B, const u8* reorder, u8* level, hipStream_t st) {
    if (B.n_tiles) hipLaunchKernelGGL(k_level_init, dim3(B.n_tiles), dim3(kThreads), 0, st, B, reorder, level);
}

void level_sweep(const BatchView& B, const u8* reorder, u32 l, u8* level, u32* marked, hipStream_t st) {
    if (B.n_tiles) hipLaunchKernelGGL(k_level_sweep, dim3(B.n_tiles), dim3(kThreads), 0, st, B, reorder, l, level, marked);
}

std::size_t level_sort_temp_bytes(u64 rows) {
    std::size_t bytes = 0;
    (void)hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, static_cast<const u32*>(nullptr), static_cast<u32*>(nullptr),
                                             static_cast<const u32*>(nullptr), static_cast<u32*>(nullptr),
                                             static_cast<unsigned>(rows));
    return bytes;
}

hipError_t level_order(const BatchView& B, const u8* level, u32* key, u32* key2, u32* row, u32* order, u32* place, void* temp,
                       std::size_t temp_bytes, hipStream_t st) {
    if (!B.n_tiles) return hipSuccess;
    if (B.rows >> 32 != 0) return hipErrorInvalidValue;   // rows are 32-bit words
    hipLaunchKernelGGL(k_level_keys, dim3(B.n_tiles), dim3(kThreads), 0, st, B, level, key, row);
    int bits = 8;
    while (bits < 32 && (static_cast<u64>(B.n_blocks) >> (bits - 8)) != 0) ++bits;
    const hipError_t e = hipcub::DeviceRadixSort::SortPairs(temp, temp_bytes, key, key2, row, order,
                                                            static_cast<unsigned>(B.rows), 0, bits, st);
    if (e != hipSuccess) return e;   // (order is no index then)
    hipLaunchKernelGGL(k_order_invert, dim3(grid_for(B.rows)), dim3(256), 0, st, order, B.rows, place);
    return hipSuccess;
}

void order_lengths(const u64* row_ptr, const u32* order, u64 rows, u32* len, hipStream_t st) {
    if (rows) hipLaunchKernelGGL(k_order_lengths, dim3(grid_for(rows)), dim3(256), 0, st, row_ptr, order, rows, len);
}

void csr_to_dense(const CsrView& A, Zd* out, hipStream_t st) {
    const u64 n = static_cast<u64>(A.rows);
    if (!n) return;
    batch_fill_zero(out, n * n, st);
    hipLaunchKernelGGL(k_csr_to_dense, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st, A, out);
}

void batch_gram_schmidt(const BatchView& B, const Zd* basis, u64 layer, int K, int kmax, Zd* W, const int* full,
                        Zd* coef, hipStream_t st, const int* on) {
    if (!B.n_tiles || K < 1) return;
    hipLaunchKernelGGL(k_batch_gs_coef, dim3(B.n_blocks * static_cast<u32>(K)), dim3(kThreads), 0, st, B, basis, layer,
                       K, kmax, W, full, on, coef);
    hipLaunchKernelGGL(k_batch_gs_update, dim3(B.n_tiles), dim3(kThreads), 0, st, B, basis, layer, K, kmax, W, full,
                       on, coef);
}

void batch_dgks_gate(const BatchView& B, const double* before, const double* after, const int* full, double kappa,
                     int* on, hipStream_t st) {
    if (!B.n_blocks) return;
    hipLaunchKernelGGL(k_batch_dgks_gate, dim3(B.n_blocks * static_cast<u32>(B.R)), dim3(kThreads), 0, st, B, before,
                       after, full, kappa, on);
}

void batch_norm_partial(const BatchView& B, const Zd* V, double* partial, hipStream_t st) {
    if (!B.n_tiles) return;
    hipLaunchKernelGGL(k_batch_norm_partial, dim3(B.n_tiles), dim3(kThreads), 0, st, B, V, partial);
}

void batch_layers_transpose(const Zd* in, u64 rows, int R, int K, Zd* out, hipStream_t st) {
    const u64 n = rows * static_cast<u64>(R) * static_cast<u64>(K);
    if (!n) return;
    hipLaunchKernelGGL(k_batch_layers_transpose, dim3(grid_for(n)), dim3(256), 0, st, in, rows, R, K, out);
}

void overlap_chunks(const Zd* X, u64 ldx, const Zd* Y, u64 ldy, const OverlapChunk* chunks, u32 n_chunks,
                    const int* ma, const int* mb, int kmax, Zd* partial, hipStream_t st) {
    if (!n_chunks) return;
    const int tiles = (kmax + kOvTile - 1) / kOvTile;
    const u64 groups = (static_cast<u64>(n_chunks) + kXcds - 1) / kXcds * kXcds * static_cast<u64>(tiles * tiles);
    hipLaunchKernelGGL(k_overlap_mfma, dim3(static_cast<unsigned>(groups)), dim3(256), 0, st, X, ldx, Y, ldy, chunks,
                       n_chunks, tiles, ma, mb, kmax, partial);
}

void overlap_reduce(const Zd* partial, const u32* chunk_begin, const int* ma, const int* mb, u32 n_pairs, int kmax,
                    Zd* omega, hipStream_t st) {
    if (!n_pairs) return;
    hipLaunchKernelGGL(k_overlap_reduce, dim3(grid_for(static_cast<u64>(n_pairs) * kmax * kmax)), dim3(256), 0, st,
                       partial, chunk_begin, ma, mb, n_pairs, kmax, omega);
}

void batch_advance(const BatchView& B, hipStream_t st) {
    hipLaunchKernelGGL(k_batch_advance, dim3(1), dim3(64), 0, st, B);
}

void batch_fill_zero(Zd* x, u64 n, hipStream_t st) {
    if (!n) return;
    hipLaunchKernelGGL(k_fill_zd, dim3(grid_for(n)), dim3(256), 0, st, x, n);
}

void place_lengths(const CsrView& A, u64 row_off, const u32* place, u32* len, hipStream_t st) {
    if (!A.rows) return;
    hipLaunchKernelGGL(k_place_lengths, dim3(static_cast<unsigned>((static_cast<u64>(A.rows) + 255) / 256)), dim3(256), 0, st,
                       A, row_off, place, len);
}

void pack_csr(const CsrView& A, u64 row_off, const u32* row_place, u64 col_off, const u32* col_place, u64 nnz_off,
              u64* row_ptr, u32* col, Zd* val, u16* vid, u32 dict_off, hipStream_t st) {
    if (!A.rows) return;
    hipLaunchKernelGGL(k_pack_csr, dim3(grid_for(static_cast<u64>(A.rows) * 8)), dim3(kThreads), 0, st, A, row_off, row_place,
                       col_off, col_place, nnz_off, row_ptr, col, val, vid, dict_off);
}

}  // namespace qsa::dev
