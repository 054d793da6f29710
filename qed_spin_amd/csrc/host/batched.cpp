#include "batched.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdlib>
#include <thread>

#include "lanczos.h"
#include "tridiag.h"

namespace qsa {

namespace {

using clock_t_ = std::chrono::steady_clock;
double secs(clock_t_::time_point a, clock_t_::time_point b) { return std::chrono::duration<double>(b - a).count(); }

/// Host worker threads for the per-pair host work (seeds, tridiagonals): at most 16.
unsigned host_threads() {
    const unsigned hc = std::max(1u, std::thread::hardware_concurrency());
    return std::min(16u, hc);
}

/// fn(i) for i < n on the host worker threads (dynamic schedule); the first exception is rethrown.
template <class Fn> void parallel_for(std::size_t n, Fn&& fn) {
    const unsigned T = static_cast<unsigned>(std::min<std::size_t>(host_threads(), n));
    if (T <= 1) {
        for (std::size_t i = 0; i < n; ++i) fn(i);
        return;
    }
    std::atomic<std::size_t> next{0};
    std::exception_ptr failure;
    std::atomic<bool> failed{false};
    std::vector<std::thread> pool;
    for (unsigned t = 0; t < T; ++t)
        pool.emplace_back([&] {
            for (;;) {
                const std::size_t i = next.fetch_add(1);
                if (i >= n || failed.load()) return;
                try {
                    fn(i);
                } catch (...) {
                    if (!failed.exchange(true)) failure = std::current_exception();
                    return;
                }
            }
        });
    for (auto& th : pool) th.join();
    if (failure) std::rethrow_exception(failure);
}

template <class T> void put(DeviceBuffer& b, const std::vector<T>& h, hipStream_t st) {
    b.reset(h.size() * sizeof(T));
    if (!h.empty()) QSA_HIP(hipMemcpyAsync(b.get(), h.data(), h.size() * sizeof(T), hipMemcpyHostToDevice, st));
    QSA_HIP(hipStreamSynchronize(st));
}

/// Bytes that the row order and the R = 1 slices may take beyond the packed CSR
/// (QED_SPIN_AMD_BATCH_EXTRA_BYTES; without it, what can be allocated).
std::uint64_t extra_bytes() {
    const char* e = std::getenv("QED_SPIN_AMD_BATCH_EXTRA_BYTES");
    return e ? std::strtoull(e, nullptr, 10) : ~std::uint64_t{0};
}

/// fn(), or false when it ran out of device memory.
template <class Fn> bool if_it_fits(Fn&& fn) {
    try {
        return fn();
    } catch (const Error& e) {
        if (e.code != kResourceLimit) throw;
        return false;
    }
}

/// A pooled stream at the default priority (graph capture needs a stream other than the null one).
struct OwnStream {
    hipStream_t s = nullptr;
    OwnStream() : s(pooled_stream_acquire()) {}
    ~OwnStream() { pooled_stream_release(s); }
};

}  // namespace

void parallel_blocks(std::size_t n, const std::function<void(std::size_t)>& fn) { parallel_for(n, fn); }

BatchedLanczos::BatchedLanczos(std::vector<std::shared_ptr<const SectorOperator>> blocks, int R)
    : ops_(std::move(blocks)), R_(R) {
    if (ops_.empty()) throw Error(kInvalid, "batched lanczos: no blocks");
    if (R_ < 1 || R_ > dev::kBatchMaxR)
        throw Error(kInvalid, "batched lanczos: vectors per block must be 1.." + std::to_string(dev::kBatchMaxR));
    row_off_.assign(1, 0);
    std::vector<std::uint64_t> nnz_off(1, 0);
    for (const auto& op : ops_) {
        if (!op) throw Error(kInvalid, "batched lanczos: null block");
        if (!op->same()) throw Error(kInvalid, "batched lanczos: a block must map its sector to itself");
        if (op->lane() != kLaneCsr)
            throw Error(kDeviceUnsupported, "batched lanczos: every block needs its device CSR (csr lane)");
        if (op->dim() <= 0) throw Error(kInvalid, "batched lanczos: empty block");
        row_off_.push_back(row_off_.back() + static_cast<std::uint64_t>(op->dim()));
        nnz_off.push_back(nnz_off.back() + static_cast<std::uint64_t>(op->csr_info().nnz));
    }
    rows_ = row_off_.back();
    nnz_ = nnz_off.back();
    if (rows_ >= (std::uint64_t{1} << 32)) throw Error(kInvalid, "batched lanczos: more than 2^32 rows in one batch");
    const hipStream_t st = engine_stream();
    // Values: when every block stores dictionary ids and the dictionaries hold at most 2^16 values
    // together, 16-bit ids into their concatenation (2 bytes per entry instead of 16); else in full.
    std::vector<std::uint32_t> dict_off(ops_.size() + 1, 0);
    bool ids = true;
    std::uint64_t dict_total = 0;
    for (std::size_t b = 0; ids && b < ops_.size(); ++b) {
        const dev::CsrView A = ops_[b]->device_csr();
        if (A.width < 1 || A.width > 3 || A.dict_n < 1 || !A.dict_re || (!A.values_real && !A.dict_im)) {
            ids = false;
            break;
        }
        dict_off[b] = static_cast<std::uint32_t>(dict_total);
        dict_total += static_cast<std::uint64_t>(A.dict_n);
        dict_max_ = std::max(dict_max_, static_cast<std::uint32_t>(A.dict_n));
    }
    if (dict_total > (std::uint64_t{1} << 16)) ids = false;
    if (ids) {
        dict_n_ = static_cast<std::uint32_t>(dict_total);
        dict_off.back() = dict_n_;
        put(dict_begin_, dict_off, st);
        dict_re_.reset(dict_total * 8);
        dict_im_.reset(dict_total * 8);
        for (std::size_t b = 0; b < ops_.size(); ++b) {
            const dev::CsrView A = ops_[b]->device_csr();
            const std::size_t n = static_cast<std::size_t>(A.dict_n) * 8;
            QSA_HIP(hipMemcpyAsync(dict_re_.get<double>() + dict_off[b], A.dict_re, n, hipMemcpyDeviceToDevice, st));
            if (A.values_real)
                dev::fill_zero(false, dict_im_.get<double>() + dict_off[b], static_cast<std::size_t>(A.dict_n), st);
            else
                QSA_HIP(hipMemcpyAsync(dict_im_.get<double>() + dict_off[b], A.dict_im, n, hipMemcpyDeviceToDevice, st));
        }
    }
    // Tiles: every block cut into runs of at most kBatchTileRows rows, blocks in order.
    tile_begin_.assign(1, 0);
    for (std::size_t b = 0; b < ops_.size(); ++b) {
        for (std::uint64_t r = row_off_[b]; r < row_off_[b + 1]; r += dev::kBatchTileRows) {
            dev::Tile t{};
            t.row_begin = r;
            t.row_end = std::min<std::uint64_t>(r + dev::kBatchTileRows, row_off_[b + 1]);
            t.block = static_cast<std::uint32_t>(b);
            tiles_.push_back(t);
        }
        tile_begin_.push_back(static_cast<std::uint32_t>(tiles_.size()));
    }
    put(tiles_d_, tiles_, st);
    put(tile_begin_d_, tile_begin_, st);
    // The matrix: the row pointers, and (where rows will move) the columns that the order is found from;
    // then the entries, straight from the blocks to where they stay, so that no second copy exists at
    // any time. R = 1: into slices, unless these do not fit.
    std::vector<std::uint8_t> reorder(ops_.size(), 0);
    bool any = false;
    const std::uint64_t wide = static_cast<std::uint64_t>(std::min(R_, 8)) * sizeof(dev::Zd);
    for (std::size_t b = 0; b < ops_.size(); ++b) {
        reorder[b] = dim(static_cast<int>(b)) * wide > kOrderMinBytes ? 1 : 0;
        any = any || reorder[b];
    }
    const bool slices = R_ == 1;
    row_ptr_.reset((rows_ + 1) * 8);
    auto room = [&] {
        col_.reset(std::max<std::uint64_t>(nnz_, 1) * 4);
        if (ids) vid_.reset(std::max<std::uint64_t>(nnz_, 1) * 2);
        else val_.reset(std::max<std::uint64_t>(nnz_, 1) * sizeof(dev::Zd));
    };
    auto pack = [&](std::size_t b, const std::uint32_t* place, bool values) {
        dev::pack_csr(ops_[b]->device_csr(), row_off_[b], place, row_off_[b], place, nnz_off[b], row_ptr_.get<std::uint64_t>(),
                      col_.get<std::uint32_t>(), values && !ids ? val_.get<dev::Zd>() : nullptr,
                      values && ids ? vid_.get<std::uint16_t>() : nullptr, dict_off[b], st);
    };
    if (!slices) room();
    else if (any) col_.reset(std::max<std::uint64_t>(nnz_, 1) * 4);
    for (std::size_t b = 0; b < ops_.size(); ++b) pack(b, nullptr, !slices && !reorder[b]);
    QSA_HIP(hipGetLastError());
    const auto t_order = clock_t_::now();
    if (any && !if_it_fits([&] { return order_rows(reorder); })) {
        order_.release();
        place_.release();
    }
    if (slices) {
        col_.release();
        one_ = if_it_fits([&] { return slice_rows(ids); });
        if (!one_) room();
    }
    for (std::size_t b = 0; b < ops_.size() && !one_; ++b)
        if (slices || reorder[b]) pack(b, place_.get<std::uint32_t>(), true);
    order_.release();
    QSA_HIP(hipGetLastError());
    const char* pinned = std::getenv("QED_SPIN_AMD_BATCH_SCHEDULE");   // 0 or 1
    set_schedule(pinned ? (std::atoi(pinned) == 1 ? 1 : 0) : 1);
    order_s_ = secs(t_order, clock_t_::now());
    const std::size_t vec_bytes = rows_ * static_cast<std::size_t>(R_) * sizeof(dev::Zd);
    V0_.reset(vec_bytes);
    V1_.reset(vec_bytes);
    W_.reset(vec_bytes);
    partial_.reset(tiles_.size() * 64 * 2 * sizeof(double));
    partial2_.reset(tiles_.size() * 64 * 2 * sizeof(double));
    fix_.reset(ops_.size() * static_cast<std::size_t>(R_) * sizeof(int));
    put(fix_, std::vector<int>(ops_.size() * static_cast<std::size_t>(R_), 0), st);
    const std::size_t pairs = ops_.size() * static_cast<std::size_t>(R_);
    ov_.reset(pairs * sizeof(dev::Zd));
    cur_a_.reset(pairs * 8);
    cur_b_.reset(pairs * 8);
    inv_b_.reset(pairs * 8);
    active_d_.reset(pairs * sizeof(int));
    steps_d_.reset(pairs * sizeof(int));
    step_d_.reset(sizeof(int));
    cap_d_.reset(ops_.size() * sizeof(int));
    tol_d_.reset(ops_.size() * sizeof(double));
    dev::batch_fill_zero(V1_.get<dev::Zd>(), rows_ * R_, st);
    dev::batch_fill_zero(W_.get<dev::Zd>(), rows_ * R_, st);
    QSA_HIP(hipStreamSynchronize(st));
}

// A row's columns are gathered R at a time, so an XCD's L2 should hold the part of X that the rows in
// flight on it read. In the order of a momentum sector's states that is nearly the whole block: at
// N = 24, R = 4 (112,632 states, 7.2 MB) the counters gave 870 bytes of X fetched per row of 64. In
// breadth-first level order a row's columns lie within one level of its own (21 to 42 levels on
// rings of 22 to 26 sites, the widest 6 to 14% of a block). Blocks below 2 MB fit an L2 as they are.
// (Rows of a level by their least column of the level before, so that neighbours share columns in the
// L1, took a fifth of the L1's misses at R = 1 for 2% of the step, and made the J1-J2 rings' step at
// R = 4 9% slower.)
bool BatchedLanczos::order_rows(const std::vector<std::uint8_t>& reorder) {
    // (the sort and the scan count rows in 32 bits; 33 bytes a row and the sort's own at the peak)
    if (rows_ >= (std::uint64_t{1} << 31) || ops_.size() >= (std::size_t{1} << 24) || rows_ * 33 > extra_bytes()) return false;
    const hipStream_t st = engine_stream();
    dev::BatchView B = view();
    DeviceBuffer flags, level(rows_), marked(256 * 4);
    put(flags, reorder, st);
    const auto* on = flags.get<std::uint8_t>();
    dev::level_init(B, on, level.get<std::uint8_t>(), st);
    dev::fill_zero(false, marked.get(), marked.bytes() / 8, st);
    std::vector<std::uint32_t> hit(256, 0);
    constexpr std::uint32_t kSweeps = 16;   // between looks at whether the last ones marked anything
    for (std::uint32_t l = 0; l + 1 < 255;) {
        const std::uint32_t end = std::min<std::uint32_t>(l + kSweeps, 254);
        for (; l < end; ++l) dev::level_sweep(B, on, l, level.get<std::uint8_t>(), marked.get<std::uint32_t>(), st);
        QSA_HIP(hipGetLastError());
        copy_to_host(hit.data(), marked.get(), marked.bytes());
        if (!hit[l - 1]) break;
    }
    order_.reset(rows_ * 4);
    place_.reset(rows_ * 4);
    {
        DeviceBuffer key(rows_ * 4), key2(rows_ * 4), row(rows_ * 4);
        const std::size_t tb = dev::level_sort_temp_bytes(rows_);
        DeviceBuffer temp(tb ? tb : 8);
        QSA_HIP(dev::level_order(B, level.get<std::uint8_t>(), key.get<std::uint32_t>(), key2.get<std::uint32_t>(),
                         row.get<std::uint32_t>(), order_.get<std::uint32_t>(), place_.get<std::uint32_t>(), temp.get(), tb,
                         st));
        QSA_HIP(hipGetLastError());
    }
    DeviceBuffer len(rows_ * 4), ptr((rows_ + 1) * 8);
    dev::order_lengths(row_ptr_.get<std::uint64_t>(), order_.get<std::uint32_t>(), rows_, len.get<std::uint32_t>(), st);
    const std::size_t tb = dev::row_scan_temp_bytes(static_cast<std::int64_t>(rows_));
    DeviceBuffer temp(tb ? tb : 8);
    QSA_HIP(dev::row_scan(len.get<std::uint32_t>(), static_cast<std::int64_t>(rows_), ptr.get<std::uint64_t>(), temp.get(), tb, st));
    QSA_HIP(hipGetLastError());
    row_ptr_ = std::move(ptr);   // the old one is freed on this stream, after the kernels that read it
    return true;
}

/// The matrix in the R = 1 layout, straight from the blocks, in place of the row pointers; false when
/// rows of very different lengths would fill it to more than twice the entries.
bool BatchedLanczos::slice_rows(bool ids) {
    const hipStream_t st = engine_stream();
    const dev::BatchView B = view();
    const std::int64_t slices = static_cast<std::int64_t>(tiles_.size()) * (dev::kBatchTileRows / 64);
    DeviceBuffer words(static_cast<std::size_t>(slices + 1) * 8);
    DeviceBuffer len(rows_ * 4), ptr(static_cast<std::size_t>(slices + 1) * 8);
    dev::fill_zero(false, words.get(), static_cast<std::size_t>(slices + 1), st);
    dev::one_lengths(B, len.get<std::uint32_t>(), words.get<std::uint64_t>(), st);
    const std::size_t tb = dev::sell_scan_temp_bytes(slices);
    DeviceBuffer temp(tb ? tb : 8);
    QSA_HIP(dev::sell_scan(words.get<std::uint64_t>(), slices, ptr.get<std::uint64_t>(), temp.get(), tb, st));
    QSA_HIP(hipGetLastError());
    std::uint64_t total = 0;
    copy_to_host(&total, ptr.get<std::uint64_t>() + slices, 8);
    const std::uint64_t least = rows_ * 8;   // (short rows fill whole groups of eight)
    if (total > 2 * std::max(nnz_, least) || total * 6 > extra_bytes()) return false;
    DeviceBuffer col(std::max<std::uint64_t>(total, 1) * 4), vid(ids ? std::max<std::uint64_t>(total, 1) * 2 : 0),
        val(ids ? 0 : std::max<std::uint64_t>(total, 1) * sizeof(dev::Zd));
    for (std::size_t b = 0; b < ops_.size(); ++b)
        dev::one_fill(ops_[b]->device_csr(), row_off_[b], tile_begin_[b], order_.get<std::uint32_t>(), place_.get<std::uint32_t>(),
                      ptr.get<std::uint64_t>(), col.get<std::uint32_t>(), vid.get<std::uint16_t>(), val.get<dev::Zd>(), st);
    QSA_HIP(hipGetLastError());
    one_ptr_ = std::move(ptr);
    one_len_ = std::move(len);
    col_ = std::move(col);
    vid_ = std::move(vid);
    val_ = std::move(val);
    row_ptr_.release();
    return true;
}

void BatchedLanczos::set_schedule(int kind) {
    sched_kind_ = 0;
    sched_d_.release();
    n_sched_ = 0;
    if (kind != 1 || tiles_.empty()) return;
    // Workgroup w runs on XCD w % 8: each XCD gets one eighth of the tiles, neighbours in order, so that
    // the columns of the rows in flight share its L2; with several runs of vectors, a block's tiles
    // take one run after the other. A rule and not a trial: in level order the two are within 2% of
    // each other (all steps, in order / in runs: N = 24, 4 samples 118.5 / 117.3 ms; continued fractions,
    // N = 26, 155.4 / 154.4; N = 22, 40 samples 229.3 / 233.8).
    constexpr std::size_t kXcd = 8;
    const std::size_t nt = tiles_.size(), chunks = static_cast<std::size_t>(dev::batch_chunks(R_));
    const std::size_t longest = (nt + kXcd - 1) / kXcd * chunks;
    std::vector<std::uint32_t> sched(longest * kXcd, ~0u);
    for (std::size_t x = 0; x < kXcd; ++x) {
        const std::size_t t0 = x * nt / kXcd, t1 = (x + 1) * nt / kXcd;
        std::size_t w = x;
        for (std::size_t a = t0; a < t1;) {
            std::size_t b = a;
            while (b < t1 && tiles_[b].block == tiles_[a].block) ++b;
            for (std::size_t c = 0; c < chunks; ++c)
                for (std::size_t t = a; t < b; ++t, w += kXcd) sched[w] = static_cast<std::uint32_t>(t * chunks + c);
            a = b;
        }
    }
    put(sched_d_, sched, engine_stream());
    n_sched_ = static_cast<std::uint32_t>(sched.size());
    sched_kind_ = 1;
}

dev::BatchView BatchedLanczos::view() const {
    dev::BatchView B;
    B.rows = rows_;
    B.n_blocks = static_cast<std::uint32_t>(ops_.size());
    B.n_tiles = static_cast<std::uint32_t>(tiles_.size());
    B.R = R_;
    B.tiles = tiles_d_.get<dev::Tile>();
    B.sched = sched_d_ ? sched_d_.get<std::uint32_t>() : nullptr;
    B.n_sched = n_sched_;
    B.tile_begin = tile_begin_d_.get<std::uint32_t>();
    if (one_) {
        B.one.ptr = one_ptr_.get<std::uint64_t>();
        B.one.len = one_len_.get<std::uint32_t>();
        B.one.col = col_.get<std::uint32_t>();
        B.one.vid = vid_.get<std::uint16_t>();
        B.one.val = val_.get<dev::Zd>();
    } else {
        B.row_ptr = row_ptr_.get<std::uint64_t>();
        B.col = col_.get<std::uint32_t>();
        B.val = val_.get<dev::Zd>();
        B.vid = vid_.get<std::uint16_t>();
    }
    if (dict_n_) {
        B.dict_re = dict_re_.get<double>();
        B.dict_im = dict_im_.get<double>();
        B.dict_n = dict_n_;
        B.dict_begin = dict_begin_.get<std::uint32_t>();
        B.dict_max = dict_max_;
    }
    B.step = step_d_.get<int>();
    B.active = active_d_.get<int>();
    B.steps = steps_d_.get<int>();
    B.cap = cap_d_.get<int>();
    B.fix = fix_.get<int>();
    return B;
}

void BatchedLanczos::set_start(const cplx* host) {
    if (place_) {   // through W, into the engine's row order
        copy_to_device(W_.get(), host, rows_ * R_ * sizeof(dev::Zd));
        dev::batch_reorder(W_.get<dev::Zd>(), rows_, R_, place_.get<std::uint32_t>(), V0_.get<dev::Zd>(), engine_stream());
        QSA_HIP(hipGetLastError());
    } else {
        copy_to_device(V0_.get(), host, rows_ * R_ * sizeof(dev::Zd));
    }
    normalize(nullptr);
}

void BatchedLanczos::clear_start() {
    dev::batch_fill_zero(V0_.get<dev::Zd>(), rows_ * R_, engine_stream());
    QSA_HIP(hipGetLastError());
}

void BatchedLanczos::place(int b, int s, const cplx* device_vector) {
    if (b < 0 || b >= n_blocks() || s < 0 || s >= R_) throw Error(kInvalid, "batched lanczos: no such pair");
    dev::batch_place(V0_.get<dev::Zd>(), R_, row_off_[b], s, reinterpret_cast<const dev::Zd*>(device_vector), dim(b),
                     place_.get<std::uint32_t>(), engine_stream());
    QSA_HIP(hipGetLastError());
}

void BatchedLanczos::normalize(std::vector<double>* norm2) {
    const hipStream_t st = engine_stream();
    dev::BatchView B = view();
    B.active = nullptr;
    const std::size_t pairs = ops_.size() * static_cast<std::size_t>(R_);
    DeviceBuffer n2(norm2 ? pairs * 8 : 0);
    dev::batch_normalize(B, V0_.get<dev::Zd>(), partial_.get<double>(), inv_b_.get<double>(),
                         norm2 ? n2.get<double>() : nullptr, st);
    QSA_HIP(hipGetLastError());
    QSA_HIP(hipStreamSynchronize(st));
    if (norm2) {
        norm2->resize(pairs);
        copy_to_host(norm2->data(), n2.get(), pairs * 8);
    }
}

void BatchedLanczos::sample_start(const std::vector<std::uint32_t>& seeds) {
    const std::size_t nb = ops_.size(), pairs = nb * static_cast<std::size_t>(R_);
    if (seeds.size() != pairs) throw Error(kInvalid, "batched lanczos: one seed per pair");
    const hipStream_t st = engine_stream();
    std::vector<std::uint64_t> dims(nb);
    for (std::size_t b = 0; b < nb; ++b) dims[b] = row_off_[b + 1] - row_off_[b];
    DeviceBuffer rb_d, dim_d, seed_d;
    put(rb_d, row_off_, st);
    put(dim_d, dims, st);
    put(seed_d, seeds, st);
    dev::sample_gauss(V0_.get<dev::Zd>(), R_, rb_d.get<std::uint64_t>(), dim_d.get<std::uint64_t>(),
                      seed_d.get<std::uint32_t>(), static_cast<std::uint32_t>(pairs), place_.get<std::uint32_t>(), st);
    QSA_HIP(hipGetLastError());
    normalize(nullptr);
}

void BatchedLanczos::run(int M, const std::vector<double>& breakdown_tol, bool local, bool use_graph,
                         std::vector<double>& alpha, std::vector<double>& beta, std::vector<int>& steps,
                         BatchedTimings& t, const std::vector<int>* live) {
    if (M < 1) throw Error(kInvalid, "batched lanczos: at least one step");
    if (breakdown_tol.size() != ops_.size()) throw Error(kInvalid, "batched lanczos: one breakdown tolerance per block");
    const std::size_t nb = ops_.size(), pairs = nb * static_cast<std::size_t>(R_);
    const std::size_t hist = static_cast<std::size_t>(M) * pairs;
    // Graph capture needs a stream other than the null one: a stream of its own when the engine
    // runs on the null stream (everything before it on the null stream is finished first).
    const hipStream_t outer = engine_stream();
    std::unique_ptr<OwnStream> own;
    if (!outer) {
        QSA_HIP(hipStreamSynchronize(nullptr));
        own = std::make_unique<OwnStream>();
    }
    const hipStream_t st = outer ? outer : own->s;
    StreamScope scope(st);
    std::vector<int> cap(nb), ones(pairs, 1), zeros(pairs, 0);
    if (live) {
        if (live->size() != pairs) throw Error(kInvalid, "batched lanczos: one live flag per pair");
        ones = *live;
    }
    for (std::size_t b = 0; b < nb; ++b) cap[b] = static_cast<int>(std::min<std::uint64_t>(M, dim(static_cast<int>(b))));
    put(cap_d_, cap, st);
    put(tol_d_, breakdown_tol, st);
    put(active_d_, ones, st);
    put(steps_d_, zeros, st);
    put(step_d_, std::vector<int>{0}, st);
    alpha_h_.reset(hist * 8);
    beta_h_.reset(hist * 8);
    dev::fill_zero(false, alpha_h_.get(), hist, st);
    dev::fill_zero(false, beta_h_.get(), hist, st);
    dev::fill_zero(false, cur_b_.get(), pairs, st);
    put(scale_, std::vector<double>(3 * pairs, 1.0), st);
    QSA_HIP(hipStreamSynchronize(st));

    const dev::BatchView B = view();
    dev::Zd* V[3] = {V1_.get<dev::Zd>(), V0_.get<dev::Zd>(), W_.get<dev::Zd>()};
    double* partial = partial_.get<double>();
    double* partial2 = partial2_.get<double>();
    double* ah = alpha_h_.get<double>();
    double* bh = beta_h_.get<double>();
    dev::Zd* ov = ov_.get<dev::Zd>();
    double* ca = cur_a_.get<double>();
    double* cb = cur_b_.get<double>();
    double* ib = inv_b_.get<double>();
    const double* tol = tol_d_.get<double>();
    const double thr = 1.49011611938476562e-08;   // sqrt(eps): LocalDGKS3's overlap threshold
    // The next vector is never scaled in place: each of the three buffers keeps a per-pair factor
    // (1 / beta of the step that wrote it; 1 for the normalised start) that every read applies, which
    // rounds as a scaling pass would (same results, one pass over the vectors fewer per step).
    const std::size_t np = pairs;
    double* S[3] = {scale_.get<double>(), scale_.get<double>() + np, scale_.get<double>() + 2 * np};
    auto step = [&](int phase) {
        dev::Zd* p = V[phase % 3];
        dev::Zd* c = V[(phase + 1) % 3];
        dev::Zd* w = V[(phase + 2) % 3];
        const double* sp = S[phase % 3];
        const double* sc = S[(phase + 1) % 3];
        double* sw = S[(phase + 2) % 3];
        dev::batch_spmv_fused(B, p, c, w, cb, partial, st, sp, sc);
        dev::batch_finish(B, 0, partial, ah, bh, ov, ca, cb, ib, tol, st);
        if (local) {
            // W -= alpha V with the local overlap and ||W||^2 in one pass; the correction pass then
            // touches only the pairs whose overlap asks for one (their norms are summed again)
            dev::batch_vec(B, 5, c, w, ca, nullptr, 0.0, partial, st, partial2, sc);
            dev::batch_finish(B, 1, partial, ah, bh, ov, ca, cb, ib, tol, st, thr);
            dev::batch_vec(B, 2, c, w, nullptr, ov, thr, partial, st, partial2, sc);
            dev::batch_finish(B, 2, partial2, ah, bh, ov, ca, cb, sw, tol, st);
        } else {
            dev::batch_vec(B, 4, c, w, ca, nullptr, 0.0, partial, st, nullptr, sc);
            dev::batch_finish(B, 2, partial, ah, bh, ov, ca, cb, sw, tol, st);
        }
        dev::batch_advance(B, st);
    };
    const int Mrun = *std::max_element(cap.begin(), cap.end());
    hipEvent_t e0, e1;
    QSA_HIP(hipEventCreate(&e0));
    QSA_HIP(hipEventCreate(&e1));
    hipGraphExec_t exec[3] = {nullptr, nullptr, nullptr};
    hipGraph_t graph[3] = {nullptr, nullptr, nullptr};
    auto cleanup = [&] {
        for (int i = 0; i < 3; ++i) {
            if (exec[i]) (void)hipGraphExecDestroy(exec[i]);
            if (graph[i]) (void)hipGraphDestroy(graph[i]);
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
    };
    try {
        if (use_graph) {
            for (int ph = 0; ph < 3 && ph < Mrun; ++ph) {
                {
                    const auto no_fence = capture_guard();   // no fence touches st while it captures
                    QSA_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
                    try {
                        step(ph);
                    } catch (...) {
                        hipGraph_t broken = nullptr;
                        (void)hipStreamEndCapture(st, &broken);
                        if (broken) (void)hipGraphDestroy(broken);
                        throw;
                    }
                    QSA_HIP(hipStreamEndCapture(st, &graph[ph]));
                }
                QSA_HIP(hipGraphInstantiate(&exec[ph], graph[ph], nullptr, nullptr, 0));
            }
        }
        QSA_HIP(hipEventRecord(e0, st));
        for (int j = 0; j < Mrun; ++j) {
            if (use_graph) QSA_HIP(hipGraphLaunch(exec[j % 3], st));
            else step(j % 3);
        }
        QSA_HIP(hipEventRecord(e1, st));
        QSA_HIP(hipGetLastError());
        QSA_HIP(hipEventSynchronize(e1));
        float ms = 0.0f;
        QSA_HIP(hipEventElapsedTime(&ms, e0, e1));
        t.steps_s += ms * 1e-3;
        t.steps += Mrun;
        t.graph = use_graph;
    } catch (...) {
        (void)hipStreamSynchronize(st);
        cleanup();
        throw;
    }
    cleanup();
    alpha.resize(hist);
    beta.resize(hist);
    steps.resize(pairs);
    copy_to_host(alpha.data(), ah, hist * 8);
    copy_to_host(beta.data(), bh, hist * 8);
    copy_to_host(steps.data(), steps_d_.get(), pairs * sizeof(int));
    for (int s : steps) t.applies += static_cast<std::uint64_t>(s);
    t.rows = rows_;
    t.nnz = nnz_;
}

void BatchedLanczos::run_kept(int M, const std::vector<double>& breakdown_tol, const std::vector<int>& full,
                              cplx* basis_c, std::vector<double>& alpha, std::vector<double>& beta,
                              std::vector<int>& steps, BatchedTimings& t, const std::vector<int>* live) {
    if (M < 1) throw Error(kInvalid, "batched lanczos: at least one step");
    const std::size_t nb = ops_.size(), pairs = nb * static_cast<std::size_t>(R_);
    if (breakdown_tol.size() != nb || full.size() != nb)
        throw Error(kInvalid, "batched lanczos: one breakdown tolerance and one reorthogonalisation flag per block");
    if (live && live->size() != pairs) throw Error(kInvalid, "batched lanczos: one live flag per pair");
    const hipStream_t st = engine_stream();
    const auto t0 = clock_t_::now();
    const std::size_t hist = static_cast<std::size_t>(M) * pairs;
    std::vector<int> cap(nb), zeros(pairs, 0);
    for (std::size_t b = 0; b < nb; ++b) cap[b] = static_cast<int>(std::min<std::uint64_t>(M, dim(static_cast<int>(b))));
    put(cap_d_, cap, st);
    put(tol_d_, breakdown_tol, st);
    put(active_d_, live ? *live : std::vector<int>(pairs, 1), st);
    put(steps_d_, zeros, st);
    put(step_d_, std::vector<int>{0}, st);
    put(fix_, zeros, st);
    DeviceBuffer full_d;
    put(full_d, full, st);
    const bool any_full = std::any_of(full.begin(), full.end(), [](int f) { return f != 0; });
    DeviceBuffer coef(any_full ? nb * static_cast<std::size_t>(M + 1) * R_ * sizeof(dev::Zd) : 8);
    DeviceBuffer gs2(pairs * sizeof(int));   // per pair: the second Gram-Schmidt pass of this step
    alpha_h_.reset(hist * 8);
    beta_h_.reset(hist * 8);
    dev::fill_zero(false, alpha_h_.get(), hist, st);
    dev::fill_zero(false, beta_h_.get(), hist, st);
    dev::fill_zero(false, cur_b_.get(), pairs, st);
    const std::uint64_t layer = rows_ * static_cast<std::uint64_t>(R_);
    auto* basis = reinterpret_cast<dev::Zd*>(basis_c);
    QSA_HIP(hipMemcpyAsync(basis, V0_.get(), layer * sizeof(dev::Zd), hipMemcpyDeviceToDevice, st));
    const dev::BatchView B = view();
    double* partial = partial_.get<double>();
    double* partial2 = partial2_.get<double>();
    double* ah = alpha_h_.get<double>();
    double* bh = beta_h_.get<double>();
    dev::Zd* ov = ov_.get<dev::Zd>();
    double* ca = cur_a_.get<double>();
    double* cb = cur_b_.get<double>();
    double* ib = inv_b_.get<double>();
    const double* tol = tol_d_.get<double>();
    const double thr = 1.49011611938476562e-08;   // sqrt(eps): LocalDGKS3's overlap threshold
    const int Mrun = *std::max_element(cap.begin(), cap.end());
    for (int j = 0; j < Mrun; ++j) {
        const dev::Zd* Vp = basis + static_cast<std::uint64_t>(j > 0 ? j - 1 : 0) * layer;
        const dev::Zd* Vc = basis + static_cast<std::uint64_t>(j) * layer;
        dev::Zd* W = basis + static_cast<std::uint64_t>(j + 1) * layer;
        // the kept layers are stored normalised (the overlaps read them later), so only the first
        // recurrence pass is fused here, not the deferred scaling of run()
        dev::batch_spmv_fused(B, Vp, Vc, W, cb, partial, st);
        dev::batch_finish(B, 0, partial, ah, bh, ov, ca, cb, ib, tol, st);
        dev::batch_vec(B, 5, Vc, W, ca, nullptr, 0.0, partial, st, partial2);
        dev::batch_finish(B, 1, partial, ah, bh, ov, ca, cb, ib, tol, st, thr);
        dev::batch_vec(B, 2, Vc, W, nullptr, ov, thr, partial, st, partial2);
        if (any_full) {
            // CGS2 against every kept layer; the second pass only where the first removed more than
            // 1 - kappa of ||W|| (DGKS, as the reference's FullCGS2 gates it): partial2 holds the
            // norms before the first pass, partial those after it
            dev::batch_gram_schmidt(B, basis, layer, j + 1, M + 1, W, full_d.get<int>(), coef.get<dev::Zd>(), st);
            dev::batch_norm_partial(B, W, partial, st);
            dev::batch_dgks_gate(B, partial2, partial, full_d.get<int>(), kDgksKappa, gs2.get<int>(), st);
            dev::batch_gram_schmidt(B, basis, layer, j + 1, M + 1, W, full_d.get<int>(), coef.get<dev::Zd>(), st,
                                    gs2.get<int>());
            dev::batch_norm_partial(B, W, partial2, st);
        }
        dev::batch_finish(B, 2, partial2, ah, bh, ov, ca, cb, ib, tol, st);
        dev::batch_vec(B, 3, nullptr, W, ib, nullptr, 0.0, partial, st);
        dev::batch_advance(B, st);
    }
    QSA_HIP(hipGetLastError());
    QSA_HIP(hipStreamSynchronize(st));
    t.steps_s += secs(t0, clock_t_::now());
    t.steps += Mrun;
    alpha.resize(hist);
    beta.resize(hist);
    steps.resize(pairs);
    copy_to_host(alpha.data(), ah, hist * 8);
    copy_to_host(beta.data(), bh, hist * 8);
    copy_to_host(steps.data(), steps_d_.get(), pairs * sizeof(int));
    for (int s : steps) t.applies += static_cast<std::uint64_t>(s);
    t.rows = rows_;
    t.nnz = nnz_;
}

std::vector<Curves> batched_ftlm(const std::vector<std::shared_ptr<const SectorOperator>>& blocks,
                                 const BatchedFtlmOptions& o, BatchedTimings& t) {
    const auto t_all = clock_t_::now();
    const std::size_t nb = blocks.size();
    if (nb == 0) return {};
    if (o.samples < 1 || o.krylov < 1 || o.betas.empty()) throw Error(kInvalid, "ftlm: bad sizes");
    if (o.block_seeds.size() != nb || o.breakdown_tol.size() != nb)
        throw Error(kInvalid, "ftlm: one seed and one breakdown tolerance per block");
    const auto t_pack = clock_t_::now();
    const int R = std::min(o.samples, dev::kBatchMaxR);
    BatchedLanczos L(blocks, R);
    t.pack_s += secs(t_pack, clock_t_::now());
    t.schedule = L.schedule();
    t.order_s = L.order_seconds();
    std::vector<RitzPool> pools(nb);
    std::vector<double> alpha, beta;
    std::vector<int> steps;
    for (int s0 = 0; s0 < o.samples; s0 += R) {
        const int Rc = std::min(R, o.samples - s0);
        // Samples of this round: pair (block, s) starts from sample s0 + s of the block's stream (the
        // 32-bit Mersenne Twister seed of sample_engine), drawn on the device; the unused columns of
        // a short last round repeat its first sample (never read back).
        const auto t_seed = clock_t_::now();
        std::vector<std::uint32_t> seeds(nb * static_cast<std::size_t>(R));
        for (std::size_t b = 0; b < nb; ++b)
            for (int s = 0; s < R; ++s) {
                const int sample = s0 + (s < Rc ? s : 0);
                seeds[b * R + s] = static_cast<std::uint32_t>(
                    splitmix_seed(o.block_seeds[b], static_cast<std::uint64_t>(sample)));
            }
        L.sample_start(seeds);
        t.seed_s += secs(t_seed, clock_t_::now());
        L.run(o.krylov, o.breakdown_tol, /*local=*/true, o.use_graph, alpha, beta, steps, t);
        const auto t_post = clock_t_::now();
        const std::size_t pairs = nb * static_cast<std::size_t>(R);
        std::vector<std::vector<double>> ritz(nb * static_cast<std::size_t>(Rc)), weight(ritz.size());
        parallel_for(nb * static_cast<std::size_t>(Rc), [&](std::size_t i) {
            const std::size_t b = i / Rc, s = i % Rc;
            const std::size_t pr = b * R + s;
            const int m = steps[pr];
            std::vector<double> a(static_cast<std::size_t>(m)), bn(static_cast<std::size_t>(m));
            for (int j = 0; j < m; ++j) {
                a[j] = alpha[static_cast<std::size_t>(j) * pairs + pr];
                bn[j] = beta[static_cast<std::size_t>(j) * pairs + pr];
            }
            tridiag_weights(a.data(), bn.data(), static_cast<std::size_t>(m), ritz[i], weight[i]);
        });
        for (std::size_t b = 0; b < nb; ++b)   // samples pooled in sample order
            for (int s = 0; s < Rc; ++s)
                if (!ritz[b * Rc + s].empty()) pools[b].add_sample(ritz[b * Rc + s], weight[b * Rc + s]);
        t.post_s += secs(t_post, clock_t_::now());
    }
    std::vector<Curves> out(nb);
    for (std::size_t b = 0; b < nb; ++b) out[b] = pools[b].curves(L.dim(static_cast<int>(b)), o.betas);
    t.total_s += secs(t_all, clock_t_::now());
    return out;
}

}  // namespace qsa
