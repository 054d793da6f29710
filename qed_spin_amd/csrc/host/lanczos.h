// The Lanczos recurrence on device vectors: the reference's single Lanczos algorithm
// (include/ed/krylov/lanczos.h:266-576) with its three reorthogonalisation policies, breakdown rule and
// convergence hook, on the HIP backend. The kept basis is one contiguous column block in HBM, so a full
// Gram-Schmidt pass is one tall-skinny dot kernel and one update kernel over it (each streaming the
// block once), with the norms before and after folded in.
//
// The scalars stay on the device: a step's coefficients, its norm, the gate of the second Gram-Schmidt
// pass and of the local correction are read there by the kernels that need them, so steps are enqueued
// one behind the other, at most eight ahead of the device (StepsInFlight), and the host looks at alpha
// and beta a batch of steps at a time (a few with a convergence check). What lies past the step that
// ends a run (breakdown, convergence) is not returned. (200 steps with full reorthogonalisation on 9252
// states: 190 us a step when the host waited five times a step for a scalar and the Gram-Schmidt
// kernels left the card idle, 49 to 60 us so; 100 on 2.6 million, without the basis column's copy: 832
// -> 713 us.)
#pragma once

#include <chrono>
#include <cmath>
#include <functional>
#include <stdexcept>
#include <type_traits>
#include <utility>
#include <vector>

#include "backend.h"

namespace qsa {

enum class Reorth : int { None = 0, FullCGS2 = 1, LocalDGKS3 = 2 };

/// DGKS "twice is enough": a second pass only when the first removed more than 1 - 1/sqrt 2 of ||w||.
inline constexpr double kDgksKappa = 0.7071067811865476;

template <class Scalar> struct LanczosOptions {
    std::size_t max_iter = 100;
    double breakdown_tol = 1e-300;
    Reorth reorth = Reorth::FullCGS2;
    bool keep_basis = true;
    std::function<bool(const std::vector<double>&, const std::vector<double>&)> convergence_check;
    std::size_t convergence_check_interval = 0;
    double local_ortho_threshold = 1.49011611938476562e-08;
    bool random_start = false;   ///< a start that lies in no small invariant subspace: no early look
};

/// Seconds of a run: apply_s, reorth_s and vector_s from events around the phases of every eighth of its
/// steps or so, scaled to all of them.
struct LanczosTimings {
    double apply_s = 0.0, reorth_s = 0.0, vector_s = 0.0, total_s = 0.0;
    std::size_t applies = 0;
};

template <class Scalar> struct LanczosResult {
    std::vector<double> alpha;   ///< iters
    std::vector<double> beta;    ///< iters + 1, beta[0] = 0
    std::size_t iters = 0;
    LanczosTimings timings;
};

/// A matvec that can also run a step's first pass fused (first_pass(v, v_prev, beta, w, alpha, scratch):
/// w = H v - *beta v_prev, *alpha = <v, w> on the device, false when it cannot).
template <class M, class S, class = void> struct HasFirstPass : std::false_type {};
template <class M, class S>
struct HasFirstPass<M, S,
                    std::void_t<decltype(std::declval<const M&>().first_pass(
                        static_cast<const S*>(nullptr), static_cast<const S*>(nullptr), static_cast<const double*>(nullptr),
                        static_cast<S*>(nullptr), static_cast<dev::Zd*>(nullptr), std::declval<DeviceBuffer&>()))>>
    : std::true_type {};

namespace detail {

/// Events around the phases of the timed steps; read once the stream has passed them.
class StepClock {
public:
    explicit StepClock(std::size_t steps) : every_(std::max<std::size_t>(1, steps / 8)) {}
    ~StepClock() {
        for (auto& e : ev_) (void)hipEventDestroy(e);
    }
    StepClock(const StepClock&) = delete;
    StepClock& operator=(const StepClock&) = delete;
    void mark(std::size_t step) {
        if (step % every_) return;
        hipEvent_t e;
        QSA_HIP(hipEventCreate(&e));
        ev_.push_back(e);
        QSA_HIP(hipEventRecord(e, engine_stream()));
    }
    /// Four marks a timed step: before and after the apply, after the vector work, at its end.
    void read(std::size_t steps, LanczosTimings& t) const {
        double part[3] = {0.0, 0.0, 0.0};
        const std::size_t timed = ev_.size() / 4;
        if (!timed) return;
        for (std::size_t q = 0; q < timed; ++q)
            for (std::size_t k = 0; k < 3; ++k) {
                float ms = 0.0f;
                QSA_HIP(hipEventElapsedTime(&ms, ev_[4 * q + k], ev_[4 * q + k + 1]));
                part[k] += ms * 1e-3;
            }
        const double f = static_cast<double>(steps) / static_cast<double>(timed);
        t.apply_s = part[0] * f;
        t.vector_s = part[1] * f;
        t.reorth_s = part[2] * f;
    }

private:
    std::size_t every_;
    std::vector<hipEvent_t> ev_;
};

/// Bounds the steps that lie enqueued and not yet run: every `stride` steps an event, and a wait for the
/// event before it (two in turn), so at most 2 stride steps lie there: the device always has the next
/// ones, while a release on another thread, which waits for all that every engine stream holds
/// (fence_engine_streams), and the short kernels of streams that share a hardware queue wait for a few
/// steps and not for a run. (100 mixed requests on 8 slots, mean latency: 4.73 s without a bound, 4.27
/// with; a walk of 64 streamed blocks after them in one process 12.1 and 7.8 s.) The stride is what costs
/// nothing: an event a step from 2^19 rows on took an estimate of 716,000 rows from 4.6 to 4.8 ms, every
/// other step 4.65; from 2^22 on a step is long beside its event.
class StepsInFlight {
public:
    explicit StepsInFlight(std::size_t n)
        : stride_(n < (std::size_t{1} << 19) ? 4 : n < (std::size_t{1} << 22) ? 2 : 1) {}
    ~StepsInFlight() {
        for (auto& e : ev_)
            if (e) (void)hipEventDestroy(e);
    }
    StepsInFlight(const StepsInFlight&) = delete;
    StepsInFlight& operator=(const StepsInFlight&) = delete;
    /// A step has been enqueued.
    void step() {
        if (++count_ % stride_) return;
        const std::size_t s = count_ / stride_ % 2;
        if (!ev_[s]) QSA_HIP(hipEventCreateWithFlags(&ev_[s], hipEventDisableTiming));
        QSA_HIP(hipEventRecord(ev_[s], engine_stream()));
        if (ev_[s ^ 1]) QSA_HIP(hipEventSynchronize(ev_[s ^ 1]));
    }

private:
    std::size_t stride_, count_ = 0;
    hipEvent_t ev_[2] = {nullptr, nullptr};
};

}  // namespace detail

template <class Scalar, class Matvec>
LanczosResult<Scalar> lanczos_run(const HipBackend<Scalar>& be, Matvec&& matvec, std::size_t n, const Scalar* v0,
                                  const LanczosOptions<Scalar>& o) {
    using clock = std::chrono::steady_clock;
    const auto t_start = clock::now();
    LanczosResult<Scalar> R;
    const bool cgs = o.reorth == Reorth::FullCGS2;
    if (cgs && !o.keep_basis) throw Error(kInvalid, "lanczos: FullCGS2 requires keep_basis");
    if (o.max_iter == 0) return R;
    const std::size_t cap = std::min<std::size_t>(o.max_iter, n);
    // v_j: column j of the kept basis, or three vectors in turn
    typename HipBackend<Scalar>::UniqueVec block(be.allocate(n * (cgs ? cap : 3)));
    auto col = [&](std::size_t j) { return block.get() + (cgs ? j : j % 3) * n; };
    typename HipBackend<Scalar>::UniqueVec work;   // w of a kept-basis run (else the vector after next)
    if (cgs) work.reset(be.allocate(n));
    R.beta.push_back(0.0);
    be.copy(v0, col(0), n);
    const double n0 = be.nrm2(col(0), n);
    if (!(n0 > 0.0)) throw Error(kInvalid, "lanczos: initial vector has non-positive norm");
    be.scale(Scalar(1.0 / n0), col(0), n);
    // alpha_j (complex) and beta_{j+1} of each step, side by side for one copy; the local overlap; the SELL
    // first pass's partial sums
    struct Step {
        dev::Zd alpha;
        double beta, unused;
    };
    DeviceBuffer scalars((cap + 1) * sizeof(Step)), sums;
    Step* const step = scalars.get<Step>();
    dev::Zd* const overlap = &step[cap].alpha;
    const bool check = o.convergence_check && o.convergence_check_interval > 0;
    // steps enqueued before the host looks: without a check enough to hide the look (some 60 us), fewer at
    // first where the run may break down early; with one a few, the smaller the costlier a step that
    // turns out not to be needed
    const std::size_t look = check ? (n < (std::size_t{1} << 16) ? 8 : n < (std::size_t{1} << 19) ? 3 : 1)
                                   : (n < (std::size_t{1} << 19) ? 64 : 16);
    const std::size_t first = check || o.random_start ? look : look / 4;
    detail::StepClock phases(cap);
    detail::StepsInFlight flight(n);
    std::vector<Step> host(cap);
    std::size_t timed_steps = 0;
    bool done = false;
    for (std::size_t j0 = 0; j0 < cap && !done;) {
        const std::size_t j1 = std::min(cap, j0 + (j0 == 0 ? first : look));
        for (std::size_t j = j0; j < j1; ++j) {
            const Scalar* v = col(j);
            const Scalar* prev = j > 0 ? col(j - 1) : nullptr;
            const double* beta = j > 0 ? &step[j - 1].beta : nullptr;
            dev::Zd* const alpha = &step[j].alpha;
            double* const norm = &step[j].beta;
            Scalar* w = cgs ? work.get() : col(j + 1);
            phases.mark(j);
            // alpha_j = <v_j, H v_j - beta_j v_{j-1}>: in the apply's epilogue when the matvec offers it
            bool fused = false;
            if constexpr (HasFirstPass<std::decay_t<Matvec>, Scalar>::value)
                fused = matvec.first_pass(v, prev, beta, w, alpha, sums);
            if (!fused) matvec(v, w);
            phases.mark(j);
            if (!fused) {
                if (prev) be.axpy_dot(dev::minus(beta), prev, w, v, n, alpha);
                else be.dot(v, w, n, alpha);
            }
            const dev::Coef by_alpha = dev::minus(&alpha->re);
            if (cgs) {
                be.axpy(by_alpha, v, w, n);
                phases.mark(j);
                be.cgs_gated(block.get(), n, j + 1, w, n, kDgksKappa, norm);
            } else if (o.reorth == Reorth::LocalDGKS3 && j > 0) {
                be.axpy_dot(by_alpha, v, w, v, n, overlap);
                phases.mark(j);
                be.axpy_nrm2(dev::minus_above(overlap, o.local_ortho_threshold), v, w, n, norm);
            } else {
                be.axpy_nrm2(by_alpha, v, w, n, norm);
                phases.mark(j);
            }
            phases.mark(j);
            if (j + 1 < cap) be.scale_by(w, norm, col(j + 1), n);
            flight.step();
        }
        QSA_HIP(hipGetLastError());
        copy_to_host(host.data() + j0, step + j0, (j1 - j0) * sizeof(Step));
        timed_steps = j1;
        for (std::size_t j = j0; j < j1 && !done; ++j) {
            R.alpha.push_back(host[j].alpha.re);
            R.beta.push_back(host[j].beta);
            if (host[j].beta < o.breakdown_tol) done = true;
            else if (check && (j + 1) % o.convergence_check_interval == 0) done = o.convergence_check(R.alpha, R.beta);
        }
        j0 = j1;
    }
    R.iters = R.alpha.size();
    R.timings.applies = R.iters;
    phases.read(timed_steps, R.timings);
    R.timings.total_s = std::chrono::duration<double>(clock::now() - t_start).count();
    return R;
}

}  // namespace qsa
