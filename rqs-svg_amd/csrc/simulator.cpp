// Host core of libqcs.so.
//
// Semantics follow the reference simulator core (src/qcs.cu:1685-2899):
//  - lazy measurement: measured, non-targeted qubits become implicit controls of their
//    measured value; a contradicting explicit control skips the gate; targets leave the
//    measured lists (src/qcs.cu:2161-2204, 2480-2484, 2679-2703);
//  - measurement: cached result, {p0,p1} over the subspace consistent with earlier
//    measurements, r = std::uniform_real_distribution<double>(0, p0+p1)(std::mt19937_64),
//    result = p0 < r, collapse without renormalisation unless enabled
//    (src/qcs.cu:2545-2677);
//  - mapping perm_p2l / perm_l2p and the swap-in of "global" targets
//    (src/qcs.cu:1860-1885, 2206-2332) -- here the data movement is an in-HBM qubit swap;
//  - capacity check n <= floor(log2(free / 16)) (src/qcs.cu:1895-1908), no swap buffer.
// What differs by design: the operand descriptor is a kernel argument (no per-gate
// __constant__ copy), reductions use the canonical order documented in qcs_ext.h, and all
// work is on one stream owned by the simulator.
#include "simulator.hpp"

#include "fused.hpp"
#include "pass.hpp"

#include <algorithm>
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <functional>
#include <mutex>
#include <new>
#include <stdexcept>
#include <thread>

#include <qcs_ext.h>

namespace qcore
{
    namespace
    {
        std::string fmt(const char *f, int a, int b = 0)
        {
            char buf[256];
            snprintf(buf, sizeof buf, f, a, b);
            return buf;
        }

        bool contains(const std::vector<int> &v, int x) { return std::find(v.begin(), v.end(), x) != v.end(); }

        qsv::c128 to_c(cd z) { return qsv::c128{z.real(), z.imag()}; }

        qsv::Subspace make_sub(std::vector<int> ops, uint64_t set_bits)
        {
            std::sort(ops.begin(), ops.end());
            qsv::Subspace s{};
            s.set_bits = set_bits;
            s.nops = (int)ops.size();
            if (s.nops > qsv::kMaxQubits)
                throw std::runtime_error("too many operands");
            for (int k = 0; k < s.nops; ++k)
                s.ops[k] = ops[k];
            return s;
        }
    } // namespace

    // Runs f on the state pointer of the current precision (complex128 or complex64).
    template <class F>
    void Simulator::with_state(F &&f)
    {
        if (fused_ && fused_->f64())
            f(fused_->state128());
        else if (fused_)
            f(fused_->state());
        else
            f(state_);
    }

    Simulator::Simulator()
    {
        qsv::check(hipGetDevice(&device_), "hipGetDevice");
        qsv::check(hipStreamCreate(&stream_), "hipStreamCreate");
        qsv::check(hipHostMalloc((void **)&pinned_, kPinnedResults * sizeof(double) + kRing, hipHostMallocDefault), "hipHostMalloc");
        std::random_device rd; // src/qcs.cu:1845-1852
        seed_ = rd();
        engine_.seed(seed_);
    }

    Simulator::~Simulator()
    {
        try
        {
            free_memory();
        }
        catch (...)
        {
        }
        for (auto e : events_)
            (void)hipEventDestroy(e);
        for (auto &r : recs_)
        {
            (void)hipEventDestroy(r.a);
            (void)hipEventDestroy(r.b);
        }
        for (auto e : free_events_)
            (void)hipEventDestroy(e);
        for (auto e : stage_events_)
            (void)hipEventDestroy(e);
        if (open_a_)
            (void)hipEventDestroy(open_a_);
        for (auto e : ring_read_)
            if (e)
                (void)hipEventDestroy(e);
        for (auto e : shots_there_)
            if (e)
                (void)hipEventDestroy(e);
        if (pinned_)
            (void)hipHostFree(pinned_);
        if (stream_)
            (void)hipStreamDestroy(stream_);
    }

    void Simulator::need_alloc() const
    {
        if (!allocated_)
            throw std::runtime_error("allocate_memory has not been called");
    }

    void Simulator::set_seed(uint64_t s)
    {
        seed_ = s;
        engine_.seed(s);
    }

    void Simulator::set_precision(int mode, int k)
    {
        if (allocated_)
            throw std::runtime_error("set_precision must be called before allocate_memory");
        if (mode < 0 || mode > 3)
            throw std::runtime_error("precision mode must be 0 (complex128 per gate), 1 (complex64 fused, FP32), 2 (complex128 fused) or 3 (complex64 fused, BF16x3)");
        if (mode != 0 && (k < 1 || k > 5))
            throw std::runtime_error("fused block size must be in [1, 5]");
        precision_ = mode;
        block_qubits_ = k;
    }

    void Simulator::set_stage_bits(int m)
    {
        if (m != 0 && (m < 11 || m > 14))
            throw std::runtime_error("stage tile bits must be 0 (one sweep per block), 11, 12, 13 or 14");
        stage_bits_ = m;
        stages_asked_ = true;
        if (fused_)
        {
            fused_->set_stage_bits(m);
            fused_->set_passes(false);
        }
    }

    void Simulator::set_stage_stream(int on)
    {
        if (on != 0 && on != 1)
            throw std::runtime_error("stage stream setting must be 0 or 1");
        stage_stream_ = on;
        if (fused_)
            fused_->set_stage_stream(on != 0);
    }

    void Simulator::set_planner_check(int on)
    {
        if (on != 0 && on != 1)
            throw std::runtime_error("planner check setting must be 0 or 1");
        flush();
        planner_check_ = on;
        if (fused_)
            fused_->set_check(on != 0);
    }

    void Simulator::reinitialize_mapping()
    { // src/qcs.cu:1860-1885
        state_changed();
        // the data stays where it is, so the measured qubits' zeros are not at their new places
        if (!m0_.empty() || !m1_.empty())
            consistent_ = false;
        p2l_.assign(n_, 0);
        l2p_.assign(n_, 0);
        if (initial_p2l.empty())
        {
            for (int q = 0; q < n_; ++q)
                p2l_[q] = l2p_[q] = q;
        }
        else
        {
            if ((int)initial_p2l.size() != n_)
                throw std::runtime_error(fmt("mapping size %d does not match num_qubits %d", (int)initial_p2l.size(), n_));
            p2l_ = initial_p2l;
            for (int q = 0; q < n_; ++q)
                l2p_[p2l_[q]] = q;
        }
    }

    void Simulator::allocate()
    { // src/qcs.cu:1887-1998
        if (allocated_)
            throw std::runtime_error(fmt("num_qubits is already set %d > 0", n_));
        int nq = num_qubits_cfg;
        if (nq < 1 || nq > qsv::kMaxQubits)
            throw std::runtime_error(fmt("num_qubits %d out of range [1, %d]", nq, qsv::kMaxQubits));
        size_t free_b = 0, total_b = 0;
        qsv::check(hipMemGetInfo(&free_b, &total_b), "hipMemGetInfo");
        const uint64_t S = c64_state() ? 8 : 16;
        int cap = 0;
        while ((uint64_t(1) << (cap + 1)) <= free_b / S)
            ++cap;
        if (nq > cap)
            throw std::runtime_error(fmt("num_qubits(%d) > max_num_qubits_local_device(%d)", nq, cap));
        n_ = nq;
        n_local_ = nq;
        reinitialize_mapping();
        const uint64_t count = uint64_t(1) << n_;
        if (precision_ == 0)
        {
            qsv::check(hipMalloc((void **)&state_, count * sizeof(qsv::c128)), "hipMalloc state");
        }
        else
        {
            fused_ = new FusedEngine(*this, block_qubits_, precision_);
            fused_->set_stage_bits(stage_bits_);
            fused_->set_passes(!stages_asked_);
            fused_->set_stage_stream(stage_stream_ != 0);
            fused_->set_check(planner_check_ != 0);
        }
        work_len_ = std::max(qsv::reduce_workspace(count), qsv::expz_workspace(count)) + 16;
        // the reductions' workspace, and behind it the device's copies of pass programs
        work_len_ = (work_len_ + 31) & ~uint64_t(31);
        qsv::check(hipMalloc((void **)&work_, work_len_ * sizeof(double) + kRing), "hipMalloc workspace");
        allocated_ = true;
        set_zero_state();
    }

    void Simulator::free_memory()
    {
        if (fused_)
        {
            delete fused_;
            fused_ = nullptr;
        }
        if (state_)
        {
            (void)hipStreamSynchronize(stream_);
            (void)hipFree(state_);
            state_ = nullptr;
        }
        if (work_)
        {
            (void)hipFree(work_);
            work_ = nullptr;
        }
        if (shots_)
            (void)hipHostFree(shots_);
        shots_ = nullptr;
        shots_cap_ = 0;
        for (auto p : levels_)
            (void)hipFree(p);
        levels_.clear();
        if (stage_)
            (void)hipHostFree(stage_);
        if (stage_dev_)
            (void)hipFree(stage_dev_);
        stage_ = stage_dev_ = nullptr;
        allocated_ = false;
        n_ = 0;
        state_changed();
    }

    void Simulator::set_zero_state()
    { // src/qcs.cu:2065-2079
        need_alloc();
        state_changed();
        clear_measurement_state();
        if (fused_)
            fused_->drop(); // queued gates act on a state that is being overwritten
        prof_begin(QCS_EXT_K_INIT, (c64_state() ? 8.0 : 16.0) * (1ull << n_));
        with_state([&](auto *st) { qsv::launch_fill_basis(stream_, st, uint64_t(1) << n_, 0); });
        prof_end();
    }

    void Simulator::set_sequential_state()
    { // src/qcs.cu:71-76, 2025-2043
        need_alloc();
        state_changed();
        clear_measurement_state();
        if (fused_)
            fused_->drop();
        with_state([&](auto *st) { qsv::launch_fill_sequential(stream_, st, uint64_t(1) << n_); });
    }

    void Simulator::set_flat_state()
    { // src/qcs.cu:78-82, 2045-2063
        need_alloc();
        state_changed();
        clear_measurement_state();
        if (fused_)
            fused_->drop();
        with_state([&](auto *st) { qsv::launch_fill_flat(stream_, st, uint64_t(1) << n_); });
    }

    void Simulator::set_entangled_state()
    { // src/qcs.cu:2081-2095 with one rank: amp[0] = 1, nothing else written
        need_alloc();
        state_changed();
        clear_measurement_state();
        flush(); // amp[0] = 1 on top of the current state
        with_state([&](auto *st) { qsv::launch_set_one(stream_, st, 0); });
    }

    void Simulator::set_random_state()
    { // src/qcs.cu:2097-2119: curand normals there; this build's own generator here.
      // The measured lists are kept, as in the reference.
        need_alloc();
        state_changed();
        if (fused_)
            fused_->drop();
        consistent_ = m0_.empty() && m1_.empty();
        with_state([&](auto *st) { qsv::launch_fill_random(stream_, st, uint64_t(1) << n_, seed_); });
    }

    void Simulator::clear_measurement_state()
    {
        m0_.clear();
        m1_.clear();
        consistent_ = true;
    }

    void Simulator::check_operands(const std::vector<int> &t, const std::vector<int> &ng, const std::vector<int> &ps) const
    {
        std::vector<int> all;
        all.insert(all.end(), t.begin(), t.end());
        all.insert(all.end(), ng.begin(), ng.end());
        all.insert(all.end(), ps.begin(), ps.end());
        for (int q : all)
            if (q < 0 || q >= n_)
                throw std::runtime_error(fmt("qubit %d out of range [0, %d)", q, n_));
        std::sort(all.begin(), all.end());
        if (std::adjacent_find(all.begin(), all.end()) != all.end())
            throw std::runtime_error("a qubit appears more than once among targets and controls");
    }

    // The in-HBM replacement of the reference's NCCL global<->local exchange for one pair:
    // swap the data of physical qubits a and b with the SWAP pair kernel (it reads and writes
    // only the half of the state the swap changes).  complex128 per-gate state only.
    void Simulator::swap_physical(int a, int b)
    {
        if (a == b)
            return;
        qsv::Subspace sub = make_sub({a, b}, 0);
        qsv::PairOp op{};
        op.offA = uint64_t(1) << a;
        op.offB = uint64_t(1) << b;
        op.m[0] = {0, 0};
        op.m[1] = {1, 0};
        op.m[2] = {1, 0};
        op.m[3] = {0, 0};
        prof_begin(QCS_EXT_K_PERMUTE, 2.0 * 16.0 * (1ull << (n_ - 1)));
        qsv::launch_pair(stream_, state_, n_, sub, op);
        prof_end();
    }

    // The mapping after the data of physical qubit q moved to physical qubit dst[q].
    void Simulator::remap_physical(const std::vector<int> &dst)
    {
        std::vector<int> p2l(n_);
        for (int q = 0; q < n_; ++q)
            p2l[dst[q]] = p2l_[q];
        p2l_ = p2l;
        for (int q = 0; q < n_; ++q)
            l2p_[p2l_[q]] = q;
    }

    // Moves the data of every physical qubit q to physical qubit dst[q]: one sweep of the
    // LDS-tiled permutation kernel per pass (a pass moves up to 6 qubits above the low run
    // that every tile keeps contiguous: 64 complex128 or 128 complex64 amplitudes, 1 KiB),
    // then the mapping follows the data.
    void Simulator::move_physical(const std::vector<int> &dst)
    {
        bool any = false;
        for (int q = 0; q < n_; ++q)
            any = any || dst[q] != q;
        if (!any)
            return;
        flush();
        state_changed();
        const int tb = c64_state() ? qsv::permute_tile_bits<qsv::c64>() : qsv::permute_tile_bits<qsv::c128>();
        const int low = c64_state() ? 7 : 6;
        const auto passes = n_ <= tb ? std::vector<std::vector<int>>{dst} : qsv::plan_permute_passes(dst, tb - low, low);
        const double S = c64_state() ? 8.0 : 16.0;
        for (const auto &p : passes)
        {
            prof_begin(QCS_EXT_K_PERMUTE, 2.0 * S * (1ull << n_));
            with_state([&](auto *st) { qsv::launch_permute(stream_, st, n_, p); });
            prof_end();
        }
        remap_physical(dst);
    }

    void Simulator::ensure_local(std::vector<int> &tphys)
    { // src/qcs.cu:2206-2332 (bookkeeping) with the data move done in HBM
        // Slot for the i-th global target: n_local-1-i as in the reference, except that
        // slots holding a local target of the same gate are skipped (the reference would move
        // that target away and apply the gate to the wrong qubit).
        std::vector<int> glob, loc;
        int next_slot = n_local_ - 1;
        for (auto &t : tphys)
        {
            if (t >= n_local_)
            {
                while (std::find(tphys.begin(), tphys.end(), next_slot) != tphys.end())
                    --next_slot;
                glob.push_back(t);
                loc.push_back(next_slot);
                t = next_slot--;
            }
        }
        if (glob.empty())
            return;
        std::vector<int> dst(n_);
        for (int q = 0; q < n_; ++q)
            dst[q] = q;
        for (size_t i = 0; i < glob.size(); ++i)
        {
            dst[glob[i]] = loc[i];
            dst[loc[i]] = glob[i];
        }
        // one swap of two qubits at 3 or above: the SWAP kernel moves half the state,
        // coalesced; anything else takes one permutation sweep for all the swaps
        if (!fused_ && glob.size() == 1 && std::min(glob[0], loc[0]) >= 3)
        {
            state_changed();
            swap_physical(glob[0], loc[0]);
            remap_physical(dst);
        }
        else
        {
            move_physical(dst);
        }
    }

    void Simulator::operate(const GateSpec &g, std::vector<int> targets, std::vector<int> neg, std::vector<int> pos)
    {
        need_alloc();
        state_changed();
        if ((int)targets.size() != g.ntargets)
            throw std::runtime_error(fmt("gate needs %d target qubit(s), %d given", g.ntargets, (int)targets.size()));
        check_operands(targets, neg, pos);
        // lazy measurement (src/qcs.cu:2161-2204)
        std::vector<int> *ctrl[2] = {&neg, &pos};
        const std::vector<int> *meas[2] = {&m0_, &m1_};
        std::vector<int> keep[2];
        bool condition = true;
        for (int v = 0; v < 2; ++v)
        {
            for (int q : *meas[v])
            {
                if (contains(targets, q))
                    continue;
                keep[v].push_back(q);
                bool same = contains(*ctrl[v], q), other = contains(*ctrl[1 - v], q);
                if (!same && !other)
                    ctrl[v]->push_back(q);
                else if (other)
                    condition = false;
            }
        }
        if (!condition)
            return; // src/qcs.cu:2690-2691
        ResolvedGate r;
        r.spec = g;
        r.tphys.resize(targets.size());
        for (size_t j = 0; j < targets.size(); ++j)
            r.tphys[j] = l2p_[targets[j]];
        ensure_local(r.tphys);
        for (int q : pos)
            r.pphys.push_back(l2p_[q]);
        for (int q : neg)
            r.nphys.push_back(l2p_[q]);
        for (size_t j = 0; j < targets.size(); ++j)
        {
            if (contains(m0_, targets[j]))
                r.mmask |= 1u << j;
            else if (contains(m1_, targets[j]))
            {
                r.mmask |= 1u << j;
                r.mval |= 1u << j;
            }
        }
        if (fused_)
        {
            // matrix products over more qubits than the gate's own: zeros stay zero only while
            // every amplitude is finite
            if (!m0_.empty() || !m1_.empty())
                consistent_ = false;
            fused_->enqueue(r);
        }
        else
            apply_resolved(r);
        m0_ = keep[0];
        m1_ = keep[1];
    }

    void Simulator::resolve(ResolvedGate &r, const GateSpec &g, const std::vector<int> &targets, const std::vector<int> &neg, const std::vector<int> &pos) const
    {
        if ((int)targets.size() != g.ntargets)
            throw std::runtime_error(fmt("gate needs %d target qubit(s), %d given", g.ntargets, (int)targets.size()));
        check_operands(targets, neg, pos);
        r.spec = g;
        for (int q : targets)
            r.tphys.push_back(l2p_[q]);
        for (int q : pos)
            r.pphys.push_back(l2p_[q]);
        for (int q : neg)
            r.nphys.push_back(l2p_[q]);
    }

    void Simulator::run_circuit(const std::vector<CircuitGate> &gates, size_t *applied)
    {
        need_alloc();
        *applied = 0;
        // Measured qubits (implicit controls, zeroed branches), a window of local qubits and
        // the fused modes (their own queue) go gate by gate.
        if (precision_ != 0 || !m0_.empty() || !m1_.empty() || n_local_ != n_)
        {
            for (const auto &g : gates)
            {
                operate(g.spec, g.targets, g.neg, g.pos);
                ++*applied;
            }
            return;
        }
        constexpr size_t kRun = 4096; // gates planned together: bounds the program's size
        std::vector<ResolvedGate> run;
        run.reserve(std::min(kRun, gates.size()));
        for (size_t i = 0; i < gates.size();)
        {
            run.clear();
            std::string refused;
            bool stop = false;
            for (; i < gates.size() && run.size() < kRun; ++i)
            {
                try
                {
                    run.emplace_back();
                    resolve(run.back(), gates[i].spec, gates[i].targets, gates[i].neg, gates[i].pos);
                }
                catch (const std::exception &e)
                {
                    run.pop_back();
                    refused = e.what();
                    stop = true;
                    break;
                }
            }
            apply_run(run);
            *applied += run.size();
            if (stop)
                throw std::runtime_error(refused);
        }
    }

    void Simulator::leave_segment(size_t segment)
    {
        if (!ring_read_[segment])
            qsv::check(hipEventCreateWithFlags(&ring_read_[segment], hipEventDisableTiming), "hipEventCreate");
        qsv::check(hipEventRecord(ring_read_[segment], stream_), "hipEventRecord");
        ring_pending_[segment] = true;
    }

    void Simulator::enter_segments(size_t bytes)
    {
        // the segments that begin inside the part
        for (size_t i = (ring_at_ + kSegment - 1) / kSegment; i * kSegment < ring_at_ + bytes; ++i)
            if (ring_pending_[i])
            {
                qsv::check(hipEventSynchronize(ring_read_[i]), "hipEventSynchronize");
                ring_pending_[i] = false;
            }
    }

    // Whether a gate may be in a pass: a controlled 2x2 needs 4 register bits clear of its
    // controls.
    bool Simulator::pass_takes(const ResolvedGate &g) const { return int(g.pphys.size() + g.nphys.size() + g.tphys.size()) <= pass_tile_bits(n_) - 4; }

    // What a kernel of its own for the gate moves, in sweeps of the state.
    static double sweeps_alone(const ResolvedGate &g)
    {
        const Kind kd = g.spec.kind;
        return kd == Kind::Identity ? 0.0 : std::ldexp(kd == Kind::PhaseOne || kd == Kind::PairSub ? 0.5 : 1.0, -int(g.pphys.size() + g.nphys.size()));
    }

    int Simulator::run_passes(const ResolvedGate *gates, size_t count)
    {
        const int m = pass_tile_bits(n_);
        const int amp_bytes = fused_ && !fused_->f64() ? 8 : 16;
        PassLowering lowering(n_);
        double bytes = 0; // what one kernel per gate would move, in sweeps of the state
        for (size_t i = 0; i < count; ++i)
        {
            if (!pass_takes(gates[i]) || !lowering.add(gates[i]))
                return -1;
            bytes += sweeps_alone(gates[i]);
        }
        const std::vector<PassGate> low = lowering.finish();
        if (low.empty())
            return 0;
        static_assert((kPinnedResults * sizeof(double)) % alignof(qsv::PassOp) == 0 && (32 * sizeof(double)) % alignof(qsv::PassOp) == 0, "pass program alignment");
        // With 3 low qubits in each tile instead of 4 a tile has room for one more other qubit, but
        // a pass over a large complex128 state is 3 % slower.  Up to 23 qubits the tiles have 3 (20
        // qubits, 20 layers: 405 and 372 us; 23 qubits, QAOA: 280 and 246); above, the plan with 4
        // is taken unless one with 3 has fewer passes (30 qubits, brick depth 3: 5 passes 33.2 ms,
        // 4 passes 27.5 ms; QFT: 7 either way, 56.2 and 58.0 ms), and from 28 qubits on, where a
        // pass takes longer (1.4 ms at 28, 5.5 at 30) than the search for it (0.05 to 0.15 ms in plans
        // of up to 10 passes, 0.2 to 0.3 in those of 100), more sequences of tiles are tried (30
        // qubits, 4 RY/RZ/CNOT layers: 6 passes 54.2 ms, 4 passes 42.3 ms; brick depth 24: 15 and
        // 13, 179 and 162 ms; 28 qubits, two-qubit gates: 6 and 5, 10.2 and 8.8 ms).
        // Complex64 lines are 16 amplitudes, and its passes are bound by arithmetic: 25 qubits, 6
        // layers in 6 or 7 passes, both 1.9 ms.
        const int low_bits = amp_bytes == 8 ? 4 : 3;
        std::vector<uint64_t> tiles; // above 22 qubits
        if (n_ > 22)
        {
            tiles = n_ >= 28 && low_bits == 3 ? search_tiles(low, n_, m, 3, 4, n_ >= 30 ? 8 : 4, 6) : search_tiles(low, n_, m, low_bits, low_bits, 1, 1);
            if (n_ > 23 && low_bits == 3)
            {
                std::vector<uint64_t> four = search_tiles(low, n_, m, 4, 4, 1, 1);
                if (!four.empty() && (tiles.empty() || four.size() <= tiles.size()))
                    tiles = std::move(four);
            }
            // A pass moves the whole state once, so few gates with many controls are cheaper one
            // by one.
            if (bytes < double(tiles.size()))
                return -1;
        }
        // Passes are copied and launched in groups as they are planned, the first of 2 and each of
        // two more than all before it, so that they run while others are planned and there are
        // few copies (20 qubits, 20 layers in 13 passes: 905 -> 761 us a call; 13 qubits, 6 layers:
        // 222 -> 200).  Nothing is allocated once a pass has been launched, since a run that ends
        // between its passes is a state that no gates leave: the ring is there before, a group
        // longer than what is free of it goes in parts, and a pass longer than the ring in several
        // sweeps.
        static_assert(kRing >= qsv::pass_rounds_bytes(1) + (kProgramRoundOps + qsv::kPassOpPad) * sizeof(qsv::PassOp), "the ring holds every round");
        char *const host = reinterpret_cast<char *>(pinned_ + kPinnedResults), *const dev = reinterpret_cast<char *>(work_ + work_len_);
        uint32_t done = 0; // rounds launched
        int sweeps = 0;
        auto launch = [&](const PassPlan &P) {
            while (done < P.rounds.size())
            {
                const ProgramPart part = program_part(P, done, kRing - ring_at_, ring_at_ == 0);
                if (part.end == done)
                {
                    if (ring_at_ == 0)
                        throw std::runtime_error("pass: a round does not fit the program ring");
                    if (ring_at_ < kRing)
                        leave_segment(ring_at_ / kSegment);
                    ring_at_ = 0;
                    continue;
                }
                const size_t bytes = part.bytes(P), from = ring_at_;
                enter_segments(bytes);
                part.write(P, host + from);
                qsv::launch_program_copy(stream_, dev + from, host + from, bytes);
                ring_at_ += bytes;
                for (size_t i = from / kSegment; i < ring_at_ / kSegment; ++i)
                    leave_segment(i);
                const auto *rounds = reinterpret_cast<const qsv::PassRound *>(dev + from);
                const auto *ops = reinterpret_cast<const qsv::PassOp *>(dev + from + qsv::pass_rounds_bytes(part.end - part.first));
                for (const auto &ps : P.passes)
                {
                    const uint32_t a = std::max(ps.first_round, part.first), b = std::min(ps.first_round + ps.nrounds, part.end);
                    if (a >= b)
                        continue;
                    prof_begin(QCS_EXT_K_FUSED, 2.0 * amp_bytes * (1ull << n_));
                    with_state([&](auto *st) { qsv::launch_pass(stream_, st, n_, m, ps.tq, rounds + (a - part.first), int(b - a), ops); });
                    prof_end();
                    ++sweeps;
                }
                done = part.end;
            }
        };
        size_t launched = 0; // passes
        PassPlan P;
        try
        {
            P = plan_passes(
                low, n_, m, amp_bytes, low_bits,
                [&](const PassPlan &so_far, bool last) {
                    if (last || so_far.passes.size() < 2 * (launched + 1))
                        return;
                    launch(so_far);
                    launched = so_far.passes.size();
                },
                tiles);
            launch(P);
        }
        catch (...)
        {
            (void)hipStreamSynchronize(stream_);
            throw;
        }
        return sweeps;
    }

    void Simulator::apply_run(const std::vector<ResolvedGate> &gates)
    {
        if (gates.empty())
            return;
        state_changed();
        // Up to 22 qubits a pass is worth its program's copy and its sweep where the gates' own
        // kernels take longer, in us: 3.4 a launch, or on larger states twice their share of a sweep
        // (they touch parts of lines), against 6.5 more for the first pass, 0.5 a gate, and of the
        // sweep what its launch does not cover.  (Calls that are waited for, gates' kernels and
        // passes: 10 qubits, 2 Hadamards 21.1 and 22.9 us, 3 23.4 and 23.7, 5 30.4 and 23.4; 22
        // qubits, X with 6 controls, 2 24.6 and 41.2, 6 37.6 and 43.6, 8 44.0 and 45.9, 12 57.9 and
        // 48.4, with 2 controls, 2 32.4 and 37.4, 3 52.0 and 41.0, Hadamards, 2 54.7 and 51.9.)
        const double sweep = std::ldexp(32.0, n_) / 6.2e6;
        auto worth = [&](size_t first, size_t end) {
            if (n_ > 22)
                return end - first > 1;
            double alone = 0;
            for (size_t i = first; i < end; ++i)
                if (const double share = sweeps_alone(gates[i]))
                    alone += std::max(3.4, std::min(1.0, 2 * share) * sweep);
            return alone > 6.5 + 0.5 * double(end - first) + std::max(0.0, sweep - 5.0);
        };
        for (size_t i = 0; i < gates.size();)
        {
            // the next gates that passes take, and those that they don't
            size_t end = i;
            while (end < gates.size() && pass_takes(gates[end]))
                ++end;
            if (end > i && worth(i, end) && run_passes(&gates[i], end - i) >= 0)
                i = end;
            for (; i < end || (i < gates.size() && !pass_takes(gates[i])); ++i)
                apply_resolved(gates[i]);
        }
    }

    void Simulator::apply_resolved(const ResolvedGate &r)
    {
        const GateSpec &g = r.spec;
        uint64_t setb = 0;
        for (int q : r.pphys)
            setb |= uint64_t(1) << q;
        std::vector<int> ctrl_ops = r.pphys;
        ctrl_ops.insert(ctrl_ops.end(), r.nphys.begin(), r.nphys.end());
        auto readable = [&](unsigned pattern) { return ((pattern ^ r.mval) & r.mmask) == 0; };
        const int nc = (int)ctrl_ops.size();
        switch (g.kind)
        {
        case Kind::Identity:
            return;
        case Kind::GlobalPhase:
        {
            auto sub = make_sub(ctrl_ops, setb);
            prof_begin(QCS_EXT_K_PHASE, 32.0 * (1ull << (n_ - nc)));
            qsv::launch_phase(stream_, state_, n_, sub, to_c(g.phase[0]));
            prof_end();
            return;
        }
        case Kind::PhaseOne:
        {
            int t = r.tphys[0];
            std::vector<int> ops = ctrl_ops;
            ops.push_back(t);
            auto sub = make_sub(ops, setb | (uint64_t(1) << t));
            // a target measured as 0 makes the |1> input read as zero (src/qcs.cu:1153-1171)
            cd ph = readable(1) ? g.phase[1] : cd(0.0, 0.0);
            prof_begin(QCS_EXT_K_PHASE, 32.0 * (1ull << (n_ - nc - 1)));
            qsv::launch_phase(stream_, state_, n_, sub, to_c(ph));
            prof_end();
            return;
        }
        case Kind::Diag1:
        case Kind::Diag2:
        {
            auto sub = make_sub(ctrl_ops, setb);
            qsv::DiagOp op{};
            op.ntargets = g.ntargets;
            for (int j = 0; j < g.ntargets; ++j)
                op.t[j] = r.tphys[j];
            for (int k = 0; k < (1 << g.ntargets); ++k)
                op.phase[k] = readable(k) ? to_c(g.phase[k]) : qsv::c128{0.0, 0.0};
            prof_begin(QCS_EXT_K_DIAG, 32.0 * (1ull << (n_ - nc)));
            qsv::launch_diag(stream_, state_, n_, sub, op);
            prof_end();
            return;
        }
        case Kind::Pair1:
        case Kind::PairSub:
        {
            std::vector<int> ops = ctrl_ops;
            ops.insert(ops.end(), r.tphys.begin(), r.tphys.end());
            auto sub = make_sub(ops, setb);
            qsv::PairOp op{};
            int pa = g.kind == Kind::Pair1 ? 0 : g.pat[0];
            int pb = g.kind == Kind::Pair1 ? 1 : g.pat[1];
            auto off = [&](int pat) {
                uint64_t o = 0;
                for (int j = 0; j < g.ntargets; ++j)
                    if ((pat >> j) & 1)
                        o |= uint64_t(1) << r.tphys[j];
                return o;
            };
            op.offA = off(pa);
            op.offB = off(pb);
            for (int i = 0; i < 4; ++i)
                op.m[i] = to_c(g.m[i]);
            op.zero_mask = (readable(pa) ? 0u : 1u) | (readable(pb) ? 0u : 2u);
            prof_begin(QCS_EXT_K_PAIR, 64.0 * (1ull << (n_ - (int)ops.size())));
            qsv::launch_pair(stream_, state_, n_, sub, op);
            prof_end();
            return;
        }
        case Kind::Dense4:
        case Kind::Mono:
        {
            std::vector<int> ops = ctrl_ops;
            ops.insert(ops.end(), r.tphys.begin(), r.tphys.end());
            auto sub = make_sub(ops, setb);
            const int K = 1 << g.ntargets;
            uint64_t offs[16];
            for (int k = 0; k < K; ++k)
            {
                offs[k] = 0;
                for (int j = 0; j < g.ntargets; ++j)
                    if ((k >> j) & 1)
                        offs[k] |= uint64_t(1) << r.tphys[j];
            }
            unsigned rmask = 0;
            for (int k = 0; k < K; ++k)
                if (readable(k))
                    rmask |= 1u << k;
            const uint64_t items = 1ull << (n_ - (int)ops.size());
            if (g.kind == Kind::Dense4)
            {
                qsv::Dense4Op op{};
                for (int k = 0; k < 4; ++k)
                    op.off[k] = offs[k];
                for (int i = 0; i < 16; ++i)
                    op.m[i] = to_c(g.m[i]);
                // rows equal to the identity row are not written (the reference's apply()
                // skips them too)
                op.write_mask = 0;
                unsigned needed = 0;
                for (int row = 0; row < 4; ++row)
                {
                    bool ident = true;
                    for (int c = 0; c < 4; ++c)
                        if (g.m[4 * row + c] != (row == c ? cd(1.0, 0.0) : cd(0.0, 0.0)))
                            ident = false;
                    if (!ident)
                    {
                        op.write_mask |= 1u << row;
                        for (int c = 0; c < 4; ++c)
                            if (g.m[4 * row + c] != cd(0.0, 0.0))
                                needed |= 1u << c;
                    }
                }
                op.read_mask = rmask & needed;
                double bytes = 16.0 * (__builtin_popcount(op.read_mask) + __builtin_popcount(op.write_mask)) * items;
                prof_begin(QCS_EXT_K_DENSE4, bytes);
                qsv::launch_dense4(stream_, state_, n_, sub, op);
                prof_end();
            }
            else
            {
                qsv::MonoOp op{};
                op.ntargets = g.ntargets;
                op.nrows = g.nrows;
                for (int k = 0; k < K; ++k)
                    op.off[k] = offs[k];
                for (int k = 0; k < g.nrows; ++k)
                {
                    op.row[k] = g.row[k];
                    op.src[k] = g.src[k];
                    op.coef[k] = to_c(g.coef[k]);
                }
                op.read_mask = rmask;
                prof_begin(QCS_EXT_K_MONO, 32.0 * g.nrows * items);
                qsv::launch_mono(stream_, state_, n_, sub, op);
                prof_end();
            }
            return;
        }
        }
    }

    int Simulator::measure(int q)
    { // src/qcs.cu:2545-2677
        need_alloc();
        if (q < 0 || q >= n_)
            throw std::runtime_error(fmt("qubit %d out of range [0, %d)", q, n_));
        if (contains(m0_, q))
            return 0;
        if (contains(m1_, q))
            return 1;
        flush();
        state_changed();
        std::vector<int> tphys = {l2p_[q]};
        ensure_local(tphys);
        const int tq = tphys[0];
        std::vector<int> ops = {tq};
        uint64_t setb = 0;
        for (int x : m1_)
        {
            ops.push_back(l2p_[x]);
            setb |= uint64_t(1) << l2p_[x];
        }
        for (int x : m0_)
            ops.push_back(l2p_[x]);
        auto sub = make_sub(ops, setb);
        const uint64_t items = uint64_t(1) << (n_ - sub.nops);
        const double S = c64_state() ? 8.0 : 16.0;
        prof_begin(QCS_EXT_K_REDUCE, 2.0 * S * items);
        with_state([&](auto *st) { qsv::reduce_pair_probs(stream_, st, sub, uint64_t(1) << tq, items, work_, pinned_); });
        prof_end();
        const double p0 = pinned_[0], p1 = pinned_[1];
        std::uniform_real_distribution<double> dist(0, p0 + p1);
        const double rnd = dist(engine_);
        const int result = p0 < rnd;
        (result ? m1_ : m0_).push_back(q);
        const double pk = result ? p1 : p0;
        const double scale = (renormalize_ && pk > 0) ? 1.0 / std::sqrt(pk) : 1.0;
        // qubits measured before whose other halves are zero already
        std::vector<int> fixed;
        if (consistent_)
            for (int x : ops)
                if (x != tq)
                    fixed.push_back(x);
        std::sort(fixed.begin(), fixed.end());
        prof_begin(QCS_EXT_K_COLLAPSE, S * std::ldexp(0.5, n_ - int(fixed.size())) * (scale != 1.0 ? 3.0 : 1.0));
        with_state([&](auto *st) { qsv::launch_collapse(stream_, st, n_, tq, result, scale, fixed.data(), int(fixed.size()), setb); });
        prof_end();
        return result;
    }

    // Amplitudes pass between the state and a caller's buffer through a ring of pinned slots,
    // which the gather kernel writes over the link itself, and threads copy between the slots
    // and the caller's pages, which is what takes longest (64 MiB: 1.2 ms over the link; one
    // thread 2.1 ms, 4.8 ms into pages touched first, 8 threads 1.4 ms).  22 qubits, set 3.4 ->
    // 2.0 ms, get 6.2 -> 1.9 ms.
    uint64_t Simulator::stage_len() const { return std::min<uint64_t>(uint64_t(1) << n_, kSlotLen * kSlots); }

    void Simulator::ensure_stage()
    {
        if (!stage_)
            qsv::check(hipHostMalloc((void **)&stage_, stage_len() * sizeof(qsv::c128), hipHostMallocDefault), "hipHostMalloc stage");
        while (stage_events_.size() < kSlots)
        {
            hipEvent_t e;
            qsv::check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
            stage_events_.push_back(e);
        }
    }

    namespace
    {
        // The i-th part of the state to go (a power of two of them): the threads at work at one
        // time are in 8 separate regions, since first touches within one huge page wait for
        // each other.
        uint64_t spread(uint64_t i, uint64_t parts)
        {
            const uint64_t regions = std::min<uint64_t>(parts, 8);
            return (i % regions) * (parts / regions) + i / regions;
        }

        // Copies slots 0 .. count - 1, in order of their numbers but several at a time, each
        // once open() has covered it; done(i) waits for one.  The destructor ends the threads.
        class CopyCrew
        {
        public:
            CopyCrew(size_t count, std::function<void(size_t)> copy) : count_(count), done_(count, 0), copy_(std::move(copy))
            {
                const size_t threads = count < 4 ? 0 : std::min<size_t>({size_t(8), std::max(1u, std::thread::hardware_concurrency()), count / 2});
                pool_.reserve(threads);
                try
                {
                    for (size_t t = 0; t < threads; ++t)
                        pool_.emplace_back([this] { work(); });
                }
                catch (const std::exception &)
                { // fewer threads, then: done() copies too
                }
            }
            ~CopyCrew()
            {
                {
                    std::lock_guard<std::mutex> lock(mu_);
                    next_ = count_;
                }
                cv_.notify_all();
                for (auto &t : pool_)
                    t.join();
            }
            void open(size_t slots)
            {
                {
                    std::lock_guard<std::mutex> lock(mu_);
                    open_ = std::max(open_, slots);
                }
                cv_.notify_all();
            }
            // whether slot i (an open one) is copied; waits until it is if asked to
            bool done(size_t i, bool wait = true)
            {
                std::unique_lock<std::mutex> lock(mu_);
                while (wait && !done_[i])
                    if (next_ < open_)
                        one(lock);
                    else
                        cv_.wait(lock);
                return done_[i];
            }

        private:
            void one(std::unique_lock<std::mutex> &lock)
            {
                const size_t i = next_++;
                lock.unlock();
                copy_(i);
                lock.lock();
                done_[i] = 1;
                cv_.notify_all();
            }
            void work()
            {
                std::unique_lock<std::mutex> lock(mu_);
                while (next_ < count_)
                    if (next_ < open_)
                        one(lock);
                    else
                        cv_.wait(lock);
            }
            std::mutex mu_;
            std::condition_variable cv_;
            size_t next_ = 0, open_ = 0;
            const size_t count_;
            std::vector<char> done_;
            std::function<void(size_t)> copy_;
            std::vector<std::thread> pool_;
        };
    } // namespace

    void Simulator::save_statevector(const char *path)
    { // src/qcs.cu:2494-2543: raw little-endian complex<double>, logical order, no header
        need_alloc();
        flush();
        if (path == nullptr)
            throw std::runtime_error("output file name must not be NULL");
        FILE *fp = std::fopen(path, "wb");
        if (!fp)
            throw std::runtime_error("open failed");
        try
        {
            const uint64_t count = uint64_t(1) << n_;
            ensure_stage();
            const uint64_t chunk = stage_len();
            for (uint64_t first = 0; first < count; first += chunk)
            {
                with_state([&](auto *st) { qsv::launch_gather_logical(stream_, st, stage_, first, chunk, l2p_.data(), n_); });
                qsv::check(hipStreamSynchronize(stream_), "save sync");
                if (std::fwrite(stage_, sizeof(qsv::c128), chunk, fp) != chunk)
                    throw std::runtime_error("fwrite failed");
            }
        }
        catch (...)
        {
            std::fclose(fp);
            throw;
        }
        if (std::fclose(fp) != 0)
            throw std::runtime_error("close failed");
    }

    void Simulator::get_statevector(double *out, uint64_t count)
    {
        need_alloc();
        flush();
        if (out == nullptr || count != (uint64_t(1) << n_))
            throw std::runtime_error("statevector buffer size mismatch");
        ensure_stage();
        const uint64_t len = std::min(count, kSlotLen), slots = count / len;
        auto slot = [&](uint64_t i) { return stage_ + (i % kSlots) * kSlotLen; };
        auto part = [&](uint64_t i) { return len * spread(i, slots); };
        CopyCrew crew(slots, [&](size_t i) { std::memcpy(out + 2 * part(i), slot(i), len * sizeof(qsv::c128)); });
        for (uint64_t issued = 0, arrived = 0; arrived < slots;)
        {
            // keep every slot that has been copied out busy; wait for one only with none on its way
            for (; issued < slots && issued < arrived + kSlots; ++issued)
            {
                if (issued >= kSlots && !crew.done(issued - kSlots, arrived == issued))
                    break;
                with_state([&](auto *st) { qsv::launch_gather_logical(stream_, st, slot(issued), part(issued), len, l2p_.data(), n_); });
                qsv::check(hipEventRecord(stage_events_[issued % kSlots], stream_), "hipEventRecord");
            }
            qsv::check(hipEventSynchronize(stage_events_[arrived % kSlots]), "hipEventSynchronize");
            crew.open(++arrived);
        }
        for (uint64_t i = 0; i < slots; ++i)
            crew.done(i);
    }

    void Simulator::set_statevector(const double *in, uint64_t count)
    {
        need_alloc();
        flush();
        if (in == nullptr || count != (uint64_t(1) << n_))
            throw std::runtime_error("statevector buffer size mismatch");
        state_changed();
        if (fused_)
            fused_->drop();
        ensure_stage();
        consistent_ = m0_.empty() && m1_.empty(); // a failure on the way leaves part of the new state
        const uint64_t len = std::min(count, kSlotLen), slots = count / len;
        auto slot = [&](uint64_t i) { return stage_ + (i % kSlots) * kSlotLen; };
        qsv::check(hipStreamSynchronize(stream_), "sync"); // no earlier work reads the slots
        // a kernel reads host memory at 37 GB/s, the copy engine at 57 (it writes at 49); a part
        // of a slot is faster without the copy's launch
        const bool dma = len == kSlotLen;
        if (dma && !stage_dev_)
            qsv::check(hipMalloc((void **)&stage_dev_, stage_len() * sizeof(qsv::c128)), "hipMalloc stage");
        auto part = [&](uint64_t i) { return len * spread(i, slots); };
        CopyCrew crew(slots, [&](size_t i) { std::memcpy(slot(i), in + 2 * part(i), len * sizeof(qsv::c128)); });
        crew.open(std::min(slots, kSlots));
        // copies in groups: between a copy and the scatter that follows it the engines wait for
        // each other (15 us)
        const uint64_t group = std::min<uint64_t>(slots, 4);
        for (uint64_t i = 0; i < slots; i += group)
        {
            for (uint64_t j = i; j < i + group; ++j)
            {
                crew.done(j);
                if (dma)
                    qsv::check(hipMemcpyAsync(stage_dev_ + (j % kSlots) * kSlotLen, slot(j), len * sizeof(qsv::c128), hipMemcpyHostToDevice, stream_), "copy");
            }
            for (uint64_t j = i; j < i + group; ++j)
                with_state([&](auto *st) { qsv::launch_scatter_logical(stream_, st, dma ? stage_dev_ + (j % kSlots) * kSlotLen : slot(j), part(j), len, l2p_.data(), n_); });
            qsv::check(hipEventRecord(stage_events_[i % kSlots], stream_), "hipEventRecord");
            // the slots of the group two back take their next amplitudes
            const uint64_t back = 2 * group;
            if (i >= back && i - back + kSlots < slots)
            {
                qsv::check(hipEventSynchronize(stage_events_[(i - back) % kSlots]), "hipEventSynchronize");
                crew.open(i - back + group + kSlots);
            }
        }
        qsv::check(hipStreamSynchronize(stream_), "sync");
        // a new state: earlier measurement results no longer describe it
        clear_measurement_state();
    }

    void Simulator::load_statevector(const char *path)
    { // src/qcs.cu:2121-2159 (reads physical order from a fixed name); here: any path, the
      // logical-order format save_statevector writes, streamed through the pinned stage
        need_alloc();
        flush();
        if (path == nullptr)
            throw std::runtime_error("input file name must not be NULL");
        FILE *fp = std::fopen(path, "rb");
        if (!fp)
            throw std::runtime_error("open failed");
        try
        {
            const uint64_t count = uint64_t(1) << n_;
            if (std::fseek(fp, 0, SEEK_END) != 0)
                throw std::runtime_error("fseek failed");
            const long long size = std::ftell(fp);
            if (size < 0 || uint64_t(size) != count * sizeof(qsv::c128))
                throw std::runtime_error("statevector file holds " + std::to_string(size) + " bytes, expected " + std::to_string(count * sizeof(qsv::c128)));
            std::rewind(fp);
            state_changed();
            if (fused_)
                fused_->drop();
            ensure_stage();
            consistent_ = m0_.empty() && m1_.empty(); // as in set_statevector
            const uint64_t chunk = stage_len();
            for (uint64_t first = 0; first < count; first += chunk)
            {
                qsv::check(hipStreamSynchronize(stream_), "sync");
                if (std::fread(stage_, sizeof(qsv::c128), chunk, fp) != chunk)
                    throw std::runtime_error("fread failed");
                with_state([&](auto *st) { qsv::launch_scatter_logical(stream_, st, stage_, first, chunk, l2p_.data(), n_); });
            }
            qsv::check(hipStreamSynchronize(stream_), "sync");
        }
        catch (...)
        {
            std::fclose(fp);
            throw;
        }
        std::fclose(fp);
        clear_measurement_state();
    }

    void Simulator::ensure_levels()
    {
        auto sz = qsv::fold_level_sizes(uint64_t(1) << n_);
        if (levels_.size() + 1 == sz.size())
            return;
        for (auto p : levels_)
            (void)hipFree(p);
        levels_.clear();
        for (size_t lev = 1; lev < sz.size(); ++lev)
        {
            double *p = nullptr;
            qsv::check(hipMalloc((void **)&p, sz[lev] * sizeof(double)), "hipMalloc levels");
            levels_.push_back(p);
        }
    }

    double Simulator::probability_total()
    {
        need_alloc();
        flush();
        // the levels are built once per state: sample() after probability_total() (or a
        // second probability_total()) on an unchanged state reuses them
        if (levels_valid_)
            return levels_total_;
        ensure_levels();
        prof_begin(QCS_EXT_K_REDUCE, (c64_state() ? 8.0 : 16.0) * (1ull << n_));
        std::vector<double *> levels = levels_;
        levels.back() = pinned_; // the total; a search starts one level below
        with_state([&](auto *st) { qsv::build_fold_levels(stream_, st, uint64_t(1) << n_, levels); });
        prof_end();
        qsv::check(hipStreamSynchronize(stream_), "sync");
        levels_total_ = pinned_[0];
        levels_valid_ = true;
        return levels_total_;
    }

    void Simulator::sample(uint64_t seed, uint64_t shots, uint64_t *out)
    {
        need_alloc();
        if (shots > 0 && out == nullptr)
            throw std::runtime_error("outcome buffer must not be NULL");
        flush();
        const double total = probability_total();
        if (shots == 0)
            return;
        // through pinned memory that the search writes: an allocation, a copy and a release each
        // call took 40 us.  More outcomes than one fetch come in turn to its two halves, and
        // one is searched while the other is copied out (8388608 outcomes of 10 qubits: 8.2 ms
        // one after the other, 5.3 so).
        const uint64_t cap = std::min(shots, kShotChunk), halves = shots > cap ? 2 : 1;
        if (halves * cap > shots_cap_)
        {
            if (shots_)
                (void)hipHostFree(shots_);
            shots_ = nullptr;
            shots_cap_ = 0;
            uint64_t want = 1024;
            while (want < halves * cap)
                want *= 2;
            qsv::check(hipHostMalloc((void **)&shots_, want * sizeof(uint64_t), hipHostMallocDefault), "hipHostMalloc outcomes");
            shots_cap_ = want;
        }
        auto search = [&](uint64_t chunk) {
            const uint64_t first = chunk * cap;
            prof_begin(QCS_EXT_K_SAMPLE, 0.0);
            with_state([&](auto *st) { qsv::launch_sample_search(stream_, st, uint64_t(1) << n_, levels_, total, seed, first, std::min(cap, shots - first), p2l_.data(), n_, shots_ + chunk % 2 * cap); });
            prof_end();
            if (halves == 1)
                return;
            hipEvent_t &e = shots_there_[chunk % 2];
            if (!e)
                qsv::check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
            qsv::check(hipEventRecord(e, stream_), "hipEventRecord");
        };
        search(0);
        for (uint64_t chunk = 0, first = 0; first < shots; ++chunk, first += cap)
        {
            if (first + cap < shots)
                search(chunk + 1);
            qsv::check(halves == 1 ? hipStreamSynchronize(stream_) : hipEventSynchronize(shots_there_[chunk % 2]), "sync");
            std::memcpy(out + first, shots_ + chunk % 2 * cap, std::min(cap, shots - first) * sizeof(uint64_t));
        }
    }

    void Simulator::sample_noalloc(uint64_t seed, uint64_t shots, uint64_t *out)
    {
        need_alloc();
        if (fused_ && fused_->has_queued())
            throw std::runtime_error("sample_noalloc: fused gates are queued and their flush may allocate; call qcs_ext_flush first");
        with_state([&](auto *st) { qsv::sample_noalloc(stream_, device_, st, n_, seed, shots, p2l_.data(), pinned_, out); });
    }

    double Simulator::norm()
    {
        need_alloc();
        flush();
        prof_begin(QCS_EXT_K_REDUCE, (c64_state() ? 8.0 : 16.0) * (1ull << n_));
        with_state([&](auto *st) { qsv::reduce_probs(stream_, st, uint64_t(1) << n_, work_, pinned_); });
        prof_end();
        return pinned_[0];
    }

    void Simulator::expect_z(double *out, int count)
    {
        need_alloc();
        flush();
        if (count < 0 || count > n_ || (count > 0 && out == nullptr))
            throw std::runtime_error("expect_z count out of range");
        if (count == 0)
            return;
        prof_begin(QCS_EXT_K_REDUCE, (c64_state() ? 8.0 : 16.0) * (1ull << n_));
        with_state([&](auto *st) { qsv::expect_z(stream_, st, n_, work_, pinned_, l2p_.data(), count, out); });
        prof_end();
    }

    void Simulator::set_local_qubits(int nl)
    {
        need_alloc();
        if (nl < 1 || nl > n_)
            throw std::runtime_error(fmt("num_local_qubits %d out of range [1, %d]", nl, n_));
        n_local_ = nl;
    }

    void Simulator::get_mapping(int16_t *out, int count) const
    {
        need_alloc();
        if (out == nullptr || count != n_)
            throw std::runtime_error("mapping buffer size mismatch");
        for (int q = 0; q < n_; ++q)
            out[q] = (int16_t)p2l_[q];
    }

    void Simulator::permute(const std::vector<int> &want)
    {
        need_alloc();
        flush();
        state_changed();
        if ((int)want.size() != n_)
            throw std::runtime_error("mapping size mismatch");
        std::vector<bool> used(n_, false);
        for (int l : want)
        {
            if (l < 0 || l >= n_ || used[l])
                throw std::runtime_error("not a permutation");
            used[l] = true;
        }
        // logical qubit want[q] goes to physical slot q
        std::vector<int> dst(n_);
        for (int q = 0; q < n_; ++q)
            dst[l2p_[want[q]]] = q;
        move_physical(dst);
    }

    void Simulator::overlap(Simulator &other, double out[3])
    {
        need_alloc();
        other.need_alloc();
        flush();
        other.flush();
        if (n_ != other.n_ || p2l_ != other.p2l_)
            throw std::runtime_error("overlap needs two states of the same size and qubit mapping");
        if (device_ != other.device_)
            throw std::runtime_error("overlap needs both simulators on the same device");
        qsv::check(hipStreamSynchronize(other.stream_), "hipStreamSynchronize");
        const uint64_t count = uint64_t(1) << n_;
        double *work = nullptr;
        qsv::check(hipMalloc((void **)&work, qsv::overlap_workspace(count) * sizeof(double)), "hipMalloc overlap");
        try
        {
            with_state([&](auto *a) { other.with_state([&](auto *b) { qsv::overlap(stream_, a, b, count, work, out); }); });
        }
        catch (...)
        {
            (void)hipFree(work);
            throw;
        }
        (void)hipFree(work);
    }

    void Simulator::set_plan(bool enable, int tile_bits, int k, int tiles, int window, int rule)
    {
        if (!fused_)
            throw std::runtime_error("a fixed fusion plan needs a fused precision mode (1, 2 or 3, allocated)");
        fused_->set_plan(enable, tile_bits, k, tiles, window, rule);
    }

    void Simulator::set_planner_model(CostModel *m)
    {
        if (!fused_)
            throw std::runtime_error("the fusion planner needs a fused precision mode (1, 2 or 3, allocated)");
        flush();
        fused_->set_model(m);
    }

    void Simulator::planner_stats(double out[5])
    {
        if (!fused_)
            throw std::runtime_error("the fusion planner needs a fused precision mode (1, 2 or 3, allocated)");
        flush();
        fused_->planner_stats(out);
    }

    int Simulator::planner_record_plans(int capacity, float *features, float *log2_us)
    {
        if (!fused_)
            throw std::runtime_error("recording plan timings needs a fused precision mode (1, 2 or 3, allocated)");
        state_changed();
        consistent_ = m0_.empty() && m1_.empty();
        return fused_->record_plans(capacity, features, log2_us);
    }

    void Simulator::planner_last_choice(int out[5])
    {
        if (!fused_)
            throw std::runtime_error("the fusion planner needs a fused precision mode (1, 2 or 3, allocated)");
        const PlanOption o = fused_->last_choice();
        out[0] = o.stage_bits;
        out[1] = o.k;
        out[2] = o.tiles;
        out[3] = o.window;
        out[4] = o.rule;
    }

    void Simulator::planner_record(int count, uint64_t seed, float *features, float *log2_us)
    {
        if (!fused_)
            throw std::runtime_error("recording block timings needs a fused precision mode (1, 2 or 3, allocated)");
        if (count < 0 || (count > 0 && (!features || !log2_us)))
            throw std::runtime_error("planner_record: bad output buffers");
        state_changed();
        consistent_ = m0_.empty() && m1_.empty();
        fused_->record(count, seed, features, log2_us);
    }

    void Simulator::fusion_stats(uint64_t *gates, uint64_t *blocks)
    {
        flush();
        *gates = fused_ ? fused_->gates_applied() : 0;
        *blocks = fused_ ? fused_->blocks_applied() : 0;
    }

    void Simulator::flush()
    {
        if (fused_)
            fused_->flush();
    }

    int Simulator::event_create()
    {
        hipEvent_t e;
        qsv::check(hipEventCreate(&e), "hipEventCreate");
        events_.push_back(e);
        return (int)events_.size() - 1;
    }

    void Simulator::event_record(int e)
    {
        if (e < 0 || e >= (int)events_.size())
            throw std::runtime_error(fmt("event %d does not exist", e));
        flush();
        qsv::check(hipEventRecord(events_[e], stream_), "hipEventRecord");
    }

    double Simulator::event_elapsed(int a, int b)
    { // src/qcs.cu:2862-2897: seconds from the float milliseconds of the runtime
        if (a < 0 || a >= (int)events_.size() || b < 0 || b >= (int)events_.size())
            throw std::runtime_error("event does not exist");
        qsv::check(hipEventSynchronize(events_[a]), "hipEventSynchronize");
        qsv::check(hipEventSynchronize(events_[b]), "hipEventSynchronize");
        float ms = 0.0f;
        qsv::check(hipEventElapsedTime(&ms, events_[a], events_[b]), "hipEventElapsedTime");
        return ms * 1e-3;
    }

    // ---- profiling ----
    hipEvent_t Simulator::pool_event()
    {
        if (!free_events_.empty())
        {
            hipEvent_t e = free_events_.back();
            free_events_.pop_back();
            return e;
        }
        hipEvent_t e;
        qsv::check(hipEventCreate(&e), "hipEventCreate");
        return e;
    }

    void Simulator::prof_begin(int cls, double bytes)
    {
        if (!profile_)
            return;
        open_cls_ = cls;
        open_bytes_ = bytes;
        open_a_ = pool_event();
        qsv::check(hipEventRecord(open_a_, stream_), "hipEventRecord");
    }

    void Simulator::prof_end()
    {
        if (!profile_ || open_cls_ < 0)
            return;
        hipEvent_t b = pool_event();
        qsv::check(hipEventRecord(b, stream_), "hipEventRecord");
        recs_.push_back(Rec{open_cls_, open_bytes_, open_a_, b});
        open_cls_ = -1;
        open_a_ = nullptr;
        if (recs_.size() > 4096)
            prof_resolve();
    }

    void Simulator::prof_resolve()
    {
        for (auto &r : recs_)
        {
            qsv::check(hipEventSynchronize(r.b), "hipEventSynchronize");
            float ms = 0.0f;
            qsv::check(hipEventElapsedTime(&ms, r.a, r.b), "hipEventElapsedTime");
            prof_launches_[r.cls] += 1;
            prof_seconds_[r.cls] += ms * 1e-3;
            prof_bytes_[r.cls] += r.bytes;
            free_events_.push_back(r.a);
            free_events_.push_back(r.b);
        }
        recs_.clear();
    }

    void Simulator::profile_enable(bool on)
    {
        if (!on)
            prof_resolve();
        profile_ = on;
    }

    void Simulator::profile_get(int cls, uint64_t *launches, double *seconds, double *bytes)
    {
        if (cls < 0 || cls >= QCS_EXT_K_COUNT)
            throw std::runtime_error("kernel class out of range");
        flush();
        prof_resolve();
        if (!launches || !seconds || !bytes)
            throw std::runtime_error("result pointer must not be NULL");
        *launches = prof_launches_[cls];
        *seconds = prof_seconds_[cls];
        *bytes = prof_bytes_[cls];
    }

    void Simulator::profile_reset()
    {
        prof_resolve();
        for (int i = 0; i < 16; ++i)
        {
            prof_launches_[i] = 0;
            prof_seconds_[i] = 0;
            prof_bytes_[i] = 0;
        }
    }
} // namespace qcore
