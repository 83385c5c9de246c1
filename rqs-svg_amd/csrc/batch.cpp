// Batching form host side: partition, plan, capture into one hipGraph, autotune.
//
// By default circuits run as circuit passes (pass_kernels.hpp): one of up to 12 qubits as one
// tile in the registers of one workgroup, from |0...0> to its sums for <Z>; a larger one as
// passes over a complex64 state, batched across circuits: one launch per pass round covers the
// r-th pass of every such circuit.  BF16x3 products are asked for by set_precision(3): circuits
// of more than lds_max_qubits qubits then run as stages (below).
// With a tuning set, circuits of up to `lds_max_qubits` qubits go to the persistent
// LDS-resident kernel (one workgroup per circuit, work-counter driven); larger ones keep a
// complex64 state in HBM.  Those of at least stage_bits + 4 qubits run as stages on LDS tiles,
// batched across circuits in the same way.  The rest run as fused k-qubit blocks, one launch
// each, spread over several streams.
// Everything -- counter reset, the persistent kernel, the stage rounds, the fills and
// block sequences of the smaller HBM circuits, the <Z> reductions -- is captured once into
// a hipGraph and replayed with a single launch.
#include "batch.hpp"
#include "pass.hpp"
#include "simulator.hpp"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <thread>

namespace qcore
{
    namespace
    {
        using cd = std::complex<double>;

        void mat2(const BatchGate &g, cd m[4])
        {
            GateSpec s = make_gate(g.name, g.params);
            if (s.ntargets != 1)
                throw std::runtime_error("batch: only 1-target gates (with at most one control) are batched: " + g.name);
            auto u = dense_matrix(s);
            for (int i = 0; i < 4; ++i)
                m[i] = u[i];
        }

        // f(0) .. f(count - 1), each once, on up to `threads` threads; first meanwhile(), on this one
        // beside the others
        template <class F, class M>
        void for_each_circuit(size_t count, size_t threads, F f, M meanwhile)
        {
            std::exception_ptr err;
            std::mutex err_mu;
            std::atomic<size_t> next{0};
            auto work = [&] {
                try
                {
                    for (size_t i = next++; i < count; i = next++)
                        f(i);
                }
                catch (...)
                {
                    std::lock_guard<std::mutex> lock(err_mu);
                    err = std::current_exception();
                }
            };
            threads = std::min<size_t>({threads, std::max(1u, std::thread::hardware_concurrency()), count});
            std::vector<std::thread> pool;
            pool.reserve(threads);
            try
            {
                for (size_t t = 1; t < threads; ++t)
                    pool.emplace_back(work);
            }
            catch (const std::exception &)
            { // fewer threads, then
            }
            try
            {
                meanwhile();
            }
            catch (...)
            {
                std::lock_guard<std::mutex> lock(err_mu);
                err = std::current_exception();
            }
            work();
            for (auto &th : pool)
                th.join();
            if (err)
                std::rethrow_exception(err);
        }

        qsv::BatchOp to_op(int target, int control, const cd m[4])
        {
            qsv::BatchOp op{};
            op.target = target;
            op.control = control;
            for (int i = 0; i < 4; ++i)
            {
                op.m[2 * i] = float(m[i].real());
                op.m[2 * i + 1] = float(m[i].imag());
            }
            return op;
        }
    } // namespace

    Batch::Batch()
    {
        qsv::check(hipGetDevice(&device_), "hipGetDevice");
        qsv::check(hipEventCreate(&t0_), "hipEventCreate");
        qsv::check(hipEventCreate(&t1_), "hipEventCreate");
    }

    Batch::~Batch()
    {
        try
        {
            release();
        }
        catch (...)
        {
        }
        (void)hipEventDestroy(t0_);
        (void)hipEventDestroy(t1_);
    }

    void Batch::release()
    {
        for (auto s : streams_)
            (void)hipStreamSynchronize(s);
        if (exec_)
            (void)hipGraphExecDestroy(exec_);
        if (graph_)
            (void)hipGraphDestroy(graph_);
        exec_ = nullptr;
        graph_ = nullptr;
        work_ = nullptr;
        for (void *p : {(void *)d_circs_, (void *)d_ops_, (void *)d_out_, (void *)d_counter_, (void *)d_states_, (void *)d_partials_, (void *)d_mats_, (void *)d_sums_, d_prog_})
            if (p)
                (void)hipFree(p);
        d_circs_ = nullptr;
        d_ops_ = nullptr;
        d_out_ = nullptr;
        d_counter_ = nullptr;
        d_states_ = nullptr;
        d_partials_ = nullptr;
        d_mats_ = nullptr;
        d_sums_ = nullptr;
        d_prog_ = nullptr;
        for (auto e : fork_join_)
            (void)hipEventDestroy(e);
        fork_join_.clear();
        for (auto s : streams_)
            (void)hipStreamDestroy(s);
        streams_.clear();
        prepared_ = false;
    }

    int Batch::add_circuit(int n, const std::vector<BatchGate> &gates)
    {
        if (n < 1 || n > 30)
            throw std::runtime_error("batch: circuits must have 1..30 qubits");
        for (const auto &g : gates)
        {
            if (g.target < 0 || g.target >= n || g.control >= n || g.control == g.target)
                throw std::runtime_error("batch: qubit index out of range or control equal to target");
            cd m[4];
            mat2(g, m); // validates the gate name and arity
        }
        release();
        circuits_.push_back(Circuit{n, gates, total_qubits_});
        total_qubits_ += n;
        return (int)circuits_.size() - 1;
    }

    void Batch::set_tuning(const BatchTuning &t)
    {
        if (t.lds_max_qubits < 0 || t.lds_max_qubits > qsv::kBatchMaxLdsQubits)
            throw std::runtime_error("batch: lds_max_qubits must be in [0, 14]");
        if (t.block_size != 256 && t.block_size != 512 && t.block_size != 1024)
            throw std::runtime_error("batch: block size must be 256, 512 or 1024");
        if (t.block_qubits != 4 && t.block_qubits != 5)
            throw std::runtime_error("batch: block qubits must be 4 or 5");
        if (t.streams < 1 || t.streams > 4)
            throw std::runtime_error("batch: streams must be in [1, 4]");
        if (t.stage_bits != 0 && (t.stage_bits < 11 || t.stage_bits > 13))
            throw std::runtime_error("batch: stage bits must be 0, 11, 12 or 13");
        release();
        tuning_ = t;
        passes_ = false;
    }

    void Batch::set_precision(int mode)
    {
        if (mode != 1 && mode != 3)
            throw std::runtime_error("batch: precision must be 1 (FP32 MFMA) or 3 (BF16x3 MFMA)");
        release();
        x3_ = mode == 3;
    }

    void Batch::prepare()
    {
        if (prepared_)
            return;
        if (circuits_.empty())
            throw std::runtime_error("batch: no circuits");
        release(); // what a preparation that failed left
        const BatchTuning &T = tuning_;
        auto make_streams = [&](int count) {
            while ((int)streams_.size() < std::clamp(count, 1, T.streams))
            {
                hipStream_t s;
                qsv::check(hipStreamCreateWithFlags(&s, hipStreamNonBlocking), "hipStreamCreate");
                streams_.push_back(s);
            }
        };
        // ---- small circuits: op lists for the persistent kernel ----
        std::vector<qsv::BatchCircuit> small;
        std::vector<qsv::BatchOp> ops;
        int small_max_n = 1;
        std::vector<int> large;
        struct Passed
        {
            int ci;
            PassPlan plan;
        };
        std::vector<Passed> passed;
        // The circuits' pass plans (no passes: a circuit without such a plan), on up to 16 host threads
        // of at least 512 gates each, some 200 us of work.  The streams are created beside them,
        // one a kind of circuit as far as the sizes tell: several take 0.3 to 2 ms.  (First run,
        // before passes, with 8 circuits a thread and the streams afterwards, and so: 8 circuits of
        // 4-6 qubits and 150 layers 2.4, 4.0 and 1.8 ms; 256 of 8-14 and 6 layers 4.7, 6.1 and 4.5.)
        std::vector<PassPlan> plans(circuits_.size());
        size_t gates = 0;
        int kinds[5] = {}; // up to 10, 11, 12 and more qubits, and those that run as stages
        for (const Circuit &C : circuits_)
        {
            gates += C.gates.size();
            ++kinds[x3_ && C.n > T.lds_max_qubits ? 4 : std::clamp(C.n, qsv::kPassMinBits, qsv::kPassMaxBits + 1) - qsv::kPassMinBits];
        }
        if (passes_)
            for_each_circuit(circuits_.size(), std::min<size_t>(16, gates / 512), [&](size_t ci) {
                const Circuit &C = circuits_[ci];
                if (x3_ && C.n > T.lds_max_qubits)
                    return;
                PassLowering lowering(C.n);
                ResolvedGate r;
                for (const auto &g : C.gates)
                {
                    r.spec = make_gate(g.name, g.params);
                    r.tphys.assign(1, g.target);
                    r.pphys.assign(g.control >= 0 ? 1 : 0, g.control);
                    if (!lowering.add(r))
                        return;
                }
                const auto low = lowering.finish();
                // A launch takes tiles of one size from all circuits.  2^12 is the better one, from
                // 13 qubits on as well, where single complex128 states take 2^11: one circuit of
                // 13, 16, 18, 20 qubits and 8 layers 124, 161, 189, 222 us (2^11: 127, 163, 190,
                // 255), 64 of 13-18 396 (418), 256 of 13-15 380 (415).
                if (!low.empty())
                    plans[ci] = plan_passes(low, C.n, std::clamp(C.n, qsv::kPassMinBits, qsv::kPassMaxBits), 8);
            }, [&] { make_streams(std::min(kinds[0], 1) + std::min(kinds[1], 1) + std::min(kinds[2], 1) + std::min(kinds[3], 2) + std::min(kinds[4], 1)); });
        for (int ci = 0; ci < (int)circuits_.size(); ++ci)
        {
            const Circuit &C = circuits_[ci];
            if (!plans[ci].passes.empty())
            {
                passed.push_back(Passed{ci, std::move(plans[ci])});
                continue;
            }
            if (C.n > T.lds_max_qubits)
            {
                large.push_back(ci);
                continue;
            }
            qsv::BatchCircuit bc{C.n, 0, (int)ops.size(), C.out_offset};
            // adjacent uncontrolled gates on the same qubit are multiplied together (FP64)
            int last_t = -1;
            cd acc[4];
            auto emit = [&]() {
                if (last_t >= 0)
                    ops.push_back(to_op(last_t, -1, acc));
                last_t = -1;
            };
            for (const auto &g : C.gates)
            {
                cd m[4];
                mat2(g, m);
                if (g.control < 0)
                {
                    if (last_t == g.target)
                    {
                        cd r[4] = {m[0] * acc[0] + m[1] * acc[2], m[0] * acc[1] + m[1] * acc[3],
                                   m[2] * acc[0] + m[3] * acc[2], m[2] * acc[1] + m[3] * acc[3]};
                        for (int i = 0; i < 4; ++i)
                            acc[i] = r[i];
                    }
                    else
                    {
                        emit();
                        last_t = g.target;
                        for (int i = 0; i < 4; ++i)
                            acc[i] = m[i];
                    }
                }
                else
                {
                    emit();
                    ops.push_back(to_op(g.target, g.control, m));
                }
            }
            emit();
            bc.nops = (int)ops.size() - bc.op_offset;
            small.push_back(bc);
            small_max_n = std::max(small_max_n, C.n);
        }
        // ---- large circuits: complex64 states in HBM ----
        // Circuits of >= stage_bits + 4 qubits run in stage rounds: launch r applies stage r
        // of every such circuit (tiles numbered across the circuits), after one basis-state
        // fill for all of them and before one <Z> reduction for all of them.  The others run
        // their fused blocks one launch each, spread over the streams.
        struct Staged
        {
            int ci;
            std::vector<PreparedStage> stages;
        };
        struct Blocked
        {
            int ci;
            std::vector<PreparedBlock> blocks;
        };
        std::vector<Staged> staged;
        std::vector<Blocked> blocked;
        std::vector<float> mats;
        ComposeList compose;
        compose.apart = true;
        for (int ci : large)
        {
            const Circuit &C = circuits_[ci];
            std::vector<ResolvedGate> rg;
            rg.reserve(C.gates.size());
            for (const auto &g : C.gates)
            {
                ResolvedGate r;
                r.spec = make_gate(g.name, g.params);
                r.tphys = {g.target};
                if (g.control >= 0)
                    r.pphys = {g.control};
                rg.push_back(r);
            }
            const int kq = (C.n >= 5 && T.block_qubits == 5) ? 5 : 4;
            if (C.n < kq)
                throw std::runtime_error("batch: circuit too small for the HBM path");
            // A tuned batch launches the blocks of states of less than 16 tiles one by one; in
            // rounds with others they fill the chip as well (256 circuits of 6-16 qubits, the
            // 15-qubit ones in BF16x3: 5033 launches before, 26 now).
            if (T.stage_bits > 0 && C.n >= T.stage_bits + (passes_ ? 1 : 4) && !rg.empty())
            {
                const auto plan = plan_stages(rg, C.n, T.stage_bits, kq);
                // batched gates span at most 2 qubits, so every stage has a tile
                bool all_tiled = true;
                for (const auto &st : plan)
                    all_tiled = all_tiled && !st.tile.empty();
                if (all_tiled)
                {
                    Staged sc{ci, {}};
                    for (const auto &st : plan)
                        sc.stages.push_back(prepare_stage(rg, st, kq, T.stage_bits, C.n, mats, x3_, false, &compose));
                    staged.push_back(std::move(sc));
                    continue;
                }
            }
            blocked.push_back(Blocked{ci, prepare_blocks(rg, plan_greedy(rg, kq), kq, C.n, mats, x3_, &compose)});
        }
        // largest first: round launches hand out the biggest states' tiles first, and with
        // sizes descending every state starts at a multiple of its own size
        std::stable_sort(staged.begin(), staged.end(), [&](const Staged &a, const Staged &b) { return circuits_[a.ci].n > circuits_[b.ci].n; });
        std::stable_sort(blocked.begin(), blocked.end(), [&](const Blocked &a, const Blocked &b) { return circuits_[a.ci].n > circuits_[b.ci].n; });
        uint64_t state_total = 0;
        size_t partial_total = 0;
        std::vector<uint64_t> state_off, partial_off; // staged circuits, then blocked ones
        auto place = [&](int ci) {
            state_off.push_back(state_total);
            partial_off.push_back(partial_total);
            state_total += uint64_t(1) << circuits_[ci].n;
            partial_total += size_t(qsv::zsum_blocks(circuits_[ci].n)) * 32;
        };
        for (const auto &sc : staged)
            place(sc.ci);
        for (const auto &bc : blocked)
            place(bc.ci);
        // ---- circuit passes: one program for all circuits, tasks per launch ----
        // Biggest circuits first: they have most passes, and most tiles to spread.
        std::stable_sort(passed.begin(), passed.end(), [&](const Passed &a, const Passed &b) {
            const int na = circuits_[a.ci].n, nb = circuits_[b.ci].n;
            return na != nb ? na > nb : a.plan.work > b.plan.work;
        });
        struct PassLaunch
        {
            int m;
            uint32_t tiles = 0;
            std::vector<qsv::PassTask> tasks;
            size_t offset = 0; // of the tasks in the program
        };
        // launches 0 .. 2: whole circuits on tiles of 2^10 .. 2^12; from 3 on: the rounds, of even
        // and odd circuits in turn, two chains that fill the ends of each other's launches
        // (96 circuits of 10-20 qubits: 1272 -> 1137 us)
        std::vector<PassLaunch> plaunch{{10}, {11}, {12}};
        size_t large_passed = 0;
        uint64_t sums_total = 0;
        // Circuits of one tile write their <Z> themselves where the batch has no others; with larger
        // ones there is a launch that adds up tiles' sums, and it does theirs too.  (12 circuits of
        // 7-9 qubits: 64.5 -> 62.4 us; 24 of 4-10: 28.4 -> 26.8.)
        const bool one_launch = passed.size() == circuits_.size() && std::all_of(passed.begin(), passed.end(), [&](const Passed &p) { return circuits_[p.ci].n <= p.plan.m; });
        std::vector<uint64_t> pass_state; // per passed circuit
        std::vector<size_t> pass_sums;
        for (const auto &pc : passed)
        {
            pass_state.push_back(state_total);
            pass_sums.push_back(sums_total);
            const int n = circuits_[pc.ci].n, m = pc.plan.m;
            if (n > m)
                state_total += uint64_t(1) << n;
            sums_total += (n > m ? uint64_t(1) << (n - m) : 1) * qsv::kPassSums;
        }
        // ---- device buffers (addresses go into the task arrays below) ----
        auto upload = [](void **dst, const void *src, size_t bytes) {
            if (bytes == 0)
                return;
            qsv::check(hipMalloc(dst, bytes), "hipMalloc batch");
            qsv::check(hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice), "batch upload");
        };
        upload((void **)&d_circs_, small.data(), small.size() * sizeof(qsv::BatchCircuit));
        upload((void **)&d_ops_, ops.data(), ops.size() * sizeof(qsv::BatchOp));
        qsv::check(hipMalloc((void **)&d_out_, std::max(1, total_qubits_) * sizeof(double)), "hipMalloc batch");
        qsv::check(hipMalloc((void **)&d_counter_, sizeof(unsigned)), "hipMalloc batch");
        if (state_total)
            qsv::check(hipMalloc((void **)&d_states_, state_total * sizeof(qsv::c64)), "hipMalloc batch states");
        if (partial_total)
            qsv::check(hipMalloc((void **)&d_partials_, partial_total * sizeof(double)), "hipMalloc batch");
        if (sums_total)
            qsv::check(hipMalloc((void **)&d_sums_, sums_total * sizeof(double)), "hipMalloc batch");
        // the program, written once: rounds, padding, operations, tasks of each launch, <Z> entries
        // (all multiples of 16 bytes)
        static_assert(sizeof(qsv::PassRound) % 16 == 0 && sizeof(qsv::PassOp) % 16 == 0 && sizeof(qsv::PassTask) % 16 == 0 && sizeof(qsv::PassZ) % 16 == 0, "pass program alignment");
        size_t nrounds = 0, nops = 0, ntasks = 0, nz = 0;
        for (const auto &pc : passed)
        {
            nrounds += pc.plan.rounds.size();
            nops += pc.plan.ops.size();
            ntasks += pc.plan.passes.size();
            nz += one_launch ? 0 : size_t(circuits_[pc.ci].n);
        }
        const size_t pops_off = qsv::pass_rounds_bytes(nrounds), tasks_off = pops_off + nops * sizeof(qsv::PassOp), pz_off = tasks_off + ntasks * sizeof(qsv::PassTask);
        // (one small circuit's task and entries are less than the padding of its operations)
        const size_t prog_bytes = passed.empty() ? 0 : std::max(pz_off + nz * sizeof(qsv::PassZ), pops_off + (nops + qsv::kPassOpPad) * sizeof(qsv::PassOp));
        const std::unique_ptr<char[]> prog(new char[prog_bytes]);
        auto put = [&](size_t at, const void *src, size_t bytes) { std::memcpy(prog.get() + at, src, bytes); };
        uint32_t first_round = 0, first_op = 0, pz_count = 0;
        for (size_t i = 0; i < passed.size(); ++i)
        {
            const Circuit &C = circuits_[passed[i].ci];
            const PassPlan &P = passed[i].plan;
            const int n = C.n, m = P.m;
            const uint32_t tiles = n > m ? uint32_t(1) << (n - m) : 1;
            put(pops_off + first_op * sizeof(qsv::PassOp), P.ops.data(), P.ops.size() * sizeof(qsv::PassOp));
            for (size_t k = 0; k < P.rounds.size(); ++k)
            {
                qsv::PassRound r = P.rounds[k];
                r.first += first_op;
                put((first_round + k) * sizeof r, &r, sizeof r);
            }
            for (size_t p = 0; p < P.passes.size(); ++p)
            {
                const auto &ps = P.passes[p];
                const size_t li = n > m ? 3 + 2 * p + large_passed % 2 : size_t(m - qsv::kPassMinBits);
                while (li >= plaunch.size())
                    plaunch.push_back(PassLaunch{qsv::kPassMaxBits});
                PassLaunch &L = plaunch[li];
                qsv::PassTask t{};
                t.state = n > m ? d_states_ + pass_state[i] : nullptr;
                t.sums = one_launch ? d_out_ + C.out_offset : d_sums_ + pass_sums[i];
                t.tile_begin = L.tiles;
                t.first_round = first_round + ps.first_round;
                t.nrounds = ps.nrounds;
                for (int b = 0; b < m; ++b)
                    t.tq[b / 4] |= uint32_t(ps.tq[b]) << (8 * (b % 4));
                auto bit_of = [&](uint32_t q) { return uint8_t(std::find(ps.tq, ps.tq + m, q) - ps.tq); };
                const qsv::PassRound &R = P.rounds[ps.first_round + ps.nrounds - 1];
                for (int j = 0; j < m; ++j)
                    t.zb[j] = bit_of(j < 4 ? R.rq[j] : R.tq[j - 4]);
                if (p == 0)
                    t.flags |= qsv::kPassZeroState;
                if (p + 1 == P.passes.size())
                {
                    t.flags |= qsv::kPassExpectZ | (one_launch ? uint32_t(n) << qsv::kPassQubits : 0);
                    uint32_t outside = 0; // qubits below q that are not tile qubits
                    for (int q = 0; q < n && !one_launch; ++q)
                    {
                        const int b = bit_of(q);
                        qsv::PassZ z{};
                        z.sums = t.sums;
                        z.out = d_out_ + C.out_offset + q;
                        z.ntiles = tiles;
                        z.slot = b < m ? 1 + b : 0;
                        z.sign = b < m ? 0 : uint32_t(1) << outside++;
                        put(pz_off + pz_count++ * sizeof z, &z, sizeof z);
                    }
                }
                L.tiles += tiles;
                L.tasks.push_back(t);
            }
            large_passed += n > m;
            first_round += uint32_t(P.rounds.size());
            first_op += uint32_t(P.ops.size());
        }
        size_t at = tasks_off;
        for (auto &L : plaunch)
        {
            L.offset = at;
            put(at, L.tasks.data(), L.tasks.size() * sizeof(qsv::PassTask));
            at += L.tasks.size() * sizeof(qsv::PassTask);
        }
        upload(&d_prog_, prog.get(), prog_bytes);
        // states within the 256 MB memory-side cache keep cached accesses
        const bool pass_nt = state_total * sizeof(qsv::c64) > (uint64_t(256) << 20);
        // ---- staged circuits: task arrays of the rounds, the fill and the reduction ----
        struct Round
        {
            size_t task_offset;
            int ntasks;
            uint64_t tiles;
        };
        std::vector<Round> rounds;
        size_t zsum_offset = 0;
        uint32_t zsum_blocks_total = 0, zsum_qubits_total = 0;
        const int kq_staged = T.block_qubits;
        if (!staged.empty())
        {
            size_t nrounds = 0;
            for (const auto &sc : staged)
                nrounds = std::max(nrounds, sc.stages.size());
            for (size_t r = 0; r < nrounds; ++r)
            {
                std::vector<qsv::StageTask> tasks;
                uint64_t tiles = 0;
                for (size_t i = 0; i < staged.size(); ++i)
                {
                    if (r >= staged[i].stages.size())
                        continue;
                    const PreparedStage &p = staged[i].stages[r];
                    if (p.kq != kq_staged)
                        throw std::runtime_error("batch: stage round with mixed block sizes");
                    tasks.push_back(stage_task(p, d_states_ + state_off[i], tiles));
                    if (r == 0)
                        tasks.back().flags = qsv::kStageZeroState; // the first stage starts from |0...0>
                    tiles += uint64_t(1) << (p.n - p.m);
                }
                rounds.push_back(Round{append_stage_tasks(mats, tasks), (int)tasks.size(), tiles});
            }
            std::vector<qsv::ZsumTask> zt;
            for (size_t i = 0; i < staged.size(); ++i)
            {
                const int n = circuits_[staged[i].ci].n;
                qsv::ZsumTask z{};
                z.state = d_states_ + state_off[i];
                z.part = d_partials_ + partial_off[i];
                z.out = d_out_ + circuits_[staged[i].ci].out_offset;
                z.block_begin = zsum_blocks_total;
                z.qubit_begin = zsum_qubits_total;
                z.n = n;
                z.nblocks = qsv::zsum_blocks(n);
                zsum_blocks_total += uint32_t(z.nblocks);
                zsum_qubits_total += uint32_t(n);
                zt.push_back(z);
            }
            static_assert(sizeof(qsv::ZsumTask) % 16 == 0, "ZsumTask keeps 16-B alignment");
            auto append = [&](const void *src, size_t bytes) {
                while (mats.size() % 4)
                    mats.push_back(0.f);
                const size_t off = mats.size();
                mats.resize(off + (bytes + sizeof(float) - 1) / sizeof(float));
                std::memcpy(mats.data() + off, src, bytes);
                return off;
            };
            zsum_offset = append(zt.data(), zt.size() * sizeof(qsv::ZsumTask));
        }
        const size_t room_at = compose.append(mats);
        for (const auto &sc : staged)
            for (const auto &st : sc.stages)
                move_matrices(st, room_at, mats);
        for (auto &bc : blocked)
            for (auto &b : bc.blocks)
                b.matrix_offset += room_at;
        if (!mats.empty())
        {
            qsv::check(hipMalloc((void **)&d_mats_, (compose.room > 0 ? room_at + compose.room : mats.size()) * sizeof(float)), "hipMalloc batch");
            qsv::check(hipMemcpy(d_mats_, mats.data(), mats.size() * sizeof(float), hipMemcpyHostToDevice), "batch upload");
        }
        // algorithmic traffic and launches of one run (see qcs_ext_batch_traffic)
        hbm_bytes_ = 0;
        launches_ = small.empty() ? 0 : 2;
        if (!staged.empty())
        {
            for (const auto &sc : staged)
            {
                // the first stage writes without reading; the reduction reads once
                const double amps = double(uint64_t(1) << circuits_[sc.ci].n);
                hbm_bytes_ += 16.0 * amps * double(sc.stages.size()) - 8.0 * amps + 8.0 * amps;
            }
            launches_ += rounds.size() + 2;
        }
        for (const auto &bc : blocked)
        {
            const double amps = double(uint64_t(1) << circuits_[bc.ci].n);
            hbm_bytes_ += 16.0 * amps * double(bc.blocks.size()) + 8.0 * amps + 8.0 * amps;
            launches_ += 1 + bc.blocks.size() + 2;
        }
        for (const auto &pc : passed)
        {
            // the first pass does not read, the last does not write
            const double amps = double(uint64_t(1) << circuits_[pc.ci].n);
            if (circuits_[pc.ci].n > pc.plan.m)
                hbm_bytes_ += 16.0 * amps * double(pc.plan.passes.size() - 1);
        }
        for (const auto &L : plaunch)
            launches_ += L.tasks.empty() ? 0 : 1;
        launches_ += pz_count > 0;
        int grid = 0;
        if (!small.empty())
        {
            qsv::batch_prepare(T.block_size, small_max_n);
            grid = std::min<int>(qsv::batch_lds_grid(T.block_size, small_max_n), (int)small.size());
        }
        // ---- streams and graph capture ----
        // no more streams than chains of launches
        int chains = int(!small.empty()) + int(!staged.empty()) + (blocked.empty() ? 0 : T.streams) + int(std::min<size_t>(large_passed, 2));
        for (int i = 0; i < 3; ++i)
            chains += int(!plaunch[i].tasks.empty());
        const int ns = std::clamp(chains, 1, T.streams);
        make_streams(ns);
        for (int i = 0; i < 2 * ns; ++i)
        {
            hipEvent_t e;
            qsv::check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
            fork_join_.push_back(e);
        }
        hipStream_t s0 = streams_[0];
        compose.launch(s0, d_mats_);
        qsv::check(hipStreamSynchronize(s0), "hipStreamSynchronize");
        const int nsmall = (int)small.size();
        const int nstaged = (int)staged.size();
        std::vector<uint64_t> blocked_state(state_off.begin() + nstaged, state_off.end());
        std::vector<uint64_t> blocked_partial(partial_off.begin() + nstaged, partial_off.end());
        // the whole batch as launches on the streams: captured once into the graph below,
        // or issued directly by run_direct
        work_ = [this, blocked = std::move(blocked), blocked_state, blocked_partial, rounds, nstaged, kq_staged,
                 stage_bits = T.stage_bits, zsum_offset, zsum_blocks_total, zsum_qubits_total, grid, nsmall,
                 small_max_n, ns, block_size = T.block_size, x3 = x3_, plaunch, plaunch_empty = passed.empty(), pops_off, pz_off, pz_count, pass_nt]() mutable {
            hipStream_t s0 = streams_[0];
            qsv::check(hipEventRecord(fork_join_[0], s0), "hipEventRecord");
            for (int i = 1; i < ns; ++i)
                qsv::check(hipStreamWaitEvent(streams_[i], fork_join_[0], 0), "hipStreamWaitEvent");
            if (nsmall > 0)
                qsv::launch_batch_lds(s0, block_size, grid, small_max_n, d_circs_, nsmall, d_ops_, d_out_, d_counter_);
            // the LDS kernel occupies s0; the stage rounds take the next stream, the blocked
            // circuits (biggest first) the ones after it
            int next = 0;
            auto stream = [&]() { return streams_[ns == 1 ? 0 : 1 + (next++) % (ns - 1)]; };
            // the longest chains first, each on its own stream while there are some: the pass
            // rounds, the stage rounds, each kind of whole circuits
            const auto *prog = static_cast<const char *>(d_prog_);
            auto launch_tasks = [&](hipStream_t s, const PassLaunch &L) {
                qsv::launch_pass_tasks(s, L.m, pass_nt, reinterpret_cast<const qsv::PassTask *>(prog + L.offset), int(L.tasks.size()), L.tiles,
                                       reinterpret_cast<const qsv::PassRound *>(prog), reinterpret_cast<const qsv::PassOp *>(prog + pops_off));
            };
            int chain = 0;
            auto chain_stream = [&] { return streams_[size_t(chain++) % size_t(ns)]; };
            for (size_t g = 3; g < 5 && g < plaunch.size(); ++g)
            {
                hipStream_t s = chain_stream();
                for (size_t i = g; i < plaunch.size(); i += 2)
                    if (!plaunch[i].tasks.empty())
                        launch_tasks(s, plaunch[i]);
            }
            if (nstaged > 0)
            {
                hipStream_t s = plaunch_empty ? stream() : chain_stream();
                for (const auto &r : rounds)
                    launch_stage_tasks(s, kq_staged, stage_bits, x3, d_mats_, r.task_offset, r.ntasks, r.tiles);
                qsv::launch_zsum_tasks(s, reinterpret_cast<const qsv::ZsumTask *>(d_mats_ + zsum_offset), nstaged, zsum_blocks_total, zsum_qubits_total);
            }
            for (size_t i = 3; i-- > 0;)
                if (!plaunch[i].tasks.empty())
                    launch_tasks(chain_stream(), plaunch[i]);
            for (size_t i = 0; i < blocked.size(); ++i)
            {
                const Circuit &C = circuits_[blocked[i].ci];
                hipStream_t s = stream();
                qsv::c64 *st = d_states_ + blocked_state[i];
                qsv::launch_fill_zero_c64(s, st, uint64_t(1) << C.n);
                for (auto &b : blocked[i].blocks)
                    launch_prepared(s, st, C.n, b, d_mats_);
                qsv::launch_zsum(s, st, C.n, d_partials_ + blocked_partial[i], d_out_ + C.out_offset);
            }
            for (int i = 1; i < ns; ++i)
            {
                qsv::check(hipEventRecord(fork_join_[ns + i], streams_[i]), "hipEventRecord");
                qsv::check(hipStreamWaitEvent(s0, fork_join_[ns + i], 0), "hipStreamWaitEvent");
            }
            if (pz_count > 0)
                qsv::launch_pass_z(s0, reinterpret_cast<const qsv::PassZ *>(prog + pz_off), pz_count);
        };
        qsv::check(hipStreamBeginCapture(s0, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
        try
        {
            work_();
        }
        catch (...)
        {
            hipGraph_t g = nullptr;
            (void)hipStreamEndCapture(s0, &g);
            if (g)
                (void)hipGraphDestroy(g);
            throw;
        }
        qsv::check(hipStreamEndCapture(s0, &graph_), "hipStreamEndCapture");
        size_t nodes = 0;
        qsv::check(hipGraphGetNodes(graph_, nullptr, &nodes), "hipGraphGetNodes");
        graph_nodes_ = nodes;
        qsv::check(hipGraphInstantiate(&exec_, graph_, nullptr, nullptr, 0), "hipGraphInstantiate");
        prepared_ = true;
    }

    double Batch::run(double *expz)
    {
        prepare();
        hipStream_t s0 = streams_[0];
        qsv::check(hipEventRecord(t0_, s0), "hipEventRecord");
        qsv::check(hipGraphLaunch(exec_, s0), "hipGraphLaunch");
        qsv::check(hipEventRecord(t1_, s0), "hipEventRecord");
        qsv::check(hipEventSynchronize(t1_), "hipEventSynchronize");
        float ms = 0;
        qsv::check(hipEventElapsedTime(&ms, t0_, t1_), "hipEventElapsedTime");
        if (expz)
            qsv::check(hipMemcpy(expz, d_out_, total_qubits_ * sizeof(double), hipMemcpyDeviceToHost), "batch copy");
        return ms * 1e-3;
    }

    double Batch::run_direct(double *expz)
    {
        prepare();
        hipStream_t s0 = streams_[0];
        qsv::check(hipEventRecord(t0_, s0), "hipEventRecord");
        work_();
        qsv::check(hipEventRecord(t1_, s0), "hipEventRecord");
        qsv::check(hipEventSynchronize(t1_), "hipEventSynchronize");
        float ms = 0;
        qsv::check(hipEventElapsedTime(&ms, t0_, t1_), "hipEventElapsedTime");
        if (expz)
            qsv::check(hipMemcpy(expz, d_out_, total_qubits_ * sizeof(double), hipMemcpyDeviceToHost), "batch copy");
        return ms * 1e-3;
    }

    double Batch::run_plain(double *expz)
    {
        std::map<int, std::unique_ptr<Simulator>> sims;
        const auto t0 = std::chrono::steady_clock::now();
        for (const auto &c : circuits_)
        {
            auto &sim = sims[c.n];
            if (!sim)
            {
                sim = std::make_unique<Simulator>();
                sim->num_qubits_cfg = c.n;
                sim->allocate();
            }
            else
                sim->set_zero_state();
            for (const auto &g : c.gates)
            {
                std::vector<int> pos;
                if (g.control >= 0)
                    pos.push_back(g.control);
                sim->operate(make_gate(g.name.c_str(), g.params), {g.target}, {}, pos);
            }
            std::vector<double> z(c.n);
            sim->expect_z(z.data(), c.n);
            if (expz)
                std::copy(z.begin(), z.end(), expz + c.out_offset);
        }
        return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    }

    BatchTuning Batch::autotune()
    {
        auto time = [&] {
            run(nullptr); // warm-up (first replay)
            double best = 1e30;
            for (int r = 0; r < 2; ++r)
                best = std::min(best, run(nullptr));
            return best;
        };
        auto measure = [&](const BatchTuning &t) {
            set_tuning(t);
            return time();
        };
        const BatchTuning untuned = tuning_;
        const double passes_s = passes_ ? time() : 1e30;
        BatchTuning best = tuning_;
        double best_s = measure(best);
        auto try_set = [&](auto setter, std::initializer_list<int> values) {
            for (int v : values)
            {
                BatchTuning t = best;
                setter(t, v);
                double s = measure(t);
                if (s < best_s)
                {
                    best_s = s;
                    best = t;
                }
            }
        };
        try_set([](BatchTuning &t, int v) { t.lds_max_qubits = v; }, {12, 13, 14});
        try_set([](BatchTuning &t, int v) { t.block_size = v; }, {256, 512, 1024});
        // block size and stage tile size together: the better block size depends on the
        // tile (FP32 products favour 4-qubit blocks, BF16x3 ones 5-qubit blocks on some tiles)
        try_set([](BatchTuning &t, int v) { t.block_qubits = v / 16; t.stage_bits = v % 16; },
                {4 * 16 + 0, 4 * 16 + 11, 4 * 16 + 12, 4 * 16 + 13, 5 * 16 + 0, 5 * 16 + 11, 5 * 16 + 12, 5 * 16 + 13});
        try_set([](BatchTuning &t, int v) { t.streams = v; }, {1, 2, 4});
        if (passes_s <= best_s)
        { // as before the search
            set_tuning(untuned);
            passes_ = true;
            return untuned;
        }
        set_tuning(best);
        return best;
    }
} // namespace qcore
