// Pass launches refuse programs off their types' alignment before anything is launched (the
// pointers here are never read: with aligned ones the tile's qubits are refused next).
#include "pass_kernels.hpp"

#include <cstdio>
#include <stdexcept>
#include <string>

template <class F>
static std::string refusal(F f)
{
    try
    {
        f();
    }
    catch (const std::exception &e)
    {
        return e.what();
    }
    return "accepted";
}

int main()
{
    static_assert(alignof(qsv::PassOp) == 64 && alignof(qsv::PassRound) == 16 && sizeof(qsv::PassOp) == 64, "sizes of the program's parts");
    for (size_t count = 1; count < 40; ++count)
        if (qsv::pass_rounds_bytes(count) % 64 || qsv::pass_rounds_bytes(count) < count * sizeof(qsv::PassRound) || qsv::pass_rounds_bytes(count) >= count * sizeof(qsv::PassRound) + 64)
            return std::printf("rounds of %zu\n", count), 1;
    auto *state = reinterpret_cast<qsv::c128 *>(uintptr_t(1) << 20);
    auto *tasks = reinterpret_cast<qsv::PassTask *>(uintptr_t(1) << 20);
    const uint8_t tq[16] = {}; // not ascending: refused after the program
    for (uintptr_t r : {0, 16, 64, 8, 4})
        for (uintptr_t o : {0, 64, 128, 16, 32, 48, 8})
        {
            const auto *rounds = reinterpret_cast<const qsv::PassRound *>((uintptr_t(1) << 20) + r);
            const auto *ops = reinterpret_cast<const qsv::PassOp *>((uintptr_t(1) << 21) + o);
            const bool bad = r % 16 || o % 64;
            const std::string one = refusal([&] { qsv::launch_pass(nullptr, state, 12, 12, tq, rounds, 1, ops); });
            if ((one.find("aligned") != std::string::npos) != bad || (!bad && one.find("ascending") == std::string::npos))
                return std::printf("launch_pass, rounds + %d, operations + %d: %s\n", int(r), int(o), one.c_str()), 1;
            const std::string many = refusal([&] { qsv::launch_pass_tasks(nullptr, 9, false, tasks, 1, 1, rounds, ops); });
            if ((many.find("aligned") != std::string::npos) != bad || (!bad && many.find("tile size") == std::string::npos))
                return std::printf("launch_pass_tasks, rounds + %d, operations + %d: %s\n", int(r), int(o), many.c_str()), 1;
        }
    std::printf("ok\n");
    return 0;
}
