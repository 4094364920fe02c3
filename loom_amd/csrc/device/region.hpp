// -*- C++ -*-
/// @file region.hpp
/// @brief Regions of a kernel's control-flow graph: groups of blocks that a
/// sweep runs as one piece of structured lane code.
///
/// A sweep dispatches blocks one by one: a compare of the program counter, a
/// ballot, a branch, the block under its mask, a select of the next program
/// counter.  For a kernel of small blocks that bookkeeping is most of the
/// work (Collatz: 22 vector and as many scalar instructions per trip of a
/// loop that needs nine).  A region is entered only at its leader, so its
/// other blocks need no dispatch of their own: their conditions are branches
/// within the lane code, which the compiler turns into selects and masks,
/// and a region that is a loop keeps looping on the spot.  Measured on runs
/// without statistics: Collatz, 2^24 threads, 3.2 ms by blocks and 1.42 ms by
/// regions (11 vector instructions a trip); fib, 2^20 threads, 48 and 25 us.
///
/// Leaders are START, the targets of back edges, and every block whose
/// predecessors lie in different regions or in another loop (or in a START
/// that is pooled, pool.hpp).  A block joins
/// the region of its predecessors only within the same set of loops: the
/// code after a loop is a region of its own, which lanes leaving the loop at
/// different trips reach together.
#pragma once

#include "pool.hpp"

namespace loom::hipvm
{
template <typename K>
struct Regions
{
    static constexpr std::size_t nb = ir::table_of<K>.nb;

    struct Map
    {
        std::array<std::uint8_t, 64>  of{};      ///< region (its leader) of each block
        std::array<std::uint8_t, 64>  rpo{};     ///< blocks in reverse post-order
        std::array<std::uint8_t, 64>  count{};   ///< blocks of the region of a leader
        std::array<bool, 64>          loops{};   ///< the leader has a back edge from its region
        std::array<bool, 64>          outer{};   ///< no loop but the leader's own contains it
        std::array<std::uint32_t, 64> exit{};    ///< the only successor outside, NONE if several
    };

    static constexpr Map map = []
    {
        constexpr const auto& T = ir::table_of<K>;
        Map                   m;
        // reverse post-order of a depth-first walk from START; blocks that
        // are never reached follow it
        std::array<std::uint8_t, 64> state{}, stack{}, next{}, post{};
        std::size_t                  sp = 0, np = 0, n = 0;
        stack[sp++] = 0;
        state[0]    = 1;
        while(sp)
        {
            const std::uint8_t b = stack[sp - 1];
            if(next[b] < T.block[b].ns)
            {
                const auto s = T.succ[T.block[b].s0 + next[b]++];
                if(s == ir::halt16 || state[s]) continue;
                state[s]    = 1;
                stack[sp++] = static_cast<std::uint8_t>(s);
            }
            else
            {
                post[np++] = b;
                --sp;
            }
        }
        for(std::size_t k = np; k-- > 0;) m.rpo[n++] = post[k];
        for(std::size_t b = 0; b < nb; ++b)
            if(!state[b]) m.rpo[n++] = static_cast<std::uint8_t>(b);
        // loops that hold each block, as a mask over the loop heads
        std::array<std::uint64_t, 64> in_loops{};
        std::array<bool, 64>          head{};
        for(std::size_t h = 0; h < T.nhead; ++h)
        {
            head[T.head[h]] = true;
            for(std::size_t b = 0; b < nb; ++b)
                if(b == T.head[h] || ((T.body[h] >> b) & 1u)) in_loops[b] |= 1ull << h;
        }
        for(std::size_t k = 0; k < nb; ++k)
        {
            const std::uint8_t b = m.rpo[k];
            // the region of its predecessors, if they agree; a block that is
            // no loop head has all of them before it in this order
            std::uint32_t r = NONE;
            if(b != 0 && !head[b] && state[b])
                for(std::size_t p = 0; p < nb; ++p)
                    for(std::size_t j = 0; j < T.block[p].ns; ++j)
                        if(T.succ[T.block[p].s0 + j] == b)
                            r = (r == NONE || r == m.of[p]) && in_loops[m.of[p]] == in_loops[b] ?
                                    m.of[p] :
                                    64u;
            // a pooled START runs alone: its threads enter the sweep after it
            if(r == 0 && StartPool<K>::used) r = 64u;
            m.of[b] = r < 64u ? static_cast<std::uint8_t>(r) : b;
            ++m.count[m.of[b]];
        }
        for(std::size_t l = 0; l < nb; ++l)
        {
            if(m.of[l] != l) continue;
            std::uint64_t other = in_loops[l];
            for(std::size_t h = 0; h < T.nhead; ++h)
                if(T.head[h] == l) other &= ~(1ull << h);
            m.outer[l] = other == 0;
            std::uint32_t out = HALT + 1; // none yet
            for(std::size_t b = 0; b < nb; ++b)
            {
                if(m.of[b] != l) continue;
                bool halts = T.block[b].ns == 0;
                for(std::size_t j = 0; j < T.block[b].ns; ++j)
                {
                    const auto s = T.succ[T.block[b].s0 + j];
                    if(s == ir::halt16)
                        halts = true;
                    else if(s == l)
                        m.loops[l] = true;
                    else if(m.of[s] != l)
                        out = out == HALT + 1 || out == s ? s : NONE;
                }
                // a jump table goes to HALT past its last label
                const auto& blk = T.block[b];
                for(std::size_t i = blk.i0; i < std::size_t(blk.i0 + blk.ni); ++i)
                    if(T.instr[i].kind == SK::pjump && T.instr[i].nt != 2) halts = true;
                if(halts) out = out == HALT + 1 || out == HALT ? HALT : NONE;
            }
            m.exit[l] = out == HALT + 1 ? NONE : out;
        }
        return m;
    }();
};

/// @brief Run the blocks of the region of leader @p L on a lane at L: L
/// itself, then the others in reverse post-order where the lane is at them.
template <typename K, std::size_t L>
LOOM_DEVICE void
exec_region(Regs<K>& r, std::uint32_t& pc, std::uint32_t& err)
{
    exec_block<K, L>(r, pc, err);
    [&]<std::size_t... I>(std::index_sequence<I...>)
    {
        (
            [&]
            {
                constexpr std::size_t B = Regions<K>::map.rpo[I];
                if constexpr(B != L && Regions<K>::map.of[B] == L)
                    if(pc == B) exec_block<K, B>(r, pc, err);
            }(),
            ...);
    }(std::make_index_sequence<ir::table_of<K>.nb>{});
}
} // namespace loom::hipvm
