// -*- C++ -*-
/// @file pool.hpp
/// @brief A wave's pool of started threads, in LDS.
///
/// A wave that refills its free lanes runs START on those lanes alone: the
/// path tracer's START is a quarter of a bounce's instructions and ran on 16
/// of 64 lanes, which also kept the refill threshold low (48).  With a pool
/// START runs on 64 new threads at once; what is live after it (the registers
/// live into its successors, the thread id, the next block if there are
/// several) waits in LDS, one column of 64 words each, and a refill reads it
/// from there.  Registers that START sets to a literal are set again at the
/// refill instead.  Threads that halt in START never enter the pool.
///
/// The path tracer's 1024x768x64 frame: 7.18 ms without the pool (refilled at 48
/// lanes, 72% of the lanes active), 6.44 with it (refilled at 60, 81%).
///
/// Used where it pays: START of at least kPoolMinOps operations that no other
/// block jumps back to, with few enough words live after it (lds_per_wave), in
/// waves that own their workgroup's LDS.
#pragma once

#include "exec.hpp"

namespace loom::hipvm
{
/// Operations of a START worth pooling.  Below, reading the pool costs about
/// what START does (fib and Collatz with 3 operations, pooled: 2-14% slower;
/// the cubic with 4: even).  From 26 to 98 operations the pool pays where the
/// threads do work between refills: loops of 32 or 68 operations and 1 to 32
/// trips, refilled at 48 lanes, took 0.68 to 0.96 of the time without it
/// (12,000,003 threads; 3,000,017: 0.86 to 1.00; 200,003, where few refills
/// happen: 0.98 to 1.04).  Where the columns are the cost (8 operations and a
/// few trips) it is up to 10% slower, at 26 as at 98 operations; trip counts
/// are not known here.
inline constexpr std::uint32_t kPoolMinOps = 24;

/// @brief 32-bit words of the registers in @p live.
template <typename K>
constexpr std::size_t
words_of(const ir::Bits& live)
{
    std::size_t n = 0;
    for(std::size_t r = 0; r < ir::table_of<K>.nr; ++r)
        if(live.test(r)) n += ir::table_of<K>.reg[r].width == 8 ? 2 : 1;
    return n;
}

/// @brief LDS that a one-wave workgroup of @p K may use before it holds fewer
/// waves than registers allow.  What is live at a block is in VGPRs there, 512
/// a lane for all waves of a SIMD, of which eight fit at most; a CU has four
/// SIMDs and 160 KB of LDS in granules of 1280 bytes: 5120 bytes (20 words a
/// lane) where all eight fit, more for kernels with much live state.
template <typename K>
inline constexpr std::size_t lds_per_wave = []
{
    std::size_t words = 1;
    for(std::size_t b = 0; b < ir::table_of<K>.nb; ++b)
    {
        const std::size_t w = words_of<K>(ir::table_of<K>.block[b].live_in);
        words               = w > words ? w : words;
    }
    const std::size_t fit   = 512 / ((words + 7) / 8 * 8);
    const std::size_t waves = fit < 1 ? 1 : (fit > 8 ? 8 : fit);
    return 160 * 1024 / (4 * waves) / 1280 * 1280;
}();

template <typename K>
struct StartPool
{
    static constexpr std::size_t none = ~std::size_t(0);

    /// the instruction that sets register @p r to a literal for good in START
    static constexpr std::size_t
    literal(std::size_t r)
    {
        constexpr const auto& T  = ir::table_of<K>;
        std::size_t           at = none;
        for(std::size_t i = T.block[0].i0; i < std::size_t(T.block[0].i0 + T.block[0].ni); ++i)
        {
            const ir::Instr& in = T.instr[i];
            if(in.kind != SK::compute || T.opnd[in.dst].slot != r) continue;
            at = in.op == Op::mov && T.opnd[in.a0].lit ? i : none;
        }
        return at;
    }

    struct Map
    {
        std::array<std::uint16_t, 2 * ir::max_regs> reg{};  ///< register of each word
        std::array<std::uint8_t, 2 * ir::max_regs>  half{}; ///< upper half of a 64-bit one
        std::array<bool, ir::max_regs>              live{}; ///< live after START
        std::size_t                                 n    = 0;
        std::size_t                                 succ = 0; ///< successors but HALT
        std::uint32_t                               next = 0; ///< the last of them
        bool                                        back = false;
    };

    static constexpr Map map = []
    {
        constexpr const auto& T = ir::table_of<K>;
        Map                   m;
        ir::Bits              any{};
        for(std::size_t j = 0; j < T.block[0].ns; ++j)
        {
            const auto s = T.succ[T.block[0].s0 + j];
            if(s == ir::halt16) continue;
            any = any | T.block[s].live_in;
            if(m.succ == 0 || m.next != s) ++m.succ;
            m.next = s;
        }
        for(std::size_t b = 0; b < T.nb; ++b)
            for(std::size_t j = 0; j < T.block[b].ns; ++j)
                m.back |= T.succ[T.block[b].s0 + j] == 0;
        for(std::size_t r = 0; r < T.nr; ++r)
        {
            m.live[r] = any.test(r);
            if(!m.live[r] || literal(r) != none) continue;
            for(std::uint8_t h = 0; h < (T.reg[r].width == 8 ? 2 : 1); ++h)
            {
                m.reg[m.n]    = static_cast<std::uint16_t>(r);
                m.half[m.n++] = h;
            }
        }
        return m;
    }();

    /// columns: the words of the registers, the thread id, the next block
    static constexpr std::size_t columns = map.n + 1 + (map.succ > 1 ? 1 : 0);

    static constexpr bool used =
        ir::table_of<K>.block[0].ops >= kPoolMinOps && map.succ != 0 && !map.back &&
        columns * 256 + SctTable<K>::words * 4 <= lds_per_wave<K>;
};

/// @brief Columns of the pool of a wave that runs the kernels @p Ks one after
/// the other: the largest of theirs.
template <typename... Ks>
inline constexpr std::size_t pool_columns = []
{
    std::size_t n = 1;
    ((n = StartPool<Ks>::used && StartPool<Ks>::columns > n ? StartPool<Ks>::columns : n), ...);
    return n;
}();

template <std::size_t Columns>
__shared__ std::uint32_t start_pool[Columns * 64];

/// @brief Put this lane's thread, started, into row @p row of the pool @p C.
template <typename K, std::size_t C>
LOOM_DEVICE void
pool_write(const Regs<K>& r, std::uint32_t pc, std::uint32_t tid, std::uint32_t row)
{
    using M = StartPool<K>;
    [&]<std::size_t... W>(std::index_sequence<W...>)
    {
        ((start_pool<C>[W * 64 + row] = static_cast<std::uint32_t>(
              r.template raw<M::map.reg[W]>() >> (M::map.half[W] ? 32 : 0))),
         ...);
    }(std::make_index_sequence<M::map.n>{});
    start_pool<C>[M::map.n * 64 + row] = tid;
    if constexpr(M::map.succ > 1) start_pool<C>[(M::map.n + 1) * 64 + row] = pc;
}

/// @brief Take the thread of row @p row into this lane; returns its id.
template <typename K, std::size_t C>
LOOM_DEVICE std::uint32_t
pool_read(Regs<K>& r, std::uint32_t& pc, std::uint32_t row)
{
    using M = StartPool<K>;
    [&]<std::size_t... W>(std::index_sequence<W...>)
    {
        (
            [&]
            {
                constexpr std::size_t R = M::map.reg[W];
                const std::uint64_t   v = start_pool<C>[W * 64 + row];
                if constexpr(M::map.half[W] != 0)
                    r.template set_raw<R>((r.template raw<R>() & 0xFFFFFFFFull) | (v << 32));
                else
                    r.template set_raw<R>(v);
            }(),
            ...);
    }(std::make_index_sequence<M::map.n>{});
    std::uint32_t none = HALT, err = 0;
    [&]<std::size_t... R>(std::index_sequence<R...>)
    {
        (
            [&]
            {
                if constexpr(M::map.live[R] && M::literal(R) != M::none)
                    exec_instr<K, M::literal(R)>(r, none, err);
            }(),
            ...);
    }(std::make_index_sequence<ir::table_of<K>.nr>{});
    if constexpr(M::map.succ > 1)
        pc = start_pool<C>[(M::map.n + 1) * 64 + row];
    else
        pc = M::map.next;
    return start_pool<C>[M::map.n * 64 + row];
}
} // namespace loom::hipvm
