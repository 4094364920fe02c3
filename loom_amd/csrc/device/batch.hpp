// -*- C++ -*-
/// @file batch.hpp
/// @brief Many launches of different kernels and uneven thread counts in one
/// persistent gfx950 kernel.
///
/// The reference runs several kernels of uneven sizes concurrently with its
/// multi-stream Shop: CPU worker threads round-robin over a bench of
/// per-kernel streams (mp.hpp:158-190, 316-385).  Here one persistent launch
/// takes a table of jobs (kernel, thread range, input/output columns) whose
/// kernels all belong to one compiled batch set.  A wave claims guided
/// chunks of one job, runs them with in-wave refill from the same job, and
/// moves to another job when that one is exhausted; waves start on
/// different jobs (spread by workgroup index) so small and large jobs run
/// side by side.  The register file of a wave is the union of the member
/// kernels' (the largest sets the occupancy).
#pragma once

#include "sched.hpp"

namespace loom::hipvm
{
inline constexpr std::uint32_t kMaxJobs = 64;

/// @brief Waves per SIMD that the sweep policy's batch kernels with member
/// @p K are compiled to allow at least (as waves_hint;
/// LOOM_HIP_BATCH_WAVES_HINT): the largest of their members' hints.  The
/// other policies keep more registers live across a dispatch and are left to
/// the compiler: held to the path tracer's hint they spill 40 to 52 bytes a
/// lane (16 mixed jobs of 20,011 threads, left alone and held: 698 and 828 us
/// under the topological policy, 888 and 1064 under successor-major).
template <typename K>
inline constexpr int batch_waves_hint = 1;
template <int P, typename... Ks>
inline constexpr int batch_waves = []
{
    int w = 1;
    if constexpr(P == POLICY_SWEEP) ((w = batch_waves_hint<Ks> > w ? batch_waves_hint<Ks> : w), ...);
    return w;
}();

/// @brief One job of a batch (device copy of loom_job).
struct JobDesc
{
    std::uint32_t member = 0; ///< index of the kernel in the batch set
    std::uint32_t pad    = 0;
    std::uint64_t begin = 0, end = 0;
    const void*   in[kMaxIO]{};
    void*         out[kMaxIO]{};
};

struct BatchCtl
{
    Slot64 next[kMaxJobs]; ///< claim cursor of each job, one per 256-byte block
};

struct BatchArgs
{
    const JobDesc* jobs    = nullptr;
    BatchCtl*      ctl     = nullptr;
    std::uint32_t  njobs   = 0;
};

/// @brief Claim a guided chunk of job @p j: returns the count.
LOOM_DEVICE std::uint32_t
claim_job_chunk(BatchCtl* ctl, const JobDesc* J, std::uint32_t j, std::uint32_t chunk,
                std::uint64_t& base)
{
    std::uint64_t b = 0;
    std::uint32_t got = 0;
    if(lane_id() == 0)
    {
        const std::uint64_t e = J[j].end;
        const std::uint64_t k = atomicAdd(reinterpret_cast<unsigned long long*>(&ctl->next[j].v),
                                          static_cast<unsigned long long>(chunk));
        if(k < e)
        {
            b   = k;
            got = static_cast<std::uint32_t>(e - k < chunk ? e - k : chunk);
        }
    }
    base = uniform64(b);
    return uniform(got);
}

/// @brief Run job @p j (kernel K) on this wave until the job has no more
/// threads to admit and every lane halted: its pool of started threads is
/// empty again then, so all jobs share one.
template <typename K, int P, bool CNT, std::size_t Columns>
LOOM_DEVICE void
run_job(const BatchArgs& a, std::uint32_t j, const CtlArgs& c, CtxOf<CNT>& w, std::uint64_t& admitted)
{
    const JobDesc*      J   = a.jobs;
    const std::uint64_t len = J[j].end - J[j].begin;
    // chunk: the job spread over about four claims per wave that starts on
    // it (gridDim.x / njobs waves do), one batch at least, 512 at most
    const std::uint64_t per = len * a.njobs / (4ull * gridDim.x);
    const std::uint32_t chunk = static_cast<std::uint32_t>(per < 64 ? 64 : (per > 512 ? 512 : per));
    std::uint64_t rbase = 0;
    std::uint32_t rcount = 0;
    bool          exhausted = false;

    Lanes<K, P, RegsOf<K, CNT>, Columns> l;
    bool                                 force = true;

    auto input = [&](std::uint32_t want)
    {
        if(rcount == 0 && !exhausted)
        {
            rcount    = claim_job_chunk(a.ctl, J, j, chunk, rbase);
            exhausted = rcount == 0;
        }
        Taken t;
        t.count = t.head = rcount < want ? rcount : want;
        t.base           = static_cast<std::uint32_t>(rbase);
        rbase += t.count;
        rcount -= t.count;
        return t;
    };

    for(;;)
    {
        if constexpr(CNT) flush_if_high(w);
        const std::uint64_t live = ballot(l.has);
        if(~live && l.input_left() && l.refill(~live, J[j], w, input, admitted)) force = true;
        if((l.pooled && CNT && w.over) || !ballot(l.has)) return;
        run_policy<K, P, l.pooled>(l.r, l.pc, 0, l.input_left() ? c.live_thr : 0u, force, w);
        force = false;
        if(l.has && l.pc == HALT)
        {
            store_outputs<K>(l.r, J[j].out, l.tid);
            l.has = false;
        }
        if(w.over) return;
    }
}

template <typename... Ks>
struct BatchSet
{
    static constexpr std::uint32_t size = sizeof...(Ks);
};

/// @brief The persistent batch kernel over the kernels @p Ks (policy @p P;
/// CNT: with work counts, else for runs that count none, see plain_run).
template <int P, bool CNT, typename... Ks>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(batch_waves<P, Ks...>))) void
batch_kernel(CtlArgs c, BatchArgs a)
{
    (sct_table_init<Ks>(), ...);
    CtxOf<CNT> w(c);
    std::uint64_t admitted = 0;
    const std::uint32_t nj = a.njobs;
    // each wave walks the job list from its own start, so jobs of every size
    // are worked on from the beginning
    for(std::uint32_t step = 0; step < nj && !w.over; ++step)
    {
        const std::uint32_t j = (blockIdx.x + step) % nj;
        // skip exhausted jobs cheaply
        if(uniform64(__hip_atomic_load(&a.ctl->next[j].v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) >=
           a.jobs[j].end)
            continue;
        const std::uint32_t m = a.jobs[j].member;
        std::uint32_t       idx = 0;
        (
            [&]
            {
                if(m == idx) run_job<Ks, P, CNT, pool_columns<Ks...>>(a, j, c, w, admitted);
                ++idx;
            }(),
            ...);
    }
    flush_stats(w);
    if(CNT && c.stats && lane_id() == 0)
        atomicAdd(&stat_slot(c)[ST_ADMITTED], static_cast<unsigned long long>(admitted));
    raise_errors(w.err, w.over, c);
}
} // namespace loom::hipvm
