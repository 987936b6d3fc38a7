#pragma once
// The device code of the lifted matching (lifted.hpp) and the kernels built on it: the env step, the counts, the flat
// expansion and the successor listing. A block holds up to kMaxWaves wavefronts; each wave works on one state at a time
// in its own LDS region. Waves of a block run different states, so every barrier inside the per-state work is a
// wavefront barrier. Included by one translation unit per MYA_GENERAL_TASKS: 0, for tasks whose preconditions are all read
// as candidate words and whose schemas have at most kLaneDepth + 1 parameters (TaskDev::simple); 1, for any task: literals
// checked one by one (k-ary, repeated variables, ground) and nested counts that go on past kLaneDepth levels with cursors
// in LDS. Kept apart because the checks' tables and the deeper levels cost the common tasks registers in every loop.

#include "env.hpp"
#include "state_set.hpp"

#include <type_traits>

namespace mya
{
namespace
{
constexpr int kMaxWaves = 4;
constexpr bool kGeneral = MYA_GENERAL_TASKS;


/// LDS-qualified types (32-bit LDS addresses) and constant-address-space types: loads of the latter are invariant, so
/// with a wave-uniform address they are scalar loads, and the branches on their values scalar branches.
template<class X>
using lds = __attribute__((address_space(3))) X;
template<class X>
using cst = const __attribute__((address_space(4))) X;

/// A copy of the record at p.
template<class X>
__device__ __forceinline__ X ld(cst<X>* p)
{
    static_assert(sizeof(X) % 4 == 0, "records are whole 32-bit words");
    u32 w[sizeof(X) / 4];
    cst<u32>* src = (cst<u32>*)p;
#pragma unroll
    for (u32 i = 0; i < sizeof(X) / 4; ++i)
        w[i] = src[i];
    X x;
    __builtin_memcpy(&x, w, sizeof(X));
    return x;
}

/// A value that every lane holds, in a scalar register.
__device__ __forceinline__ u32 uni(u32 v) { return static_cast<u32>(__builtin_amdgcn_readfirstlane(static_cast<int>(v))); }
__device__ __forceinline__ u64 uni(u64 v) { return static_cast<u64>(uni(static_cast<u32>(v))) | (static_cast<u64>(uni(static_cast<u32>(v >> 32))) << 32); }

/// The image's tables. Steps and terms (records of 32 bytes) are indexed from the image's start, as are the words of
/// the terms' dom0 and static rows.
struct Tab
{
    cst<u64>* image;
    cst<DevStep>* steps;
    cst<DevTerm>* terms;
    cst<DevSchema>* schemas;
    cst<DevDelta>* deltas;
    cst<DevCheck>* checks;
    cst<DevEffect>* effects;
    cst<DevPair>* pairs;
    cst<DevPredDecode>* decode;
    cst<u32>* goal_pos;
    cst<u32>* goal_neg;
    cst<u32>* pred_arity;
    cst<u32>* pos_begin;
    cst<u64>* pred_pairs;
    cst<u64>* pred_offset;
};

__device__ __forceinline__ Tab tab_of(const TaskDev& T)
{
    cst<u64>* img = (cst<u64>*)T.image;
    Tab t;
    t.schemas = (cst<DevSchema>*)(img + T.off_schemas);
    t.image = img;
    t.steps = (cst<DevStep>*)img;
    t.terms = (cst<DevTerm>*)img;
    t.deltas = (cst<DevDelta>*)(img + T.off_deltas);
    t.checks = (cst<DevCheck>*)(img + T.off_checks);
    t.effects = (cst<DevEffect>*)(img + T.off_effects);
    t.pairs = (cst<DevPair>*)(img + T.off_pairs);
    t.decode = (cst<DevPredDecode>*)(img + T.off_decode);
    t.goal_pos = (cst<u32>*)(img + T.off_goal_pos);
    t.goal_neg = (cst<u32>*)(img + T.off_goal_neg);
    t.pred_arity = (cst<u32>*)(img + T.off_pred_arity);
    t.pos_begin = (cst<u32>*)(img + T.off_pos_begin);
    t.pred_pairs = img + T.off_pred_pairs;
    t.pred_offset = img + T.off_pred_offset;
    return t;
}

/// A wave's LDS region.
struct Lds
{
    lds<u64>* row;     // [W] the state
    lds<u64>* view;    // [view_words] rows of the non-bulk view pairs
    lds<u32>* ub;      // [A] the wave-uniform binding (the picked action, the enumeration's prefix)
    lds<u32>* bind;    // [A][64]: the lanes' bindings (parameter p of lane l at p * 64 + l)
    lds<u32>* counts;  // [num_schemas]
    lds<u64>* dfs_m;   // [A] the successor enumeration's per-parameter candidates left in the current word
    lds<u32>* dfs_w;   // [A] and that word
    lds<u32>* eff;     // [kMaxEff]: effect slots of a successor (lane k: effect k)
    lds<u32>* before;  // [kMaxEff]: their bits before the move
    lds<u64>* cur_m;   // [A][64]: the lanes' enumeration cursors (candidate bits left) of plans deeper than kLaneDepth
    lds<u32>* cur_w;   // [A][64]: and their word indices
};

__device__ __forceinline__ Lds lds_of(lds<u64>* region, const TaskDev& T)
{
    Lds l;
    l.view = region;
    l.row = region + T.l_row;
    l.dfs_m = region + T.l_dfs_m;
    l.ub = reinterpret_cast<lds<u32>*>(region + T.l_ub);
    l.bind = reinterpret_cast<lds<u32>*>(region + T.l_bind);
    l.counts = reinterpret_cast<lds<u32>*>(region + T.l_counts);
    l.dfs_w = reinterpret_cast<lds<u32>*>(region + T.l_dfs_w);
    l.eff = reinterpret_cast<lds<u32>*>(region + T.l_eff);
    l.before = reinterpret_cast<lds<u32>*>(region + T.l_before);
    l.cur_m = region + T.l_cur;
    l.cur_w = reinterpret_cast<lds<u32>*>(region + T.l_cur + 64 * (T.label_width ? T.label_width : 1));
    return l;
}

/// The kernel's argument record (its first argument) behind a pointer the compiler knows nothing about: loads through it
/// are made where they are used. The kernels have more invariant fields (arguments, table pointers, LDS offsets) than
/// scalar registers, and hoisted to the kernel's start they spill into vector lanes (900 spills in the step, a third of
/// its vector instructions); a scalar load again is one cached access.
template<class X>
__device__ __forceinline__ const X& kernel_args()
{
    cst<X>* p = (cst<X>*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const X*)p;
}

/// Orders the wave's LDS accesses before and after this point (lanes of one wave run in lockstep).
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template<class P>
__device__ __forceinline__ bool row_bit(P row, u32 slot) { return (row[slot >> 6] >> (slot & 63)) & 1; }

/// The candidate bits of step `st` for objects [st.lo + 64 w, + 64) under the lane's binding. The terms are records of a
/// uniform index (scalar loads); w and the bound objects may differ from lane to lane.
__device__ __forceinline__ u64 cand_word(const Tab& H, const Lds& L, const DevStep& st, u32 w, u32 lane)
{
    u64 a = ~u64{0};
    for (u32 ti = st.term_begin; ti < st.cons_end; ++ti)
    {
        const DevTerm c = ld(H.terms + ti);
        u32 ri = c.row0;
        if (c.src != kNone)
            ri = L.bind[c.src * 64 + lane] - c.row0;
        bool in = true;
        if (c.rows != kNone)
        {
            in = ri < c.rows;
            ri = in ? ri : 0;
        }
        const u32 at = c.base + ri * c.stride;
        u64 v;
        if (c.path == static_cast<u32>(TermPath::Words))
            v = L.view[at + w];
        else if (c.path == static_cast<u32>(TermPath::Image))
            v = H.image[at + w];
        else
        {
            // 64 bits from bit `rel` of the row on, those outside the row cleared
            const RowBits b = row_bits(c, w);
            const u32 pos = at + b.skip, sh = pos & 63;
            const auto r = L.view + (pos >> 6);
            v = (r[0] >> sh) | ((r[1] << 1) << (63 - sh));
            v = b.keep >= 64 ? v : b.keep > 0 ? v & ((u64{1} << b.keep) - 1) : 0;
            if (c.delta < 0 && b.rel < 0)
                v = b.rel > -64 ? v << -b.rel : 0;
        }
        if (c.rows != kNone)
            v = in ? v : 0;
        a &= v ^ (c.neg ? ~u64{0} : 0);
    }
    return a;
}

/// The binding of the lane (column `lane` of the bindings) or of the whole wave (L.ub): parameter p.
struct LaneBinding
{
    lds<u32>* b;
    __device__ __forceinline__ u32 operator[](u32 p) const { return b[p * 64]; }
};
struct WaveBinding
{
    lds<u32>* b;
    __device__ __forceinline__ u32 operator[](u32 p) const { return b[p]; }
};

template<class B>
__device__ __forceinline__ bool check_holds(const TaskDev& T, const Tab& H, const Lds& L, const DevCheck& c, B b)
{
    u32 objs[6];
#pragma unroll
    for (int i = 0; i < 6; ++i)
    {
        const i32 t = c.terms[i];
        objs[i] = (static_cast<u32>(i) < c.nterms) ? (t < 0 ? static_cast<u32>(-(t + 1)) : b[static_cast<u32>(t)]) : 0;
    }
    bool h;
    if (c.kind == static_cast<u32>(CheckKind::Fluent))
    {
        u64 key = H.pred_offset[c.pred];
        const u32 pb = H.pos_begin[c.pred];
#pragma unroll
        for (int i = 0; i < 6; ++i)
            if (static_cast<u32>(i) < c.nterms)
                key += T.rs[static_cast<u64>(pb + i) * T.n + objs[i]];
        if (key >= T.fluent_count)
            h = false;
        else
        {
            const u32 slot = T.dense ? static_cast<u32>(key) : T.slot_of[key];
            h = slot != kNone && row_bit(L.row, slot);
        }
    }
    else
    {
        const DevStaticMeta m = T.static_meta[c.pred];
        u64 key = 0;
#pragma unroll
        for (int i = 0; i < 6; ++i)
            if (static_cast<u32>(i) < c.nterms)
                key = key * T.n + objs[i];
        const u64* keys = T.static_words + m.keys;
        u64 lo = 0, hi = m.count;
        while (lo < hi)
        {
            const u64 mid = lo + (hi - lo) / 2;
            if (keys[mid] < key)
                lo = mid + 1;
            else
                hi = mid;
        }
        h = lo < m.count && keys[lo] == key;
    }
    return h == (c.pos != 0);
}

template<class B>
__device__ __forceinline__ bool checks_ok(const TaskDev& T, const Tab& H, const Lds& L, u32 cb, u32 ce, B b)
{
    if constexpr (!kGeneral)
        return true;
    for (u32 k = cb; k < ce; ++k)
        if (!check_holds(T, H, L, ld(H.checks + k), b))
            return false;
    return true;
}

/// A task and a wave region as plain values, for the functions that are calls: code that many places need is kept once
/// (the instruction cache holds 64 KiB for two CUs), and a call's registers are its own.
struct Where
{
    u64 task;
    u32 region;
    __device__ __forceinline__ Where(const TaskDev& T, const Lds& L)
        : task(reinterpret_cast<u64>(&T)), region(static_cast<u32>(reinterpret_cast<std::uintptr_t>(L.view)))
    {
    }
};
__device__ __forceinline__ const TaskDev& task_at(u64 t) { return *(const TaskDev*)(cst<TaskDev>*)uni(t); }
__device__ __forceinline__ lds<u64>* region_at(u32 r) { return (lds<u64>*)uni(r); }

/// Bindings completing steps [si, se) sequentially in this lane (its own binding column): an iterative nested loop whose
/// per-level cursor (current word index and remaining candidate bits) lives in the lane's LDS columns; the lanes may be
/// at different levels. The levels past kLaneDepth of count_lanes.
__device__ __noinline__ u32 count_deep(u64 task, u32 region, u32 si, u32 se)
{
    const TaskDev& T = task_at(task);
    const Tab H = tab_of(T);
    const Lds L = lds_of(region_at(region), T);
    const u32 lane = lane_id();
    const LaneBinding b{L.bind + lane};
    u32 total = 0;
    u32 d = 0;  // level: step si + d
    L.cur_w[lane] = 0;
    L.cur_m[lane] = cand_word(H, L, ld(H.steps + si), 0, lane);
    for (;;)
    {
        const DevStep st = ld(H.steps + si + d);
        u64 m = L.cur_m[d * 64 + lane];
        const bool last = si + d + 1 == se;
        const bool chk = kGeneral && st.check_begin != st.check_end;
        if (last && !chk)
        {
            total += static_cast<u32>(__popcll(m));
            m = 0;
        }
        if (m == 0)
        {
            // next word of this level, or back to the level above
            const u32 w = L.cur_w[d * 64 + lane] + 1;
            if (w < st.words)
            {
                L.cur_w[d * 64 + lane] = w;
                L.cur_m[d * 64 + lane] = cand_word(H, L, st, w, lane);
                continue;
            }
            if (d == 0)
                break;
            --d;
            continue;
        }
        const u32 bit = static_cast<u32>(__builtin_ctzll(m));
        L.cur_m[d * 64 + lane] = m & (m - 1);
        L.bind[st.param * 64 + lane] = st.lo + 64 * L.cur_w[d * 64 + lane] + bit;
        if (chk && !checks_ok(T, H, L, st.check_begin, st.check_end, b))
            continue;
        if (last)
        {
            ++total;
            continue;
        }
        ++d;
        L.cur_w[d * 64 + lane] = 0;
        L.cur_m[d * 64 + lane] = cand_word(H, L, ld(H.steps + si + d), 0, lane);
    }
    return total;
}

/// Bindings completing steps [si, se) from this lane's binding. The lanes walk the levels together: the level's step is
/// the same record in every lane (scalar loads and branches), a level's words follow each other, and each lane takes
/// its own candidates of a word one after the other. D levels nest as code, deeper ones in count_deep.
template<u32 D>
__device__ __forceinline__ u32 count_lanes(const TaskDev& T, const Tab& H, const Lds& L, u32 si, u32 se, u32 lane)
{
    if (si == se)
        return 1;
    const DevStep st = ld(H.steps + si);
    const bool last = si + 1 == se, chk = kGeneral && st.check_begin != st.check_end;
    u32 total = 0;
    for (u32 w = 0; w < st.words; ++w)
    {
        u64 m = cand_word(H, L, st, w, lane);
        if (last && !chk)
        {
            total += static_cast<u32>(__popcll(m));
            continue;
        }
        while (m)
        {
            L.bind[st.param * 64 + lane] = st.lo + 64 * w + static_cast<u32>(__builtin_ctzll(m));
            m &= m - 1;
            if (chk && !checks_ok(T, H, L, st.check_begin, st.check_end, LaneBinding{L.bind + lane}))
                continue;
            if (last)
                ++total;
            else if constexpr (D > 1)
                total += count_lanes<D - 1>(T, H, L, si + 1, se, lane);
            else if constexpr (kGeneral)
                total += count_deep(Where(T, L).task, Where(T, L).region, si + 1, se);
        }
    }
    return total;
}

/// Calls f(w, m) for the window words of step st from w0 on whose candidate word m is nonzero, ascending, until f
/// returns true (then returns true). Every lane must hold the same binding of the parameters before st's: the words
/// are evaluated 64 at a time, one per lane, and the nonzero ones taken from a ballot. w and m are wave-uniform.
template<class F>
__device__ __forceinline__ bool for_nonzero_words(const TaskDev& T, const Tab& H, const Lds& L, const DevStep& st, u32 w0, u32 lane, F&& f)
{
    for (u32 base = w0; base < st.words; base += kWave)
    {
        const u32 wl = base + lane;
        u64 mine = 0;
        if (wl < st.words)
            mine = cand_word(H, L, st, wl, lane);
        for (u64 nz = __ballot(mine != 0); nz; nz &= nz - 1)
        {
            const u32 k = static_cast<u32>(__builtin_ctzll(nz));
            if (f(base + k, lane_value(mine, k)))
                return true;
        }
    }
    return false;
}

/// Binds parameter p to object o in every lane's column.
__device__ __forceinline__ void bind_all(const Lds& L, u32 p, u32 o, u32 lane) { L.bind[p * 64 + lane] = o; }

/// Whether the candidates m of a word before a last step of `next_words` words are counted one by one, each with the lanes
/// side by side over that step's window, instead of one per lane: the candidates' trips over the window are then fewer
/// than the lanes' word-by-word trips (a grid cell's 16-word row of neighbours after one cell).
__device__ __forceinline__ bool one_by_one(u64 m, u32 next_words)
{
    return next_words > 1 && static_cast<u32>(__popcll(m)) * ((next_words + kWave - 1) / kWave) < next_words;
}

/// The words of step st's candidates side by side over the lanes: the lane's part of their number.
__device__ __forceinline__ u32 count_window(const Tab& H, const Lds& L, const DevStep& st, u32 lane)
{
    u32 acc = 0;
    for (u32 w = lane; w < st.words; w += kWave)
        acc += static_cast<u32>(__popcll(cand_word(H, L, st, w, lane)));
    return acc;
}

/// The words of the last step of a plan [pb, pe) of one step without checks, else 0 (one_by_one's window).
__device__ __forceinline__ u32 last_window(const Tab& H, u32 pb, u32 pe)
{
    return pb + 1 == pe && !(kGeneral && H.steps[pb].check_begin != H.steps[pb].check_end) ? H.steps[pb].words : 0;
}

/// Bindings completing steps [si, se) from a binding that every lane holds, as per-lane parts (their sum over the wave
/// is the count).
__device__ __forceinline__ u32 count_part(const TaskDev& T, const Tab& H, const Lds& L, u32 si, u32 se, u32 lane)
{
    if (si == se)
        return lane == 0 ? 1 : 0;
    const DevStep st = ld(H.steps + si);
    const bool last = si + 1 == se, chk = kGeneral && st.check_begin != st.check_end;
    if (last && !chk)
        return count_window(H, L, st, lane);
    u32 acc = 0;
    const u32 next_words = last ? 0 : last_window(H, si + 1, se);
    for_nonzero_words(T, H, L, st, 0, lane, [&](u32 w, u64 m) {
        if (one_by_one(m, next_words))
        {
            const DevStep next = ld(H.steps + si + 1);
            for (u64 x = m; x; x &= x - 1)
            {
                bind_all(L, st.param, st.lo + 64 * w + static_cast<u32>(__builtin_ctzll(x)), lane);
                if (!chk || checks_ok(T, H, L, st.check_begin, st.check_end, LaneBinding{L.bind + lane}))
                    acc += count_window(H, L, next, lane);
            }
        }
        else if ((m >> lane) & 1)
        {
            bind_all(L, st.param, st.lo + 64 * w + lane, lane);
            if (!chk || checks_ok(T, H, L, st.check_begin, st.check_end, LaneBinding{L.bind + lane}))
                acc += count_lanes<kLaneDepth>(T, H, L, si + 1, se, lane);
        }
        return false;
    });
    return acc;
}

/// Position of the k-th (from 0) set bit of m (k < popcount(m)).
__device__ __forceinline__ u32 kth_bit(u64 m, u32 k)
{
    u32 pos = 0;
    u32 c = static_cast<u32>(__popc(static_cast<u32>(m)));
    if (k >= c)
    {
        k -= c;
        m >>= 32;
        pos += 32;
    }
#pragma unroll
    for (u32 sh = 16; sh; sh >>= 1)
    {
        c = static_cast<u32>(__popc(static_cast<u32>(m) & ((1u << sh) - 1)));
        if (k >= c)
        {
            k -= c;
            m >>= sh;
            pos += sh;
        }
    }
    return pos;
}

/// The successor counts of the schemas of `mask` (bit s, every schema past 32) into LDS (witness pruning off).
__device__ __forceinline__ void count_schemas(const TaskDev& T, const Tab& H, const Lds& L, u32 mask, u32 lane)
{
    for (u32 s = 0; s < T.num_schemas; ++s)
    {
        if (s < 32 && !((mask >> s) & 1))
            continue;
        const auto& S = H.schemas[s];
        u32 c = 0;
        if (!S.never && checks_ok(T, H, L, S.ground_begin, S.ground_end, WaveBinding{L.ub}))
            c = wave_sum(count_part(T, H, L, S.plan_begin[0], S.plan_begin[1], lane));
        if (lane == 0)
            L.counts[s] = c;
    }
    wave_sync();
}

/// The sum of the per-schema counts.
__device__ __forceinline__ u32 total_count(const TaskDev& T, const Lds& L, u32 lane)
{
    u32 part = 0;
    for (u32 s = lane; s < T.num_schemas; s += kWave)
        part += L.counts[s];
    return wave_sum(part);
}

/// Successors of the state (witness pruning off); the per-schema counts into LDS.
__device__ __forceinline__ u32 count_all(const TaskDev& T, const Tab& H, const Lds& L, u32 lane)
{
    count_schemas(T, H, L, ~0u, lane);
    return total_count(T, L, lane);
}

/// The counts that the move's changed effects (bit e of `changed`: effect e's atom changes) take away (the deltas before
/// the move, on the state it leaves) or add (after it, on the state it reaches), in L.counts; L.ub holds the action.
/// An action touches few bindings of a schema, so this replaces counting the schema again.
__device__ __forceinline__ void apply_deltas(const TaskDev& T, const Tab& H, const Lds& L, u32 begin, u32 end, u32 changed, bool add, u32 lane)
{
    for (u32 k = begin; k < end; ++k)
    {
        const DevDelta d = ld(H.deltas + k);
        if (!((changed >> d.effect) & 1))
            continue;
        auto object = [&](i32 t) { return t < 0 ? static_cast<u32>(-(t + 1)) : uni(L.ub[t]); };
        bool ok = true;
#pragma unroll
        for (u32 q = 0; q < kMaxDeltaTerms; ++q)
            if (q < d.neq)
                ok = ok && object(d.eq[2 * q]) == object(d.eq[2 * q + 1]);
        if (!ok)
            continue;
#pragma unroll
        for (u32 q = 0; q < kMaxDeltaTerms; ++q)
            if (q < d.nbound)
                bind_all(L, static_cast<u32>(d.param[q]), object(d.term[q]), lane);
        if (d.tests)
        {
#pragma unroll
            for (u32 q = 0; q < kMaxDeltaTerms; ++q)
                if (q < d.nbound && ok)
                {
                    const DevStep st = ld(H.steps + d.test_begin + q);
                    const u32 o = object(d.term[q]) - st.lo;
                    ok = o < 64 * st.words && ((uni(cand_word(H, L, st, o >> 6, lane)) >> (o & 63)) & 1) &&
                         uni(checks_ok(T, H, L, st.check_begin, st.check_end, LaneBinding{L.bind + lane}) ? 1u : 0u);
                }
            if (!ok)
                continue;
        }
        const u32 c = count_part(T, H, L, d.plan_begin, d.plan_end, lane);
        if (c)
            __hip_atomic_fetch_add(L.counts + d.schema, add ? c : 0u - c, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    }
    wave_sync();
}

/// The per-env goal test (mask_goal, src/mymyr/rl/env.cpp:55-61): the LDS row against a row of goal masks.
__device__ __forceinline__ bool mask_goal(const lds<u64>* row, const u64* gp, const u64* gn, u32 W, u32 lane)
{
    bool ok = true;
    for (u32 w = lane; w < W; w += kWave)
    {
        const u64 x = row[w];
        ok = ok && (x & gp[w]) == gp[w] && (x & gn[w]) == 0;
    }
    return __ballot(!ok) == 0;
}

/// Whether a row of goal masks sets only the task's fluent slots (words past W and bits past the last slot clear).
__device__ __forceinline__ bool goal_masks_fit(const u64* gp, const u64* gn, u32 words, const TaskDev& T, u32 lane)
{
    bool fit = true;
    for (u32 w = lane; w < words; w += kWave)
    {
        const u64 x = gp[w] | gn[w];
        if (w >= T.W)
            fit = fit && x == 0;
        else if (w == T.W - 1 && (T.fluent_slots & 63))
            fit = fit && (x >> (T.fluent_slots & 63)) == 0;
    }
    return __ballot(!fit) == 0;
}

/// A 64-bit fingerprint of the state (the count cache's check that a row still holds the state its counts are of): the
/// sum over the words of fingerprint_word.
__device__ __forceinline__ u64 fingerprint_word(u64 x, u32 w) { return mix64(x ^ (static_cast<u64>(w + 1) * 0x9E3779B97F4A7C15ull)); }
__device__ __forceinline__ u64 state_fingerprint(const lds<u64>* row, u32 W, u32 lane)
{
    u64 acc = 0;
    for (u32 w = lane; w < W; w += kWave)
        acc += fingerprint_word(row[w], w);
    return wave_sum64(acc);
}

/// The per-schema counts of a count-cache row into LDS.
__device__ __forceinline__ void load_counts(const TaskDev& T, const Lds& L, const u32* crow, u32 lane)
{
    for (u32 s = lane; s < T.num_schemas; s += kWave)
        L.counts[s] = crow[s];
    wave_sync();
}

/// A count-cache row of `cw` words from the per-schema counts in LDS (zeros past the instance's schemas, as for a
/// suite's narrower domains) and the state's fingerprint plus the instance's salt in its last two words.
__device__ __forceinline__ void store_counts(const TaskDev& T, const Lds& L, u32* crow, u32 cw, u32 lane, u64 fp)
{
    for (u32 s = lane; s < cw - 2; s += kWave)
        crow[s] = s < T.num_schemas ? L.counts[s] : 0;
    if (lane == 0)
    {
        crow[cw - 2] = static_cast<u32>(fp);
        crow[cw - 1] = static_cast<u32>(fp >> 32);
    }
}

/// The schema holding successor `a` (< total) and the rank within it.
__device__ __forceinline__ void select_schema(const TaskDev& T, const Lds& L, u32 a, u32* schema, u32* rank)
{
    for (u32 s = 0; s < T.num_schemas; ++s)
    {
        const u32 c = uni(L.counts[s]);
        if (a < c)
        {
            *schema = s;
            *rank = a;
            return;
        }
        a -= c;
    }
    *schema = kNone;
    *rank = 0;
}

/// The rank-th applicable binding of schema s in lexicographic order into L.ub (and the lanes' columns). false: not
/// found. Per parameter i in order, the window words of its candidates given parameters [0, i) are taken 64 at a time,
/// one per lane; in a nonzero word each lane counts the completions of its candidate over the rest of the plan
/// (count_lanes), or few candidates are counted one by one (one_by_one), and the prefix over the candidates in object
/// order locates the rank. The last parameter's candidates have one completion each.
__device__ __forceinline__ bool pick(const TaskDev& T, const Tab& H, const Lds& L, u32 s, u32 rank, u32 lane)
{
    const auto& S = H.schemas[s];
    const u32 arity = S.arity;
    u32 a = rank;
    for (u32 i = 0; i < arity; ++i)
    {
        const DevStep F = ld(H.steps + S.filter_step[i]);
        const u32 pb = S.plan_begin[i + 1], pe = S.plan_begin[i + 2];
        const bool chk = kGeneral && F.check_begin != F.check_end;
        const u32 next_words = last_window(H, pb, pe);
        const bool found = for_nonzero_words(T, H, L, F, 0, lane, [&](u32 w, u64 m) {
            const u32 o0 = F.lo + 64 * w;
            if (chk)
            {
                // lane b checks candidate b
                bool ok = false;
                if ((m >> lane) & 1)
                {
                    bind_all(L, i, o0 + lane, lane);
                    ok = checks_ok(T, H, L, F.check_begin, F.check_end, LaneBinding{L.bind + lane});
                }
                m = __ballot(ok);
            }
            u32 o = kNone;
            if (pb == pe)
            {
                const u32 n = static_cast<u32>(__popcll(m));
                if (a >= n)
                {
                    a -= n;
                    return false;
                }
                o = o0 + kth_bit(m, a);
                a = 0;
            }
            else if (one_by_one(m, next_words))
            {
                for (u64 x = m; x; x &= x - 1)
                {
                    const u32 cand = o0 + static_cast<u32>(__builtin_ctzll(x));
                    bind_all(L, i, cand, lane);
                    const u32 c = wave_sum(count_window(H, L, ld(H.steps + pb), lane));
                    if (a < c)
                    {
                        o = cand;
                        break;
                    }
                    a -= c;
                }
                if (o == kNone)
                    return false;
            }
            else
            {
                u32 c = 0;
                if ((m >> lane) & 1)
                {
                    bind_all(L, i, o0 + lane, lane);
                    c = count_lanes<kLaneDepth>(T, H, L, pb, pe, lane);
                }
                const u32 incl = wave_inclusive(c);
                const u32 tot = lane_value(incl, kWave - 1);
                if (a >= tot)
                {
                    a -= tot;
                    return false;
                }
                const u32 win = static_cast<u32>(__builtin_ctzll(__ballot(incl > a)));
                a -= lane_value(incl - c, win);
                o = o0 + win;
            }
            bind_all(L, i, o, lane);
            if (lane == 0)
                L.ub[i] = o;
            return true;
        });
        if (!found)
            return false;
    }
    wave_sync();
    return true;
}

/// Whether the binding in L.ub (parameters [0, arity)) of schema s is applicable, for a schema with at least one
/// applicable binding (its ground preconditions hold): parameter i's object is a candidate of its filter step given
/// parameters [0, i), the test that makes a picked binding applicable (every precondition is checked at the step of its
/// last parameter). Wave-uniform; the lanes' columns take the binding on the way.
__device__ __forceinline__ bool label_applicable(const TaskDev& T, const Tab& H, const Lds& L, u32 s, u32 lane)
{
    const auto& S = H.schemas[s];
    for (u32 i = 0; i < S.arity; ++i)
    {
        const DevStep F = ld(H.steps + S.filter_step[i]);
        const u32 o = uni(L.ub[i]);
        if (o < F.lo || o - F.lo >= 64 * F.words)
            return false;
        const u32 w = (o - F.lo) >> 6, b = (o - F.lo) & 63;
        bind_all(L, i, o, lane);
        if (!((uni(cand_word(H, L, F, w, lane)) >> b) & 1))
            return false;
        if (F.check_begin != F.check_end && !checks_ok(T, H, L, F.check_begin, F.check_end, WaveBinding{L.ub}))
            return false;
    }
    return true;
}

/// Witness pruning (include/mymyr/successor/detail/engine.hpp:345-356): whether the witness objects of the full binding
/// in L.ub are the ones the reference's matcher binds first for its effect-relevant objects, i.e. the first completion
/// of the witnesses in the matcher's witness order, each witness taking its lowest object that the later ones can
/// complete. Per witness t, lane b tests candidate b of each window word (its checks, then whether the count plan of
/// the later witnesses finds a completion); the lowest passing candidate is the matcher's, and the binding is not the
/// one emitted as soon as one differs. The lanes' binding columns hold L.ub again on return. Wave-uniform.
__device__ __forceinline__ bool witness_first(const TaskDev& T, const Tab& H, const Lds& L, const DevWitness* Xg, u32 arity, u32 lane)
{
    cst<DevWitness>* X = (cst<DevWitness>*)Xg;
    for (u32 q = 0; q < arity; ++q)
        L.bind[q * 64 + lane] = L.ub[q];
    const u32 n = X->n;
    bool first = true;
    for (u32 t = 0; t < n && first; ++t)
    {
        const u32 v = X->param[t];
        const DevStep F = ld(H.steps + X->filter[t]);
        const u32 lo = X->plan_lo[t], hi = X->plan_hi[t];
        u32 found = kNone;
        for (u32 w = 0; w < F.words && found == kNone; ++w)
        {
            const u64 m = cand_word(H, L, F, w, lane);
            bool ok = false;
            if ((m >> lane) & 1)
            {
                L.bind[v * 64 + lane] = F.lo + 64 * w + lane;
                ok = F.check_begin == F.check_end || checks_ok(T, H, L, F.check_begin, F.check_end, LaneBinding{L.bind + lane});
                if (ok && lo != hi)
                    ok = count_lanes<kLaneDepth>(T, H, L, lo, hi, lane) != 0;
            }
            const u64 okm = __ballot(ok);
            if (okm)
                found = F.lo + 64 * w + static_cast<u32>(__builtin_ctzll(okm));
        }
        first = found == uni(L.ub[v]);
        L.bind[v * 64 + lane] = found;
    }
    for (u32 q = 0; q < arity; ++q)
        L.bind[q * 64 + lane] = L.ub[q];
    wave_sync();
    return first;
}

/// Calls emit(k, s) for the successors of the state in canonical order (schema, then lexicographic binding),
/// k = 0, 1, ...; L.ub holds the binding during the call, and emit returns false to stop. Each schema with successors
/// (L.counts from count_all) is enumerated depth first over its parameters in order, so the bindings come in the order
/// pick(rank) finds them for rank 0, 1, .... A level takes the window words of its parameter's filter step, evaluated 64
/// at a time: in a nonzero word lane b tests candidate b against the step's checks and counts its completions over the
/// rest of the plan (as pick does), and only candidates with completions are visited, lowest first; the leaf level
/// emits its candidates. Counting thus happens once per node of the binding tree instead of once per successor and
/// parameter. The levels' words and candidates left live in L.dfs_w / L.dfs_m; L.bind holds the binding's prefix in
/// every lane's column. Returns the successors enumerated.
template<bool kWitness = false, class Emit>
__device__ __forceinline__ u32 for_each_successor(const TaskDev& T, const Tab& H, const Lds& L, u32 lane, Emit&& emit, u32 s_begin = 0,
                                                  u32 s_end = kNone)
{
    const u32 A = T.label_width ? T.label_width : 1;
    u32 k = 0;
    for (u32 s = s_begin; s < T.num_schemas && s < s_end; ++s)
    {
        if (uni(L.counts[s]) == 0)
            continue;
        const auto& S = H.schemas[s];
        const u32 arity = S.arity;
        // witness pruning: only the full bindings whose witnesses the matcher binds first are successors
        [[maybe_unused]] const DevWitness* X = nullptr;
        if constexpr (kWitness)
            X = (T.witness && ((cst<DevWitness>*)T.witness)[s].n) ? T.witness + s : nullptr;
        if (arity == 0)
        {
            if (!emit(k++, s))
                return k;
            continue;
        }
        // parameter i from its first word at or past w0 with live candidates (false: none)
        auto open = [&](u32 i, u32 w0) -> bool {
            const DevStep F = ld(H.steps + S.filter_step[i]);
            const u32 pb = S.plan_begin[i + 1], pe = S.plan_begin[i + 2];
            const bool chk = kGeneral && F.check_begin != F.check_end;
            return for_nonzero_words(T, H, L, F, w0, lane, [&](u32 w, u64 m) {
                if (chk || pb != pe)
                {
                    // the candidates with at least one completion
                    bool live = false;
                    if ((m >> lane) & 1)
                    {
                        bind_all(L, i, F.lo + 64 * w + lane, lane);
                        live = !chk || checks_ok(T, H, L, F.check_begin, F.check_end, LaneBinding{L.bind + lane});
                        if (live && pb != pe)
                            live = count_lanes<kLaneDepth>(T, H, L, pb, pe, lane) != 0;
                    }
                    m = __ballot(live);
                }
                if (!m)
                    return false;
                wave_sync();
                if (lane == 0)
                {
                    L.dfs_m[i] = m;
                    L.dfs_w[i] = w;
                }
                wave_sync();
                return true;
            });
        };
        u32 i = 0;
        bool have = open(0, 0);
        for (;;)
        {
            if (!have)
            {
                if (i == 0)
                    break;
                --i;
                have = uni(L.dfs_m[i]) != 0 || open(i, uni(L.dfs_w[i]) + 1);
                continue;
            }
            // the level's lowest live candidate
            const u64 m = uni(L.dfs_m[i]);
            const u32 w = uni(L.dfs_w[i]);
            const u32 o = H.steps[S.filter_step[i]].lo + 64 * w + static_cast<u32>(__builtin_ctzll(m));
            wave_sync();
            if (lane == 0)
            {
                L.dfs_m[i] = m & (m - 1);
                L.ub[i] = o;
            }
            L.bind[i * 64 + lane] = o;
            for (u32 q = 0; q < i && q < A; ++q)
                L.bind[q * 64 + lane] = L.ub[q];
            wave_sync();
            if (i + 1 == arity)
            {
                bool take = true;
                if constexpr (kWitness)
                    take = !X || witness_first(T, H, L, X, arity, lane);
                if (take && !emit(k++, s))
                    return k;
                have = uni(L.dfs_m[i]) != 0 || open(i, w + 1);
                continue;
            }
            ++i;
            have = open(i, 0);
        }
    }
    return k;
}

/// The slot of an effect's atom under the wave's binding (kNone: none); its canonical id in *cid.
__device__ __forceinline__ u32 effect_slot(const TaskDev& T, const Lds& L, const DevEffect& e, u64* cid_out)
{
    u64 cid = e.arith ? e.arith_base : e.base;
#pragma unroll
    for (u32 v = 0; v < 4; ++v)
        if (v < e.nvar)
        {
            const u32 o = L.ub[e.var_param[v]];
            cid += e.arith ? o * e.mul[v] : T.rs[static_cast<u64>(e.var_pos[v]) * T.n + o];
        }
    *cid_out = cid;
    if (cid >= T.fluent_count)
        return kNone;
    return T.dense ? static_cast<u32>(cid) : T.slot_of[cid];
}

/// An added atom without a slot: an error under frozen slots; lazy slots record it for the host to intern (the
/// successor written is then incomplete, and the launch is repeated once the atom has a slot).
__device__ __forceinline__ void missing_atom(const TaskDev& T, u64 cid, u32* status)
{
    if (T.missing && cid < T.fluent_count)
        atomicOr(reinterpret_cast<unsigned long long*>(T.missing + (cid >> 6)), 1ull << (cid & 63));
    atomicOr(status, kStatusNoSlot);
}

/// The view word and bit of atom (pred, a0, a1) in the non-bulk pairs of its predicate: calls f(word pointer, bit).
template<class F>
__device__ __forceinline__ void for_view_bits(const Tab& H, const Lds& L, u32 pred, u32 a0, u32 a1, F&& f)
{
    const u64 pp = H.pred_pairs[pred];
    if (pp == ~u64{0})
        return;
    const u32 ar = H.pred_arity[pred];
    for (int d = 0; d < 2; ++d)
    {
        const u32 pi = d == 0 ? static_cast<u32>(pp) : static_cast<u32>(pp >> 32);
        if (pi == kNone)
            continue;
        const auto& P = H.pairs[pi];
        if (P.bulk)
            continue;
        u32 ri, bi;
        if (ar == 1)
        {
            ri = 0;
            bi = a0 - P.dst_lo;
        }
        else if (d == 0)
        {
            ri = a0 - P.src_lo;
            bi = a1 - P.dst_lo;
        }
        else
        {
            ri = a1 - P.src_lo;
            bi = a0 - P.dst_lo;
        }
        f(L.view + P.offset + static_cast<u64>(ri) * P.dst_words + (bi >> 6), u64{1} << (bi & 63));
    }
}

/// Builds the view of the wave's row (all lanes). With arithmetic slot decoding the row is read predicate by predicate:
/// only the slot ranges of predicates with scattered view rows, each with its decoding and its two pairs read once;
/// otherwise every set bit is decoded from its slot's record.
__device__ __forceinline__ void build_view(const TaskDev& T, const Tab& H, const Lds& L, u32 lane)
{
    for (u32 k = lane; k < T.view_words; k += kWave)
        L.view[k] = 0;
    wave_sync();
    if (T.decode_arith)
    {
        for (u32 k = 0; k < T.num_decode; ++k)
        {
            const DevPredDecode d = ld(H.decode + k);
            const u64 end = min(d.offset + d.size, static_cast<u64>(T.fluent_slots));
            if (!d.has_scatter || end <= d.offset)
                continue;
            // the predicate's scattered pairs: forward (or unary) and backward
            const u64 pp = H.pred_pairs[d.pred];
            const u32 ar = H.pred_arity[d.pred];
            u32 on[2], off[2], src_lo[2], dst_lo[2], dst_words[2];
#pragma unroll
            for (int q = 0; q < 2; ++q)
            {
                const u32 pi = q == 0 ? static_cast<u32>(pp) : static_cast<u32>(pp >> 32);
                on[q] = 0;
                off[q] = src_lo[q] = dst_lo[q] = dst_words[q] = 0;
                if (pp != ~u64{0} && pi != kNone)
                {
                    const DevPair P = ld(H.pairs + pi);
                    on[q] = P.bulk ? 0 : 1;
                    off[q] = P.offset;
                    src_lo[q] = P.src_lo;
                    dst_lo[q] = P.dst_lo;
                    dst_words[q] = P.dst_words;
                }
            }
            const u32 w0 = static_cast<u32>(d.offset >> 6), w1 = static_cast<u32>((end - 1) >> 6);
            for (u32 w = w0 + lane; w <= w1; w += kWave)
            {
                u64 x = L.row[w];
                if (w == w0)
                    x &= ~u64{0} << (d.offset & 63);
                if (w == w1 && (end & 63))
                    x &= (u64{1} << (end & 63)) - 1;
                while (x)
                {
                    const u32 rem = static_cast<u32>(w * 64 + static_cast<u32>(__builtin_ctzll(x)) - d.offset);
                    x &= x - 1;
                    u32 a0, a1;
                    if (d.arity >= 2)
                    {
                        const u32 r0 = d.magic ? mulhi32(rem, d.magic) : rem / d.d1;
                        a0 = d.lo0 + r0;
                        a1 = d.lo1 + (rem - r0 * d.d1);
                    }
                    else
                    {
                        a0 = d.lo0 + rem;
                        a1 = 0;
                    }
                    // the atom's bits in the pairs' rows, as for_view_bits places them
#pragma unroll
                    for (int q = 0; q < 2; ++q)
                    {
                        if (!on[q])
                            continue;
                        u32 ri, bi;
                        if (ar == 1)
                        {
                            ri = 0;
                            bi = a0 - dst_lo[q];
                        }
                        else if (q == 0)
                        {
                            ri = a0 - src_lo[q];
                            bi = a1 - dst_lo[q];
                        }
                        else
                        {
                            ri = a1 - src_lo[q];
                            bi = a0 - dst_lo[q];
                        }
                        __hip_atomic_fetch_or(L.view + off[q] + static_cast<u64>(ri) * dst_words[q] + (bi >> 6), u64{1} << (bi & 63),
                                              __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                    }
                }
            }
        }
        wave_sync();
        return;
    }
    for (u32 w = lane; w < T.W; w += kWave)
    {
        u64 x = L.row[w];
        while (x)
        {
            const u32 s = w * 64 + static_cast<u32>(__builtin_ctzll(x));
            x &= x - 1;
            if (s >= T.fluent_slots)
                break;  // bits past the task's slots belong to no atom
            const u64 rec = T.records[s];
            for_view_bits(H, L, static_cast<u32>(rec & 0xFFFF), static_cast<u32>((rec >> 16) & 0xFFFF), static_cast<u32>((rec >> 32) & 0xFFFF),
                          [](lds<u64>* word, u64 bit) {
                              __hip_atomic_fetch_or(word, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
                          });
        }
    }
    wave_sync();
}

/// Loads row i (W words of `words`) into the wave's LDS row.
__device__ __forceinline__ void load_row_lds(const TaskDev& T, const Lds& L, const u64* src, u32 lane)
{
    if (T.W <= kWave)  // one load per lane
    {
        if (lane < T.W)
            L.row[lane] = src[lane];
        wave_sync();
        return;
    }
    // up to 8 loads of a lane in flight before their LDS stores: a wide row arrives in about one load latency
    constexpr u32 kBatch = 8;
    for (u32 k0 = 0; k0 < T.W; k0 += kBatch * kWave)
    {
        u64 v[kBatch];
#pragma unroll
        for (u32 j = 0; j < kBatch; ++j)
        {
            const u32 k = k0 + j * kWave + lane;
            v[j] = k < T.W ? src[k] : 0;
        }
#pragma unroll
        for (u32 j = 0; j < kBatch; ++j)
        {
            const u32 k = k0 + j * kWave + lane;
            if (k < T.W)
                L.row[k] = v[j];
        }
    }
    wave_sync();
}

/// Loads the first n words of a row into the wave's LDS row and zeroes the rest of its T.W words (rows narrower than
/// the task: a lazy task's rows grow as atoms intern).
__device__ __forceinline__ void load_row_lds_n(const TaskDev& T, const Lds& L, const u64* src, u32 n, u32 lane)
{
    for (u32 k = lane; k < T.W; k += kWave)
        L.row[k] = k < n ? src[k] : 0;
    wave_sync();
}

/// dst[k] = k < n ? src[k] : 0 for k < z (global to global), up to 8 loads of a lane in flight.
__device__ __forceinline__ void copy_words(u64* dst, const u64* src, u32 n, u32 z, u32 lane)
{
    if (z <= kWave)  // one word per lane
    {
        if (lane < z)
            dst[lane] = lane < n ? src[lane] : 0;
        return;
    }
    constexpr u32 kBatch = 8;
    for (u32 k0 = 0; k0 < z; k0 += kBatch * kWave)
    {
        u64 v[kBatch];
#pragma unroll
        for (u32 j = 0; j < kBatch; ++j)
        {
            const u32 k = k0 + j * kWave + lane;
            v[j] = k < n ? src[k] : 0;
        }
#pragma unroll
        for (u32 j = 0; j < kBatch; ++j)
        {
            const u32 k = k0 + j * kWave + lane;
            if (k < z)
                dst[k] = v[j];
        }
    }
}

/// The ascending set-bit slots of `row` (W words) into out[0, max_atoms), -1 padded (all lanes). A lane takes kPer
/// consecutive words per round (one wave scan per kPer * 64 words; wide rows take 4); a lane's atoms are consecutive
/// in the output, and the lanes' ranges follow each other.
template<u32 kPer = 1, class P>
__device__ __forceinline__ void encode_row(P row, u32 W, i32* out, u32 max_atoms, u32 lane, u32* status)
{
    u32 base = 0;
    for (u32 w0 = 0; w0 < W; w0 += kWave * kPer)
    {
        const u32 wl = w0 + lane * kPer;
        u64 x[kPer];
        u32 c = 0;
#pragma unroll
        for (u32 j = 0; j < kPer; ++j)
        {
            x[j] = wl + j < W ? row[wl + j] : 0;
            c += static_cast<u32>(__popcll(x[j]));
        }
        const u32 incl = wave_inclusive(c);
        u32 k = base + incl - c;
#pragma unroll
        for (u32 j = 0; j < kPer; ++j)
            for (u64 y = x[j]; y; y &= y - 1)
            {
                if (k < max_atoms)
                    out[k] = static_cast<i32>((wl + j) * 64 + static_cast<u32>(__builtin_ctzll(y)));
                ++k;
            }
        base += lane_value(incl, kWave - 1);
    }
    for (u32 k = base + lane; k < max_atoms; k += kWave)
        out[k] = -1;
    if (base > max_atoms && lane == 0)
        atomicOr(status, kStatusCapacity);
}

template<class P>
__device__ __forceinline__ bool goal_test(const TaskDev& T, const Tab& H, P row, u32 lane)
{
    bool ok = true;
    for (u32 i = lane; i < T.ngp; i += kWave)
        ok = ok && row_bit(row, H.goal_pos[i]);
    for (u32 i = lane; i < T.ngn; i += kWave)
        ok = ok && !row_bit(row, H.goal_neg[i]);
    return !T.goal_unsat && __ballot(!ok) == 0;
}

/// A move applied to the LDS row and the view.
struct Moved
{
    u32 slot;     // the lane's effect slot (kNone: no effect or no slot): the row words that can have changed are theirs
    u64 fp_diff;  // the change of the row's fingerprint
};

/// Applies the effects of the picked binding of schema s to the LDS row and the view (delete, then add), and what they
/// change in the successor counts (DevDelta). One effect per lane: its slot (the table reads of the effects overlap
/// instead of following each other), whether its atom's bit really changes (lanes that list one atom agree on one of
/// them), then the deletes, the adds, and the view bits of the atoms that change. View pairs exist for predicates of
/// arity 1 and 2 only, so a view bit stands for one atom.
__device__ __forceinline__ Moved apply_effects(const TaskDev& T, const Tab& H, const Lds& L, u32 s, bool deltas, u32 lane, u32* status)
{
    const auto& S = H.schemas[s];
    const u32 eff = S.eff_begin, nadd = S.nadd;
    const u32 ne = min(S.eff_end - eff, kMaxEff);
    if (lane == 0 && S.eff_end - eff > kMaxEff)
        atomicOr(status, kStatusCapacity);
    const bool mine = lane < ne;
    const bool add = lane < nadd;
    u32 sl = kNone, pred = 0, a0 = 0, a1 = 0;
    bool before = false;
    u64 old = 0;
    if (mine)
    {
        const DevEffect e = ld(H.effects + eff + lane);
        u64 cid;
        sl = effect_slot(T, L, e, &cid);
        if (sl != kNone)
        {
            old = L.row[sl >> 6];
            before = (old >> (sl & 63)) & 1;
        }
        if (add && sl == kNone)
            missing_atom(T, cid, status);
        pred = e.pred;
        a0 = e.terms[0] < 0 ? static_cast<u32>(-(e.terms[0] + 1)) : L.ub[e.terms[0]];
        a1 = e.terms[1] < 0 ? static_cast<u32>(-(e.terms[1] + 1)) : L.ub[e.terms[1]];
    }
    // an atom's bit changes in the first lane that lists it: a delete of a set atom that no effect adds, an add of a clear one
    bool changes = mine && sl != kNone && before != add;
    bool first_word = mine && sl != kNone;  // the first lane that lists its row word
    for (u32 q = 0; q < ne; ++q)
    {
        const u32 sq = lane_value(sl, q);
        if (sq == kNone || q == lane)
            continue;
        if (sq == sl && ((q < nadd) == add ? q < lane : q < nadd))
            changes = false;
        if ((sq >> 6) == (sl >> 6) && q < lane)
            first_word = false;
    }
    const u32 changed = static_cast<u32>(__ballot(changes));
    if (deltas)
        apply_deltas(T, H, L, S.del_begin, S.add_begin, changed, false, lane);
    wave_sync();
    if (mine && !add && sl != kNone)
        __hip_atomic_fetch_and(L.row + (sl >> 6), ~(u64{1} << (sl & 63)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    wave_sync();
    if (mine && add && sl != kNone)
        __hip_atomic_fetch_or(L.row + (sl >> 6), u64{1} << (sl & 63), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    if (changes)
        for_view_bits(H, L, pred, a0, a1, [add](lds<u64>* word, u64 bit) {
            if (add)
                __hip_atomic_fetch_or(word, bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            else
                __hip_atomic_fetch_and(word, ~bit, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        });
    wave_sync();
    if (deltas)
        apply_deltas(T, H, L, S.add_begin, S.add_end, changed, true, lane);
    u64 diff = 0;
    if (first_word)
        diff = fingerprint_word(L.row[sl >> 6], sl >> 6) - fingerprint_word(old, sl >> 6);
    return Moved{sl, wave_sum64(diff)};
}

/// hash_state of a row (its trimmed words; include/mymyr/core/hash.hpp:56-60), one lane.
template<class P>
__device__ __forceinline__ u64 row_hash(P row, u32 W)
{
    u32 n = W;
    while (n > 0 && row[n - 1] == 0)
        --n;
    u64 h = kHashSeed ^ (static_cast<u64>(n) * kHashP1);
    u32 k = 0;
    for (; k + 1 < n; k += 2)
        h = mulfold(h ^ row[k] ^ kHashP1, row[k + 1] ^ kHashP2);
    if (k < n)
        h = mulfold(h ^ row[k] ^ kHashP1, kHashP2);
    return mix64(h);
}

constexpr u64 kVisitedZero = 0x9E3779B97F4A7C15ull;  // the key of hash 0 (0 marks an empty slot)

/// visited_insert (include/mymyr/rl/visited.hpp:31-52), one lane: whether the key was present; a new key above
/// floor(3H/4) entries is skipped and the count saturates at H.
__device__ __forceinline__ bool visited_insert(u64* table, u32 H, i32& count, u64 hash)
{
    const u64 key = hash ? hash : kVisitedZero;
    u32 at = static_cast<u32>(key) & (H - 1);
    for (u32 probe = 0; probe < H; ++probe, at = (at + 1) & (H - 1))
    {
        const u64 x = table[at];
        if (x == key)
            return true;
        if (!x)
        {
            if (count >= static_cast<i32>((static_cast<u64>(H) * 3) / 4))
                count = static_cast<i32>(H);
            else
            {
                table[at] = key;
                ++count;
            }
            return false;
        }
    }
    count = static_cast<i32>(H);
    return false;
}

/// visited_clear + visited_insert of one hash over a row's table (all lanes; every slot written once, the key's own
/// slot with the key); the count becomes 1 (lane 0).
__device__ __forceinline__ void visited_restart(u64* table, u32 H, i32* count, u64 hash, u32 lane)
{
    const u64 key = hash ? hash : kVisitedZero;
    const u32 at = static_cast<u32>(key) & (H - 1);
    for (u32 q = lane; q < H; q += kWave)
        table[q] = q == at ? key : 0;
    if (lane == 0)
        *count = 1;
}

/// One environment's step (HostEnv::step_row_impl, src/mymyr/rl/env.cpp:351-528): row i of instance k, whose tables
/// are T / H and whose wave region is L. An autoreset restarts the row in next_task_ids[i] when that names an instance
/// (else in k), writing the new instance's initial state and goal masks over the words the row may have dirtied
/// (TaskSuite::initial_row, src/mymyr/rl/task_suite.cpp:130-138) and its id into task_ids.
template<bool kOne, bool kVisited, bool kPlain>
__device__ __forceinline__ void step_row(const EnvArgs& A, const TaskDev& T, const Tab& H, const Lds& L, u64 i, u32 k, u32 lane)
{
    static_assert(!kPlain || (kOne && !kVisited), "the plain step is a one-instance step without visited tables");
    // the plain step (an env pool's step: the random policy over one instance, the env's RNG key and env ids first_env +
    // row, the task's goal, steps and draws kept, no labels or final states) knows the optional inputs it does not
    // take at compile time, so their pointers and tests take no registers
    const i64* const actions = kPlain ? nullptr : A.actions;
    const i32* const label_schema = kPlain ? nullptr : A.label_schema;
    const u64* const seeds = kPlain ? nullptr : A.seeds;
    const u32* const env_ids = kPlain ? nullptr : A.env_ids;
    const u64* const goal_pos = kPlain ? nullptr : A.goal_pos;
    u64* const final_states = kPlain ? nullptr : A.final_states;
    u32* const reset_counts = kPlain ? nullptr : A.reset_counts;
    i32* const steps = A.steps;
    u64* const draws = A.draws;
    const bool have_steps = kPlain || A.steps != nullptr;
    const bool have_draws = kPlain || A.draws != nullptr;
    const u32 Lw = A.label_width;
    u64* grow = A.states + i * A.words;
    // the row's scalars are read before its words, so that their latencies overlap with the row's
    const bool already_goal = A.at_goal[i] != 0;
    const i64 act_in = actions ? actions[i] : 0;
    const u64 draws0 = have_draws ? draws[i] : 0;
    const i32 steps0 = have_steps ? steps[i] : 0;
    const i32 next_in = (!kOne && A.next_task_ids) ? A.next_task_ids[i] : 0;
    const i32 label_in = label_schema ? label_schema[i] : -1;
    // the count cache row: its counts stand for the row's state (and instance) when its fingerprint matches (reset,
    // refresh and step write it; a state written directly since is counted again)
    const u32 cw = A.cache_width;
    u32* crow = A.counts ? A.counts + i * cw : nullptr;
    const u64 fp_cached = crow ? (static_cast<u64>(crow[cw - 2]) | (static_cast<u64>(crow[cw - 1]) << 32)) : 0;
    load_row_lds(T, L, grow, lane);
    build_view(T, H, L, lane);
    u64 fp = 0;  // the fingerprint of the LDS row plus the instance's salt
    bool cached = false;
    if (crow)
    {
        fp = state_fingerprint(L.row, T.W, lane) + instance_salt(k);
        cached = uni(fp_cached) == fp;
    }
    enum
    {
        kOk = 0,
        kStuck = 1,
        kInvalid = 2,
        kGoal = 3
    };
    // phase 0 counts s, chooses, picks and moves; phase 1 counts again what the move's deltas did not bring up to date
    u32 c = 0, c2 = 0, st = kOk, schema = kNone;
    u32 moved_slot = kNone;  // the lane's effect slot of the applied move (its word is the only one it can change)
    bool g = already_goal;
    for (u32 phase = 0; phase < 2; ++phase)
    {
        if (phase == 0 && cached)
            load_counts(T, L, crow, lane);
        const u32 recount = phase == 1 ? H.schemas[schema].recount : (cached ? 0u : ~0u);
        if (recount)
            count_schemas(T, H, L, recount, lane);
        const u32 cc = total_count(T, L, lane);
        if (phase == 1)
        {
            c2 = cc;
            break;
        }
        c = c2 = cc;
        // 2. the choice (env.cpp:416-440)
        st = already_goal ? kGoal : kOk;
        u32 a = 0;
        bool labelled = false;  // the move is the row's label (no pick)
        if (!already_goal && c == 0)
            st = kStuck;
        else if (!already_goal && label_schema)
        {
            // label mode (env.cpp:376-398, 423-425): the label moves where it is applicable, else the row is invalid
            bool ok = label_in >= 0 && static_cast<u32>(label_in) < T.num_schemas && uni(L.counts[label_in]) > 0;
            if (ok)
            {
                const u32 arity = H.schemas[label_in].arity;
                if (lane < arity)
                    L.ub[lane] = static_cast<u32>(A.label_binding[i * A.label_stride + lane]);
                wave_sync();
                ok = label_applicable(T, H, L, static_cast<u32>(label_in), lane);
            }
            if (ok)
            {
                schema = static_cast<u32>(label_in);
                labelled = true;
            }
            else
                st = kInvalid;
        }
        else if (!already_goal && actions)
        {
            const i64 act = act_in;
            if (act < 0 || static_cast<u64>(act) >= c)
                st = kInvalid;
            else
                a = static_cast<u32>(act);
        }
        else if (!already_goal)
        {
            const u64 key = seeds ? seeds[i] : *A.seed;  // the row's own key, or the env's
            a = successor_index(key, env_ids ? static_cast<u64>(env_ids[i]) : A.first_env + i, draws0, c);
        }
        u32 rank = 0;
        if (st == kOk && !labelled)
        {
            select_schema(T, L, a, &schema, &rank);
            if (schema == kNone || !pick(T, H, L, schema, rank, lane))
            {
                if (lane == 0)
                    atomicOr(A.status, kStatusPickFailed);
                st = kStuck;
            }
        }
        if (lane == 0)
        {
            if (have_draws)
                draws[i] = draws0 + 1;
            if (A.schema)
                A.schema[i] = st == kOk ? static_cast<i32>(schema) : -1;
            if (A.invalid)
                A.invalid[i] = st == kInvalid ? 1 : 0;
        }
        if (A.binding)
        {
            const u32 arity = st == kOk ? H.schemas[schema].arity : 0;
            for (u32 q = lane; q < Lw; q += kWave)
                A.binding[i * Lw + q] = (st == kOk && q < arity) ? static_cast<i32>(L.ub[q]) : -1;
        }
        if (st != kOk)
            break;
        // 3. the move, goal and (next phase) the successor count of the reached state
        const Moved mv = apply_effects(T, H, L, schema, T.num_schemas <= 32, lane, A.status);
        moved_slot = mv.slot;
        fp += mv.fp_diff;
        g = goal_pos ? mask_goal(L.row, goal_pos + i * A.words, A.goal_neg + i * A.words, T.W, lane)
                     : goal_test(T, H, L.row, lane);
    }
    // 4. rewards, termination, truncation (env.cpp:466-485)
    const bool dead = !A.cfg.dead_end_none && !g && ((st == kOk && c2 == 0) || st == kStuck);
    const bool term = g || (dead && A.cfg.dead_end_terminal);
    const bool absorbed = already_goal || (st == kStuck && dead && A.cfg.dead_end_terminal);
    const i32 t2 = have_steps ? steps0 + (absorbed ? 0 : 1) : 0;
    const bool trunc = !term && A.cfg.max_steps && t2 >= static_cast<i32>(A.cfg.max_steps);
    if (lane == 0)
    {
        if (A.reward)
        {
            float r = 0.0f;
            if (!absorbed)
            {
                r = A.cfg.step_reward + (g ? A.cfg.goal_reward : 0.0f);
                r = r + (dead ? A.cfg.dead_end_reward : 0.0f);
            }
            A.reward[i] = r;
        }
        if (A.terminated)
            A.terminated[i] = term ? 1 : 0;
        if (A.truncated)
            A.truncated[i] = trunc ? 1 : 0;
        if (A.goal)
            A.goal[i] = g ? 1 : 0;
    }
    if (final_states)
    {
        const u32 FW = A.final_words;
        u64* f = final_states + i * FW;
        for (u32 q = lane; q < FW; q += kWave)
            f[q] = q < T.W ? L.row[q] : 0;
    }
    // the reached state's key into the row's visited table unless its episode is over without autoreset (env.cpp:487-499)
    if (kVisited && (A.visited.capacity || A.revisited))
    {
        bool revisited = false;
        const bool over = !A.cfg.autoreset && (absorbed || (A.cfg.max_steps && steps0 >= static_cast<i32>(A.cfg.max_steps)));
        if (lane == 0 && A.visited.capacity && !over)
        {
            const u32 H = A.visited.capacity;
            i32 cnt = A.visited.count[i];
            revisited = visited_insert(A.visited.table + i * H, H, cnt, row_hash(L.row, T.W));
            A.visited.count[i] = cnt;
            if (cnt == static_cast<i32>(H))
                atomicOr(A.visited.status + (A.visited.status_per_row ? i : 0), 1);
        }
        if (lane == 0 && A.revisited)
            A.revisited[i] = revisited ? 1 : 0;
        wave_sync();
    }
    // 5. the autoreset, or the bookkeeping of the move (the LDS row holds s'). The instance an autoreset restarts in:
    // next_task_ids[i], where an id outside the table sets the status (in every row, as the reference checks the whole
    // array) and keeps the row's instance
    u32 next = k;
    if (!kOne && A.next_task_ids)
    {
        const i32 v = next_in;
        if (v < 0 || static_cast<u32>(v) >= A.instances)
        {
            if (lane == 0)
                atomicOr(A.status, kStatusTaskId);
        }
        else
            next = static_cast<u32>(v);
    }
    const bool reset = A.cfg.autoreset && (term || trunc);
    if (reset)
    {
        // every autoreset advances the row's reset counter (a sampled restart comes in as next_task_ids, drawn before the
        // step with the counter's value before this advance)
        if (reset_counts && lane == 0)
            reset_counts[i] += 1;
        const InstDev& J = A.inst[next];  // a one-instance env restarts in instance 0
        const u32 z = min(A.words, max(J.W, T.W));  // the words the row may have dirtied: its old and new instance's
        copy_words(grow, J.initial, J.W, z, lane);
        if (goal_pos)
        {
            copy_words(A.goal_pos + i * A.words, J.goal_pos, J.W, z, lane);
            copy_words(A.goal_neg + i * A.words, J.goal_neg, J.W, z, lane);
        }
        if (lane == 0)
        {
            if (!kOne && A.task_ids)
                A.task_ids[i] = static_cast<i32>(next);
            if (A.count)
                A.count[i] = static_cast<i32>(J.init_count);
            A.at_goal[i] = J.init_goal ? 1 : 0;
            if (have_steps)
                steps[i] = 0;
        }
        if (crow)
            for (u32 q = lane; q < cw; q += kWave)
                crow[q] = J.init_cache[q];
        if (kVisited && A.visited.capacity)
            visited_restart(A.visited.table + i * A.visited.capacity, A.visited.capacity, A.visited.count + i, J.init_hash, lane);
    }
    else
    {
        // a move changes only the words of its effects' slots: one per effect lane (lanes sharing a word write the same
        // value)
        if (st == kOk && moved_slot != kNone)
            grow[moved_slot >> 6] = L.row[moved_slot >> 6];
        if (lane == 0)
        {
            A.at_goal[i] = g ? 1 : 0;
            if (have_steps)
                steps[i] = t2;
            if (A.count)
                A.count[i] = static_cast<i32>(c2);
        }
        // the count cache of the state the row now holds: the counts in LDS (of s' after a move, of s otherwise)
        // unless they came from the cache
        if (crow && (st == kOk || !cached))
            store_counts(T, L, crow, cw, lane, fp);
    }
    // 6. the observation's encoding: true-atom slots and applicable-schema masks (LDS holds the per-schema counts of
    // the state the row holds unless the row was reset)
    if (A.atoms || A.masks)
    {
        wave_sync();
        if (A.atoms)
        {
            if (reset)
                encode_row<4>(A.inst[next].initial, A.inst[next].W, A.atoms + i * A.max_atoms, A.max_atoms, lane, A.status);
            else
                encode_row<4>(L.row, T.W, A.atoms + i * A.max_atoms, A.max_atoms, lane, A.status);
        }
        if (A.masks)
            for (u32 q = lane; q < A.mask_width; q += kWave)
                A.masks[i * A.mask_width + q] = reset ? A.inst[next].init_masks[q] : (q < T.num_schemas && L.counts[q] > 0 ? 1 : 0);
    }
    wave_sync();
}

/// Instance k's tables, read through the constant address space: loads of them are invariant, so the compiler
/// re-reads a field with a scalar load where it needs it instead of holding the whole record in registers.
__device__ __forceinline__ const TaskDev& instance_tables(const TaskDev* tasks, u32 k)
{
    return *(const TaskDev*)((cst<TaskDev>*)tasks + k);
}

/// Waves per SIMD the env step is compiled for.
constexpr int kEnvStepWaves = 4;

/// The step of a batch in batch order, a wave per row: with kOne every row as instance 0 (the host checks given task ids
/// and next_task_ids with launch_check_ids first), else each row with the tables of its own instance (the rows whose
/// task id names no instance set kStatusTaskId and stay as they are). The waves read the tables through the caches, so
/// rows of different instances need no grouping.
template<bool kOne, bool kVisited, bool kPlain>
__global__ __launch_bounds__(kMaxWaves * kWave) __attribute__((amdgpu_waves_per_eu(kEnvStepWaves))) void k_env_step(EnvArgs A)
{
    extern __shared__ u64 smem[];
    const u32 lane = lane_id(), wave = uni(threadIdx.x / kWave), nw = blockDim.x / kWave;
    lds<u64>* const region = (lds<u64>*)smem + static_cast<u64>(wave) * A.wave_words;
    for (u64 i = static_cast<u64>(blockIdx.x) * nw + wave; i < A.rows; i += static_cast<u64>(gridDim.x) * nw)
    {
        u32 k = 0;
        if constexpr (!kOne)
        {
            k = uni(static_cast<u32>(A.task_ids[i]));
            if (k >= A.instances)
            {
                if (lane == 0)
                    atomicOr(A.status, kStatusTaskId);
                continue;
            }
        }
        const EnvArgs& a = kernel_args<EnvArgs>();
        const TaskDev& T = kOne ? a.T : instance_tables(a.tasks, k);
        step_row<kOne, kVisited, kPlain>(a, T, tab_of(T), lds_of(region, T), i, k, lane);
    }
}

/// The count of row i of instance k (HostEnv::refresh / count_row, src/mymyr/rl/env.cpp:283-322): successors, goal
/// (per-env masks, checked against the instance's slots, or the instance's goal test), masks and the count cache.
__device__ __forceinline__ void count_row(const CountArgs& A, const TaskDev& T, const Tab& H, const Lds& L, u64 i, u32 k, u32 lane)
{
    load_row_lds(T, L, A.states + i * A.words, lane);
    build_view(T, H, L, lane);
    const u32 c = count_all(T, H, L, lane);
    bool g;
    if (A.goal_pos)
    {
        const u64* gp = A.goal_pos + i * A.words;
        const u64* gn = A.goal_neg + i * A.words;
        if (!goal_masks_fit(gp, gn, A.words, T, lane) && lane == 0 && A.status)
            atomicOr(A.status, kStatusGoalMask);
        g = mask_goal(L.row, gp, gn, T.W, lane);
    }
    else
        g = goal_test(T, H, L.row, lane);
    if (lane == 0)
    {
        if (A.count)
            A.count[i] = static_cast<i32>(c);
        if (A.goal)
            A.goal[i] = g ? 1 : 0;
    }
    if (A.masks)
        for (u32 q = lane; q < A.mask_width; q += kWave)
            A.masks[i * A.mask_width + q] = q < T.num_schemas && L.counts[q] > 0 ? 1 : 0;
    if (A.cache)
        store_counts(T, L, A.cache + i * A.cache_width, A.cache_width, lane, state_fingerprint(L.row, T.W, lane) + instance_salt(k));
    wave_sync();
}

/// The count of a batch in batch order: with kOne every row as instance A.instance (T's), else each row with the tables
/// of its own instance. Rows whose task id names no instance (with kOne: is not 0) set kStatusTaskId and are not counted.
template<bool kOne>
__global__ __launch_bounds__(kMaxWaves * kWave) void k_env_count(CountArgs A)
{
    extern __shared__ u64 smem[];
    const u32 lane = lane_id(), wave = uni(threadIdx.x / kWave), nw = blockDim.x / kWave;
    lds<u64>* const region = (lds<u64>*)smem + static_cast<u64>(wave) * A.wave_words;
    for (u64 i = static_cast<u64>(blockIdx.x) * nw + wave; i < A.rows; i += static_cast<u64>(gridDim.x) * nw)
    {
        const u32 k = A.task_ids ? uni(static_cast<u32>(A.task_ids[i])) : 0u;
        if (k >= (kOne ? 1u : A.instances))
        {
            if (lane == 0 && A.status)
                atomicOr(A.status, kStatusTaskId);
            continue;
        }
        const CountArgs& a = kernel_args<CountArgs>();
        const TaskDev& T = kOne ? a.T : instance_tables(a.tasks, k);
        count_row(a, T, tab_of(T), lds_of(region, T), i, kOne ? A.instance : k, lane);
    }
}

/// Applies the effects of the picked binding of schema s to the LDS row only (the view stays the parent's), keeping
/// the effect slots and their prior bits for succ_revert. Returns whether no bit changed (a no-op successor). One effect
/// per lane (lane k: slot L.eff[k], prior bit L.before[k]); deletes, then adds.
__device__ __forceinline__ bool succ_apply(const TaskDev& T, const Tab& H, const Lds& L, u32 s, u32 lane, u32* status)
{
    const auto& S = H.schemas[s];
    const u32 ne = min(S.eff_end - S.eff_begin, kMaxEff);
    if (lane == 0 && S.eff_end - S.eff_begin > kMaxEff)
        atomicOr(status, kStatusCapacity);
    const bool mine = lane < ne;
    const bool add = lane < S.nadd;
    u32 sl = kNone;
    bool before = false;
    if (mine)
    {
        u64 cid;
        sl = effect_slot(T, L, ld(H.effects + S.eff_begin + lane), &cid);
        before = sl != kNone && row_bit(L.row, sl);
        L.eff[lane] = sl;
        L.before[lane] = before ? 1u : 0u;
        if (add && sl == kNone)
            missing_atom(T, cid, status);
    }
    wave_sync();
    if (mine && !add && sl != kNone)
        __hip_atomic_fetch_and(L.row + (sl >> 6), ~(u64{1} << (sl & 63)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    wave_sync();
    if (mine && add && sl != kNone)
        __hip_atomic_fetch_or(L.row + (sl >> 6), u64{1} << (sl & 63), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    wave_sync();
    const bool changed = mine && sl != kNone && row_bit(L.row, sl) != before;
    return __ballot(changed) == 0;
}

/// Restores the parent row after succ_apply (lanes listing one slot hold the same prior bit).
__device__ __forceinline__ void succ_revert(const Tab& H, const Lds& L, u32 s, u32 lane)
{
    const auto& S = H.schemas[s];
    const u32 ne = min(S.eff_end - S.eff_begin, kMaxEff);
    if (lane < ne)
    {
        const u32 sl = L.eff[lane];
        if (sl != kNone)
        {
            if (L.before[lane])
                __hip_atomic_fetch_or(L.row + (sl >> 6), u64{1} << (sl & 63), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
            else
                __hip_atomic_fetch_and(L.row + (sl >> 6), ~(u64{1} << (sl & 63)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
        }
    }
    wave_sync();
}

/// 1 + the index of the highest nonzero word of the LDS row (0 for an empty row), on every lane.
__device__ __forceinline__ u32 trimmed_words(const lds<u64>* row, u32 W, u32 lane)
{
    u32 top = 0;
    for (u32 w = lane; w < W; w += kWave)
        if (row[w])
            top = w + 1;
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1)
        top = max(top, static_cast<u32>(__shfl_xor(static_cast<int>(top), d, kWave)));
    return top;
}

/// Witness pruning (include/mymyr/successor/successors.hpp:154-248 with witness pruning on): the successor counts of
/// the schemas with witness parameters become the number of full bindings whose witnesses the matcher binds first (one
/// per effect-relevant binding), counted by enumerating those schemas; `total` (count_all's) is corrected to match.
__device__ __forceinline__ u32 witness_counts(const TaskDev& T, const Tab& H, const Lds& L, u32 lane, u32 total)
{
    if (!T.witness)
        return total;
    for (u32 s = 0; s < T.num_schemas; ++s)
    {
        const u32 all = uni(L.counts[s]);
        if (T.witness[s].n == 0 || all == 0)
            continue;
        const u32 kept = for_each_successor<true>(T, H, L, lane, [](u32, u32) { return true; }, s, s + 1);
        wave_sync();
        if (lane == 0)
            L.counts[s] = kept;
        wave_sync();
        total = total - all + kept;
    }
    return total;
}

/// A lane's bindings of schema parameters [I, arity) that complete its binding, in lexicographic order: packed (16 bits
/// per object) into list[index - lo] for the indices in [lo, hi), the first of them `index`.
template<u32 I>
__device__ __forceinline__ void list_lanes(const Tab& H, const Lds& L, const auto& S, u32 arity, u64 prefix, u32& index, u32 lo, u32 hi,
                                           lds<u64>* list, u32 lane)
{
    const DevStep F = ld(H.steps + S.filter_step[I]);
    for (u32 w = 0; w < F.words; ++w)
        for (u64 m = cand_word(H, L, F, w, lane); m; m &= m - 1)
        {
            const u32 o = F.lo + 64 * w + static_cast<u32>(__builtin_ctzll(m));
            const u64 e = prefix | (static_cast<u64>(o) << (16 * I));
            if (I + 1 == arity)
            {
                if (index >= lo && index < hi)
                    list[index - lo] = e;
                ++index;
            }
            else if constexpr (I < kLaneDepth)
            {
                L.bind[I * 64 + lane] = o;
                list_lanes<I + 1>(H, L, S, arity, e, index, lo, hi, list, lane);
            }
        }
}

/// The successors of the state in canonical order, kListCap at a time, for listable tasks (TaskDev::listable). Each schema's
/// first parameter's candidates are spread over the lanes, which count their completions (their places in the list) and
/// then write their bindings there; the list is handed on 64 successors at a time: flush(s, first, n) with the bindings
/// of successors [0, n) at list[first ..].
template<class Flush>
__device__ __forceinline__ void for_each_listed(const TaskDev& T, const Tab& H, const Lds& L, lds<u64>* list, u32 lane, Flush&& flush)
{
    for (u32 s = 0; s < T.num_schemas; ++s)
    {
        if (uni(L.counts[s]) == 0)
            continue;
        const auto& S = H.schemas[s];
        const u32 arity = S.arity;
        if (arity == 0)
        {
            if (lane == 0)
                list[0] = 0;
            wave_sync();
            flush(s, 0u, 1u);
            continue;
        }
        const DevStep F = ld(H.steps + S.filter_step[0]);
        const u32 pb = S.plan_begin[1], pe = S.plan_begin[2];
        for_nonzero_words(T, H, L, F, 0, lane, [&](u32 w, u64 m) {
            const u32 o = F.lo + 64 * w + lane;
            u32 c = 0;
            if ((m >> lane) & 1)
            {
                L.bind[lane] = o;
                c = count_lanes<kLaneDepth>(T, H, L, pb, pe, lane);
            }
            const u32 incl = wave_inclusive(c), total = lane_value(incl, kWave - 1), at = incl - c;
            for (u32 lo = 0; lo < total; lo += kListCap)
            {
                const u32 hi = min(total, lo + kListCap);
                wave_sync();
                if (c && at < hi && incl > lo)
                {
                    if (arity == 1)
                        list[at - lo] = o;
                    else
                    {
                        u32 index = at;
                        list_lanes<1>(H, L, S, arity, o, index, lo, hi, list, lane);
                    }
                }
                wave_sync();
                for (u32 b = lo; b < hi; b += kWave)
                    flush(s, b - lo, min(static_cast<u32>(kWave), hi - b));
            }
            return false;
        });
    }
}

/// The expansion of a row of a listable task (as expand_row), 64 successors at a time: each lane forms one successor's
/// effect slots, flags and label from its binding, then the wave writes the successor rows one after the other, the
/// parent's words with the effects' bits patched in registers.
__device__ __forceinline__ void expand_listed(const ExpandArgs& A, const TaskDev& T, const Tab& H, const Lds& L, lds<u64>* list, u64 i, u32 c,
                                              u32 lane)
{
    const bool drop = A.drop_noops != 0;
    const bool write = A.pass == 1;
    const bool keep_all = write && drop && uni(A.noops[i]) == c;
    const u64 out0 = write ? A.offsets[i] - A.offset_base : 0;
    u32 listed = 0, kept = 0, noops = 0;
    for_each_listed(T, H, L, list, lane, [&](u32 s, u32 first, u32 n) {
        const auto& S = H.schemas[s];
        const u32 eff = S.eff_begin, ne = S.eff_end - eff, nadd = S.nadd;
        const bool mine = lane < n;
        const u64 bind = mine ? list[first + lane] : 0;
        // the lane's successor: its effects' slots, and whether it changes a bit (delete, then add)
        u32 sl[kListEff];
        bool changed = false;
#pragma unroll
        for (u32 j = 0; j < kListEff; ++j)
        {
            sl[j] = kNone;
            if (j >= ne)
                continue;
            const DevEffect e = ld(H.effects + eff + j);
            u64 cid = e.arith ? e.arith_base : e.base;
#pragma unroll
            for (u32 v = 0; v < 4; ++v)
                if (v < e.nvar)
                {
                    const u32 o = static_cast<u32>(bind >> (16 * e.var_param[v])) & 0xFFFF;
                    cid += e.arith ? o * e.mul[v] : T.rs[static_cast<u64>(e.var_pos[v]) * T.n + o];
                }
            if (mine && cid < T.fluent_count)
                sl[j] = T.dense ? static_cast<u32>(cid) : T.slot_of[cid];
            if (mine && j < nadd && sl[j] == kNone)
                missing_atom(T, cid, A.status);
        }
        auto bit = [&](u32 q) {  // bit q of the lane's successor
            bool v = q < 64 * T.W && row_bit(L.row, q);
#pragma unroll
            for (u32 j = kListEff; j-- > 0;)  // deletes (last) first, so that the adds win
                if (j < ne && sl[j] == q)
                    v = j < nadd;
            return v;
        };
#pragma unroll
        for (u32 j = 0; j < kListEff; ++j)
            if (j < ne && sl[j] != kNone)
                changed = changed || bit(sl[j]) != row_bit(L.row, sl[j]);
        const bool noop = !changed;
        noops += static_cast<u32>(__popcll(__ballot(mine && noop)));
        const bool take = mine && (!drop || !noop || keep_all);
        const u64 took = __ballot(take);
        const u32 k = listed + lane;
        const u64 pos = out0 + (drop ? kept + static_cast<u32>(__popcll(took & ((u64{1} << lane) - 1))) : k);
        listed += n;
        kept += static_cast<u32>(__popcll(took));
        const bool out = write && take && pos < A.capacity;
        if (out)
        {
            if (A.goal)
            {
                bool g;
                if (A.any_goal.any)
                    g = any_of_holds_dev(A.any_goal, bit);
                else
                {
                    g = !T.goal_unsat;
                    for (u32 q = 0; q < T.ngp; ++q)
                        g = g && bit(H.goal_pos[q]);
                    for (u32 q = 0; q < T.ngn; ++q)
                        g = g && !bit(H.goal_neg[q]);
                }
                A.goal[pos] = g ? 1 : 0;
            }
            if (A.noop)
                A.noop[pos] = noop ? 1 : 0;
            if (A.index)
                A.index[pos] = static_cast<i32>(k);
            if (A.parent)
                A.parent[pos] = static_cast<i32>(i);
            if (A.schema)
                A.schema[pos] = static_cast<i32>(s);
            if (A.binding)
                for (u32 q = 0; q < A.label_width; ++q)
                    A.binding[pos * A.label_width + q] = q < S.arity ? static_cast<i32>((bind >> (16 * q)) & 0xFFFF) : -1;
        }
        if (!A.succ)
            return;
        if (A.out_words <= kListRegs * kWave)
        {
            // the parent's words stay in registers, and an effect's word and bit are scalars: read from LDS for each
            // successor and compared with every effect in every word, the rows of 176-word transport states were written
            // slower (10^6-state search 5.77 -> 5.46 ms, 8,195 states expanded 1.81 -> 1.73 ms)
            u64 row[kListRegs];
#pragma unroll
            for (u32 r = 0; r < kListRegs; ++r)
                row[r] = r * kWave + lane < T.W ? L.row[r * kWave + lane] : 0;
            for (u64 x = __ballot(out); x; x &= x - 1)
            {
                const u32 j = static_cast<u32>(__builtin_ctzll(x));
                u64* const dst = A.succ + lane_value(pos, j) * A.out_words;
                u64 v[kListRegs];
#pragma unroll
                for (u32 r = 0; r < kListRegs; ++r)
                    v[r] = row[r];
#pragma unroll
                for (u32 q = kListEff; q-- > 0;)
                {
                    if (q >= ne)
                        continue;
                    const u32 e = lane_value(sl[q], j);
                    if (e == kNone)
                        continue;
                    const u64 b = lane == ((e >> 6) & (kWave - 1)) ? u64{1} << (e & 63) : 0;
#pragma unroll
                    for (u32 r = 0; r < kListRegs; ++r)
                        if (e >> 12 == r)
                            v[r] = q < nadd ? v[r] | b : v[r] & ~b;
                }
#pragma unroll
                for (u32 r = 0; r < kListRegs; ++r)
                    if (r * kWave + lane < A.out_words)
                        dst[r * kWave + lane] = v[r];
            }
            return;
        }
        for (u64 x = __ballot(out); x; x &= x - 1)
        {
            const u32 j = static_cast<u32>(__builtin_ctzll(x));
            u64* const dst = A.succ + lane_value(pos, j) * A.out_words;
            u32 es[kListEff];
#pragma unroll
            for (u32 q = 0; q < kListEff; ++q)
                es[q] = q < ne ? lane_value(sl[q], j) : kNone;
            for (u32 w = lane; w < A.out_words; w += kWave)
            {
                u64 v = w < T.W ? L.row[w] : 0;
#pragma unroll
                for (u32 q = kListEff; q-- > 0;)
                    if (q < ne && w == es[q] >> 6 && es[q] != kNone)
                    {
                        const u64 b = u64{1} << (es[q] & 63);
                        v = q < nadd ? v | b : v & ~b;
                    }
                dst[w] = v;
            }
        }
    });
    if (listed != c && lane == 0)
        atomicOr(A.status, kStatusPickFailed);
    if (A.pass == 0 && lane == 0)
    {
        A.counts[i] = c;
        A.noops[i] = noops;
    }
    wave_sync();
}

/// The expansion of row i (pass 0: its counts and the validation of its words; pass 1: its successors from
/// offsets[i] on) with the tables of its instance.
template<bool kWitness>
__device__ __forceinline__ void expand_row(const ExpandArgs& A, const TaskDev& T, const Tab& H, const Lds& L, [[maybe_unused]] lds<u64>* list, u64 i,
                                           u32 lane)
{
    const u32 Lw = A.label_width;
    const u64* src = A.states + i * A.words;
    if (A.pass == 0)
    {
        // rows must hold no atoms past the task's slots (ExpandOptions::validate)
        bool wide = false;
        for (u32 w = lane; w < A.words; w += kWave)
        {
            const u64 x = src[w];
            if (w >= T.W)
                wide = wide || x != 0;
            else if (w == T.W - 1 && (T.fluent_slots & 63))
                wide = wide || (x >> (T.fluent_slots & 63)) != 0;
        }
        if (__ballot(wide) && lane == 0)
            atomicOr(A.status, kStatusWideRow);
    }
    load_row_lds_n(T, L, src, min(A.words, T.W), lane);
    build_view(T, H, L, lane);
    u32 c = count_all(T, H, L, lane);
    if constexpr (kWitness)
        c = witness_counts(T, H, L, lane, c);
    if (A.pass == 0 && !A.drop_noops)
    {
        if (lane == 0)
            A.counts[i] = c;
        return;
    }
    if constexpr (!kGeneral && !kWitness)
        if (A.list)
        {
            expand_listed(A, T, H, L, list, i, c, lane);
            return;
        }
    const bool keep_all = A.pass == 1 && A.drop_noops && A.noops[i] == c;
    u32 noops = 0, kept = 0;
    const u32 listed = for_each_successor<kWitness>(T, H, L, lane, [&](u32 k, u32 s) {
        const bool noop = succ_apply(T, H, L, s, lane, A.status);
        noops += noop ? 1 : 0;
        if (A.pass == 1 && (!A.drop_noops || !noop || keep_all))
        {
            const u64 pos = A.offsets[i] - A.offset_base + (A.drop_noops ? kept : k);
            ++kept;
            const u32 n = (A.succ_hash || (A.succ && A.out_words < T.W)) ? trimmed_words(L.row, T.W, lane) : 0;
            const bool fits = n <= A.out_words;
            if (A.succ && !fits && lane == 0)
                atomicMax(A.words_needed, n);
            if (pos < A.capacity)
            {
                if (A.succ)
                {
                    u64* dst = A.succ + pos * A.out_words;
                    for (u32 w = lane; w < A.out_words; w += kWave)
                        dst[w] = (fits && w < T.W) ? L.row[w] : 0;
                }
                if (A.goal)
                {
                    const bool g = A.any_goal.any
                                       ? any_of_holds_dev(A.any_goal, [&](u32 s) { return s < 64 * T.W && row_bit(L.row, s); })
                                       : goal_test(T, H, L.row, lane);
                    if (lane == 0)
                        A.goal[pos] = g ? 1 : 0;
                }
                if (lane == 0)
                {
                    if (A.succ_hash)
                    {
                        // hash_state over the trimmed words: the pairs chained in order
                        u64 h = kHashSeed ^ (static_cast<u64>(n) * kHashP1);
                        for (u32 w = 0; w < n; w += 2)
                            h = mulfold(h ^ L.row[w] ^ kHashP1, (w + 1 < n ? L.row[w + 1] : 0) ^ kHashP2);
                        A.succ_hash[pos] = mix64(h);
                    }
                    if (A.noop)
                        A.noop[pos] = noop ? 1 : 0;
                    if (A.index)
                        A.index[pos] = static_cast<i32>(k);
                    if (A.parent)
                        A.parent[pos] = static_cast<i32>(i);
                    if (A.schema)
                        A.schema[pos] = static_cast<i32>(s);
                }
                if (A.binding)
                {
                    const u32 arity = H.schemas[s].arity;
                    for (u32 q = lane; q < Lw; q += kWave)
                        A.binding[pos * Lw + q] = q < arity ? static_cast<i32>(L.ub[q]) : -1;
                }
            }
        }
        succ_revert(H, L, s, lane);
        return true;
    });
    if (listed != c && lane == 0)
        atomicOr(A.status, kStatusPickFailed);
    if (A.pass == 0 && lane == 0)
    {
        A.counts[i] = c;
        A.noops[i] = noops;
    }
    wave_sync();
}

/// The expansion of a batch in batch order: with kOne every row with T's tables, else each row with its own instance's
/// (rows whose task id names no instance set kStatusTaskId and count no successors).
template<bool kOne, bool kWitness>
__global__ __launch_bounds__(kMaxWaves * kWave) void k_expand(ExpandArgs A)
{
    extern __shared__ u64 smem[];
    const u32 lane = lane_id(), wave = uni(threadIdx.x / kWave), nw = blockDim.x / kWave;
    lds<u64>* const region = (lds<u64>*)smem + static_cast<u64>(wave) * (A.wave_words + (A.list ? kListCap : 0));
    for (u64 i = static_cast<u64>(blockIdx.x) * nw + wave; i < A.rows; i += static_cast<u64>(gridDim.x) * nw)
    {
        u32 k = 0;
        if constexpr (!kOne)
        {
            k = uni(static_cast<u32>(A.task_ids[i]));
            if (k >= A.instances)
            {
                if (lane == 0)
                {
                    atomicOr(A.status, kStatusTaskId);
                    if (A.pass == 0)
                    {
                        A.counts[i] = 0;
                        if (A.drop_noops)
                            A.noops[i] = 0;
                    }
                }
                continue;
            }
        }
        const ExpandArgs& a = kernel_args<ExpandArgs>();
        const TaskDev& T = kOne ? a.T : instance_tables(a.tasks, k);
        expand_row<kWitness>(a, T, tab_of(T), lds_of(region, T), region + A.wave_words, i, lane);
    }
}

// Successor listing: successor k of row i is pick(k) applied to a copy of the row.
__global__ __launch_bounds__(kMaxWaves * kWave) void k_successors(TaskDev T0, const u64* states, u64 rows, u32 words, u32 cap, i32* count,
                                                                  i32* schema, i32* binding, u64* succ, u32* status)
{
    extern __shared__ u64 smem[];
    const u32 lane = lane_id(), wave = uni(threadIdx.x / kWave), nw = blockDim.x / kWave;
    const TaskDev& T = kernel_args<TaskDev>();
    const Tab H = tab_of(T);
    const Lds L = lds_of((lds<u64>*)smem + static_cast<u64>(wave) * T.l_words, T);
    const u32 Lw = T.label_width;
    for (u64 i = static_cast<u64>(blockIdx.x) * nw + wave; i < rows; i += static_cast<u64>(gridDim.x) * nw)
    {
        load_row_lds_n(T, L, states + i * words, min(words, T.W), lane);
        build_view(T, H, L, lane);
        const u32 c = count_all(T, H, L, lane);
        if (lane == 0 && count)
            count[i] = static_cast<i32>(c);
        const u32 listed = cap == 0 ? 0 : for_each_successor<false>(T, H, L, lane, [&](u32 k, u32 s) {
            const u64 o = i * cap + k;
            if (lane == 0 && schema)
                schema[o] = static_cast<i32>(s);
            const auto& S = H.schemas[s];
            if (binding)
                for (u32 q = lane; q < Lw; q += kWave)
                    binding[o * Lw + q] = q < S.arity ? static_cast<i32>(L.ub[q]) : -1;
            if (succ)
            {
                // the successor on the LDS row (one effect per lane), copied out, then the row restored
                succ_apply(T, H, L, s, lane, status);
                u64* dst = succ + o * words;
                for (u32 q = lane; q < words; q += kWave)
                    dst[q] = q < T.W ? L.row[q] : 0;
                // a successor with atoms past the rows' words (a lazy task's rows outgrew them) is an error
                bool wide = false;
                for (u32 q = words + lane; q < T.W; q += kWave)
                    wide = wide || L.row[q] != 0;
                if (__ballot(wide) && lane == 0)
                    atomicOr(status, kStatusWideRow);
                succ_revert(H, L, s, lane);
            }
            wave_sync();
            return k + 1 < cap;
        });
        if (listed != min(c, cap) && lane == 0)
            atomicOr(status, kStatusPickFailed);
        wave_sync();
    }
}


EnvKernels env_kernels()
{
    EnvKernels k{};
    if constexpr (!kGeneral)
        k.step_plain = k_env_step<true, false, true>;
    k.step = k_env_step<true, kGeneral, false>;
    k.step_visited = k_env_step<true, true, false>;
    k.step_table = k_env_step<false, true, false>;
    k.count = k_env_count<true>;
    k.count_table = k_env_count<false>;
    k.expand = k_expand<true, false>;
    k.expand_witness = k_expand<true, true>;
    k.expand_table = k_expand<false, false>;
    k.successors = k_successors;
    return k;
}
}  // namespace
}  // namespace mya
