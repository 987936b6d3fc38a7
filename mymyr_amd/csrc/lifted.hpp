#pragma once
// Device-side lifted matching over one state, executed by one wavefront (64 lanes) per state:
//   - the view: per fluent predicate of arity 1 one row, of arity 2 forward / backward rows, each row an object bitset
//     over the window of the other position's domain. Rows that are contiguous slices of the state (dense slots over
//     contiguous domains, forward direction) are read from the state row itself; the others are built in LDS from
//     the state's set bits;
//   - count(schema, plan j): the number of applicable full bindings extending a bound prefix, a nested loop over the
//     plan's parameters whose candidates are ANDs of 64-bit words (dom0, view rows, static rows), with k-ary literals
//     checked at the level that binds their last parameter;
//   - pick(schema, rank): the rank-th applicable binding in lexicographic parameter order, by prefix counting.
// The set of bindings is the reference's (all literals of the precondition hold; witness pruning off), and the
// lexicographic order is its canonical order (include/mymyr/successor/successors.hpp:8-10, 154-248).
//
// The plans are the same for every lane, so the kernels read them (schemas, steps, terms, checks) through the constant
// address space with wave-uniform indices: scalar loads and scalar branches, while the vector units do only the
// candidates' bit work. Each wave has its own LDS region (state row, view, lane bindings).

#include "device_common.hpp"
#include "scan.hpp"
#include "task.hpp"

namespace mya
{
/// The task as the kernels see it: sections by word offset in the image, tables read lane by lane by pointer.
struct TaskDev
{
    u64 off_schemas, off_deltas, off_checks, off_effects, off_pairs, off_decode;
    u64 off_goal_pos, off_goal_neg, off_pred_arity, off_pos_begin, off_pred_pairs, off_pred_offset;
    const u64* image;
    const u64* rs;
    const u32* slot_of;
    const u64* records;
    const DevStaticMeta* static_meta;
    const u64* static_words;  // image base (static keys are image offsets)
    const u64* initial;
    u64 fluent_count;
    u32 n, ow, W, num_schemas, num_pairs, view_words, ngp, ngn, goal_unsat, dense, label_width, fluent_slots;
    u32 num_decode, decode_arith;
    u32 simple;    // no literal is checked one by one and no schema has more than kLaneDepth + 1 parameters
    u32 listable;  // simple, at most kListEff effects per schema and objects of 16 bits: successors are listed (expand_listed)
    u32 lazy;      // lazy slots: an added atom without a slot is recorded in `missing`
    u64* missing;  // lazy slots: bit per canonical fluent atom (device; set by the successor kernels), else null
    u32 l_row, l_dfs_m, l_ub, l_bind, l_counts, l_dfs_w, l_eff, l_before, l_cur, l_step, l_words;  // a wave's LDS region (set_region)
    const DevWitness* witness;  // per schema its witness parameters and plans (null: no schema has a witness)
};

/// Pointers into an uploaded image (host helper).
TaskDev task_dev(const u64* image_dev, const DevTaskHeader& h);

constexpr u32 kMaxEnvSchemas = 8192;  // schemas whose per-state counts a wave keeps in LDS
constexpr u32 kListCap = 128;      // successors listed at a time (a word each in the expansion's LDS)
constexpr u32 kMaxEff = 32;        // effects per schema the step applies (more set kStatusCapacity)

/// The word offsets of a wave's LDS region: the view, the state row, then the uniform binding, the 64 lanes' bindings
/// (A = the largest schema arity, at least 1), the per-schema counts, for plans deeper than kLaneDepth the lanes'
/// enumeration cursors (so far l_step words: the step's and the count's region), the successor enumeration's level
/// cursors (A masks, A words) and its effect scratch. A read of two words at a bit position (row_bits) ends at most at
/// the word after the row, the binding's. A step's region is what limits the waves of wide states: a
/// transport_xl wave takes 22,816 bytes without the enumeration's scratch and 23,120 with it, seven waves to a CU or six
/// (the allocation's granularity rounds the latter up past a seventh of the 160 KiB): 6.21 -> 5.38 ms per step.
inline void set_region(TaskDev& t)
{
    const u32 A = t.label_width ? t.label_width : 1;
    u32 w = t.view_words;
    auto next = [&](u32 words) {
        const u32 at = w;
        w += words;
        return at;
    };
    t.l_row = next(t.W);
    t.l_ub = next((A + 1) / 2);
    t.l_bind = next(32 * A);
    t.l_counts = next((t.num_schemas + 1) / 2);
    t.l_cur = next(A > kLaneDepth ? 64 * A + 32 * A : 0);
    t.l_step = (w + 1) & ~1u;
    t.l_dfs_m = next(A);
    t.l_dfs_w = next((A + 1) / 2);
    t.l_eff = next(kMaxEff / 2);
    t.l_before = next(kMaxEff / 2);
    t.l_words = (w + 1) & ~1u;
}
}  // namespace mya
