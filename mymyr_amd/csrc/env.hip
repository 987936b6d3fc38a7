// Lifted matching (lifted.hpp) and the device env step (env.hpp). A block holds up to kMaxWaves wavefronts; each wave
// works on one state at a time in its own LDS region. Waves of a block run different states, so every barrier inside the
// per-state work is a wavefront barrier.

#define MYA_GENERAL_TASKS 0
#include "env_device.hpp"
#include "runtime.hpp"
#include "state_set.hpp"

#include <algorithm>
#include <mutex>
#include <type_traits>
#include <unordered_map>

namespace mya
{
TaskDev task_dev(const u64* img, const DevTaskHeader& h)
{
    TaskDev t{};
    t.off_schemas = h.off_schemas;
    t.off_deltas = h.off_deltas;
    t.off_checks = h.off_checks;
    t.off_effects = h.off_effects;
    t.off_pairs = h.off_pairs;
    t.off_decode = h.off_decode;
    t.off_goal_pos = h.off_goal_pos;
    t.off_goal_neg = h.off_goal_neg;
    t.off_pred_arity = h.off_pred_arity;
    t.off_pos_begin = h.off_pos_begin;
    t.off_pred_pairs = h.off_pred_pairs;
    t.off_pred_offset = h.off_pred_offset;
    t.image = img;
    t.rs = img + h.off_rs;
    t.slot_of = reinterpret_cast<const u32*>(img + h.off_slot_of);
    t.records = img + h.off_records;
    t.static_meta = reinterpret_cast<const DevStaticMeta*>(img + h.off_static_meta);
    t.static_words = img;
    t.initial = img + h.off_initial;
    t.witness = h.off_witness ? reinterpret_cast<const DevWitness*>(img + h.off_witness) : nullptr;
    t.fluent_count = h.fluent_count;
    t.n = h.num_objects;
    t.ow = h.ow;
    t.W = h.words;
    t.num_schemas = h.num_schemas;
    t.num_pairs = h.num_pairs;
    t.view_words = h.view_words;
    t.ngp = h.num_goal_pos;
    t.ngn = h.num_goal_neg;
    t.goal_unsat = h.goal_unsat;
    t.dense = h.dense;
    t.label_width = h.label_width;
    t.fluent_slots = h.fluent_slots;
    t.num_decode = h.num_decode;
    t.decode_arith = h.decode_arith;
    t.lazy = h.lazy;
    t.missing = nullptr;
    t.simple = h.simple;
    t.listable = h.listable;
    set_region(t);
    return t;
}

namespace
{
constexpr size_t kCuLds = 160 * 1024;  // a CU's LDS, and the most a workgroup can have

/// The waves per block that keep the most waves resident on a CU (its 160 KiB of LDS shared by whole blocks), for
/// `wave` bytes per wave; a smaller block is taken only for at least 1/8 more resident waves.
unsigned block_shape(size_t wave, size_t* lds_bytes)
{
    // the waves per CU that the registers of the simple tasks' steps and counts allow; of their expansions 24 and of the
    // general kernels 20 are resident, and the shape chosen against 28 holds as many of them as one chosen against these
    constexpr int kCuWaves = 28;
    int nw = 1, best = 0;
    for (int k = kMaxWaves; k >= 1; --k)
    {
        const size_t block = static_cast<size_t>(k) * wave;
        if (block > kCuLds)
            continue;
        const int resident = std::min(kCuWaves, k * static_cast<int>(kCuLds / block));
        if (8 * resident > 9 * best)
        {
            best = resident;
            nw = k;
        }
    }
    *lds_bytes = static_cast<size_t>(nw) * wave;
    if (*lds_bytes > kCuLds)
        throw std::invalid_argument("mymyr_amd: env: the task's per-state LDS (" + std::to_string(*lds_bytes) +
                                    " bytes) exceeds the 160 KiB of a gfx950 workgroup");
    return static_cast<unsigned>(nw);
}

void check_schemas(const TaskDev& T)
{
    if (T.num_schemas > kMaxEnvSchemas)
        throw std::invalid_argument("mymyr_amd: env: the device step keeps the successor counts of at most " + std::to_string(kMaxEnvSchemas) +
                                    " schemas (the task has " + std::to_string(T.num_schemas) + ")");
}

/// visited_mask (include/mymyr/rl/visited.hpp:63-74), one lane per successor: whether succ_hash[j] is in the table of
/// row parent[j] (or rows[parent[j]]). Padding (-1) and parents or rows outside the tables read as not visited.
__global__ __launch_bounds__(256) void k_visited_mask(const u64* table, const i32* count, u64 table_rows, u32 H, const u64* succ_hash,
                                                      const i32* parent, const i32* rows, u64 parents, u64 size, u8* out)
{
    const u64 stride = u64{gridDim.x} * blockDim.x;
    for (u64 j = static_cast<u64>(blockIdx.x) * blockDim.x + threadIdx.x; j < size; j += stride)
    {
        const i32 p = parent[j];
        bool hit = false;
        const i32 row = p < 0 || static_cast<u64>(p) >= parents ? -1 : rows ? rows[p] : p;
        if (row >= 0 && static_cast<u64>(row) < table_rows && count[row])
        {
            const u64 h = succ_hash[j], key = h ? h : kVisitedZero;
            const u64* t = table + static_cast<u64>(row) * H;
            u32 at = static_cast<u32>(key) & (H - 1);
            for (u32 probe = 0; probe < H; ++probe, at = (at + 1) & (H - 1))
            {
                const u64 x = t[at];
                if (x == key)
                {
                    hit = true;
                    break;
                }
                if (!x)
                    break;
            }
        }
        out[j] = hit ? 1 : 0;
    }
}

__global__ __launch_bounds__(kWave) void k_encode(const u64* states, u64 rows, u32 words, u32 W, i32* out, u32 max_atoms, u32* status)
{
    const u32 lane = threadIdx.x;
    for (u64 i = blockIdx.x; i < rows; i += gridDim.x)
        encode_row<4>(states + i * words, W, out + i * max_atoms, max_atoms, lane, status);
}

/// The instance a reset puts row i in: task_ids[i] (null: 0); an id outside the table resets into instance 0.
__device__ __forceinline__ u32 reset_instance(const i32* task_ids, u64 i, u32 instances, bool* bad)
{
    const i32 v = task_ids ? task_ids[i] : 0;
    *bad = v < 0 || static_cast<u32>(v) >= instances;
    return *bad ? 0u : static_cast<u32>(v);
}

/// One thread per state word of the batch (reset_row with a dirtied row: zeros up to the batch's words).
__global__ void k_env_reset(const InstDev* inst, u32 instances, u64* states, u64 rows, u32 words, const u8* mask, i32* task_ids,
                            i32* steps, u8* at_goal, i32* count, u32* status)
{
    const u64 total = rows * words;
    for (u64 e = static_cast<u64>(blockIdx.x) * blockDim.x + threadIdx.x; e < total; e += static_cast<u64>(gridDim.x) * blockDim.x)
    {
        const u64 i = e / words;
        const u32 w = static_cast<u32>(e - i * words);
        if (mask && !mask[i])
            continue;
        // the word-0 thread writes a corrected id (0) while the row's other threads may read it: either value they
        // see resets the row into instance 0
        bool bad = false;
        const u32 k = reset_instance(task_ids, i, instances, &bad);
        const InstDev& J = inst[k];
        states[e] = w < J.W ? J.initial[w] : 0;
        if (w == 0)
        {
            if (bad)
            {
                atomicOr(status, kStatusTaskId);
                task_ids[i] = 0;
            }
            if (steps)
                steps[i] = 0;
            if (at_goal)
                at_goal[i] = J.init_goal ? 1 : 0;
            if (count)
                count[i] = static_cast<i32>(J.init_count);
        }
    }
}

/// One wave per row: the masked rows' visited tables restarted with the initial state's key of the row's instance, or
/// (current) the key of the row's state.
__global__ __launch_bounds__(256) void k_visited_restart(VisitedDev v, const InstDev* inst, u32 instances, const u64* states, u64 rows,
                                                         u32 words, const u8* mask, const i32* task_ids, u32 current)
{
    const u32 lane = lane_id(), nw = blockDim.x / kWave;
    for (u64 i = static_cast<u64>(blockIdx.x) * nw + threadIdx.x / kWave; i < rows; i += static_cast<u64>(gridDim.x) * nw)
    {
        if (mask && !mask[i])
            continue;
        bool bad = false;
        const InstDev& J = inst[reset_instance(task_ids, i, instances, &bad)];
        u64 h = J.init_hash;
        if (current)
        {
            u64 mine = 0;
            if (lane == 0)
                mine = row_hash(states + i * words, J.W);
            h = __shfl(mine, 0, kWave);
        }
        visited_restart(v.table + i * v.capacity, v.capacity, v.count + i, h, lane);
    }
}

/// Per row before a reset: the drawn task id (sample) and the advanced reset counter.
__global__ void k_env_reset_draw(SamplerDev sampler, const u64* seed, u64 first_env, u64 rows, const u8* mask, u32 sample, i32* task_ids,
                                 u32* reset_counts, const u64* sampling_seeds, const u32* env_ids)
{
    for (u64 i = static_cast<u64>(blockIdx.x) * blockDim.x + threadIdx.x; i < rows; i += static_cast<u64>(gridDim.x) * blockDim.x)
    {
        if (mask && !mask[i])
            continue;
        if (!reset_counts)
            continue;
        const u32 rc = reset_counts[i];
        if (sample && task_ids)
            task_ids[i] = instance_draw(sampling_seeds ? sampling_seeds[i] : *seed, env_ids ? static_cast<u64>(env_ids[i]) : first_env + i, rc,
                                        sampler.instances, sampler.thresholds, sampler.indices, sampler.m);
        reset_counts[i] = rc + 1;
    }
}

/// The random policy's next choices without a step (DeviceEnv::random_actions, include/mymyr/cuda/env.hpp:189-192):
/// out[i] = successor_index(key, env id, draws[i], min(count[i], max_actions)), 0 where that is 0.
__global__ void k_env_random_actions(const u64* seed, const u64* seeds, const u32* env_ids, u64 first_env, const u64* draws, const i32* count,
                                     u64 rows, u32 max_actions, i64* out)
{
    for (u64 i = static_cast<u64>(blockIdx.x) * blockDim.x + threadIdx.x; i < rows; i += static_cast<u64>(gridDim.x) * blockDim.x)
    {
        const u32 c = min(static_cast<u32>(max(count[i], 0)), max_actions);
        out[i] = c ? static_cast<i64>(successor_index(seeds ? seeds[i] : *seed, env_ids ? static_cast<u64>(env_ids[i]) : first_env + i, draws[i], c))
                   : 0;
    }
}

/// kStatusTaskId if some ids[i] is outside [0, instances).
__global__ void k_check_ids(const i32* ids, u64 rows, u32 instances, u32* status)
{
    bool bad = false;
    for (u64 i = static_cast<u64>(blockIdx.x) * blockDim.x + threadIdx.x; i < rows; i += static_cast<u64>(gridDim.x) * blockDim.x)
        bad = bad || ids[i] < 0 || static_cast<u32>(ids[i]) >= instances;
    if (bad)
        atomicOr(status, kStatusTaskId);
}

/// The device seed word of an env, written in stream order.
__global__ void k_set_word(u64* p, u64 v) { *p = v; }

/// Per row: the instance its next autoreset would draw (with the row's current reset counter), for a step without
/// next_task_ids over a batch with reset counters and an env with a sampler.
__global__ void k_env_sample_next(SamplerDev sampler, const u64* seed, u64 first_env, u64 rows, const u32* reset_counts, const u64* sampling_seeds,
                                  const u32* env_ids, i32* next)
{
    for (u64 i = static_cast<u64>(blockIdx.x) * blockDim.x + threadIdx.x; i < rows; i += static_cast<u64>(gridDim.x) * blockDim.x)
        next[i] = instance_draw(sampling_seeds ? sampling_seeds[i] : *seed, env_ids ? static_cast<u64>(env_ids[i]) : first_env + i,
                                reset_counts[i], sampler.instances, sampler.thresholds, sampler.indices, sampler.m);
}

/// Per row: the instance's goal into the row's goal masks, or (keep) the given masks checked against the instance's
/// fluent slots and tested on its initial state. Runs after k_env_reset, so task ids are valid.
__global__ void k_env_reset_goals(const InstDev* inst, u32 instances, u64 rows, u32 words, const u8* mask, const i32* task_ids,
                                  u64* goal_pos, u64* goal_neg, u32 keep, u8* at_goal, u32* status)
{
    for (u64 i = static_cast<u64>(blockIdx.x) * blockDim.x + threadIdx.x; i < rows; i += static_cast<u64>(gridDim.x) * blockDim.x)
    {
        if (mask && !mask[i])
            continue;
        bool bad = false;
        const InstDev& J = inst[reset_instance(task_ids, i, instances, &bad)];
        u64* gp = goal_pos + i * words;
        u64* gn = goal_neg + i * words;
        if (!keep)
        {
            for (u32 w = 0; w < words; ++w)
            {
                gp[w] = w < J.W ? J.goal_pos[w] : 0;
                gn[w] = w < J.W ? J.goal_neg[w] : 0;
            }
            continue;
        }
        bool ok = true, fit = true;
        for (u32 w = 0; w < words; ++w)
        {
            const u64 p = gp[w], n = gn[w], x = w < J.W ? J.initial[w] : 0;
            ok = ok && (x & p) == p && (x & n) == 0;
            if (w >= J.W)
                fit = fit && (p | n) == 0;
            else if (w == J.W - 1 && (J.fluent_slots & 63))
                fit = fit && ((p | n) >> (J.fluent_slots & 63)) == 0;
        }
        if (!fit)
            atomicOr(status, kStatusGoalMask);
        if (at_goal)
            at_goal[i] = ok ? 1 : 0;
    }
}

/// One thread per count-cache word: the initial state's row of the row's instance. Runs after k_env_reset.
__global__ void k_env_reset_cache(const InstDev* inst, u32 instances, u64 rows, u32 width, const u8* mask, const i32* task_ids, u32* cache)
{
    const u64 total = rows * width;
    for (u64 e = static_cast<u64>(blockIdx.x) * blockDim.x + threadIdx.x; e < total; e += static_cast<u64>(gridDim.x) * blockDim.x)
    {
        const u64 i = e / width;
        if (mask && !mask[i])
            continue;
        bool bad = false;
        cache[e] = inst[reset_instance(task_ids, i, instances, &bad)].init_cache[e - i * width];
    }
}

__global__ void k_offsets_i32(const u64* src, u64 n, i32* dst)
{
    const u64 i = static_cast<u64>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n)
        dst[i] = static_cast<i32>(src[i]);
}

__global__ void k_kept_counts(const u32* counts, const u32* noops, u64 rows, u32* kept)
{
    const u64 i = static_cast<u64>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < rows)
        kept[i] = noops[i] == counts[i] ? counts[i] : counts[i] - noops[i];
}

// Padded view of a flat expansion, one wave per row: the row's k slots are contiguous in every output, so the lanes
// walk each output row (scalars over the k slots, succ over k * words, binding over k * label_width) with coalesced
// stores, reading the flat rows b .. b + k - 1 that are also contiguous.
template<class X>
__device__ __forceinline__ void pad_rows(X* dst, const X* src, u32 K, u32 n, u32 W, u32 FW, X fill, u32 lane)
{
    if (W == 0)
        return;
    const u32 dk = kWave / W, dw = kWave % W;
    u32 k = lane / W, w = lane % W;
    constexpr int kBatch = 4;  // loads of a lane in flight before their stores
    while (k < K)
    {
        X v[kBatch];
        u64 at[kBatch];
        bool live[kBatch];
#pragma unroll
        for (int q = 0; q < kBatch; ++q)
        {
            live[q] = k < K;
            at[q] = static_cast<u64>(k) * W + w;
            v[q] = fill;
            if (k < n && w < FW)
                v[q] = src[static_cast<u64>(k) * FW + w];
            k += dk;
            w += dw;
            if (w >= W)
            {
                w -= W;
                ++k;
            }
        }
#pragma unroll
        for (int q = 0; q < kBatch; ++q)
            if (live[q])
                dst[at[q]] = v[q];
    }
}

__global__ __launch_bounds__(256) void k_pad(PadArgs a)
{
    const u32 lane = lane_id();
    const u64 nw = u64{gridDim.x} * (blockDim.x / kWave);
    const u32 K = a.k;
    for (u64 i = static_cast<u64>(blockIdx.x) * (blockDim.x / kWave) + threadIdx.x / kWave; i < a.rows; i += nw)
    {
        const u64 b = static_cast<u64>(static_cast<i64>(a.offsets[i]));
        const u64 c = static_cast<u64>(static_cast<i64>(a.offsets[i + 1])) - b;
        // valid slots: k < min(c, K) with b + k < capacity
        const u64 room = b < a.capacity ? a.capacity - b : 0;
        const u32 n = static_cast<u32>(std::min<u64>(std::min<u64>(c, K), room));
        if (lane == 0)
        {
            if (a.count)
                a.count[i] = static_cast<i32>(c);
            if (c > K || n < std::min<u64>(c, K))
                atomicOr(a.overflow, 1u);
        }
        const u64 base = i * K;
        for (u32 k = lane; k < K; k += kWave)
        {
            const bool valid = k < n;
            const u64 j = b + k, at = base + k;
            if (a.out_index)
                a.out_index[at] = valid ? static_cast<i32>(j) : -1;
            if (a.mask)
                a.mask[at] = valid ? 1 : 0;
            if (a.canonical)
                a.canonical[at] = valid && a.index ? a.index[j] : -1;
            if (a.out_schema)
                a.out_schema[at] = valid && a.schema ? a.schema[j] : -1;
            if (a.out_goal)
                a.out_goal[at] = valid && a.goal ? a.goal[j] : 0;
            if (a.out_succ_hash)
                a.out_succ_hash[at] = valid && a.succ_hash ? a.succ_hash[j] : 0;
            if (a.out_noop)
                a.out_noop[at] = valid && a.noop ? a.noop[j] : 0;
        }
        if (a.out_succ)
        {
            // rows of equal even widths go 16 bytes a lane; the lanes' (slot, word) advance by a wave's stride without a
            // division per element
            const u32 W = a.words, FW = a.succ ? a.flat_words : 0;
            if (W == FW && (W & 1) == 0 && ((reinterpret_cast<std::uintptr_t>(a.out_succ) | reinterpret_cast<std::uintptr_t>(a.succ)) & 15) == 0)
                pad_rows<ulonglong2>(reinterpret_cast<ulonglong2*>(a.out_succ) + base * (W / 2), reinterpret_cast<const ulonglong2*>(a.succ) + b * (FW / 2),
                                     K, n, W / 2, FW / 2, ulonglong2{0, 0}, lane);
            else
                pad_rows<u64>(a.out_succ + base * W, a.succ + b * FW, K, n, W, FW, u64{0}, lane);
        }
        if (a.out_binding)
        {
            const u32 L = a.label_width, FL = a.binding ? a.flat_label_width : 0;
            pad_rows<i32>(a.out_binding + base * L, a.binding + b * FL, K, n, L, FL, -1, lane);
        }
    }
}

// The position of each row's label in its flat expansion (canonical order): one lane per row scans the row's successors
// for the label's schema and the objects of its binding (the flat binding's -1 columns lie past the arity and match
// anything); -1 when no successor carries the label.
__global__ __launch_bounds__(256) void k_label_actions(const i32* offsets, const i32* schema, const i32* binding, u32 L, u64 rows,
                                                       const i32* label_schema, const i32* label_binding, u32 stride, i64* actions)
{
    const u64 step = u64{gridDim.x} * blockDim.x;
    for (u64 i = static_cast<u64>(blockIdx.x) * blockDim.x + threadIdx.x; i < rows; i += step)
    {
        const i64 b = offsets[i], e = offsets[i + 1];
        const i32 ls = label_schema[i];
        const i32* lb = label_binding + i * stride;
        i64 act = -1;
        for (i64 j = b; j < e && act < 0; ++j)
        {
            if (schema[j] != ls)
                continue;
            const i32* fb = binding + static_cast<u64>(j) * L;
            bool same = true;
            for (u32 k = 0; k < L && same; ++k)
                same = fb[k] < 0 || fb[k] == lb[k];
            if (same)
                act = j - b;
        }
        actions[i] = act;
    }
}

unsigned grid_for(u64 rows, unsigned nw) { return static_cast<unsigned>(std::min<u64>((rows + nw - 1) / nw, u64{1} << 20)); }

/// Raises a kernel's dynamic LDS limit once per (kernel, size): later launches make no runtime call besides the launch,
/// so a step recorded into a HIP graph after a first eager call holds kernel nodes only.
void set_lds(const void* fn, size_t bytes)
{
    if (bytes <= 64 * 1024)
        return;
    static std::mutex mu;
    static std::unordered_map<const void*, size_t> done;
    std::lock_guard lock(mu);
    size_t& have = done[fn];
    if (bytes <= have)
        return;
    hip_check(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes)), "LDS size");
    have = bytes;
}
}  // namespace

/// Compute units of the current device (queried once per device).
unsigned device_cus()
{
    static std::mutex mu;
    static std::unordered_map<int, unsigned> cus;
    int dev = 0;
    hip_check(hipGetDevice(&dev), "device");
    std::lock_guard lock(mu);
    unsigned& n = cus[dev];
    if (n == 0)
    {
        int v = 0;
        hip_check(hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev), "compute units");
        n = static_cast<unsigned>(std::max(1, v));
    }
    return n;
}

u32 env_wave_words(const TaskDev* const* tasks, u32 n, bool step)
{
    u32 words = 0;
    for (u32 k = 0; k < n; ++k)
    {
        check_schemas(*tasks[k]);
        words = std::max(words, step ? tasks[k]->l_step : tasks[k]->l_words);
    }
    size_t lds = 0;
    block_shape(static_cast<size_t>(words) * 8, &lds);  // throws where a wave's region does not fit a workgroup
    return words;
}

namespace
{
/// The LDS words per wave of a launch: given (a table's widest instance), or those of its one instance.
u32 wave_words_of(u32 given, const TaskDev& T, bool step)
{
    if (given)
        return given;
    const TaskDev* t = &T;
    return env_wave_words(&t, 1, step);
}

/// The kernels for simple tasks (TaskDev::simple; every instance of a table), or for any.
EnvKernels kernels_for(bool simple) { return simple ? env_kernels() : env_kernels_general(); }

/// The kernel of a step, by what it takes: the visited tables' code only in the launches that use it (it keeps more
/// kernel arguments live); the plain step (an env pool's random-policy step over one instance) compiles the optional
/// inputs it does not take away.
auto step_kernel(const EnvKernels& k, bool one, bool visited, bool plain)
{
    return !one ? k.step_table : visited ? k.step_visited : plain && k.step_plain ? k.step_plain : k.step;
}
}  // namespace

void launch_env_step(const EnvArgs& args, hipStream_t stream)
{
    if (args.rows == 0)
        return;
    EnvArgs a = args;
    a.wave_words = wave_words_of(a.wave_words, a.T, true);
    size_t lds = 0;
    const unsigned nw = block_shape(static_cast<size_t>(a.wave_words) * 8, &lds);
    const bool visited = a.visited.capacity || a.revisited;
    const bool plain = !visited && !a.actions && !a.label_schema && !a.seeds && !a.env_ids && !a.goal_pos && !a.final_states &&
                       !a.reset_counts && !a.next_task_ids && a.steps && a.draws;
    const auto fn = step_kernel(kernels_for(a.T.simple && !a.general), a.instances == 1, visited, plain);
    set_lds(reinterpret_cast<const void*>(fn), lds);
    hipLaunchKernelGGL(fn, dim3(grid_for(a.rows, nw)), dim3(nw * kWave), lds, stream, a);
    launch_check("env step");
}

void launch_env_count(const CountArgs& args, hipStream_t stream)
{
    if (args.rows == 0)
        return;
    CountArgs a = args;
    a.wave_words = wave_words_of(a.wave_words, a.T, true);
    size_t lds = 0;
    const unsigned nw = block_shape(static_cast<size_t>(a.wave_words) * 8, &lds);
    const EnvKernels k = kernels_for(a.T.simple && !a.general);
    const auto fn = a.instances == 1 ? k.count : k.count_table;
    set_lds(reinterpret_cast<const void*>(fn), lds);
    hipLaunchKernelGGL(fn, dim3(grid_for(a.rows, nw)), dim3(nw * kWave), lds, stream, a);
    launch_check("env count");
}

void launch_env_count(const TaskDev& T, const u64* states, u64 rows, u32 words, i32* count, u8* goal, u8* masks, u32* cache,
                      hipStream_t stream, const u64* goal_pos, const u64* goal_neg, u32* status, u32 instance, u32 schemas)
{
    CountArgs a{};
    a.T = T;
    a.mask_width = schemas ? schemas : T.num_schemas;
    a.cache_width = a.mask_width + 2;
    a.instances = 1;
    a.states = states;
    a.rows = rows;
    a.words = words;
    a.count = count;
    a.goal = goal;
    a.masks = masks;
    a.cache = cache;
    a.goal_pos = goal_pos;
    a.goal_neg = goal_neg;
    a.status = status;
    a.instance = instance;
    launch_env_count(a, stream);
}

void prepare_env_launches(u32 wave_words, bool general, bool one)
{
    size_t lds = 0;
    block_shape(static_cast<size_t>(wave_words) * 8, &lds);
    const EnvKernels k = kernels_for(!general);
    for (const bool visited : {false, true})
        for (const bool plain : {false, true})
            set_lds(reinterpret_cast<const void*>(step_kernel(k, one, visited, plain)), lds);
    set_lds(reinterpret_cast<const void*>(one ? k.count : k.count_table), lds);
}

void launch_expand(const ExpandArgs& args, hipStream_t stream)
{
    if (args.rows == 0)
        return;
    ExpandArgs a = args;
    a.wave_words = wave_words_of(a.wave_words, a.T, false);
    const bool simple = a.T.simple && !a.general;
    // successors 64 at a time, where every instance is listable, the call asks for whole rows (rows narrower than the
    // task's need their trimmed lengths, a successor at a time) and a workgroup has room for the list beside a wave's region
    const u32 whole = a.tasks ? a.table_words : a.T.W;
    a.list = simple && a.T.listable && !a.unlistable && !a.witness && !a.succ_hash && (!a.succ || a.out_words >= whole) &&
             (u64{a.wave_words} + kListCap) * 8 <= kCuLds;
    size_t lds = 0;
    const unsigned nw = block_shape(static_cast<size_t>(a.wave_words + (a.list ? kListCap : 0)) * 8, &lds);
    if (a.witness && a.tasks)
        throw std::invalid_argument("mymyr_amd: expand: witness pruning over a task table is not supported by the device expansion");
    const EnvKernels k = kernels_for(simple);
    const auto fn = a.tasks ? k.expand_table : a.witness ? k.expand_witness : k.expand;
    set_lds(reinterpret_cast<const void*>(fn), lds);
    hipLaunchKernelGGL(fn, dim3(grid_for(a.rows, nw)), dim3(nw * kWave), lds, stream, a);
    launch_check("expand");
}

void launch_offsets_i32(const u64* src, u64 n, i32* dst, hipStream_t stream)
{
    hipLaunchKernelGGL(k_offsets_i32, dim3(blocks_for(n, 256)), dim3(256), 0, stream, src, n, dst);
    launch_check("expand offsets");
}

void launch_kept_counts(const u32* counts, const u32* noops, u64 rows, u32* kept, hipStream_t stream)
{
    if (rows == 0)
        return;
    hipLaunchKernelGGL(k_kept_counts, dim3(blocks_for(rows, 256)), dim3(256), 0, stream, counts, noops, rows, kept);
    launch_check("expand kept counts");
}

void launch_pad(const PadArgs& a, hipStream_t stream)
{
    if (a.rows == 0)
        return;
    constexpr unsigned nw = 4;
    hipLaunchKernelGGL(k_pad, dim3(grid_for(a.rows, nw)), dim3(nw * kWave), 0, stream, a);
    launch_check("pad");
}

void launch_label_actions(const i32* offsets, const i32* schema, const i32* binding, u32 L, u64 rows, const i32* label_schema,
                          const i32* label_binding, u32 stride, i64* actions, hipStream_t stream)
{
    if (rows == 0)
        return;
    hipLaunchKernelGGL(k_label_actions, dim3(static_cast<unsigned>(std::min<u64>(blocks_for(rows, 256), 16384))), dim3(256), 0, stream, offsets,
                       schema, binding, L, rows, label_schema, label_binding, stride, actions);
    launch_check("label actions");
}

void launch_encode_atoms(const u64* states, u64 rows, u32 words, u32 W, i32* out, u32 max_atoms, u32* status, hipStream_t stream)
{
    if (rows == 0)
        return;
    hipLaunchKernelGGL(k_encode, dim3(grid_for(rows, 1)), dim3(kWave), 0, stream, states, rows, words, W, out, max_atoms, status);
    launch_check("encode atoms");
}

void launch_env_reset(const InstDev* inst, u32 instances, u64* states, u64 rows, u32 words, const u8* mask, i32* task_ids, i32* steps,
                      u8* at_goal, i32* count, u32* cache, u32 cache_width, u32* status, hipStream_t stream)
{
    if (rows == 0)
        return;
    const u64 total = rows * words;
    hipLaunchKernelGGL(k_env_reset, dim3(static_cast<unsigned>(std::min<u64>(blocks_for(total, 256), 65536))), dim3(256), 0, stream, inst,
                       instances, states, rows, words, mask, task_ids, steps, at_goal, count, status);
    launch_check("env reset");
    if (cache)
    {
        const u64 cells = rows * cache_width;
        hipLaunchKernelGGL(k_env_reset_cache, dim3(static_cast<unsigned>(std::min<u64>(blocks_for(cells, 256), 65536))), dim3(256), 0,
                           stream, inst, instances, rows, cache_width, mask, task_ids, cache);
        launch_check("env reset cache");
    }
}

void launch_env_random_actions(const u64* seed, const u64* seeds, const u32* env_ids, u64 first_env, const u64* draws, const i32* count,
                               u64 rows, u32 max_actions, i64* out, hipStream_t stream)
{
    if (rows == 0)
        return;
    hipLaunchKernelGGL(k_env_random_actions, dim3(static_cast<unsigned>(std::min<u64>(blocks_for(rows, 256), 4096))), dim3(256), 0, stream,
                       seed, seeds, env_ids, first_env, draws, count, rows, max_actions, out);
    launch_check("env random actions");
}

void launch_check_ids(const i32* ids, u64 rows, u32 instances, u32* status, hipStream_t stream)
{
    if (rows == 0 || !ids)
        return;
    hipLaunchKernelGGL(k_check_ids, dim3(static_cast<unsigned>(std::min<u64>(blocks_for(rows, 256), 1024))), dim3(256), 0, stream, ids, rows,
                       instances, status);
    launch_check("check task ids");
}

void launch_set_word(u64* p, u64 v, hipStream_t stream)
{
    hipLaunchKernelGGL(k_set_word, dim3(1), dim3(1), 0, stream, p, v);
    launch_check("set word");
}

void launch_env_sample_next(const SamplerDev& sampler, const u64* seed, u64 first_env, u64 rows, const u32* reset_counts,
                            const u64* sampling_seeds, const u32* env_ids, i32* next, hipStream_t stream)
{
    if (rows == 0)
        return;
    hipLaunchKernelGGL(k_env_sample_next, dim3(static_cast<unsigned>(std::min<u64>(blocks_for(rows, 256), 4096))), dim3(256), 0, stream,
                       sampler, seed, first_env, rows, reset_counts, sampling_seeds, env_ids, next);
    launch_check("env sample next");
}

void launch_visited_restart(const VisitedDev& v, const InstDev* inst, u32 instances, const u64* states, u64 rows, u32 words,
                            const u8* mask, const i32* task_ids, bool current, hipStream_t stream)
{
    if (rows == 0 || !v.capacity)
        return;
    hipLaunchKernelGGL(k_visited_restart, dim3(static_cast<unsigned>(std::min<u64>(blocks_for(rows, 4), 16384))), dim3(256), 0, stream, v, inst,
                       instances, states, rows, words, mask, task_ids, current ? 1u : 0u);
    launch_check("visited restart");
}

void launch_visited_mask(const u64* table, const i32* count, u64 table_rows, u32 capacity, const u64* succ_hash, const i32* parent,
                         const i32* rows, u64 parents, u64 size, u8* out, hipStream_t stream)
{
    if (size == 0)
        return;
    hipLaunchKernelGGL(k_visited_mask, dim3(static_cast<unsigned>(std::min<u64>(blocks_for(size, 256), 16384))), dim3(256), 0, stream, table,
                       count, table_rows, capacity, succ_hash, parent, rows, parents, size, out);
    launch_check("visited mask");
}

void launch_env_reset_draw(const SamplerDev& sampler, const u64* seed, u64 first_env, u64 rows, const u8* mask, bool sample, i32* task_ids,
                           u32* reset_counts, const u64* sampling_seeds, const u32* env_ids, hipStream_t stream)
{
    if (rows == 0 || !reset_counts)
        return;
    hipLaunchKernelGGL(k_env_reset_draw, dim3(static_cast<unsigned>(std::min<u64>(blocks_for(rows, 256), 4096))), dim3(256), 0, stream,
                       sampler, seed, first_env, rows, mask, sample ? 1u : 0u, task_ids, reset_counts, sampling_seeds, env_ids);
    launch_check("env reset draw");
}

void launch_env_reset_goals(const InstDev* inst, u32 instances, u64 rows, u32 words, const u8* mask, const i32* task_ids, u64* goal_pos,
                            u64* goal_neg, bool keep_goals, u8* at_goal, u32* status, hipStream_t stream)
{
    if (rows == 0)
        return;
    hipLaunchKernelGGL(k_env_reset_goals, dim3(static_cast<unsigned>(std::min<u64>(blocks_for(rows, 256), 4096))), dim3(256), 0, stream, inst,
                       instances, rows, words, mask, task_ids, goal_pos, goal_neg, keep_goals ? 1u : 0u, at_goal, status);
    launch_check("env reset goals");
}

void launch_successors(const TaskDev& T, const u64* states, u64 rows, u32 words, u32 cap, i32* count, i32* schema, i32* binding,
                       u64* succ, u32* status, hipStream_t stream)
{
    if (rows == 0)
        return;
    check_schemas(T);
    size_t lds = 0;
    const unsigned nw = block_shape(static_cast<size_t>(T.l_words) * 8, &lds);
    const auto fn = kernels_for(T.simple).successors;
    set_lds(reinterpret_cast<const void*>(fn), lds);
    hipLaunchKernelGGL(fn, dim3(grid_for(rows, nw)), dim3(nw * kWave), lds, stream, T, states, rows, words, cap, count, schema,
                       binding, succ, status);
    launch_check("successors");
}
}  // namespace mya
