// Reads task texts named on the command line, compiles each and checks every word that the device's matching reads for a
// term of a plan against the wave's region (the view, the state row and the word after it) and against the image.
// Prints one line per task ("ok", or the first read out of range) and exits with the number of tasks out of range.

#include "task.cpp"

#include <cstdio>
#include <fstream>
#include <set>
#include <sstream>

using namespace mya;

namespace
{
template<class X>
const X* at(const CompiledTask& t, u64 word)
{
    return reinterpret_cast<const X*>(t.image.data() + word);
}

/// The rows that term c of schema s can read: the first and the last (a row's words follow from its number linearly).
std::set<u32> rows_of(const CompiledTask& t, u32 s, const DevTerm& c)
{
    u32 first = kNone, last = 0;
    auto add = [&](u32 r) {
        r = c.rows != kNone && r >= c.rows ? 0 : r;
        first = std::min(first, r);
        last = std::max(last, r);
    };
    if (c.src == kNone)
        add(c.row0);
    else
        for (u32 o = 0; o < t.n; ++o)
            if ((t.dom0[s][c.src][o >> 6] >> (o & 63)) & 1)
                add(o - c.row0);
    return first == kNone ? std::set<u32>{} : std::set<u32>{first, last};
}

std::string check_step(const CompiledTask& t, u32 s, u32 step, u64& reads)
{
    const DevTaskHeader& h = t.header();
    const u64 region = u64{h.view_words} + h.words;  // and one word more
    const DevStep& st = *at<DevStep>(t, u64{step} * 4);
    for (u32 k = st.term_begin; k < st.cons_end; ++k)
    {
        const DevTerm& c = *at<DevTerm>(t, u64{k} * 4);
        for (const u32 r : rows_of(t, s, c))
            for (u32 w = 0; w < st.words; ++w, ++reads)
            {
                u64 first, last, end;
                if (c.path == static_cast<u32>(TermPath::Bits))
                {
                    first = (u64{c.base} + u64{r} * c.stride + row_bits(c, w).skip) >> 6;
                    last = first + 1;
                    end = region + 1;
                }
                else
                {
                    first = last = u64{c.base} + u64{r} * c.stride + w;
                    end = c.path == static_cast<u32>(TermPath::Image) ? t.image.size() : region;
                }
                if (last >= end)
                    return "schema " + std::to_string(s) + " parameter " + std::to_string(st.param) + ": word " + std::to_string(last) +
                           " of " + std::to_string(end);
            }
    }
    return {};
}

std::string check(const CompiledTask& t, u64& reads)
{
    const DevTaskHeader& h = t.header();
    for (u32 s = 0; s < h.num_schemas; ++s)
    {
        const DevSchema& S = at<DevSchema>(t, h.off_schemas)[s];
        if (S.never)
            continue;
        std::vector<std::pair<u32, u32>> runs{{S.plan_begin[0], S.plan_begin[S.arity + 1]}};  // (schema s's steps)
        for (u32 i = 0; i < S.arity; ++i)
            runs.push_back({S.filter_step[i], S.filter_step[i] + 1});
        if (h.off_witness)
        {
            const DevWitness& x = at<DevWitness>(t, h.off_witness)[s];
            for (u32 k = 0; k < x.n; ++k)
            {
                runs.push_back({x.filter[k], x.filter[k] + 1});
                runs.push_back({x.plan_lo[k], x.plan_hi[k]});
            }
        }
        for (u32 a = 0; a < h.num_schemas; ++a)
        {
            const DevSchema& A = at<DevSchema>(t, h.off_schemas)[a];
            for (u32 k = A.del_begin; k < A.add_end; ++k)
            {
                const DevDelta& d = at<DevDelta>(t, h.off_deltas)[k];
                if (d.schema != s)
                    continue;
                if (d.tests)
                    runs.push_back({d.test_begin, d.test_begin + d.nbound});
                runs.push_back({d.plan_begin, d.plan_end});
            }
        }
        for (const auto& [b, e] : runs)
            for (u32 step = b; step < e; ++step)
                if (std::string bad = check_step(t, s, step, reads); !bad.empty())
                    return bad;
    }
    return {};
}
}  // namespace

int main(int argc, char** argv)
{
    int bad = 0;
    for (int i = 1; i < argc; ++i)
    {
        std::ifstream f(argv[i]);
        std::stringstream text;
        text << f.rdbuf();
        u64 reads = 0;
        if (const std::string out = check(*compile_task(parse_task_text(text.str()), AtomsOption::Auto), reads); !out.empty())
        {
            std::printf("%s: %s\n", argv[i], out.c_str());
            ++bad;
        }
        std::printf("%s: %llu reads\n", argv[i], static_cast<unsigned long long>(reads));
    }
    return bad;
}
