// Checks on the host that no plan of the packed attention calls leaves what the
// host provides for it: partial entries and workgroups, the arrival count, a
// split's pages, the workspace (tests/test_plan_bounds.py).  It includes the
// library's host code, and the plan as the kernels take it from the sums over
// the requests.  Prints one line per check: its name and how many random calls
// broke it.
#include "../residualquant_amd/csrc/capi.hip"
#include "../residualquant_amd/csrc/rq_multirow.h"

#include <map>
#include <random>

namespace {

std::mt19937_64 g_rng(20);

int64_t below(int64_t n) { return (int64_t)(g_rng() % (uint64_t)n); }

// Log-uniform over low..high.
int64_t spread(double low, double high) {
    std::uniform_real_distribution<double> u(std::log(low), std::log(high + 1));
    return (int64_t)std::exp(u(g_rng));
}

struct Call {
    int heads, head_dim, page_tokens;
    int64_t requests, rows, max_pages;
    std::vector<int64_t> history, count;  // tokens and rows per request
};

Call random_call(bool one_row) {
    static const int kHeads[] = {1, 2, 3, 5, 8, 16, 16, 24, 40, 55, 64, 96, 128};
    Call c;
    c.heads = kHeads[below(13)];
    c.head_dim = below(2) ? 128 : 96;
    c.page_tokens = below(2) ? 16 : 32;
    c.requests = spread(1, rq::kPlanRequests);
    const int64_t longest = below(20) ? spread(1, 60000) : spread(60000, 6000000);
    const int64_t shortest = spread(1, longest), most = spread(1, 700);
    c.rows = 0;
    for (int64_t b = 0; b < c.requests; ++b) {
        c.history.push_back(below(10) ? spread(shortest, longest) : 0);
        c.count.push_back(one_row ? (below(20) ? 1 : below(4)) : below(3) ? most : below(most + 1));
        c.rows += c.count.back();
    }
    if (c.rows == 0) c.rows = c.count[0] = 1;
    // A table as wide as the longest history, wider, or (its tail is not read) narrower.
    c.max_pages = std::max<int64_t>(1, (longest + c.page_tokens - 1) / c.page_tokens + below(3) - 1);
    if (below(50) == 0) c.max_pages *= 1 + below(40);
    return c;
}

// The splits of every request, as plan_find and plan_request count them.
struct Plan {
    int64_t items = 0, entries = 0, most_splits = 0, most_units = 0;
};

Plan take(const rq::PlanSizes& sizes, const std::vector<int64_t>& count, const std::vector<int64_t>& length,
          const std::vector<int64_t>& rows) {
    uint32_t total = 0, counts = 0, longest = 0;
    for (size_t b = 0; b < count.size(); ++b) {
        total += (uint32_t)(count[b] * length[b]);
        counts += (uint32_t)count[b];
        if (count[b] > 0) longest = std::max(longest, (uint32_t)length[b]);
    }
    const rq::PlanShare share = rq::plan_share_of(sizes, total, counts, longest);
    Plan plan;
    for (size_t b = 0; b < count.size(); ++b) {
        const int64_t splits = share.whole ? 1 : rq::plan_splits(sizes, share, (uint32_t)length[b]);
        plan.items += count[b] * splits;
        plan.entries += rows[b] * splits;
        if (count[b] == 0) continue;
        plan.most_splits = std::max(plan.most_splits, splits);
        plan.most_units = std::max(plan.most_units, (length[b] + splits - 1) / splits);
    }
    return plan;
}

std::map<std::string, int> g_broken;
void check(const char* name, bool holds) { g_broken[name] += holds ? 0 : 1; }

void several_rows() {
    const Call c = random_call(false);
    const int64_t average_tiles = std::max<int64_t>(1, (c.rows / c.requests + 31) / 32);
    const int splits = multirow_splits(c.requests * c.heads * average_tiles, c.max_pages, c.page_tokens);
    if ((int64_t)splits * ((c.rows + 31) / 32) > 65535) return;  // refused
    const size_t required = multirow_bytes(c.rows, c.heads, splits);
    const size_t full = attention_workspace_total(c.rows, c.heads, c.head_dim, c.max_pages, c.page_tokens);
    check("rows_required_within_total", required <= full);
    // What the caller gives: the total, what is required, or between; moved up to the boundary.
    const size_t given = below(3) == 0 ? full : below(2) ? required : required + (size_t)below((int64_t)(full - required) + 1);
    const size_t bytes = given - (size_t)below(16);
    rq::MultiRowParams m{};
    m.rows = c.rows;
    m.heads = c.heads;
    m.requests = c.requests;
    m.max_pages = c.max_pages;
    m.page_tokens = c.page_tokens;
    const bool chunk = takes_chunk_kernels(c.rows, c.requests);
    if (chunk) plan_chunk(m, bytes);
    else plan_multirow(m, splits, bytes);
    std::vector<int64_t> tiles, length;
    for (int64_t b = 0; b < c.requests; ++b) {
        tiles.push_back((c.count[b] + m.tile_rows - 1) / m.tile_rows);
        const int64_t tokens = std::min<int64_t>(c.history[b], c.max_pages * c.page_tokens);
        length.push_back((tokens + m.plan_unit - 1) / m.plan_unit);
    }
    const Plan plan = take(chunk ? rq::multirow_sizes<false>(m) : rq::multirow_sizes<true>(m), tiles, length, c.count);
    check("rows_entries", plan.entries <= m.entries);
    check("rows_entries_in_workspace", sizeof(float) * rq::kMultiRowEntry * c.heads * (size_t)m.entries <= bytes);
    check("rows_items", plan.items <= m.items);
    check("rows_arrivals", plan.most_splits <= rq::kMaxArrivals);
    // A split that starts inside a page holds one page more.
    const int64_t pages = (plan.most_units * m.plan_unit + c.page_tokens - 1) / c.page_tokens + (m.plan_unit % c.page_tokens ? 1 : 0);
    check("rows_split_pages", pages <= rq::kMultiRowMaxSplitPages);
    // The no-alloc scratch holds the same plan as the whole workspace.
    if (required <= RQ_ATTENTION_NOALLOC_MAX_BYTES) {
        rq::MultiRowParams a = m, b = m;
        const size_t scratch = std::min(full, kAttentionScratchBytes);
        if (chunk) plan_chunk(a, full), plan_chunk(b, scratch);
        else plan_multirow(a, splits, full), plan_multirow(b, splits, scratch);
        check("rows_scratch", a.splits == b.splits && a.plan_target == b.plan_target);
    }
}

void one_row() {
    const Call c = random_call(true);
    const bool chain = below(2) != 0;
    const int per_cu = chain ? kChainPerCu : packed_per_cu(c.head_dim);
    const int splits = split_count(c.rows, c.heads, c.max_pages, per_cu);
    const size_t required = workspace_layout(c.rows, c.heads, c.head_dim, splits).total;
    const size_t bytes = required - (size_t)below(16);
    const DecodePlan plan = decode_plan(c.rows, c.heads, c.head_dim, c.max_pages, per_cu, c.page_tokens, bytes);
    // (A chain's launch takes at most `splits` of equal lengths.)
    const int even = chain ? 1 + (int)below(splits) : splits;
    const int64_t items = std::max<int64_t>(c.rows + plan.target, c.rows * even);
    check("decode_items_in_workspace",
          plan.partials + sizeof(float) * (c.head_dim + 2) * c.heads * (size_t)items <= bytes);
    const int64_t round = std::max<int64_t>(1, 2LL * compute_units() * 3 / 4 / c.heads);
    const rq::PlanSizes sizes{plan.target, even, plan.min_pages, INT32_MAX, rq::kMaxSplits,
                              chain ? kChainRoundTokens / c.page_tokens : 0, chain ? (int)round : 1, 18};
    std::vector<int64_t> pages;
    for (int64_t b = 0; b < c.requests; ++b)
        pages.push_back(std::min<int64_t>((c.history[b] + c.page_tokens - 1) / c.page_tokens, c.max_pages));
    const Plan taken = take(sizes, c.count, pages, c.count);
    check("decode_items", taken.items <= items);
    const int64_t by_pages = std::max<int64_t>(1, (c.max_pages + plan.min_pages - 1) / plan.min_pages);
    check("decode_items_by_pages", by_pages > plan.target / c.rows || taken.items <= std::max(c.rows * by_pages, c.rows * even));
    check("decode_arrivals", taken.most_splits <= rq::kMaxSplits);
}

}  // namespace

int main() {
    for (int i = 0; i < 300000; ++i) {
        several_rows();
        one_row();
    }
    for (const auto& [name, broken] : g_broken) printf("%s %d\n", name.c_str(), broken);
}
