// CPU check of the step planner's rule and tables for RoPE factors that the kernel evaluates
// (gemma4-webgpu_amd/csrc/step_plan.h, StepTuning::rope_eval_sets), built with g++ by tests/test_rope_eval_plan.py.
// Random steps whose entries bring no table, one of a few or their own, at shared and at own positions, and steps on
// both sides of the two thresholds. Where the rule asks for it, every entry with a host table carries the flag and
// points at that table's inverse frequencies, once per table, inside the blob and the workspace's tables region, and
// the plan is otherwise the plan with the host's factors; elsewhere it is that plan, byte for byte. One planner state
// plans them all. Prints "ok <steps> <steps whose factors the kernel evaluates>".
#include <stdio.h>
#include <string.h>

#include <map>
#include <random>
#include <set>

#include "../gemma4-webgpu_amd/csrc/step_plan.h"

using namespace g4;

namespace {

constexpr uint32_t kSets = 4;
std::vector<std::vector<float>> tables;
StepPlanHost ph;  // kept between the plans, as a library thread keeps it

g4_step_entry entry(uint32_t i, uint32_t seq, uint32_t position, const float* table) {
    g4_step_entry e{};
    const uintptr_t base = uintptr_t(i + 1) << 32;  // made-up device addresses: the planner stores them
    e.q = e.k = e.v = reinterpret_cast<const float*>(base + 0x1000);
    e.q_weight = e.k_weight = reinterpret_cast<const uint16_t*>(base + 0x2000);
    e.k_cache = reinterpret_cast<uint16_t*>(base + 0x10000000);
    e.v_cache = reinterpret_cast<uint16_t*>(base + 0x20000000);
    e.out = reinterpret_cast<float*>(base + 0x30000000);
    e.seq_len = seq;
    e.position = position;
    e.store_kv = 1;
    e.scale = 1.0f;
    e.rope_inv_freq_host = table;
    return e;
}

// Returns 1 when the kernel evaluates the plan's factors, 0 when not, -1 on a failure.
int check(const std::vector<g4_step_entry>& ents, uint32_t hd) {
    const uint32_t n = (uint32_t)ents.size();
    char* const dev = reinterpret_cast<char*>(uintptr_t(1) << 40);
    const StepLayout L = step_layout(n, 1, 8, hd);
    StepTuning tune;
    tune.rope_eval_sets = kSets;
    StepPlanHost host;
    char err[256];
    if (plan_step(ents.data(), n, 8, 1, hd, 256, StepTuning{}, dev + L.tables, &host, err, sizeof err) ||
        plan_step(ents.data(), n, 8, 1, hd, 256, tune, dev + L.tables, &ph, err, sizeof err))
        return printf("FAIL %s\n", err), -1;
    std::set<std::pair<const float*, uint32_t>> pairs;
    std::set<const float*> used;
    for (const auto& e : ents)
        if (e.rope_inv_freq_host) pairs.insert({e.rope_inv_freq_host, e.position}), used.insert(e.rope_inv_freq_host);
    const bool want = pairs.size() >= kSets && 2 * pairs.size() > n;
    if (!want) {
        if (ph.blob != host.blob) return printf("FAIL the host's plan differs\n"), -1;
        return 0;
    }
    if (ph.n_wgs != host.n_wgs || ph.n_merge != host.n_merge || ph.waves != host.waves || ph.max_parts != host.max_parts ||
        ph.off_merge != host.off_merge || ph.off_ents != host.off_ents || ph.off_rope != host.off_rope)
        return printf("FAIL partition\n"), -1;
    const size_t set_bytes = hd / 2 * sizeof(float);
    if (ph.blob.size() != ph.off_rope + used.size() * set_bytes) return printf("FAIL one set per table\n"), -1;
    if (ph.blob.size() > L.part_ml - L.tables) return printf("FAIL tables region\n"), -1;
    const StepWorkDev* w = reinterpret_cast<const StepWorkDev*>(ph.blob.data());
    const StepWorkDev* h = reinterpret_cast<const StepWorkDev*>(host.blob.data());
    std::map<const float*, const float*> at;
    for (uint32_t k = 0; k < ph.n_wgs; k++) {
        const g4_step_entry& e = ents[w[k].entry];
        const bool eval = w[k].ent.flags & kRopeEval;
        if (eval != (e.rope_inv_freq_host != nullptr)) return printf("FAIL flag\n"), -1;
        if (eval) {
            const char* p = reinterpret_cast<const char*>(w[k].ent.rope_cs);
            const char* r0 = dev + L.tables + ph.off_rope;
            if (p < r0 || p + set_bytes > dev + L.tables + ph.blob.size() || (size_t)(p - r0) % set_bytes)
                return printf("FAIL set outside the blob\n"), -1;
            if (memcmp(ph.blob.data() + (p - (dev + L.tables)), e.rope_inv_freq_host, set_bytes))
                return printf("FAIL inverse frequencies\n"), -1;
            const auto it = at.emplace(e.rope_inv_freq_host, w[k].ent.rope_cs).first;
            if (it->second != w[k].ent.rope_cs) return printf("FAIL two sets of one table\n"), -1;
        } else if (w[k].ent.rope_cs) {
            return printf("FAIL set without a table\n"), -1;
        }
        StepWorkDev a = w[k], b = h[k];
        a.ent.flags &= ~kRopeEval;
        a.ent.rope_cs = b.ent.rope_cs = nullptr;
        if (memcmp(&a, &b, sizeof a)) return printf("FAIL work item\n"), -1;
    }
    if (memcmp(ph.blob.data() + ph.off_merge, host.blob.data() + ph.off_merge, ph.off_rope - ph.off_merge))
        return printf("FAIL merge or entry table\n"), -1;
    return 1;
}

}  // namespace

int main() {
    std::mt19937 rng(11);
    auto pick = [&](uint32_t lo, uint32_t hi) { return lo + rng() % (hi - lo + 1); };
    tables.assign(80, std::vector<float>(256));
    for (size_t t = 0; t < tables.size(); t++)
        for (uint32_t i = 0; i < 256; i++) tables[t][i] = 1.0f / (float)(i + 1 + t);
    int evaluated = 0, steps = 0;
    for (uint32_t hd : {256u, 512u})
        for (uint32_t n : {1u, 3u, 4u, 5u, 7u, 8u, 9u, 31u, 64u})
            for (uint32_t sets = 0; sets <= n; sets++)  // sets entries at positions of their own, the rest at the first's or bare
                for (bool bare : {false, true}) {
                    std::vector<g4_step_entry> e;
                    for (uint32_t i = 0; i < n; i++)
                        e.push_back(entry(i, 100 + 10 * i, i < sets ? 99 + 10 * i : 99,
                                          i < sets || (!bare && sets) ? tables[0].data() : nullptr));
                    const int r = check(e, hd);
                    if (r < 0 || r != (int)(sets >= kSets && 2 * sets > n)) return printf("at n %u sets %u\n", n, sets), 1;
                    evaluated += r, steps++;
                }
    for (int it = 0; it < 3000; it++) {
        const uint32_t n = pick(1, 70), hd = pick(0, 1) ? 512 : 256, kinds = pick(0, 3), positions = pick(0, 2);
        std::vector<g4_step_entry> e;
        for (uint32_t i = 0; i < n; i++) {
            const uint32_t seq = positions == 0 ? 700 : positions == 1 ? 300 + 50 * pick(0, 5) : pick(1, 9000);
            const float* table = pick(0, 7) == 0 && kinds ? nullptr : tables[kinds == 3 ? i : pick(0, kinds)].data();
            e.push_back(entry(i, seq, seq - 1, table));
        }
        const int r = check(e, hd);
        if (r < 0) return printf("at step %d\n", it), 1;
        evaluated += r, steps++;
    }
    printf("ok %d %d\n", steps, evaluated);
    return 0;
}
