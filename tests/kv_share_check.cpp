// CPU check of the step planner's work-item order for entries that share cache rows
// (gemma4-webgpu_amd/csrc/step_plan.h), built with g++ by tests/test_kv_share_plan.py. Random steps whose
// entries read a few caches over a few row ranges: every part of every entry is planned exactly once with the
// rows of the plan without sharing, and the items of one part of a group sit on one XCD (workgroup index mod 8)
// unless the group straddles the end of an XCD's workgroups. Rows are read with ordinary loads where enough of the
// step's tiles are read again. Prints "ok <steps> <shared steps> <steps that keep rows>".
#include <stdio.h>

#include <map>
#include <random>
#include <set>
#include <tuple>

#include "../gemma4-webgpu_amd/csrc/step_plan.h"

using namespace g4;

int main() {
    std::mt19937 rng(7);
    auto pick = [&](uint32_t lo, uint32_t hi) { return lo + rng() % (hi - lo + 1); };
    static char dev[1 << 16];
    uint16_t* base = reinterpret_cast<uint16_t*>(dev);
    float* f = reinterpret_cast<float*>(dev);
    int shared_steps = 0, kept_steps = 0, steps = 3000;
    for (int it = 0; it < steps; it++) {
        const uint32_t n = pick(1, 40), hd = pick(0, 1) ? 512 : 256, caches = pick(1, 6);
        std::vector<g4_step_entry> e(n);
        for (auto& s : e) {
            const uint32_t c = pick(0, caches - 1);
            s = g4_step_entry{};
            s.q = s.k = s.v = f;
            s.q_weight = s.k_weight = base;
            s.k_cache = base + 8 * c;
            s.v_cache = base + 8 * (c + (pick(0, 9) == 0));  // now and then the same K rows with other V rows
            s.out = f;
            s.seq_len = pick(0, 3) ? 300 + 977 * c : pick(1, 9000);
            s.sliding_window = pick(0, 2) ? 0 : 128;
            s.scale = 1.0f;
        }
        StepPlanHost ph, own;
        char err[256];
        if (plan_step(e.data(), n, 8, 1, hd, 256, StepTuning{}, dev, &ph, err, sizeof err)) return printf("FAIL %s\n", err), 1;
        // The same rows through caches of their own: the partition without sharing.
        std::vector<g4_step_entry> u = e;
        for (uint32_t i = 0; i < n; i++) u[i].k_cache = base + 8 * (100 + i);
        if (plan_step(u.data(), n, 8, 1, hd, 256, StepTuning{}, dev, &own, err, sizeof err)) return printf("FAIL %s\n", err), 1;
        if (own.keep_rows || own.n_wgs != ph.n_wgs) return printf("FAIL partition %d\n", it), 1;
        const StepWorkDev* w = reinterpret_cast<const StepWorkDev*>(ph.blob.data());
        const StepWorkDev* w1 = reinterpret_cast<const StepWorkDev*>(own.blob.data());
        auto rows = [](const StepWorkDev& x) { return std::make_tuple(x.entry, x.row_begin, x.row_end, x.part, x.ent.n_parts); };
        std::set<std::tuple<uint32_t, uint32_t, uint32_t, uint32_t, uint32_t>> a, b;
        std::map<std::tuple<const void*, const void*, uint32_t, uint32_t, uint32_t>, std::set<uint32_t>> xcds;
        std::map<std::tuple<const void*, const void*, uint32_t, uint32_t>, std::set<uint32_t>> groups;
        for (uint32_t i = 0; i < ph.n_wgs; i++) {
            if (w[i].ent.k_cache != e[w[i].entry].k_cache || w[i].ent.key_end != e[w[i].entry].seq_len)
                return printf("FAIL item's entry %d\n", it), 1;
            a.insert(rows(w[i]));
            b.insert(rows(w1[i]));
            const StepEntryDev& d = w[i].ent;
            xcds[{d.k_cache, d.v_cache, d.key_end, d.window, w[i].row_begin}].insert(i % 8);
            groups[{d.k_cache, d.v_cache, d.key_end, d.window}].insert(w[i].entry);
        }
        if (a != b || a.size() != ph.n_wgs) return printf("FAIL items %d\n", it), 1;
        bool shared = false;
        for (auto& g : groups) shared |= g.second.size() > 1;
        // Rows are kept where an eighth of the tiles or more read rows that an earlier entry reads.
        uint64_t total = 0, again = 0;
        std::set<std::tuple<const void*, const void*, uint32_t, uint32_t>> seen;
        for (const auto& s : e) {
            const uint32_t first = s.sliding_window && s.seq_len > s.sliding_window ? s.seq_len - s.sliding_window : 0;
            const uint32_t tiles = (s.seq_len - first + 31) / 32;
            total += tiles;
            if (!seen.insert({s.k_cache, s.v_cache, s.seq_len, s.sliding_window}).second) again += tiles;
        }
        if (ph.keep_rows != (8 * again >= total)) return printf("FAIL keep_rows %d\n", it), 1;
        kept_steps += ph.keep_rows;
        shared_steps += shared;
        size_t crossings = 0;
        for (auto& g : xcds) crossings += g.second.size() - 1;
        if (shared && crossings > 7) return printf("FAIL %zu parts across XCDs %d\n", crossings, it), 1;
        if (!shared)
            for (uint32_t i = 0; i + 1 < ph.n_wgs; i++)
                if (w[i].entry > w[i + 1].entry) return printf("FAIL order %d\n", it), 1;
    }
    // One sequence twice in a large batch, and one short window shared beside long rows: streamed.
    for (int window : {0, 1}) {
        std::vector<g4_step_entry> e(64);
        for (uint32_t i = 0; i < e.size(); i++) {
            e[i].q = e[i].k = e[i].v = f;
            e[i].q_weight = e[i].k_weight = base;
            e[i].k_cache = e[i].v_cache = base + 8 * (i < 63 ? i : 5);
            e[i].out = f;
            e[i].seq_len = i < 63 ? 1000 + 200 * i : 2000;
            e[i].sliding_window = window && (i == 5 || i == 63) ? 64 : 0;
            e[i].scale = 1.0f;
        }
        StepPlanHost ph;
        char err[256];
        if (plan_step(e.data(), 64, 8, 1, 256, 256, StepTuning{}, dev, &ph, err, sizeof err)) return printf("FAIL %s\n", err), 1;
        if (ph.kv_next[5] != 63 || ph.keep_rows) return printf("FAIL a small shared pair\n"), 1;
    }
    printf("ok %d %d %d\n", steps, shared_steps, kept_steps);
    return 0;
}
