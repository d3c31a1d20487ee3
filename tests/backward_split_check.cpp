// Host program of test_backward_split.py: for each line "dtype batch q_heads kv_heads seq head_dim
// causal limit" the split that fa::backward_split chooses, after checking its index arithmetic
// against plain loops. Prints "chunk parts slots bytes split_blocks" or "fault: ...".
#include <cstdio>
#include <map>
#include <set>
#include <utility>

#include "kernels.hpp"

static const char* fault(const fa::BackwardSplit& sp, int nkb, int group, bool causal) {
    const int n = sp.workgroups(nkb, group, causal);
    std::map<std::pair<int, int>, int> slot_of;  // (key block, chunk) -> workgroup
    for (int i = 0; i < n; ++i) {
        int kb, part;
        sp.coords(i, nkb, group, causal, kb, part);
        if (kb < 0 || kb >= nkb || part < 0 || part >= sp.parts) return "coords out of range";
        if (!slot_of.insert({{kb, part}, i}).second) return "a chunk twice";
    }
    long long want = 0;
    int several = 0;
    for (int kb = 0; kb < nkb; ++kb) {
        const long long tiles = (long long)group * (causal ? nkb - kb : nkb);
        const int chunks = (int)((tiles + sp.chunk - 1) / sp.chunk);
        want += chunks;
        if (chunks > 1) {
            if (several++ != kb) return "key blocks with several chunks are not the first ones";
            fa::BackwardSplit::Walk w(sp, kb, nkb, group, causal);
            for (int c = 0; c < chunks; ++c) {
                const auto at = slot_of.find({kb, c});
                if (at == slot_of.end() || at->second != w.slot) return "walk leaves the chunks";
                if (w.slot >= sp.slots) return "slot past the workspace";
                if (c + 1 < chunks) w.next();
            }
        }
    }
    if (want != n) return "chunks without a workgroup";
    if (several != sp.split_blocks(nkb, group, causal)) return "split_blocks";
    return nullptr;
}

int main() {
    int dt, b, hq, hkv, s, d, causal;
    unsigned long long limit;
    while (scanf("%d %d %d %d %d %d %d %llu", &dt, &b, &hq, &hkv, &s, &d, &causal, &limit) == 8) {
        fa::BackwardArgs a{};
        a.batch = b;
        a.q_heads = hq;
        a.kv_heads = hkv;
        a.group = hq / hkv;
        a.seq = s;
        a.head_dim = d;
        a.causal = causal;
        a.a64 = fa::kA64Auto;
        const fa::BackwardSplit sp = fa::backward_split((fa::Dtype)dt, a, limit);
        const int keys = dt == (int)fa::Dtype::F32 ? 32 : 128, nkb = (s + keys - 1) / keys;
        const char* f = sp.parts > 0 ? fault(sp, nkb, a.group, causal) : nullptr;
        if (!f && sp.bytes != 8ull * b * hkv * sp.slots * keys * d) f = "bytes";
        if (f) printf("fault: %s\n", f);
        else
            printf("%d %d %d %llu %d\n", sp.chunk, sp.parts, sp.slots,
                   (unsigned long long)sp.bytes,
                   sp.parts > 0 ? sp.split_blocks(nkb, a.group, causal) : 0);
    }
    return 0;
}
