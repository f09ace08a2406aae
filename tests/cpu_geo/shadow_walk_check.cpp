// CPU check of the shadow kernel's tree walk (wc_radiomap.hip, built as host
// C++ through the shim in hip/): the 64 bins of every (transmitter, edge) must
// be those of a section test against every triangle. Input directory:
// nodes.bin (64-byte wide nodes), tris.bin (48-byte triangles in leaf order),
// edges.bin (80-byte records), txs.bin (float xyz). Prints one summary line.
#include "hip/hip_runtime.h"
#include "../../witwin-channel_amd/csrc/wc_radiomap.hip"

#include <cstdio>
#include <string>
#include <vector>

int wc_fail(const char*, ...) { return 1; }
int wc_fail_hip(const char*, hipError_t) { return 1; }

using namespace wc;

template <class T> static std::vector<T> load(const std::string& path) {
    std::vector<T> v;
    FILE* f = std::fopen(path.c_str(), "rb");
    if (!f) return v;
    std::fseek(f, 0, SEEK_END);
    const long n = std::ftell(f);
    std::fseek(f, 0, SEEK_SET);
    v.resize((size_t)n / sizeof(T));
    if (std::fread(v.data(), 1, (size_t)n, f) != (size_t)n) v.clear();
    std::fclose(f);
    return v;
}

int main(int argc, char** argv) {
    if (argc < 2) return 2;
    const std::string d = argv[1];
    const auto nodes = load<WideNode>(d + "/nodes.bin");
    const auto tris = load<Tri>(d + "/tris.bin");
    const auto edges = load<Edge>(d + "/edges.bin");
    const auto txs = load<float>(d + "/txs.bin");
    if (nodes.empty() || tris.empty() || edges.empty() || txs.size() < 3) return 2;
    SceneView s{};
    s.nodes = nodes.data();
    s.tris = tris.data();
    s.tri_count = (int)tris.size();
    s.node_count = (int)nodes.size();
    s.edges = edges.data();
    s.edge_count = (int)edges.size();
    wc_solve q{};
    q.tx_pos = txs.data();
    q.tx_count = (int)txs.size() / 3;
    const long long pairs = (long long)q.tx_count * s.edge_count;
    static int list[kShadowList][256];
    blockDim = {1, 1, 1};
    threadIdx = {};
    if (kStageTop) stage_top_nodes(s);
    long wrong = 0, set = 0, full = 0, idle = 0;
    for (long long p = 0; p < pairs; ++p) {
        const Edge& e = edges[(size_t)(p % s.edge_count)];
        const ShadowFrame f = shadow_frame(e, ld3(q.tx_pos + 3 * (p / s.edge_count)));
        unsigned long long want = 0;
        if (f.valid)
            for (const Tri& t : tris) {
                const int g = __float_as_int(t.v0.w);
                if (g != e.group0 && g != e.group1) want |= triangle_shadow_bins(f, t);
            }
        // the lanes of the pair one after the other
        unsigned long long got = 0;
        for (int part = 0; part < kShadowLanes; ++part)
            got |= shadow_walk(s, f.valid, f, e.group0, e.group1, part, list, part);
        idle += shadow_walk(s, false, f, e.group0, e.group1, 0, list, 0) != 0;
        wrong += got != want;
        set += want != 0;
        full += want == ~0ull;
    }
    std::printf("pairs %lld set %ld full %ld wrong %ld idle %ld\n", pairs, set, full, wrong, idle);
    return 0;
}
