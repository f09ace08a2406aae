// CPU check of the masked path export's row kernels (wc_radiomap.hip, built as
// host C++ through the shim in hip/): what a row becomes whose dealt candidate
// the evaluating kernel does not find again, as a wall or a face border within
// the rounding of two differently compiled kernels would leave it.
//
// Straight rows: a segment through `found` walls dealt as `dealt` walls must be
// the row of a segment dealt `found` walls (a line-of-sight row without walls),
// and absent (length NaN, interactions -1) where no such row exists.
// Chains: a chain of 1 to 5 bounces whose last hit lies off the wall is absent
// too; with all zeros for its interactions it would carry the identity of a
// reflection off face 0, and the compaction would drop a real one with it.
// Input directory: nodes.bin, tris.bin (leaf order), ftris.bin (face order),
// plane.bin, goff.bin, gfaces.bin of three parallel walls at x = 10, 20, 30.
// Prints one summary line.
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

constexpr int W = kMaxDepth;

// one row of the path table
struct Row {
    int tx = 0, rx = 0, depth = -9, component = -9, primitive = -9, edge = -9, material = -9;
    float length = -9, delay = -9, gain = -9;
    int seq[W], mat[W];
    float pos[W][3], nrm[W][3], field[2], coef[2], xyz[6], arr[3], dep[3];
    wc_path_rows view() {
        wc_path_rows v{};
        v.width = W;
        v.tx_id = &tx; v.rx_id = &rx; v.depth = &depth; v.component_id = &component; v.primitive_id = &primitive;
        v.edge_id = &edge; v.material_id = &material; v.path_length_m = &length; v.delay_s = &delay;
        v.path_gain = &gain; v.primitive_sequence = seq; v.material_sequence = mat;
        v.interaction_positions = pos[0]; v.interaction_normals = nrm[0]; v.path_field = field; v.coefficient = coef;
        v.field_xyz = xyz; v.arrival_direction = arr; v.departure_direction = dep;
        return v;
    }
    bool same(const Row& o) const {
        return depth == o.depth && component == o.component && primitive == o.primitive && edge == o.edge &&
               material == o.material && length == o.length && delay == o.delay && gain == o.gain &&
               !std::memcmp(seq, o.seq, sizeof(seq)) && !std::memcmp(mat, o.mat, sizeof(mat)) &&
               !std::memcmp(pos, o.pos, sizeof(pos)) && !std::memcmp(nrm, o.nrm, sizeof(nrm)) &&
               !std::memcmp(xyz, o.xyz, sizeof(xyz)) && !std::memcmp(field, o.field, sizeof(field)) &&
               !std::memcmp(coef, o.coef, sizeof(coef));
    }
    bool absent(int comp) const {
        bool ok = std::isnan(length) && component == comp && edge == -1 && primitive == -1;
        for (int j = 0; j < W; ++j) ok = ok && seq[j] == -1 && mat[j] == -1;
        return ok;
    }
};

// the row kernel on one row dealt (component, candidate)
static Row evaluate(const SceneView& s, const wc_solve& q, int component, int candidate) {
    Row r;
    r.component = component;
    r.primitive = candidate;
    const int list[1] = {0}, dealt[2] = {0, 1};
    blockIdx = {}; threadIdx = {}; blockDim = {1, 1, 1}; gridDim = {1, 1, 1};
    export_main_kernel(s, q, r.view(), 1, list, dealt);
    return r;
}

int main(int argc, char** argv) {
    if (argc < 2) return 2;
    const std::string d = argv[1];
    const auto nodes = load<WideNode>(d + "/nodes.bin");
    const auto tris = load<Tri>(d + "/tris.bin"), faces = load<Tri>(d + "/ftris.bin");
    const auto plane = load<double>(d + "/plane.bin");
    const auto goff = load<int>(d + "/goff.bin"), gfaces = load<int>(d + "/gfaces.bin");
    if (nodes.empty() || tris.empty() || plane.empty() || goff.size() != 4) return 2;
    std::vector<int> face_group, face_material(faces.size(), 0);
    for (const Tri& t : faces) face_group.push_back(__float_as_int(t.v0.w));
    const float eps = 4.0f, sigma = 0.01f, mu = 1.0f, gain = 1.0f, thick = 0.2f;
    const int layer_offset = 0, layer_count = 1;
    SceneView s{};
    s.nodes = nodes.data(); s.tris = tris.data(); s.tri_count = (int)tris.size(); s.node_count = (int)nodes.size();
    s.faces = faces.data(); s.face_group = face_group.data(); s.face_material = face_material.data();
    s.face_count = (int)faces.size(); s.group_plane = plane.data(); s.group_face_offset = goff.data();
    s.group_faces = gfaces.data(); s.group_count = 3;
    s.mat_eps = &eps; s.mat_sigma = &sigma; s.mat_mu = &mu; s.mat_gain = &gain; s.mat_thickness = &thick;
    s.mat_layer_offset = &layer_offset; s.mat_layer_count = &layer_count; s.layer_thickness = &thick;
    s.layer_eps = &eps; s.layer_sigma = &sigma; s.layer_mu = &mu; s.material_count = 1;

    const float tx[3] = {1.0f, 2.0f, 3.0f}, up[3] = {0.0f, 0.0f, 1.0f}, power = 1.0f;
    float rx[3] = {0.0f, 4.0f, 2.5f};
    const int cell_offset[2] = {0, 1};
    wc_solve q{};
    q.tx_pos = tx; q.tx_pol = up; q.tx_power = &power; q.tx_count = 1; q.rx_pos = rx; q.rx_pol = up;
    q.cell_offset = cell_offset; q.total_cells = 1; q.frequency_hz = 3.5e9; q.lanes_per_cell = 1;
    long straight = 0, wrong = 0, gone = 0;
    for (int depth = 1; depth <= kMaxDepth; ++depth)
        for (int los = 0; los < 2; ++los)
            for (int found = 0; found <= 3; ++found)
                for (int dealt = 1; dealt <= depth; ++dealt) {
                    q.max_depth = depth;
                    q.components = kCompTrans | (los ? kCompLos : 0);
                    rx[0] = 5.0f + 10.0f * found;
                    const Row got = evaluate(s, q, kCidTrans, dealt);
                    ++straight;
                    if (found == 0 && los) {
                        wrong += !got.same(evaluate(s, q, kCidLos, 0)) || got.component != kCidLos;
                    } else if (found >= 1 && found <= depth) {
                        wrong += !got.same(evaluate(s, q, kCidTrans, found)) || got.depth != found;
                    } else {
                        ++gone;
                        wrong += !got.absent(kCidTrans);
                    }
                }

    // bounces between walls 0 and 1: wall 0 last, hit on it (y = 4) or off it (y = 400)
    std::vector<int> chain_groups(kMaxDepth * kMaxDepth, -1), chain_offset(kMaxDepth + 1);
    std::vector<double> images((size_t)kMaxDepth * kMaxDepth * 3, 0.0);
    for (int c = 0; c < kMaxDepth; ++c) {
        chain_offset[c + 1] = c + 1;
        V3<double> p{15.0, 2.0, 3.0};
        for (int b = 0; b <= c; ++b) {
            const int g = (c - b) % 2;
            chain_groups[c * kMaxDepth + b] = g;
            double off;
            const V3<double> n = group_normal(s, g, off);
            p = p - n * (2.0 * (dot(p, n) - off));
            double* im = &images[(size_t)(c * kMaxDepth + b) * 3];
            im[0] = p.x; im[1] = p.y; im[2] = p.z;
        }
    }
    const float between[3] = {15.0f, 2.0f, 3.0f};
    q.tx_pos = between; q.components = kCompRefl; q.max_depth = kMaxDepth; q.max_tx_chains = kMaxDepth;
    q.chain_offset = chain_offset.data(); q.chain_groups = chain_groups.data(); q.chain_images = images.data();
    long chains = 0, kept = 0;
    for (int c = 0; c < kMaxDepth; ++c)
        for (const float y : {4.0f, 400.0f}) {
            rx[0] = 16.0f;
            rx[1] = y;
            const Row got = evaluate(s, q, kCidRefl, c);
            ++chains;
            if (y < 40.0f) kept += got.component == kCidRefl && got.depth == c + 1 && got.length > 0.0f && got.seq[0] >= 0;
            else kept += got.absent(kCidRefl) && got.depth == c + 1;
        }
    std::printf("chains %ld chains_right %ld straight %ld gone %ld straight_wrong %ld\n", chains, kept, straight, gone, wrong);
    return 0;
}
