// CPU check of the swizzled LDS boxes of the CIC and PCS deposits (csrc/ma.hip):
//   - box_off gives every node of the box its own word inside the box;
//   - for every first node and every lane, the steps of rot_axis visit each node of the
//     footprint once, at its box_off, with its own weight;
//   - the 16 lanes of a pass are in 16 different bank pairs at every step (PCS), or in
//     the 8 (2D: 4) residues of the coordinates' parities two (four) lanes each (CIC),
//     whatever the lanes' first nodes;
//   - the partial layout of the column deposit numbers every value once, inside the slot;
//   - the tile of a node, taken by a multiplication, is the exact quotient;
//   - the PCS weights match the cubic B-spline in long double to float rounding.
// Built and run by tests/test_ma_box_emul.py (host compile only, no GPU calls).
#include "../../pylians3_amd/csrc/ma.hip"
#include <cassert>
#include <random>

using namespace pyl;

template <int MAS, int AXES>
static int check_box() {
    using D = BoxDim<MAS, AXES>;
    std::vector<int> seen(D::words, 0);
    int bad = 0;
    const int B = D::B, BZ = AXES == 3 ? B : 1;
    for (int x = 0; x < B; ++x)
        for (int y = 0; y < B; ++y)
            for (int z = 0; z < BZ; ++z) {
                const int o = box_off<MAS, AXES>(x, y, z);
                if (o < 0 || o >= D::words || seen[o]++) ++bad;
            }
    return bad;
}

// Byte offsets (and weights) of a lane's nodes in step order, as deposit_rot forms them.
template <int MAS, int AXES>
static std::vector<std::pair<int, float>> steps(const int3 &l, int lane, const float C[3][4]) {
    constexpr int F = MAS;
    using D = BoxDim<MAS, AXES>;
    float wx[4], wy[4], wz[4];
    int ox[4], oy[4], oz[4];
    std::vector<std::pair<int, float>> out;
    if (AXES == 2) {
        rot_axis<F>(C[1], l.y, lane & (F - 1), 8, 8 * D::sy, wy, oy);
        rot_axis<F>(C[0], l.x, (lane / F) & (F - 1), 8 * F, 8 * D::sx, wx, ox);
        const int b = 8 * ((l.x / F) * D::sx + (l.y / F) * D::sy);
        for (int i = 0; i < F; ++i)
            for (int m = 0; m < F; ++m) out.push_back({b + ox[i] + oy[m], wx[i] * wy[m]});
        return out;
    }
    rot_axis<F>(C[2], l.z, lane & (F - 1), 8, 8 * D::sz, wz, oz);
    rot_axis<F>(C[1], l.y, (lane / F) & (F - 1), 8 * F, 8 * D::sy, wy, oy);
    if (MAS == PYL_PCS) {
        const int b = 8 * (l.x * D::sx + (l.y / F) * D::sy + (l.z / F) * D::sz);
        for (int m = 0; m < F; ++m)
            for (int k = 0; k < F; ++k)
                for (int i = 0; i < F; ++i) out.push_back({b + oy[m] + oz[k] + 8 * i * D::sx, C[0][i] * wy[m] * wz[k]});
    } else {
        rot_axis<F>(C[0], l.x, (lane / (F * F)) & (F - 1), 8 * F * F, 8 * D::sx, wx, ox);
        const int b = 8 * ((l.x / F) * D::sx + (l.y / F) * D::sy + (l.z / F) * D::sz);
        for (int i = 0; i < F; ++i)
            for (int m = 0; m < F; ++m)
                for (int k = 0; k < F; ++k) out.push_back({b + ox[i] + oy[m] + oz[k], wx[i] * wy[m] * wz[k]});
    }
    return out;
}

template <int MAS, int AXES>
static int check_steps() {
    constexpr int F = MAS, T = AXES == 3 ? kT3 : kT2;
    const float C[3][4] = {{2, 3, 5, 7}, {11, 13, 17, 19}, {23, 29, 31, 37}};   // distinct products
    int bad = 0;
    std::mt19937 rng(5);
    for (int t = 0; t < 20000; ++t) {
        int3 l[16];
        std::vector<std::pair<int, float>> st[16];
        for (int lane = 0; lane < 16; ++lane) {
            l[lane] = make_int3(rng() % T, rng() % T, AXES == 3 ? rng() % T : 0);
            if (t % 3 == 0) l[lane] = l[0];            // a clump: one cell
            if (t % 7 == 0) l[lane].z = AXES == 3 ? T - 1 : 0;
            st[lane] = steps<MAS, AXES>(l[lane], lane, C);
            std::map<int, float> want;
            for (int i = 0; i < F; ++i)
                for (int m = 0; m < F; ++m)
                    for (int k = 0; k < (AXES == 3 ? F : 1); ++k)
                        want[8 * box_off<MAS, AXES>(l[lane].x + i, l[lane].y + m, l[lane].z + k)] =
                            C[0][i] * C[1][m] * (AXES == 3 ? C[2][k] : 1.0f);
            std::map<int, float> got(st[lane].begin(), st[lane].end());
            if (got != want || got.size() != st[lane].size()) ++bad;
        }
        constexpr int res = MAS == PYL_PCS ? 16 : AXES == 3 ? 8 : 4;
        for (size_t s = 0; s < st[0].size(); ++s) {
            int n[16] = {0};
            for (int lane = 0; lane < 16; ++lane) ++n[(st[lane][s].first / 8) % res];
            for (int r = 0; r < res; ++r)
                if (n[r] != 16 / res) ++bad;
        }
    }
    printf("box MAS %d axes %d: %s\n", MAS, AXES, bad ? "FAIL" : "ok");
    return bad + check_box<MAS, AXES>();
}

static int check_pcs_weights() {
    int bad = 0;
    std::mt19937 rng(9);
    std::uniform_real_distribution<float> U(-2.0f, 1030.0f);
    for (int t = 0; t < 500000; ++t) {
        float x = U(rng);
        if (t % 5 == 0) x = (float)(int)x;
        if (t % 11 == 0) x = std::nextafter((float)(int)x, -1e9f);
        float C[4];
        const int raw = first_node<PYL_PCS>(x);
        foot_weights<PYL_PCS>(x, raw, C);
        for (int j = 0; j < 4; ++j) {
            const long double d = std::fabs((long double)(raw + j) - (long double)x);
            const long double w = d < 1 ? (4 - 6 * d * d + 3 * d * d * d) / 6 : d < 2 ? (2 - d) * (2 - d) * (2 - d) / 6 : 0;
            // half an ulp of the rounding to float, and the double arithmetic before it
            if (!(std::fabs((long double)C[j] - w) <= 0x1p-24L * w + 0x1p-50L)) ++bad;
        }
    }
    printf("pcs weights: %s\n", bad ? "FAIL" : "ok");
    return bad;
}

// node_tile is floor(node * nt / dims) for every node of every grid size.
static int check_node_tile() {
    int bad = 0;
    auto one = [&](int dims, int axes, int step) {
        const TileGeom g = make_geom(dims, axes, PYL_TSC);
        if (g.nt == 1) return;                             // (home_tile shifts instead)
        for (int n = 0; n < dims; n += step)
            if (node_tile(n, g) != (int)((long long)n * g.nt / dims)) ++bad;
        if (node_tile(dims - 1, g) != g.nt - 1) ++bad;
    };
    for (int d = 17; d <= 2600; ++d) one(d, 3, 1);
    for (int d = 65; d <= 9000; d += 7) one(d, 2, 1);
    for (int d : {65521, 65535, 65536, 65537, 131071}) one(d, 2, 1);
    printf("node tile: %s\n", bad ? "FAIL" : "ok");
    return bad;
}

// Partial layout of the column deposit: for every pair of tile extents the ring columns
// are numbered once each (ring_col and ring_xy inverse), the four parts of a tile's slot
// do not overlap and fill at most the slot (halo_count of the largest tile).
template <int F>
static int check_ring() {
    constexpr int L = F - 1;
    int bad = 0;
    for (int zs = 8; zs <= kT3; ++zs)
        for (int ex = zs - 1; ex <= zs; ++ex)
            for (int ey = zs - 1; ey <= zs; ++ey) {
                std::vector<int> seen(ring_count<F>(ex, ey), 0);
                for (int x = 0; x < ex + L; ++x)
                    for (int y = 0; y < ey + L; ++y) {
                        if (!in_ring<F>(x, y, ex, ey)) continue;
                        const int rc = ring_col<F>(x, y, ex, ey);
                        int a, b;
                        if (rc < 0 || rc >= (int)seen.size() || seen[rc]++) { ++bad; continue; }
                        ring_xy<F>(rc, ex, ey, a, b);
                        if (a != x || b != y) ++bad;
                    }
                for (int v : seen) if (v != 1) ++bad;
                const int nr = ring_count<F>(ex, ey), ni = (ex - L) * (ey - L) * L;
                if (nr * zs > col_carry_at<F>(zs)) ++bad;
                if (col_carry_at<F>(zs) + nr * L > col_low_at<F>(zs)) ++bad;
                if (col_low_at<F>(zs) + ni > col_clow_at<F>(zs)) ++bad;
                if (col_clow_at<F>(zs) + ni > halo_count<F, 3>(zs, zs, zs)) ++bad;
            }
    for (int d = 1; d <= 19; ++d)
        for (int v = 0; v < 2048; ++v) {
            int q, r;
            small_div(v, d, q, r);
            if (q != v / d || r != v % d) ++bad;
        }
    printf("ring F %d: %s\n", F, bad ? "FAIL" : "ok");
    return bad;
}

int main() {
    int bad = check_steps<PYL_CIC, 3>() + check_steps<PYL_CIC, 2>() + check_steps<PYL_PCS, 3>() + check_steps<PYL_PCS, 2>();
    bad += check_box<PYL_NGP, 3>() + check_box<PYL_NGP, 2>() + check_box<PYL_TSC, 3>() + check_box<PYL_TSC, 2>();
    bad += check_pcs_weights() + check_node_tile() + check_ring<2>() + check_ring<3>() + check_ring<4>();
    printf(bad ? "FAILURES: %d\n" : "all ok\n", bad);
    return bad != 0;
}
