// Host side of the bead kernel (fts_bead.h): the axis matrices as operand
// tables, and the launch by plane shape.
#include <algorithm>
#include <cmath>
#include <vector>

#include "common.h"
#include "fts_bead.h"

namespace mft {

#define MFT_FOR_EACH_BEAD_SIZE(F, ...)                                                                     \
    F(16, __VA_ARGS__) F(20, __VA_ARGS__) F(24, __VA_ARGS__) F(32, __VA_ARGS__) F(40, __VA_ARGS__)         \
        F(48, __VA_ARGS__) F(64, __VA_ARGS__) F(80, __VA_ARGS__) F(96, __VA_ARGS__) F(128, __VA_ARGS__)

// Lengths the bead kernel takes.  From 160 points on a lane's orbits and their
// sums no longer fit its registers, and a 160 x 160 plane not LDS.
bool bead_length(int n)
{
    switch (n) {
#define MFT_CASE(n_, ...) case n_:
        MFT_FOR_EACH_BEAD_SIZE(MFT_CASE, 0)
#undef MFT_CASE
        return true;
    default: return false;
    }
}

// Rounds a row of block f to float so that the block's longest waves keep their
// factors: the error of every entry, largest first, is taken back by the entries that
// are still to be rounded, each by a share of the square of its own size, so that the
// row's product with each of those waves stays what it is (the smallest entries have
// the finest steps).  The waves of block f are even (cosine) or odd (sine, f & 1)
// about the orbits' reflection and of even or odd number (f & 2); a single block has
// both.  Two waves a block are the four to eight longest of the axis; more changed no
// result.  Rounded to nearest instead, each is off by 1e-8 to 4e-8 per bead and axis, which
// adds up along the chain (now 1e-10 and less; other waves keep errors of that size).
// Chains of 400 beads in a gyroid field of +-8, 64^3: last bead 1.4e-5 off 64 bits,
// now 2.0e-7 (5.4e-5 with the transforms of the plane and line kernels); 96^3, 100
// beads: 2.2e-5, now 1.5e-6 (1.1e-4).
template <int N>
static void bead_round_row(int f, const double* v, float* out)
{
    using A = BeadAxis<N>;
    constexpr int S = A::S, K = A::F == 1 ? 3 : 2;
    double u[K][S], t[S];
    int order[S];
    for (int m = 0; m < K; ++m) {
        const bool sine = A::F == 1 ? m == 2 : f & 1;
        const int first = A::F == 4 ? (f == 1 ? 2 : f >> 1) : (A::F == 2 ? f : 0);
        const int k = A::F == 1 ? (m > 0) : first + m * (A::F / 2);
        for (int i = 0; i < S; ++i) {
            const double x = 2.0 * M_PI * k * (i + 0.5) / N;
            u[m][i] = sine ? std::sin(x) : std::cos(x);
        }
    }
    for (int i = 0; i < S; ++i) {
        t[i] = v[i];
        order[i] = i;
    }
    std::stable_sort(order, order + S, [&](int a, int b) { return std::fabs(v[a]) > std::fabs(v[b]); });
    const double most = std::fabs(v[order[0]]) * 0x1p-23;
    for (int n = 0; n < S; ++n) {
        const int at = order[n];
        out[at] = (float)t[at];
        const double e = (double)out[at] - t[at];
        if (std::fabs(v[at]) < most * 0x1p-23) continue; // its rounding is below 2^-70 of the largest entry
        // least change, in units of the entries' sizes, with sum_r d_r u_m(r) = -e u_m(at):
        // orthonormal q_m from |v| u_m and forward substitution
        double q[K][S], y[K];
        for (int m = 0; m < K && n + 1 < S; ++m) {
            double norm = 0.0, rhs = -e * u[m][at];
            for (int r = n + 1; r < S; ++r) q[m][r] = std::fabs(v[order[r]]) * u[m][order[r]];
            for (int l = 0; l < m; ++l) {
                double dot = 0.0;
                for (int r = n + 1; r < S; ++r) dot += q[l][r] * q[m][r];
                for (int r = n + 1; r < S; ++r) q[m][r] -= dot * q[l][r];
                rhs -= dot * y[l];
            }
            for (int r = n + 1; r < S; ++r) norm += q[m][r] * q[m][r];
            if (norm == 0.0) break;
            for (int r = n + 1; r < S; ++r) q[m][r] /= std::sqrt(norm);
            y[m] = rhs / std::sqrt(norm);
            // few entries, or much smaller ones, cannot stand in for this one: they
            // change by less than the largest entry's rounding and than their own size
            bool fits = true;
            for (int r = n + 1; r < S && fits; ++r) {
                double z = 0.0;
                for (int l = 0; l <= m; ++l) z += q[l][r] * y[l];
                fits = std::fabs(z) < 0x1p-8 && std::fabs(z * v[order[r]]) < most;
            }
            if (!fits) break;
            for (int r = n + 1; r < S; ++r) t[order[r]] += std::fabs(v[order[r]]) * q[m][r] * y[m];
        }
    }
}

// A operands of the 16x16x4 matrix instruction for the F blocks of the circulant
// C[i][j] = c(i - j), c(d) = 1/n sum_k g_k cos(2 pi k d / n), g symmetric: block f
// couples orbits i and j by 1/F sum_h chi_f(h) C[i][h j] over the members h,
// chi_f(h) the sign member h has in sum f.  Operand (o, j, l) of a block is, for
// lane l, its entry at row orbit(4 o + l % 4, l % 16 / 4), whose result lands in
// register l % 4 of lane group l % 16 / 4, and column orbit(j, l / 16); zero past
// the last orbit.  Rows of block 0 keep their sum, 1/F, to the last bit of their
// smallest entry (the residual goes there): a constant stays the constant.
template <int N>
static void bead_table_n(const double* g, std::vector<float>& tab)
{
    using A = BeadAxis<N>;
    std::vector<double> c(N);
    for (int d = 0; d < N; ++d) {
        double s = 0.0;
        for (int k = 0; k < N; ++k) s += g[k] * std::cos(2.0 * M_PI * (double)((long)k * d % N) / N);
        c[d] = s / N;
    }
    tab.assign(A::TABLE, 0.f);
    for (int f = 0; f < A::F; ++f) {
        float blk[A::S][A::S];
        for (int i = 0; i < A::S; ++i) {
            double row[A::S], exact = 0.0, sum = 0.0;
            for (int k = 0; k < A::S; ++k) {
                double v = 0.0;
                for (int h = 0; h < A::F; ++h)
                    v += (__builtin_parity(f & h) ? -1.0 : 1.0) * c[((i - bead_row<N>(h, k)) % N + N) % N];
                row[k] = v / A::F;
            }
            bead_round_row<N>(f, row, blk[i]);
            int least = 0;
            for (int k = 0; k < A::S; ++k) {
                exact += row[k];
                sum += (double)blk[i][k];
                if (std::fabs(blk[i][k]) < std::fabs(blk[i][least])) least = k;
            }
            if (f == 0) blk[i][least] = (float)((double)blk[i][least] + (exact - sum));
        }
        for (int o = 0; o < A::RT; ++o)
            for (int j = 0; j < A::J; ++j)
                for (int l = 0; l < 64; ++l) {
                    if (l % 4 >= A::in_tile(o)) continue;
                    const int i = A::orbit(4 * o + l % 4, l % 16 / 4), k = A::orbit(j, l / 16);
                    if (i < A::S && k < A::S) tab[(size_t)f * A::BLOCK + (o * A::J + j) * 64 + l] = blk[i][k];
                }
    }
}

// operand table of an axis of n points (bead_length(n)) with the diffusion
// factors g[n]
void bead_table(int n, const double* g, std::vector<float>& tab)
{
    switch (n) {
#define MFT_CASE(n_, ...) case n_: bead_table_n<n_>(g, tab); break;
        MFT_FOR_EACH_BEAD_SIZE(MFT_CASE, 0)
#undef MFT_CASE
    default: tab.clear();
    }
}

template <int NX, int NA>
static int bead_allow_lds_n()
{
    constexpr size_t bytes = BeadShape<NX, NA>::LDS;
    if constexpr (bytes > 64 * 1024)
        MFT_HIP(hipFuncSetAttribute((const void*)k_fts_bead<NX, NA>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)bytes));
    return MFT_OK;
}

template <int NX, int NA>
static void bead_launch_n(const BeadDesc* h, const BeadDesc* d, int n, int planes, long ps, long rs, hipStream_t st)
{
    using SH = BeadShape<NX, NA>;
    BeadArgs args = {};
    if (n <= kBeadInline) {
        for (int k = 0; k < n; ++k) args.d[k] = h[k];
        d = nullptr;
    }
    k_fts_bead<NX, NA><<<dim3(planes, n), 64 * SH::W, SH::LDS, st>>>(args, d, ps, rs);
}

// raises the dynamic LDS limit of the (nx, na) plane kernel on the current
// device where it needs more than 64 KB
int bead_allow_lds(int nx, int na)
{
#define MFT_NA(na_, nx_) if (na == na_) return bead_allow_lds_n<nx_, na_>();
#define MFT_NX(nx_, ...) if (nx == nx_) { MFT_FOR_EACH_BEAD_NA(MFT_NA, nx_) }
#define MFT_FOR_EACH_BEAD_NA(F, X)                                                                         \
    F(16, X) F(20, X) F(24, X) F(32, X) F(40, X) F(48, X) F(64, X) F(80, X) F(96, X) F(128, X)
    MFT_FOR_EACH_BEAD_SIZE(MFT_NX, 0)
#undef MFT_NA
    set_error(MFT_ERR_UNSUPPORTED, "no bead kernel for %d x %d planes", nx, na);
    return MFT_ERR_UNSUPPORTED;
}

// one bead of n chains (their descriptors on the host and on the device) along axis `axis` (1: z-planes, rows along y; 2:
// y-planes, rows along z)
int bead_launch(const BeadDesc* h, const BeadDesc* d, int n, const int dims[3], int axis, hipStream_t st)
{
    const int nx = dims[0], na = dims[axis], planes = dims[3 - axis];
    const long sy = nx, sz = (long)nx * dims[1];
    const long ps = axis == 1 ? sz : sy, rs = axis == 1 ? sy : sz;
    bool done = false;
#define MFT_NA(na_, nx_) if (na == na_) { bead_launch_n<nx_, na_>(h, d, n, planes, ps, rs, st); done = true; }
    MFT_FOR_EACH_BEAD_SIZE(MFT_NX, 0)
#undef MFT_NA
    MFT_REQUIRE(done, MFT_ERR_UNSUPPORTED, "no bead kernel for %d x %d planes", nx, na);
    MFT_LAUNCH_CHECK();
    return MFT_OK;
}

} // namespace mft
