// Power spectra on gfx950: rocFFT r2c + one fused binning pass.
//
// Reference semantics: library/Pk_library/Pk_library.pyx:263-420 (Pk) and
// :529-793 (XPk).  Per mode of the half-complex FFT output the binning pass
// does, in one read of delta_k: the half-space skip rule (:324-327), integer
// bin assignment (k_index = isqrt(k^2), k_per = isqrt(k_perp^2), exact for the
// reference's (int)sqrt of integer squares), MAS deconvolution with a float
// factor equal to the double product of the per-axis corrections (:351-352),
// |delta_k|^2 in double (:355-357), mu-Legendre weights for l = 0, 2, 4 and the
// phase (:358), and the 1D / 2D / 3D accumulations (:361-378).
//
// Work decomposition.  The up to four rows (+-kx, +-ky) of one (|kx|, |ky|) form a
// row group: at every kz they share |k|, the bins, mu and the MAS factor, and differ
// only in their values.  Groups are ordered by a key that fixes the 2D bins they can
// reach: |kx| (axis 0), |ky| (axis 1) or k_per = isqrt(kx^2+ky^2) (axis 2).  A work
// item is some groups with one key; one workgroup per item accumulates into LDS: the 3D
// bins, one "line" of 2D bins (all k_per at fixed k_par for axes 0/1, all k_par at
// fixed k_per for axis 2) and the 1D bins.  Each lane handles runs of 4 consecutive kz
// of a group, adds up the group's |delta|^2 at each kz and merges equal bins along the
// run in registers before its LDS atomics.  Items write their LDS partials with plain
// stores; a reduce kernel sums them, so the result is deterministic and no global
// atomics are used.
//
// Mode counts and k sums do not depend on the data: they are computed exactly
// on the host once per (dims, axis) from Hermitian-pair counting and cached.
#include "pyl_internal.h"
#include "fixsum.h"

#include <array>

#include <algorithm>
#include <cmath>
#include <thread>

namespace pyl {

// ------------------------------------------------------------------ mode plan
// Independent modes = one of each conjugate pair plus the self-conjugate modes,
// so per bin: N_indep = (N_all + N_self) / 2, where N_all counts the full
// dims^3 cube and N_self the modes with every component in {0, dims/2}.
// Every binned quantity depends only on (|kx|, |ky|, |kz|), so the cube is
// walked over absolute values with multiplicities.
void compute_mode_plan(int dims, int axis, ModePlan *mp) {
    const int m = dims / 2;
    const bool even = dims % 2 == 0;
    const int kmax_par = m;
    const int kmax_per = (int)std::sqrt((double)(m * m + m * m));
    const int kmax = (int)std::sqrt((double)(3 * m * m));
    const long long nb2 = (long long)(kmax_par + 1) * (kmax_per + 1);
    const long long nk2 = 3LL * m * m + 1;
    auto mult = [&](int a) -> long long { return (a == 0 || (even && a == m)) ? 1 : 2; };
    auto isq = [](long long v) -> int {
        long long s = (long long)std::sqrt((double)v);
        while (s * s > v) --s;
        while ((s + 1) * (s + 1) <= v) ++s;
        return (int)s;
    };
    std::vector<int> isqrt_tab(2LL * m * m + 1);
    for (long long v = 0; v < (long long)isqrt_tab.size(); ++v) isqrt_tab[v] = isq(v);

    unsigned nth = std::max(1u, std::min(8u, std::thread::hardware_concurrency()));
    if (m < 32) nth = 1;
    struct Part {
        std::vector<long long> c3, c2, c1;
    };
    std::vector<Part> parts(nth);
    auto work = [&](unsigned t) {
        Part &P = parts[t];
        P.c3.assign(nk2, 0);
        P.c2.assign(nb2, 0);
        P.c1.assign(m + 1, 0);
        for (int a = (int)t; a <= m; a += (int)nth) {
            const long long ma = mult(a);
            for (int b = 0; b <= m; ++b) {
                const long long mab = ma * mult(b);
                for (int c = 0; c <= m; ++c) {
                    const long long w = mab * mult(c);
                    const long long k2 = (long long)a * a + (long long)b * b + (long long)c * c;
                    int kpar, kper;
                    if (axis == 0) { kpar = a; kper = isqrt_tab[b * b + c * c]; }
                    else if (axis == 1) { kpar = b; kper = isqrt_tab[a * a + c * c]; }
                    else { kpar = c; kper = isqrt_tab[a * a + b * b]; }
                    P.c3[k2] += w;
                    P.c2[(long long)(kmax_par + 1) * kper + kpar] += w;
                    if (k2 <= (long long)m * m) P.c1[kpar] += w;
                }
            }
        }
    };
    if (nth == 1) work(0);
    else {
        std::vector<std::thread> th;
        for (unsigned t = 0; t < nth; ++t) th.emplace_back(work, t);
        for (auto &x : th) x.join();
    }
    std::vector<long long> c3(nk2, 0), c2(nb2, 0), c1(m + 1, 0);
    for (auto &P : parts) {
        for (long long i = 0; i < nk2; ++i) c3[i] += P.c3[i];
        for (long long i = 0; i < nb2; ++i) c2[i] += P.c2[i];
        for (int i = 0; i <= m; ++i) c1[i] += P.c1[i];
    }
    // self-conjugate modes: components in {0} (odd) or {0, m} (even)
    std::vector<int> vals = even ? std::vector<int>{0, m} : std::vector<int>{0};
    if (even && m == 0) vals = {0};
    for (int a : vals)
        for (int b : vals)
            for (int c : vals) {
                const long long k2 = (long long)a * a + (long long)b * b + (long long)c * c;
                int kpar, kper;
                if (axis == 0) { kpar = a; kper = isq((long long)b * b + (long long)c * c); }
                else if (axis == 1) { kpar = b; kper = isq((long long)a * a + (long long)c * c); }
                else { kpar = c; kper = isq((long long)a * a + (long long)b * b); }
                c3[k2] += 1;
                c2[(long long)(kmax_par + 1) * kper + kpar] += 1;
                if (k2 <= (long long)m * m) c1[kpar] += 1;
            }
    mp->dims = dims;
    mp->axis = axis;
    mp->N3D.assign(kmax + 1, 0.0);
    mp->k3D.assign(kmax + 1, 0.0);
    for (long long k2 = 0; k2 < nk2; ++k2) {
        long long n = c3[k2] / 2;  // (N_all + N_self) / 2, always an integer
        if (!n) continue;
        int b = isq(k2);
        mp->N3D[b] += (double)n;
        mp->k3D[b] += (double)n * std::sqrt((double)k2);
    }
    mp->N2D.resize(nb2);
    for (long long i = 0; i < nb2; ++i) mp->N2D[i] = (double)(c2[i] / 2);
    mp->N1D.resize(m + 1);
    mp->k1D.resize(m + 1);
    for (int i = 0; i <= m; ++i) {
        mp->N1D[i] = (double)(c1[i] / 2);
        mp->k1D[i] = (double)i * mp->N1D[i];
    }
}

const ModePlan *get_mode_plan(Ctx *, int dims, int axis) {
    SharedTables &st = shared_tables();
    std::lock_guard<std::mutex> lk(st.mu);
    const auto key = std::make_pair(dims, axis);
    auto it = st.mode.find(key);
    if (it != st.mode.end()) return &it->second;
    ModePlan mp;
    compute_mode_plan(dims, axis, &mp);
    return &st.mode.emplace(key, std::move(mp)).first->second;
}

namespace {

constexpr int kRun = 4;          // consecutive kz per lane
constexpr int kBinBlock = 512;

struct PkDims {
    int dims, m, zlen, zpad, even, kmax, kmax_par, kmax_per;
    long long nb2;
};

PkDims pk_dims(int dims) {
    PkDims p;
    p.dims = dims;
    p.m = dims / 2;
    p.zlen = p.m + 1;
    p.zpad = (p.zlen + kRun - 1) / kRun * kRun;
    p.even = dims % 2 == 0;
    p.kmax_par = p.m;
    p.kmax_per = (int)std::sqrt((double)(p.m * p.m + p.m * p.m));
    p.kmax = (int)std::sqrt((double)(3 * p.m * p.m));
    p.nb2 = (long long)(p.kmax_par + 1) * (p.kmax_per + 1);
    return p;
}

// Key of the row group (a, b) = (|kx|, |ky|).
int group_key(int a, int b, int axis) {
    if (axis == 0) return a;
    if (axis == 1) return b;
    const long long v = (long long)a * a + (long long)b * b;
    long long s = (long long)std::sqrt((double)v);
    while (s * s > v) --s;
    while ((s + 1) * (s + 1) <= v) ++s;
    return (int)s;
}

int get_bin_plan(Ctx *c, int dims, int axis, int nreal, BinPlan **out) {
    // Groups per item.  Large grids: ~2048 items (for a batch ~16K items in total, so
    // that the partials stay small).  Small grids: at least one run per lane of the
    // workgroup, since an item's fixed cost (clearing, writing and reducing its P bins)
    // does not shrink with it: 64^3 took 513 items of four rows, 36 of 512 lanes at
    // work, and their reduction (18 us) took longer than the binning (13 us).
    const PkDims p = pk_dims(dims);
    const long long ngroups_total = (long long)(p.m + 1) * (p.m + 1);
    const int runs_per_group = p.zpad / kRun;
    const long long target = nreal > 1 ? std::max(1LL, 16384LL / nreal) : 2048LL;
    int G = c->tune_bin_rows > 0
                ? std::max(1, std::min(256, c->tune_bin_rows) / 4)
                : (int)std::max<long long>(ceil_div(kBinBlock, runs_per_group),
                                           std::min<long long>(64, ngroups_total / target));
    // an exact bin sum's low word takes at most kFixMaxAdds additions: one per run of
    // kRun modes of the item's groups
    G = std::max(1, std::min(G, kFixMaxAdds / runs_per_group));
    const ModePlan *mp = get_mode_plan(c, dims, axis);
    SharedTables &st = shared_tables();
    std::lock_guard<std::mutex> lk(st.mu);
    const auto key = std::make_tuple(c->device, dims, axis, G);
    auto it = st.bin.find(key);
    if (it != st.bin.end()) {
        *out = &it->second;
        return PYL_OK;
    }
    PYL_CHECK(!c->capturing, PYL_EINVAL, "binning plan created while a graph is captured: run the "
              "same work once on the context before capturing it");
    PYL_CHECK(p.m < 32768, PYL_EINVAL, "grid too large for the binning plan");
    const int nkeys = (axis == 2) ? p.kmax_per + 1 : p.m + 1;
    std::vector<std::vector<int>> by_key(nkeys);
    for (int a = 0; a <= p.m; ++a)
        for (int b = 0; b <= p.m; ++b) by_key[group_key(a, b, axis)].push_back(a << 16 | b);
    std::vector<int> groups;
    groups.reserve(ngroups_total);
    std::vector<int4> items;
    std::vector<int> key_items(nkeys + 1, 0);
    for (int k = 0; k < nkeys; ++k) {
        key_items[k] = (int)items.size();
        const auto &v = by_key[k];
        // equal shares of the key's groups
        const int n = (int)v.size(), ni = ceil_div(n, G);
        for (int i = 0; i < ni; ++i) {
            const int s = (int)((long long)n * i / ni), e = (int)((long long)n * (i + 1) / ni);
            items.push_back(make_int4((int)groups.size() + s, e - s, k, 0));
        }
        groups.insert(groups.end(), v.begin(), v.end());
    }
    key_items[nkeys] = (int)items.size();
    BinPlan bp;
    bp.dims = dims;
    bp.axis = axis;
    bp.G = G;
    bp.nitems = (int)items.size();
    bp.nkeys = nkeys;
    auto fail = [&](hipError_t e) {
        (void)hipFree(bp.d_groups);
        (void)hipFree(bp.d_items);
        (void)hipFree(bp.d_key_items);
        (void)hipFree(bp.d_n2);
        set_error("binning plan upload failed: %s", hipGetErrorString(e));
        return e == hipErrorOutOfMemory ? PYL_ENOMEM : PYL_EHIP;
    };
    hipError_t e;
    if ((e = hipMalloc(&bp.d_groups, groups.size() * sizeof(int))) != hipSuccess) return fail(e);
    if ((e = hipMalloc(&bp.d_items, items.size() * sizeof(int4))) != hipSuccess) return fail(e);
    if ((e = hipMalloc(&bp.d_key_items, key_items.size() * sizeof(int))) != hipSuccess) return fail(e);
    if ((e = hipMalloc(&bp.d_n2, mp->N2D.size() * sizeof(double))) != hipSuccess) return fail(e);
    if ((e = hipMemcpy(bp.d_n2, mp->N2D.data(), mp->N2D.size() * sizeof(double), hipMemcpyHostToDevice)) !=
        hipSuccess)
        return fail(e);
    if ((e = hipMemcpy(bp.d_groups, groups.data(), groups.size() * sizeof(int), hipMemcpyHostToDevice)) !=
        hipSuccess)
        return fail(e);
    if ((e = hipMemcpy(bp.d_items, items.data(), items.size() * sizeof(int4),
                       hipMemcpyHostToDevice)) != hipSuccess)
        return fail(e);
    if ((e = hipMemcpy(bp.d_key_items, key_items.data(), key_items.size() * sizeof(int),
                       hipMemcpyHostToDevice)) != hipSuccess)
        return fail(e);
    *out = &st.bin.emplace(key, bp).first->second;
    return PYL_OK;
}

// ------------------------------------------------------------------ kernels
// Spectra computed by one launch: NFL = 1 -> {auto a}; NFL = 2 -> {auto a, auto b, cross ab}.
template <int NFL> struct Spec { static constexpr int S = NFL == 1 ? 1 : 3; };

struct BinArgs {
    const float2 *dk[2];     // half-complex fields
    const double *corr[2];   // MAS correction tables [dims] per field
    float cmax[2];           // largest product of three MAS corrections per field
    const unsigned *amax[2]; // per field [realisation][64]: largest |Re|, |Im| (float bits)
    int *escale;             // [realisation][2]: E of the power and the phase sums
    int nreal;
    const int *groups;       // |kx| << 16 | |ky| per row group
    const int4 *items;
    unsigned long long *plo; // [nreal][nitems][P] low words of the item sums
    int *phi;                // [nreal][nitems][P] high words
    long long fstride;       // elements between realisations in dk[] (blockIdx.y = realisation)
    long long zs;            // elements between rows (kx, ky) of dk[] (>= zlen)
    int nitems;
    int dims, m, zlen, zpad, even, kmax, L2, L1;
    int P, off2, off1;       // partial layout: acc3 at 0, line2 at off2, line1 at off1
    int gmax;                // max groups per item (LDS group table size)
    int wide;                // rows are 16-byte aligned and padded to zpad: 16-byte loads
};

// floor(sqrt(v)) for 0 <= v < 2^24: the hardware square root (within 1 ulp)
// lands within one of the answer, and the two integer tests correct it.
__device__ __forceinline__ int isqrt_i(int v) {
    int s = (int)__builtin_amdgcn_sqrtf((float)v);
    if (s * s > v) --s;
    if ((s + 1) * (s + 1) <= v) ++s;
    return s;
}

// atan2(a, b) on the half-plane b >= |a| (the phase of Pk_library.pyx:358,
// atan2(real, |delta|)) for b in [0.5, 2): the caller scales both components by a
// power of two so that the larger has magnitude in [0.5, 1).  t = a/b (hardware
// reciprocal, 1 ulp) lies in [-1, 1] and atan(t) is t*P(t^2), P of degree 7 fitted
// to atan(t)/t on [0, 1] by iteratively reweighted least squares on Chebyshev nodes
// (max error 1.7e-7 in float, 2.3e-7 relative).
__device__ __forceinline__ float atan_halfplane(float a, float b) {
    float t = a * __builtin_amdgcn_rcpf(b);
    t = fminf(fmaxf(t, -1.0f), 1.0f);       // |a| <= b: only rounding can leave [-1, 1]
    const float u = t * t;
    float p = -0.00478044f;
    p = p * u + 0.02455707f;
    p = p * u - 0.05990465f;
    p = p * u + 0.09942755f;
    p = p * u - 0.14029419f;
    p = p * u + 0.19971375f;
    p = p * u - 0.33332094f;
    p = p * u + 0.99999991f;
    return t * p;
}

// The phase^2 of Pk_library.pyx:358, atan2(Re, |delta|)^2, from the float components
// scaled by a power of two near 1/max(|Re|, |Im|) (exact): |delta|^2 formed in float
// would overflow or underflow for |delta| beyond ~1e19 or below ~1e-19.
__device__ __forceinline__ float phase_sq(float xr, float xi) {
    float ph = 0.0f;
    const float mx = fmaxf(fabsf(xr), fabsf(xi));
    if (mx > 0.0f) {
        const int e = __builtin_amdgcn_frexp_expf(mx);
        const float xs = __builtin_ldexpf(xr, -e), ys = __builtin_ldexpf(xi, -e);
        ph = atan_halfplane(xs, __builtin_amdgcn_sqrtf(xs * xs + ys * ys));
    }
    return ph * ph;
}

__device__ __forceinline__ float masked(float x, unsigned on) { return __uint_as_float(__float_as_uint(x) & on); }

// VALU-bound: about 170 instructions per mode when every row was binned by itself
// (0.305 ms at 512^3, axis 0, against 0.1 ms for its 0.54 GB).  The symmetric rows of a
// group share everything but their values, so the geometry, the MAS factor, the
// multipole products and the flush into LDS are done once for up to four modes:
// 0.171 ms at 512^3 (3.2 TB/s of modes read), 0.092 -> 0.049 ms for two fields at 256^3
// (axis 2), 0.573 -> 0.223 ms for 32 realisations of two 128^3 fields.
template <int AXIS, int NFL, bool PHASE>
__global__ void __launch_bounds__(kBinBlock) pk_bin_kernel(BinArgs a) {
    constexpr int S = Spec<NFL>::S;
    constexpr int NA3 = 3 * S + (PHASE ? 1 : 0);   // per 3D bin: P0,P2,P4 per spectrum [+phase]
    extern __shared__ double lds[];
    // The P accumulators, fixed point: low words alo[P], high words ahi[P].  acc3
    // (indices [0, n3)) is [NA3][kmax+1] in LDS (consecutive bins in consecutive
    // banks: lanes flushing neighbouring bins do not collide), [kmax+1][NA3] in the
    // partials; the 2D line at off2, the 1D line at off1.
    unsigned long long *alo = (unsigned long long *)lds;
    int *ahi = (int *)(alo + a.P);
    const int K1 = a.kmax + 1;
    double *corrz = (double *)(ahi + ((a.P + 1) & ~1));  // [zlen*NFL]
    double *rowc = corrz + a.zlen * NFL;              // [gmax*NFL]
    int *grp = (int *)(rowc + a.gmax * NFL);          // [gmax]
    __shared__ int sE[2];

    const int4 item = a.items[blockIdx.x];
    const int ngrp = item.y;
    const int key = item.z;
    const int tid = threadIdx.x;
    const int n3 = (a.kmax + 1) * NA3;
    for (int i = tid; i < a.P; i += blockDim.x) {
        alo[i] = 0ull;
        ahi[i] = 0;
    }
    if (tid < 64) {
        // the realisation's scale: the same in every work item
        float mw[NFL];
#pragma unroll
        for (int f = 0; f < NFL; ++f) mw[f] = __uint_as_float(a.amax[f][(long long)blockIdx.y * 64 + tid]);
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
#pragma unroll
            for (int f = 0; f < NFL; ++f) mw[f] = fmaxf(mw[f], __shfl_xor(mw[f], o));
        const double nm = (double)a.dims * a.dims * a.zlen;
        double bound = 0.0;
#pragma unroll
        for (int f = 0; f < NFL; ++f) {
            const double am = (double)fmaxf(0.0f, mw[f]) * (double)a.cmax[f];
            bound = fmax(bound, 2.0 * nm * am * am);
        }
        if (tid == 0) {
            sE[0] = fix_exponent(bound * 1.01);
            sE[1] = fix_exponent(nm);
            if (blockIdx.x == 0) {
                a.escale[2 * blockIdx.y] = sE[0];
                a.escale[2 * blockIdx.y + 1] = sE[1];
            }
        }
    }
    for (int i = tid; i < a.zlen * NFL; i += blockDim.x) {
        int f = i / a.zlen, kz = i - f * a.zlen;
        corrz[i] = a.corr[f][kz];
    }
    for (int r = tid; r < ngrp; r += blockDim.x) {
        const int g = a.groups[item.x + r];
        grp[r] = g;
        for (int f = 0; f < NFL; ++f) rowc[r * NFL + f] = a.corr[f][g >> 16] * a.corr[f][g & 0xffff];
    }
    __syncthreads();
    const int Ep = sE[0], Eph = sE[1];

    const int mm = a.m * a.m;
    // 1D accumulator (axes 0/1: k_par = key): each run's sum in fixed point, added
    // up per lane in integers, so the result does not depend on which lane took which
    // run (nor on how the groups were cut into work items)
    unsigned long long p1lo[S];
    long long p1hi[S];
#pragma unroll
    for (int s = 0; s < S; ++s) {
        p1lo[s] = 0ull;
        p1hi[s] = 0;
    }

    // Lane runs start at flat index tid*kRun and advance by blockDim*kRun over the
    // item's groups x zpad (zpad is a multiple of kRun, so a run never crosses a group).
    const int step = blockDim.x * kRun;
    const int dr = step / a.zpad, dc = step - dr * a.zpad;
    int r = (tid * kRun) / a.zpad;
    int kz0 = tid * kRun - r * a.zpad;
    for (; r < ngrp; r += dr, kz0 += dc) {
        if (kz0 >= a.zpad) {
            kz0 -= a.zpad;
            ++r;
            if (r >= ngrp) break;
        }
        const int ka = grp[r] >> 16, kb = grp[r] & 0xffff;    // |kx|, |ky|
        const int kxy2 = ka * ka + kb * kb;
        // rows of the group: (ka, kb), (ka, -kb), (-ka, kb), (-ka, -kb); -ka (-kb) is a
        // row of its own unless it is 0 or the Nyquist index
        const bool hasx = ka != 0 && !(a.even && ka == a.m);
        const bool hasy = kb != 0 && !(a.even && kb == a.m);
        const unsigned rows = 1u | (hasy ? 2u : 0u) | (hasx ? 4u : 0u) | (hasx && hasy ? 8u : 0u);
        // of them, the independent ones in the kz = 0 and kz = m (even) planes
        // (Pk_library.pyx:324-327: kx < 0, and ky < 0 at the kx edges, are skipped)
        const unsigned prows = 1u | (hasy && hasx ? 2u : 0u);
        const int xn = hasx ? a.dims - ka : ka, yn = hasy ? a.dims - kb : kb;
        const long long fo = (long long)blockIdx.y * a.fstride + kz0;
        const long long ro[4] = {fo + (long long)(ka * a.dims + kb) * a.zs, fo + (long long)(ka * a.dims + yn) * a.zs,
                                 fo + (long long)(xn * a.dims + kb) * a.zs, fo + (long long)(xn * a.dims + yn) * a.zs};
        double c01[NFL];
#pragma unroll
        for (int f = 0; f < NFL; ++f) c01[f] = rowc[r * NFL + f];

        float2 v[NFL][4][kRun];
        if (a.wide) {
#pragma unroll
            for (int f = 0; f < NFL; ++f)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 *src = (const float4 *)(a.dk[f] + ro[q]);
                    const float4 x = src[0], y = src[1];
                    v[f][q][0] = make_float2(x.x, x.y);
                    v[f][q][1] = make_float2(x.z, x.w);
                    v[f][q][2] = make_float2(y.x, y.y);
                    v[f][q][3] = make_float2(y.z, y.w);
                }
        } else {
#pragma unroll
            for (int f = 0; f < NFL; ++f)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int s = 0; s < kRun; ++s)
                        v[f][q][s] = (kz0 + s < a.zlen) ? a.dk[f][ro[q] + s] : make_float2(0.f, 0.f);
        }

        int cur3 = -1, cur2 = -1;
        double r3[NA3], r2[S], p1[S];
#pragma unroll
        for (int i = 0; i < NA3; ++i) r3[i] = 0.0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
            r2[s] = 0.0;
            p1[s] = 0.0;
        }

        // |k|^2 and k_per^2 of the run's first mode; along the run kz grows by one,
        // so each square grows by 2kz-1 <= 2*isqrt+1 and each integer root by at
        // most one: one test per mode instead of a square root
        int k2 = kxy2 + kz0 * kz0;
        int kidx = isqrt_i(k2);
        int p2 = (AXIS == 0 ? kb * kb : ka * ka) + kz0 * kz0;
        int kpr = (AXIS == 2) ? key : isqrt_i(p2);
#pragma unroll
        for (int s = 0; s < kRun; ++s) {
            const int kz = kz0 + s;
            if (s > 0) {
                k2 += 2 * kz - 1;
                kidx += ((kidx + 1) * (kidx + 1) <= k2) ? 1 : 0;
                if (AXIS != 2) {
                    p2 += 2 * kz - 1;
                    kpr += ((kpr + 1) * (kpr + 1) <= p2) ? 1 : 0;
                }
            }
            if (kz >= a.zlen) continue;
            const unsigned mask = (kz == 0 || (a.even && kz == a.m)) ? prows : rows;
            const int kper = kpr;
            const int kpar = AXIS == 0 ? ka : AXIS == 1 ? kb : kz;
            // mu^2 = k_par^2 / k^2 in float (hardware reciprocal, within 2 ulp)
            const float mu2 = (k2 == 0) ? 0.0f : (float)(kpar * kpar) * __builtin_amdgcn_rcpf((float)k2);
            const float L2 = 1.5f * mu2 - 0.5f;
            const float L4 = (35.0f * mu2 * mu2 - 30.0f * mu2 + 3.0f) * 0.125f;

            float mf[NFL];
#pragma unroll
            for (int f = 0; f < NFL; ++f) mf[f] = (float)(c01[f] * corrz[f * a.zlen + kz]);
            double d2[S], ph2 = 0.0;
#pragma unroll
            for (int sp = 0; sp < S; ++sp) d2[sp] = 0.0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                // rows that are not there, or not independent, count as 0: their values are
                // masked, not multiplied by 0, since a caller's field may hold NaN or
                // infinities in them (the mask costs no more than the factor did)
                const unsigned on = (unsigned)__builtin_amdgcn_sbfe((int)mask, q, 1);   // all ones or 0
                double re[NFL], im[NFL];
                float xr0 = 0.0f, xi0 = 0.0f;
#pragma unroll
                for (int f = 0; f < NFL; ++f) {
                    const float xr = masked(v[f][q][s].x * mf[f], on);   // complex64 * float
                    const float xi = masked(v[f][q][s].y * mf[f], on);
                    re[f] = (double)xr;
                    im[f] = (double)xi;
                    if (f == 0) {
                        xr0 = xr;
                        xi0 = xi;
                    }
                }
                // the products of floats are exact in double
                d2[0] = fma(re[0], re[0], fma(im[0], im[0], d2[0]));
                if (NFL == 2) {
                    d2[1] = fma(re[1], re[1], fma(im[1], im[1], d2[1]));
                    d2[2] = fma(re[0], re[1], fma(im[0], im[1], d2[2]));
                }
                if (PHASE) ph2 += (double)phase_sq(xr0, xi0);
            }
            // 3D: merge equal bins in registers, flush on change
            if (kidx != cur3) {
                if (cur3 >= 0) {
#pragma unroll
                    for (int i = 0; i < NA3; ++i)
                        fix_add(alo, ahi, i * K1 + cur3, r3[i], (PHASE && i == NA3 - 1) ? Eph : Ep);
                }
                cur3 = kidx;
#pragma unroll
                for (int i = 0; i < NA3; ++i) r3[i] = 0.0;
            }
#pragma unroll
            for (int sp = 0; sp < S; ++sp) {
                r3[3 * sp + 0] += d2[sp];
                r3[3 * sp + 1] = fma(d2[sp], (double)L2, r3[3 * sp + 1]);
                r3[3 * sp + 2] = fma(d2[sp], (double)L4, r3[3 * sp + 2]);
            }
            if (PHASE) r3[NA3 - 1] += ph2;
            // 2D line: axes 0/1 index k_per (slowly varying), axis 2 index kz
            const int li = (AXIS == 2) ? kz : kper;
            if (AXIS == 2) {
#pragma unroll
                for (int sp = 0; sp < S; ++sp) fix_add(alo, ahi, a.off2 + li * S + sp, d2[sp], Ep);
            } else {
                if (li != cur2) {
                    if (cur2 >= 0) {
#pragma unroll
                        for (int sp = 0; sp < S; ++sp) fix_add(alo, ahi, a.off2 + cur2 * S + sp, r2[sp], Ep);
                    }
                    cur2 = li;
#pragma unroll
                    for (int sp = 0; sp < S; ++sp) r2[sp] = 0.0;
                }
#pragma unroll
                for (int sp = 0; sp < S; ++sp) r2[sp] += d2[sp];
            }
            // 1D: modes with k <= middle
            if (k2 <= mm) {
                if (AXIS == 2) {
#pragma unroll
                    for (int sp = 0; sp < S; ++sp) fix_add(alo, ahi, a.off1 + kz * S + sp, d2[sp], Ep);
                } else {
#pragma unroll
                    for (int sp = 0; sp < S; ++sp) p1[sp] += d2[sp];
                }
            }
        }
        if (cur3 >= 0) {
#pragma unroll
            for (int i = 0; i < NA3; ++i)
                fix_add(alo, ahi, i * K1 + cur3, r3[i], (PHASE && i == NA3 - 1) ? Eph : Ep);
        }
        if (AXIS != 2 && cur2 >= 0) {
#pragma unroll
            for (int sp = 0; sp < S; ++sp) fix_add(alo, ahi, a.off2 + cur2 * S + sp, r2[sp], Ep);
        }
        if (AXIS != 2) {
#pragma unroll
            for (int sp = 0; sp < S; ++sp) {
                if (p1[sp] == 0.0) continue;
                unsigned long long lo;
                int hi;
                fix_split(p1[sp], Ep, lo, hi);
                fix_acc(p1lo[sp], p1hi[sp], lo, hi);
            }
        }
    }
    if (AXIS != 2) {
#pragma unroll
        for (int sp = 0; sp < S; ++sp) {
            // exact integer sum over the wave, then one addition per wave
            unsigned long long lo = p1lo[sp];
            long long hi = p1hi[sp];
            for (int off = 32; off > 0; off >>= 1) {
                const unsigned long long olo = (unsigned long long)__shfl_xor((long long)lo, off);
                const long long ohi = __shfl_xor(hi, off);
                fix_acc(lo, hi, olo, ohi);
            }
            if ((tid & 63) == 0) fix_add_parts(alo, ahi, a.off1 + sp, lo, (int)hi);
        }
    }
    __syncthreads();
    const long long ob = ((long long)blockIdx.y * a.nitems + blockIdx.x) * a.P;
    unsigned long long *olo = a.plo + ob;
    int *ohi = a.phi + ob;
    for (int i = tid; i < n3; i += blockDim.x) {
        const int j = (i % NA3) * K1 + i / NA3;
        olo[i] = alo[j];
        ohi[i] = ahi[j];
    }
    for (int i = n3 + tid; i < a.P; i += blockDim.x) {
        olo[i] = alo[i];
        ohi[i] = ahi[i];
    }
}

// Sum the item partials (exact integer sums, so the order does not matter) and
// convert each bin to double with its realisation's scale.  Output layout per
// realisation: out3[(kmax+1)*NA3], out2[nb2*S] (reference 2D index), out1[(m+1)*S].
struct ReduceArgs {
    const unsigned long long *plo;
    const int *phi;
    const int *key_items;
    const int *escale;
    const double *n2;        // mode counts of the 2D bins
    double fact;             // (BoxSize / dims^2)^3
    double *out3, *out2, *out1;
    int nitems, nkeys, n3, na3, L2, L1, S, P, off2, off1, axis, kmax_par, nreal;
    long long nb2, n1;       // out2 / out1 elements per realisation (nb2*S, (m+1)*S)
};

// All reductions of a binning launch in one launch of kRedBlock threads, by block range:
//  * g3 blocks: columns every item contributes to (the 3D bins; the 1D line for axis
//    2), 16 columns x 64 slices of the items per block, one realisation per xb blocks;
//  * g2 blocks: the 2D line, each bin the sum of its key's items (blocks of 1024 bins
//    for axis 2, whose output order is the partials' order; tiles of 32 keys x about 32
//    line entries for axes 0 and 1, turned round in LDS, since k_par = key runs fastest
//    in the output);
//  * g1 blocks: axes 0/1, the 1D bins (k_par = key).
// The outputs go straight into the pinned host buffer the caller reads after the
// stream, in runs of whole cache lines; the 2D bins, the bulk of them, as the spectra
// themselves (sum * fact / modes: on the host their divisions took the GPU's time of
// 10 % of an XPk of two 256^3 fields), the others as sums.  Latency-bound: the chunk sums, their sum, the
// 1D line's own pair of launches (axis 2) and the download used to take 36 us at 64^3
// and 46 us at 512^3 for microseconds of data movement; now 4 and 28 us, and Pk of a 64^3
// field went from 98 to 70 us, of a 512^3 field from 1084 to 1057 us.
constexpr int kRedBlock = 1024;
constexpr int kRedCols = 16;                       // columns per block (128 B of low words)
constexpr int kRedSlices = kRedBlock / kRedCols;

// Line columns per tile of the 2D transpose: whole line entries of S spectra.
__host__ __device__ __forceinline__ int red_tile_cols(int S) { return 32 / S * S; }

__device__ __forceinline__ void reduce_key_items(const ReduceArgs &a, int key, int col, long long base,
                                                 unsigned long long &slo, long long &shi) {
    slo = 0;
    shi = 0;
    const int i1 = a.key_items[key + 1];
#pragma unroll 4
    for (int it = a.key_items[key]; it < i1; ++it) {
        const long long j = base + (long long)it * a.P + col;
        fix_acc(slo, shi, a.plo[j], a.phi[j]);
    }
}

__global__ void __launch_bounds__(kRedBlock)
pk_reduce_kernel(ReduceArgs a, int g3, int g2) {
    __shared__ unsigned long long slo_s[kRedBlock / 64][kRedCols];
    __shared__ long long shi_s[kRedBlock / 64][kRedCols];
    __shared__ double tile[32][33];
    const int b = blockIdx.x, t = threadIdx.x;
    if (b < g3) {
        const int xb = g3 / a.nreal, r = b / xb;
        const int ncol = a.n3 + (a.axis == 2 ? a.L1 * a.S : 0);
        const int c = (b - r * xb) * kRedCols + (t & (kRedCols - 1));
        unsigned long long lo = 0;
        long long hi = 0;
        if (c < ncol) {
            const long long base = (long long)r * a.nitems * a.P + (c < a.n3 ? c : a.off1 + c - a.n3);
#pragma unroll 4
            for (int it = t / kRedCols; it < a.nitems; it += kRedSlices) {
                const long long j = base + (long long)it * a.P;
                fix_acc(lo, hi, a.plo[j], a.phi[j]);
            }
        }
#pragma unroll
        for (int o = kRedCols; o < 64; o <<= 1) {
            const unsigned long long olo = (unsigned long long)__shfl_xor((long long)lo, o);
            const long long ohi = __shfl_xor(hi, o);
            fix_acc(lo, hi, olo, ohi);
        }
        if ((t & 63) < kRedCols) {
            slo_s[t >> 6][t & 63] = lo;
            shi_s[t >> 6][t & 63] = hi;
        }
        __syncthreads();
        if (t >= kRedCols || c >= ncol) return;
        for (int w = 1; w < kRedBlock / 64; ++w) fix_acc(lo, hi, slo_s[w][t], shi_s[w][t]);
        const int E = a.escale[2 * r + ((c < a.n3 && a.na3 > 0 && c % a.na3 == a.na3 - 1) ? 1 : 0)];
        const double v = fix_value(lo, hi, E);
        if (c < a.n3) a.out3[(long long)r * a.n3 + c] = v;
        else a.out1[(long long)r * a.n1 + (c - a.n3)] = v;
    } else if (b < g3 + g2) {
        const int xb = g2 / a.nreal, bb = b - g3, r = bb / xb, x = bb - r * xb;
        const long long base = (long long)r * a.nitems * a.P;
        const int E = a.escale[2 * r];
        double *out2 = a.out2 + (long long)r * a.nb2;
        const int ncol = a.L2 * a.S;
        unsigned long long lo;
        long long hi;
        if (a.axis == 2) {
            const long long i = (long long)x * kRedBlock + t;     // (key, line entry, spectrum)
            if (i >= (long long)a.nkeys * ncol) return;
            reduce_key_items(a, (int)(i / ncol), a.off2 + (int)(i % ncol), base, lo, hi);
            out2[i] = fix_value(lo, hi, E) * a.fact / a.n2[i / a.S];   // (kmax_par+1) == L2
            return;
        }
        const int tc = red_tile_cols(a.S), nct = (ncol + tc - 1) / tc;
        const int c0 = x % nct * tc, k0 = x / nct * 32;
        const int key = k0 + (t >> 5), c = c0 + (t & 31);
        if (key < a.nkeys && (t & 31) < tc && c < ncol) {
            reduce_key_items(a, key, a.off2 + c, base, lo, hi);
            tile[t >> 5][t & 31] = fix_value(lo, hi, E);
        }
        __syncthreads();
        // line entry l, keys k0.. and spectra: consecutive in the output
        if (t >= 32 * tc) return;
        const int l = t / (32 * a.S), rest = t - l * 32 * a.S, kl = rest / a.S, sp = rest - kl * a.S;
        const int cl = l * a.S + sp;
        if (k0 + kl < a.nkeys && c0 + cl < ncol) {
            const long long bin = (long long)(a.kmax_par + 1) * (c0 / a.S + l) + k0 + kl;
            out2[bin * a.S + sp] = tile[kl][cl] * a.fact / a.n2[bin];
        }
    } else {
        const int bb = b - g3 - g2, xb = (a.nkeys * a.S + kRedBlock - 1) / kRedBlock, r = bb / xb;
        const int i = (bb - r * xb) * kRedBlock + t;
        if (i >= a.nkeys * a.S) return;
        unsigned long long lo;
        long long hi;
        reduce_key_items(a, i / a.S, a.off1 + i % a.S, (long long)r * a.nitems * a.P, lo, hi);
        a.out1[(long long)r * a.n1 + i] = fix_value(lo, hi, a.escale[2 * r]);
    }
}

// FFT prologue: out = (in / scale) - shift in float32 (the reference caller's
// "delta /= mean; delta -= 1.0", Pk_snapshot.py:88), or a plain copy.  blockIdx.y
// selects one of several contiguous cubes of n elements, each with its own
// scale/shift when the device arrays are given.
__global__ void prologue_kernel(const float *__restrict__ in, float *__restrict__ out,
                                long long n, const float *__restrict__ scales,
                                const float *__restrict__ shifts, float scale, float shift,
                                int apply, int sstride = 1) {
    const long long cube = blockIdx.y;
    in += cube * n;
    out += cube * n;
    if (scales) scale = scales[cube * sstride];
    if (shifts) shift = shifts[cube * sstride];
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        float x = in[i];
        if (apply) {
            x = x / scale;
            x = x - shift;
        }
        out[i] = x;
    }
}

__global__ void rsd_kernel(float *__restrict__ pos, const float *__restrict__ vel, long long n,
                           float BoxSize, float factor, int axis) {
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        pos[3 * i + axis] = rsd_shift(pos[3 * i + axis], vel[3 * i + axis], factor, BoxSize);
    }
}

template <typename K>
int set_lds(K kernel, size_t bytes) {
    if (bytes > 64 * 1024)
        PYL_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                    (int)bytes));
    return PYL_OK;
}

// Run the binning of NFL fields (device half-complex arrays) -> reduced sums
// appended into host arrays of spectra [s_off, s_off+S).
struct HostAcc {
    int S_total;
    std::vector<double> P3;     // [(kmax+1)*3*S_total] l-major per bin: (bin*3+l)*S_total+s
    std::vector<double> phase;  // [kmax+1]
    std::vector<double> P2;     // [nb2*S_total], normalised (pk_reduce_kernel)
    std::vector<double> P1;     // [(m+1)*S_total]
    // the 2D and 1D sums to finalize: P2/P1, or the pinned download itself when one
    // launch produced every spectrum in output order (no copy of the 2D bins)
    const double *P2v = nullptr, *P1v = nullptr;
};

using AccsPtr = std::shared_ptr<std::vector<HostAcc>>;

// Copies the downloaded sums of one binning launch (h3 | h2 | h1, per realisation)
// into the spectrum columns spec_out of the host accumulators.
template <int NFL, bool PHASE>
void bin_host_part(const PkDims &p, const double *hp, size_t out3, size_t out2, size_t out1,
                   int nreal, const int *spec_out, std::vector<HostAcc> &accs) {
    constexpr int S = Spec<NFL>::S;
    constexpr int NA3 = 3 * S + (PHASE ? 1 : 0);
    const double *h3 = hp, *h2 = h3 + out3 * nreal, *h1 = h2 + out2 * nreal;
    for (int rr = 0; rr < nreal; ++rr) {
        HostAcc &acc = accs[rr];
        const double *H3 = h3 + out3 * rr, *H2 = h2 + out2 * rr, *H1 = h1 + out1 * rr;
        const int ST = acc.S_total;
        for (int b = 0; b <= p.kmax; ++b) {
            for (int sp = 0; sp < S; ++sp) {
                int so = spec_out[sp];
                if (so < 0) continue;
                for (int l = 0; l < 3; ++l)
                    acc.P3[((size_t)b * 3 + l) * ST + so] = H3[(size_t)b * NA3 + 3 * sp + l];
            }
            if (PHASE) acc.phase[b] = H3[(size_t)b * NA3 + NA3 - 1];
        }
        bool identity = ST == S;
        for (int sp = 0; sp < S; ++sp) identity = identity && spec_out[sp] == sp;
        if (identity) {
            // the only launch of this call: finalize straight from the pinned buffer
            // (valid until the next download into it)
            acc.P2v = H2;
            acc.P1v = H1;
            continue;
        }
        for (long long i = 0; i < p.nb2; ++i)
            for (int sp = 0; sp < S; ++sp)
                if (spec_out[sp] >= 0) acc.P2[(size_t)i * ST + spec_out[sp]] = H2[(size_t)i * S + sp];
        for (int i = 0; i <= p.m; ++i)
            for (int sp = 0; sp < S; ++sp)
                if (spec_out[sp] >= 0) acc.P1[(size_t)i * ST + spec_out[sp]] = H1[(size_t)i * S + sp];
        acc.P2v = acc.P2.data();
        acc.P1v = acc.P1.data();
    }
}

template <int AXIS, int NFL, bool PHASE>
int launch_bin(Ctx *c, const BinPlan *bp, const PkDims &p, const float2 *const *dk,
               long long fstride, long long zs, int nreal, const double *const *corr,
               const float *cmax, const unsigned *const *amax, const AccsPtr &accs,
               const int *spec_out, double fact, const std::function<int()> &meanwhile) {
    constexpr int S = Spec<NFL>::S;
    constexpr int NA3 = 3 * S + (PHASE ? 1 : 0);
    const int L2 = (AXIS == 2) ? p.zlen : p.kmax_per + 1;
    const int L1 = (AXIS == 2) ? p.zlen : 1;
    const int n3 = (p.kmax + 1) * NA3;
    const int P = n3 + (L2 + L1) * S;
    const int off2 = n3, off1 = n3 + L2 * S;
    const int gmax = bp->G;
    // LDS: P low words (8 B) and P high words (4 B, padded to an even count), the
    // kz corrections, the group corrections and the group table
    size_t lds = sizeof(unsigned long long) * (size_t)P + sizeof(int) * (size_t)((P + 1) & ~1) +
                 sizeof(double) * ((size_t)p.zlen * NFL + (size_t)gmax * NFL) +
                 sizeof(int) * (size_t)gmax;
    PYL_CHECK(lds <= 160 * 1024, PYL_EINVAL, "grid too large for the binning kernel (%zu B LDS)", lds);
    // scratch: partials (low words | high words), scales
    const size_t part_elems = (size_t)bp->nitems * P * nreal;
    const size_t out3 = (size_t)n3, out2 = (size_t)p.nb2 * S, out1 = (size_t)(p.m + 1) * S;
    const size_t phi_bytes = (sizeof(int) * part_elems + 7) & ~(size_t)7;
    PYL_TRY(ensure(c, BUF_BINS, sizeof(unsigned long long) * part_elems + phi_bytes +
                                    sizeof(int) * 2 * (size_t)nreal));
    unsigned long long *plo = (unsigned long long *)c->bufs[BUF_BINS].ptr;
    int *phi = (int *)(plo + part_elems);
    int *escale = (int *)((char *)phi + phi_bytes);
    // the reduced outputs (3D | 2D | 1D) are written into pinned memory by the reduction
    const size_t nout = (out3 + out2 + out1) * nreal;
    void *hp = nullptr;
    if (c->capturing) {
        // a pinned buffer of the graph's own; the host part runs after each replay
        PYL_HIP(hipHostMalloc(&hp, sizeof(double) * nout, hipHostMallocDefault));
        c->cap_host.push_back(hp);
    } else {
        PYL_TRY(pinned(c, c->pin_down, sizeof(double) * nout, &hp));
    }
    double *h3 = (double *)hp, *h2 = h3 + out3 * nreal, *h1 = h2 + out2 * nreal;

    BinArgs a{};
    for (int f = 0; f < NFL; ++f) {
        a.dk[f] = dk[f];
        a.corr[f] = corr[f];
        a.cmax[f] = cmax[f];
        a.amax[f] = amax[f];
    }
    a.escale = escale;
    a.nreal = nreal;
    a.groups = bp->d_groups;
    a.items = bp->d_items;
    a.plo = plo;
    a.phi = phi;
    a.fstride = fstride;
    a.zs = zs;
    a.nitems = bp->nitems;
    a.dims = p.dims; a.m = p.m; a.zlen = p.zlen; a.zpad = p.zpad; a.even = p.even;
    a.kmax = p.kmax; a.L2 = L2; a.L1 = L1; a.P = P; a.off2 = off2; a.off1 = off1; a.gmax = gmax;
    // 16-byte loads of a run's four modes: rows padded to zpad (the padding is read and
    // not used) and 16-byte aligned, as the own passes' buffer has them
    a.wide = zs >= p.zpad && zs % 2 == 0 && fstride % 2 == 0;
    for (int f = 0; f < NFL; ++f) a.wide = a.wide && ((uintptr_t)dk[f] & 15) == 0;
    auto kern = pk_bin_kernel<AXIS, NFL, PHASE>;
    PYL_TRY(set_lds(kern, lds));
    PYL_TRY(stage_begin(c, PYL_STAGE_PK_BIN));
    kern<<<dim3(bp->nitems, nreal), kBinBlock, lds, c->stream>>>(a);
    PYL_HIP(hipGetLastError());
    ReduceArgs r{};
    r.plo = plo; r.phi = phi; r.escale = escale;
    r.n2 = bp->d_n2; r.fact = fact;
    r.key_items = bp->d_key_items; r.out3 = h3; r.out2 = h2; r.out1 = h1;
    r.nitems = bp->nitems; r.nkeys = bp->nkeys; r.n3 = n3; r.na3 = PHASE ? NA3 : 0;
    r.L2 = L2; r.L1 = L1; r.S = S; r.P = P; r.off2 = off2; r.off1 = off1; r.axis = AXIS;
    r.kmax_par = p.kmax_par; r.nb2 = (long long)out2; r.n1 = (long long)out1; r.nreal = nreal;
    const long long g3 = (long long)ceil_div(n3 + (AXIS == 2 ? L1 * S : 0), kRedCols) * nreal;
    const long long ncol2 = (long long)L2 * S;
    const long long g2 = (AXIS == 2 ? (bp->nkeys * ncol2 + kRedBlock - 1) / kRedBlock
                                    : (long long)ceil_div((int)ncol2, red_tile_cols(S)) * ceil_div(bp->nkeys, 32)) *
                         nreal;
    const long long g1 = AXIS == 2 ? 0 : (long long)ceil_div(bp->nkeys * S, kRedBlock) * nreal;
    PYL_CHECK(g3 + g2 + g1 < (1ll << 31), PYL_EINVAL, "binning reduction too large");
    pk_reduce_kernel<<<(unsigned)(g3 + g2 + g1), kRedBlock, 0, c->stream>>>(r, (int)g3, (int)g2);
    PYL_HIP(hipGetLastError());
    PYL_TRY(stage_end(c, PYL_STAGE_PK_BIN));
    const int rc = meanwhile();               // host work beside the transform and the binning
    if (c->capturing) {
        PYL_TRY(rc);
        std::array<int, Spec<NFL>::S> so;
        for (int sp = 0; sp < Spec<NFL>::S; ++sp) so[sp] = spec_out[sp];
        const double *h = (const double *)hp;
        AccsPtr keep = accs;
        c->deferred.push_back([p, h, out3, out2, out1, nreal, so, keep]() {
            bin_host_part<NFL, PHASE>(p, h, out3, out2, out1, nreal, so.data(), *keep);
            return PYL_OK;
        });
        return PYL_OK;
    }
    PYL_HIP(hipStreamSynchronize(c->stream));
    PYL_TRY(rc);
    bin_host_part<NFL, PHASE>(p, (const double *)hp, out3, out2, out1, nreal, spec_out, *accs);
    return PYL_OK;
}

template <int NFL, bool PHASE>
int launch_bin_axis(Ctx *c, int axis, const BinPlan *bp, const PkDims &p, const float2 *const *dk,
                    long long fstride, long long zs, int nreal, const double *const *corr,
                    const float *cmax, const unsigned *const *amax, const AccsPtr &accs,
                    const int *spec_out, double fact, const std::function<int()> &meanwhile) {
    if (axis == 0)
        return launch_bin<0, NFL, PHASE>(c, bp, p, dk, fstride, zs, nreal, corr, cmax, amax, accs, spec_out, fact,
                                         meanwhile);
    if (axis == 1)
        return launch_bin<1, NFL, PHASE>(c, bp, p, dk, fstride, zs, nreal, corr, cmax, amax, accs, spec_out, fact,
                                         meanwhile);
    return launch_bin<2, NFL, PHASE>(c, bp, p, dk, fstride, zs, nreal, corr, cmax, amax, accs, spec_out, fact,
                                     meanwhile);
}

// Normalisation, Pk_library.pyx:384-418 (and :735-791 for XPk).
double pk_fact(const PkDims &p, double BoxSize) {
    return std::pow(BoxSize / ((double)p.dims * (double)p.dims), 3.0);
}

// The outputs that depend only on the mode plan (k, bin centres, mode counts):
// filled while the GPU still transforms and bins.
int finalize_modes(const ModePlan *mp, const PkDims &p, double BoxSize, pyl_pk_out *out) {
    const double kF = 2.0 * M_PI / BoxSize;
    double sumN = 0.0;
    for (double v : mp->N3D) sumN += v;
    const long long own = (p.dims % 2 == 1) ? 1 : 8;
    const long long d3 = (long long)p.dims * p.dims * p.dims;
    const long long expected = (d3 - own) / 2 + own;
    PYL_CHECK((long long)sumN == expected, PYL_EMODES,
              "WARNING: Not all modes counted (counted %lld, expected %lld)", (long long)sumN,
              expected);
    for (int i = 1; i <= p.m; ++i) {
        if (out->k1D) out->k1D[i - 1] = (mp->k1D[i] / mp->N1D[i]) * kF;
        if (out->Nmodes1D) out->Nmodes1D[i - 1] = mp->N1D[i];
    }
    // bin centres (kpar fastest: contiguous writes)
    for (int kper = 0; kper <= p.kmax_per; ++kper)
        for (int kpar = 0; kpar <= p.kmax_par; ++kpar) {
            const long long idx = (long long)(p.kmax_par + 1) * kper + kpar;
            if (out->kpar) out->kpar[idx] = 0.5 * (kpar + kpar + 1) * kF;
            if (out->kper) out->kper[idx] = 0.5 * (kper + kper + 1) * kF;
        }
    if (out->Nmodes2D) std::memcpy(out->Nmodes2D, mp->N2D.data(), sizeof(double) * p.nb2);
    for (int b = 1; b <= p.kmax; ++b) {
        if (out->k3D) out->k3D[b - 1] = (mp->k3D[b] / mp->N3D[b]) * kF;
        if (out->Nmodes3D) out->Nmodes3D[b - 1] = mp->N3D[b];
    }
    return PYL_OK;
}

// The spectra (Pk_library.pyx:384-418): 1D drops the DC bin, 2D keeps every bin
// (normalised where they were reduced), 3D drops the DC bin with the multipoles times (2l+1).
void finalize_values(const ModePlan *mp, const PkDims &p, double BoxSize, const HostAcc &acc,
                     bool want_phase, pyl_pk_out *out) {
    const int S = acc.S_total;
    const double kF = 2.0 * M_PI / BoxSize;
    const double kN = p.m * kF;
    const double fact = pk_fact(p, BoxSize);
    if (out->Pk1D)
        for (int i = 1; i <= p.m; ++i) {
            const double N = mp->N1D[i];
            const double k1 = (mp->k1D[i] / N) * kF;
            const double kmaxper = std::sqrt(kN * kN - k1 * k1);
            for (int s = 0; s < S; ++s) {
                double v = acc.P1v[(size_t)i * S + s] * fact;
                v = v * (M_PI * (kmaxper * kmaxper) / N) / ((2.0 * M_PI) * (2.0 * M_PI));
                out->Pk1D[(size_t)(i - 1) * S + s] = v;
            }
        }
    if (out->Pk2D) std::memcpy(out->Pk2D, acc.P2v, sizeof(double) * (size_t)p.nb2 * S);
    for (int b = 1; b <= p.kmax; ++b) {
        const double N = mp->N3D[b];
        if (out->Pk3D)
            for (int s = 0; s < S; ++s) {
                const size_t o = (size_t)(b - 1) * 3 * S;
                out->Pk3D[o + 0 * S + s] = (acc.P3[((size_t)b * 3 + 0) * S + s] / N) * fact;
                out->Pk3D[o + 1 * S + s] = (acc.P3[((size_t)b * 3 + 1) * S + s] * 5.0 / N) * fact;
                out->Pk3D[o + 2 * S + s] = (acc.P3[((size_t)b * 3 + 2) * S + s] * 9.0 / N) * fact;
            }
        if (want_phase && out->Pkphase) out->Pkphase[b - 1] = (acc.phase[b] / N) * fact;
    }
}

}  // namespace

__global__ void zero_u32_kernel(unsigned *__restrict__ p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

// 64 words per cube for the transforms' largest |Re|, |Im|, zeroed (a fill kernel, not
// a memset node, so that a captured call clears them on every replay) unless the own
// row pass clears them (own: one launch less).
int pk_amax_words(Ctx *c, int ncube, bool own, unsigned **out) {
    const int n = 64 * ncube;
    PYL_TRY(ensure(c, BUF_PK_AMAX, sizeof(unsigned) * (size_t)n));
    unsigned *a = (unsigned *)c->bufs[BUF_PK_AMAX].ptr;
    if (!own) {
        zero_u32_kernel<<<ceil_div(n, 256), 256, 0, c->stream>>>(a, n);
        PYL_HIP(hipGetLastError());
    }
    *out = a;
    return PYL_OK;
}

int fft_device(Ctx *c, float *in, float2 *out, int dims, int batch, long long zs = 0,
               unsigned *amax = nullptr) {
    PYL_TRY(stage_begin(c, PYL_STAGE_PK_FFT));
    PYL_TRY(fft_r2c_3d(c, in, out, dims, batch, zs, amax));
    PYL_TRY(stage_end(c, PYL_STAGE_PK_FFT));
    return PYL_OK;
}

// Own FFT passes of nfields fields of nreal cubes each (n floats per cube).  Device
// arrays are read in place; host arrays, and device arrays that are not 8-byte aligned
// (the row pass reads pairs), are brought into BUF_FFT_IN first.
int fft_fields_device(Ctx *c, const float *const *deltas, FieldSrc fs, bool dev, float2 *out, int dims,
                      long long zs, unsigned *amax) {
    const size_t cube = (size_t)dims * dims * dims * fs.nreal;
    std::vector<const float *> src(fs.nfields);
    int ncopy = 0;
    for (int f = 0; f < fs.nfields; ++f)
        if (!dev || ((uintptr_t)deltas[f] & 7)) ++ncopy;
    if (ncopy) PYL_TRY(ensure(c, BUF_FFT_IN, cube * ncopy * sizeof(float)));
    float *dst = (float *)c->bufs[BUF_FFT_IN].ptr;
    PYL_TRY(stage_begin(c, PYL_STAGE_PK_PREP));
    for (int f = 0; f < fs.nfields; ++f) {
        src[f] = deltas[f];
        if (dev && ((uintptr_t)deltas[f] & 7) == 0) continue;
        PYL_HIP(hipMemcpyAsync(dst, deltas[f], cube * sizeof(float),
                               dev ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, c->stream));
        src[f] = dst;
        dst += cube;
    }
    PYL_TRY(stage_end(c, PYL_STAGE_PK_PREP));
    fs.in = src.data();
    PYL_TRY(stage_begin(c, PYL_STAGE_PK_FFT));
    PYL_TRY(fft_r2c_fields(c, fs, out, dims, zs, amax));
    PYL_TRY(stage_end(c, PYL_STAGE_PK_FFT));
    return PYL_OK;
}

// Binning of F device half-complex fields of nreal realisations -> finalized outputs.
// Field f of realisation r is dk[f] + r*fstride.
// Device-resident MAS correction table for (dims, p), built once per device with the
// host's libm; cmax: the largest product of three axis corrections, rounded up.
int get_mas_tab(Ctx *c, int dims, int p, const double **out, float *cmax) {
    SharedTables &st = shared_tables();
    std::lock_guard<std::mutex> lk(st.mu);
    const auto key = std::make_tuple(c->device, dims, p);
    auto it = st.mas.find(key);
    if (it == st.mas.end()) {
        PYL_CHECK(!c->capturing, PYL_EINVAL, "MAS table created while a graph is captured");
        std::vector<double> tab(dims);
        mas_table(dims, p, tab.data());
        void *d = nullptr;
        PYL_HIP(hipMalloc(&d, sizeof(double) * dims));
        hipError_t e = hipMemcpy(d, tab.data(), sizeof(double) * dims, hipMemcpyHostToDevice);
        if (e != hipSuccess) {
            (void)hipFree(d);
            set_error("MAS table upload failed: %s", hipGetErrorString(e));
            return PYL_EHIP;
        }
        double mx = 1.0;
        for (double v : tab) mx = std::max(mx, v);
        it = st.mas.emplace(key, std::make_pair(d, (float)(mx * mx * mx * 1.001))).first;
    }
    *out = (const double *)it->second.first;
    *cmax = it->second.second;
    return PYL_OK;
}

// Rows of each field are zs elements apart (zs = 0: dense, dims/2+1).  amax: per
// field, realisation r's 64 words of the transform's largest |Re|, |Im| at r*64
// (fft_r2c_3d, complex_absmax).
int pk_bin_device(Ctx *c, const float2 *const *dk, long long fstride, long long zs, int nreal, int F,
                  const int *mas, int dims, double BoxSize, int axis, int flags, pyl_pk_out *outs,
                  const unsigned *const *amax) {
    if (zs <= 0) zs = dims / 2 + 1;
    const PkDims p = pk_dims(dims);
    const ModePlan *mp = get_mode_plan(c, dims, axis);
    BinPlan *bp = nullptr;
    PYL_TRY(get_bin_plan(c, dims, axis, nreal, &bp));
    std::vector<const double *> tab(F);
    std::vector<float> cmax(F);
    for (int f = 0; f < F; ++f) {
        PYL_TRY(get_mas_tab(c, dims, mas[f], &tab[f], &cmax[f]));
    }
    // the mode-plan outputs are written while the GPU works, after the first launch
    bool modes_done = false;
    const std::function<int()> meanwhile = [&]() {
        for (int r = 0; r < nreal && !modes_done; ++r) PYL_TRY(finalize_modes(mp, p, BoxSize, &outs[r]));
        modes_done = true;
        return (int)PYL_OK;
    };
    const double fact = pk_fact(p, BoxSize);
    const int S = F + F * (F - 1) / 2;
    // host accumulators reused across calls on this thread (no fresh pages per call);
    // a captured call keeps its own, used by the host steps of every replay
    static thread_local AccsPtr tl_accs;
    AccsPtr accs_p;
    if (c->capturing) {
        accs_p = std::make_shared<std::vector<HostAcc>>();
    } else {
        if (!tl_accs) tl_accs = std::make_shared<std::vector<HostAcc>>();
        accs_p = tl_accs;
    }
    std::vector<HostAcc> &accs = *accs_p;
    accs.resize(nreal);
    for (auto &acc : accs) {      // every column is written by exactly one launch below
        acc.S_total = S;
        acc.P3.resize((size_t)(p.kmax + 1) * 3 * S);
        acc.phase.assign(p.kmax + 1, 0.0);
        if (F > 2) {              // one launch: the spectra are finalized where it put them
            acc.P2.resize((size_t)p.nb2 * S);
            acc.P1.resize((size_t)(p.m + 1) * S);
        }
    }
    const bool phase = (F == 1) && !(flags & PYL_PK_NO_PHASE);
    if (F == 1) {
        const float2 *f0[1] = {dk[0]};
        const double *c0[1] = {tab[0]};
        const float m0[1] = {cmax[0]};
        const unsigned *a0[1] = {amax[0]};
        int so[1] = {0};
        if (phase)
            PYL_TRY((launch_bin_axis<1, true>(c, axis, bp, p, f0, fstride, zs, nreal, c0, m0, a0, accs_p, so,
                                              fact, meanwhile)));
        else
            PYL_TRY((launch_bin_axis<1, false>(c, axis, bp, p, f0, fstride, zs, nreal, c0, m0, a0, accs_p, so,
                                               fact, meanwhile)));
    } else {
        // pairs i<j in lexicographic order; each launch yields auto i, auto j, cross ij
        std::vector<bool> have(F, false);
        int xi = 0;
        for (int i = 0; i < F; ++i)
            for (int j = i + 1; j < F; ++j, ++xi) {
                const float2 *fp[2] = {dk[i], dk[j]};
                const double *cp[2] = {tab[i], tab[j]};
                const float mp2[2] = {cmax[i], cmax[j]};
                const unsigned *ap[2] = {amax[i], amax[j]};
                int so[3] = {have[i] ? -1 : i, have[j] ? -1 : j, F + xi};
                have[i] = have[j] = true;
                PYL_TRY((launch_bin_axis<2, false>(c, axis, bp, p, fp, fstride, zs, nreal, cp, mp2, ap,
                                                   accs_p, so, fact, meanwhile)));
            }
    }
    if (c->capturing) {
        // the caller's result structs point at host arrays that outlive the graph
        std::vector<pyl_pk_out> o(outs, outs + nreal);
        c->deferred.push_back([mp, p, BoxSize, accs_p, phase, o, nreal]() mutable {
            for (int r = 0; r < nreal; ++r) finalize_values(mp, p, BoxSize, (*accs_p)[r], phase, &o[r]);
            return PYL_OK;
        });
        return PYL_OK;
    }
    for (int r = 0; r < nreal; ++r) finalize_values(mp, p, BoxSize, accs[r], phase, &outs[r]);
    if (nreal > 16) {                            // do not keep large batch accumulators
        accs.clear();
        accs.shrink_to_fit();
    }
    return PYL_OK;
}

}  // namespace pyl

using namespace pyl;

extern "C" {

double pyl_mas_correction(double x, int p) {
    return (x == 0.0) ? 1.0 : std::pow(x / std::sin(x), (double)p);
}

int pyl_pk_get_sizes(int dims, int nfields, pyl_pk_sizes *out) {
    PYL_CHECK(out && dims >= 2 && nfields >= 1, PYL_EINVAL, "bad arguments");
    PkDims p = pk_dims(dims);
    out->n1d = p.m;
    out->n2d = p.nb2;
    out->n3d = p.kmax;
    out->nspectra = nfields + nfields * (nfields - 1) / 2;
    return PYL_OK;
}

int pyl_mode_counts(int dims, int axis, double *N1D, double *N2D, double *N3D, double *k1Dsum,
                    double *k3Dsum) {
    PYL_CHECK(dims >= 2 && axis >= 0 && axis <= 2, PYL_EINVAL, "bad dims/axis");
    ModePlan mp;
    compute_mode_plan(dims, axis, &mp);
    if (N1D) std::copy(mp.N1D.begin(), mp.N1D.end(), N1D);
    if (N2D) std::copy(mp.N2D.begin(), mp.N2D.end(), N2D);
    if (N3D) std::copy(mp.N3D.begin(), mp.N3D.end(), N3D);
    if (k1Dsum) std::copy(mp.k1D.begin(), mp.k1D.end(), k1Dsum);
    if (k3Dsum) std::copy(mp.k3D.begin(), mp.k3D.end(), k3Dsum);
    return PYL_OK;
}

int pyl_fft_r2c(pyl_ctx *ctx, const float *delta, float *delta_k, int dims, int flags) {
    TraceRange trace_("pyl_fft_r2c");
    PYL_CHECK(ctx && delta && delta_k && dims >= 2, PYL_EINVAL, "bad arguments");
    Ctx *c = &ctx->c;
    PYL_HIP(hipSetDevice(c->device));
    reset_stages(c);
    const long long n = (long long)dims * dims * dims;
    const long long nk = (long long)dims * dims * (dims / 2 + 1);
    // the own passes read a device input in place, unless it overlaps the output
    const bool apart = (const char *)(delta + n) <= (const char *)delta_k ||
                       (const char *)((const float2 *)delta_k + nk) <= (const char *)delta;
    if ((flags & PYL_PTR_DEVICE) && fft_own_size(dims) && apart) {
        FieldSrc fs;
        PYL_TRY(fft_fields_device(c, &delta, fs, true, (float2 *)delta_k, dims, 0, nullptr));
        return finish(c, flags);
    }
    PYL_TRY(ensure(c, BUF_FFT_IN, (size_t)n * sizeof(float)));
    float *in = (float *)c->bufs[BUF_FFT_IN].ptr;
    float2 *outp;
    if (flags & PYL_PTR_DEVICE) {
        if (flags & PYL_PK_DESTROY_INPUT) in = (float *)delta;
        else PYL_HIP(hipMemcpyAsync(in, delta, n * sizeof(float), hipMemcpyDeviceToDevice, c->stream));
        outp = (float2 *)delta_k;
    } else {
        PYL_TRY(ensure(c, BUF_FFT_OUT, (size_t)nk * sizeof(float2)));
        outp = (float2 *)c->bufs[BUF_FFT_OUT].ptr;
        PYL_HIP(hipMemcpyAsync(in, delta, n * sizeof(float), hipMemcpyHostToDevice, c->stream));
    }
    PYL_TRY(fft_device(c, in, outp, dims, 1));
    if (!(flags & PYL_PTR_DEVICE))
        PYL_HIP(hipMemcpyAsync(delta_k, outp, nk * sizeof(float2), hipMemcpyDeviceToHost, c->stream));
    return finish(c, flags);
}

int pyl_pk(pyl_ctx *ctx, const float *const *deltas, int nfields, const int *mas, int dims,
           double BoxSize, int axis, float scale, float shift, int flags, pyl_pk_out *out) {
    TraceRange trace_("pyl_pk");
    PYL_CHECK(ctx && deltas && mas && out, PYL_EINVAL, "NULL argument");
    PYL_CHECK(nfields >= 1, PYL_EINVAL, "need at least one field");
    PYL_CHECK(dims >= 2, PYL_EINVAL, "dims must be >= 2");
    PYL_CHECK(axis >= 0 && axis <= 2, PYL_EINVAL, "axis must be 0, 1 or 2");
    PYL_CHECK(BoxSize > 0.0, PYL_EINVAL, "BoxSize must be positive");
    for (int f = 0; f < nfields; ++f) {
        PYL_CHECK(deltas[f] != nullptr, PYL_EINVAL, "field %d is NULL", f);
        PYL_CHECK(mas[f] >= 0 && mas[f] <= 4, PYL_EINVAL, "bad MAS id %d", mas[f]);
    }
    Ctx *c = &ctx->c;
    PYL_HIP(hipSetDevice(c->device));
    reset_stages(c);
    const long long n = (long long)dims * dims * dims;
    // the library's own half-complex buffer: rows padded to 128 bytes (fft_zstride)
    const long long zs = fft_zstride(dims);
    const long long nk = (long long)dims * dims * zs;
    const bool apply = !(scale == 1.0f && shift == 0.0f);
    const bool dev = (flags & PYL_PTR_DEVICE) != 0;
    const bool destroy = dev && (flags & PYL_PK_DESTROY_INPUT);
    PYL_TRY(ensure(c, BUF_FFT_OUT, (size_t)nk * nfields * sizeof(float2)));
    float2 *dk = (float2 *)c->bufs[BUF_FFT_OUT].ptr;
    const bool own = fft_own_size(dims);
    unsigned *amax = nullptr;
    PYL_TRY(pk_amax_words(c, nfields, own, &amax));
    std::vector<const unsigned *> amf(nfields);
    for (int f = 0; f < nfields; ++f) amf[f] = amax + 64 * f;
    std::vector<const float2 *> dks(nfields);
    const int pb = 256;
    const int nb = (int)std::min<long long>((n + pb - 1) / pb, 8192);
    if (own) {
        FieldSrc fs;
        fs.nfields = nfields;
        fs.apply = apply;
        fs.scale = scale;
        fs.shift = shift;
        PYL_TRY(fft_fields_device(c, deltas, fs, dev, dk, dims, zs, amax));
        for (int f = 0; f < nfields; ++f) dks[f] = dk + (size_t)f * nk;
    } else if (destroy) {
        for (int f = 0; f < nfields; ++f) {
            float *x = (float *)deltas[f];
            if (apply) {
                PYL_TRY(stage_begin(c, PYL_STAGE_PK_PREP));
                prologue_kernel<<<nb, pb, 0, c->stream>>>(x, x, n, nullptr, nullptr, scale, shift, 1);
                PYL_HIP(hipGetLastError());
                PYL_TRY(stage_end(c, PYL_STAGE_PK_PREP));
            }
            PYL_TRY(fft_device(c, x, dk + (size_t)f * nk, dims, 1, zs, amax + 64 * f));
            dks[f] = dk + (size_t)f * nk;
        }
    } else {
        PYL_TRY(ensure(c, BUF_FFT_IN, (size_t)n * nfields * sizeof(float)));
        float *in = (float *)c->bufs[BUF_FFT_IN].ptr;
        PYL_TRY(stage_begin(c, PYL_STAGE_PK_PREP));
        for (int f = 0; f < nfields; ++f) {
            float *dst = in + (size_t)f * n;
            if (dev) {
                if (apply) {
                    prologue_kernel<<<nb, pb, 0, c->stream>>>(deltas[f], dst, n, nullptr, nullptr, scale,
                                                            shift, 1);
                    PYL_HIP(hipGetLastError());
                } else {
                    PYL_HIP(hipMemcpyAsync(dst, deltas[f], n * sizeof(float), hipMemcpyDeviceToDevice,
                                           c->stream));
                }
            } else {
                PYL_HIP(hipMemcpyAsync(dst, deltas[f], n * sizeof(float), hipMemcpyHostToDevice,
                                       c->stream));
                if (apply) {
                    prologue_kernel<<<nb, pb, 0, c->stream>>>(dst, dst, n, nullptr, nullptr, scale, shift, 1);
                    PYL_HIP(hipGetLastError());
                }
            }
        }
        PYL_TRY(stage_end(c, PYL_STAGE_PK_PREP));
        PYL_TRY(fft_device(c, in, dk, dims, nfields, zs, amax));
        for (int f = 0; f < nfields; ++f) dks[f] = dk + (size_t)f * nk;
    }
    PYL_TRY(pk_bin_device(c, dks.data(), 0, zs, 1, nfields, mas, dims, BoxSize, axis, flags, out,
                          amf.data()));
    return finish(c, flags);
}

int pyl_pk_batch(pyl_ctx *ctx, const float *const *deltas, int nreal, int nfields,
                 const int *mas, int dims, double BoxSize, int axis, const float *scales,
                 const float *shifts, int flags, pyl_pk_out *outs) {
    TraceRange trace_("pyl_pk_batch");
    PYL_CHECK(ctx && deltas && mas && outs, PYL_EINVAL, "NULL argument");
    PYL_CHECK(nreal >= 1 && nfields >= 1 && (long long)nreal * nfields <= 65535, PYL_EINVAL,
              "need 1 <= nreal*nfields <= 65535");
    PYL_CHECK(dims >= 2 && axis >= 0 && axis <= 2 && BoxSize > 0.0, PYL_EINVAL, "bad arguments");
    for (int f = 0; f < nfields; ++f) {
        PYL_CHECK(deltas[f] != nullptr, PYL_EINVAL, "field %d is NULL", f);
        PYL_CHECK(mas[f] >= 0 && mas[f] <= 4, PYL_EINVAL, "bad MAS id %d", mas[f]);
    }
    Ctx *c = &ctx->c;
    PYL_HIP(hipSetDevice(c->device));
    reset_stages(c);
    const long long n = (long long)dims * dims * dims;
    const long long zs = fft_zstride(dims);              // padded rows (fft_zstride)
    const long long nk = (long long)dims * dims * zs;
    const int ncube = nreal * nfields;                 // cube (f, r) at index f*nreal + r
    const bool dev = (flags & PYL_PTR_DEVICE) != 0;
    const bool destroy = dev && (flags & PYL_PK_DESTROY_INPUT);
    const bool apply = scales != nullptr || shifts != nullptr;
    PYL_TRY(ensure(c, BUF_FFT_OUT, (size_t)nk * ncube * sizeof(float2)));
    float2 *dk = (float2 *)c->bufs[BUF_FFT_OUT].ptr;
    unsigned *amax = nullptr;                          // cube (f, r) at (f*nreal + r)*64
    const bool own = fft_own_size(dims);
    PYL_TRY(pk_amax_words(c, ncube, own, &amax));
    std::vector<const unsigned *> amf(nfields);
    for (int f = 0; f < nfields; ++f) amf[f] = amax + (size_t)64 * nreal * f;
    float *in = nullptr;
    if (!destroy && !own) {
        PYL_TRY(ensure(c, BUF_FFT_IN, (size_t)n * ncube * sizeof(float)));
        in = (float *)c->bufs[BUF_FFT_IN].ptr;
    }
    // Per-cube scale/shift: caller order [r][f].  Device arrays are read in place
    // (stride nfields from field f); host arrays are uploaded through pinned
    // staging in cube order [f][r] (no wait for the work already queued).
    const float *dsc = nullptr, *dsh = nullptr;
    int sstride = 1;
    const bool sdev = (flags & PYL_PK_SCALES_DEVICE) != 0;
    if (apply && sdev) {
        PYL_CHECK(scales != nullptr && shifts != nullptr, PYL_EINVAL,
                  "PYL_PK_SCALES_DEVICE needs both scales and shifts");
        dsc = scales;
        dsh = shifts;
        sstride = nfields;
    } else if (apply) {
        PYL_TRY(ensure(c, BUF_SCAN_TMP, sizeof(float) * 2 * (size_t)ncube));
        float *d = (float *)c->bufs[BUF_SCAN_TMP].ptr;
        void *stage = nullptr;
        PYL_TRY(pinned(c, c->pin_scales, sizeof(float) * 2 * (size_t)ncube, &stage));
        float *sc = (float *)stage, *sh = sc + ncube;
        for (int r = 0; r < nreal; ++r)
            for (int f = 0; f < nfields; ++f) {
                sc[(size_t)f * nreal + r] = scales ? scales[(size_t)r * nfields + f] : 1.0f;
                sh[(size_t)f * nreal + r] = shifts ? shifts[(size_t)r * nfields + f] : 0.0f;
            }
        PYL_HIP(hipMemcpyAsync(d, stage, sizeof(float) * 2 * ncube, hipMemcpyHostToDevice, c->stream));
        PYL_TRY(pinned_done(c, c->pin_scales));
        dsc = d;
        dsh = d + ncube;
    }
    if (own) {
        FieldSrc fs;
        fs.nfields = nfields;
        fs.nreal = nreal;
        fs.apply = apply;
        fs.scales = dsc;
        fs.shifts = dsh;
        fs.sfield = sdev ? 1 : nreal;
        fs.sreal = sdev ? nfields : 1;
        PYL_TRY(fft_fields_device(c, deltas, fs, dev, dk, dims, zs, amax));
    } else {
        const int nbx = (int)std::max<long long>(1, std::min<long long>((n + 255) / 256, 2048));
        PYL_TRY(stage_begin(c, PYL_STAGE_PK_PREP));
        for (int f = 0; f < nfields; ++f) {
            float *dst = destroy ? (float *)deltas[f] : in + (size_t)f * nreal * n;
            if (!destroy)
                PYL_HIP(hipMemcpyAsync(dst, deltas[f], (size_t)n * nreal * sizeof(float),
                                       dev ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, c->stream));
            if (apply) {
                const size_t off = sdev ? (size_t)f : (size_t)f * nreal;
                prologue_kernel<<<dim3(nbx, nreal), 256, 0, c->stream>>>(
                    dst, dst, n, dsc + off, dsh + off, 1.0f, 0.0f, 1, sstride);
                PYL_HIP(hipGetLastError());
            }
        }
        PYL_TRY(stage_end(c, PYL_STAGE_PK_PREP));
        if (destroy) {
            for (int f = 0; f < nfields; ++f)
                PYL_TRY(fft_device(c, (float *)deltas[f], dk + (size_t)f * nreal * nk, dims, nreal, zs,
                                   amax + (size_t)64 * nreal * f));
        } else {
            PYL_TRY(fft_device(c, in, dk, dims, ncube, zs, amax));
        }
    }
    std::vector<const float2 *> dks(nfields);
    for (int f = 0; f < nfields; ++f) dks[f] = dk + (size_t)f * nreal * nk;
    PYL_TRY(pk_bin_device(c, dks.data(), nk, zs, nreal, nfields, mas, dims, BoxSize, axis, flags, outs,
                          amf.data()));
    return finish(c, flags);
}

int pyl_pk_from_fourier(pyl_ctx *ctx, const float *const *delta_k, int nfields, const int *mas,
                        int dims, double BoxSize, int axis, int flags, pyl_pk_out *out) {
    TraceRange trace_("pyl_pk_from_fourier");
    PYL_CHECK(ctx && delta_k && mas && out, PYL_EINVAL, "NULL argument");
    PYL_CHECK(nfields >= 1 && dims >= 2 && axis >= 0 && axis <= 2 && BoxSize > 0.0, PYL_EINVAL,
              "bad arguments");
    Ctx *c = &ctx->c;
    PYL_HIP(hipSetDevice(c->device));
    reset_stages(c);
    const long long nk = (long long)dims * dims * (dims / 2 + 1);
    std::vector<const float2 *> dks(nfields);
    if (flags & PYL_PTR_DEVICE) {
        for (int f = 0; f < nfields; ++f) dks[f] = (const float2 *)delta_k[f];
    } else {
        PYL_TRY(ensure(c, BUF_FFT_OUT, (size_t)nk * nfields * sizeof(float2)));
        float2 *dk = (float2 *)c->bufs[BUF_FFT_OUT].ptr;
        for (int f = 0; f < nfields; ++f) {
            PYL_HIP(hipMemcpyAsync(dk + (size_t)f * nk, delta_k[f], nk * sizeof(float2),
                                   hipMemcpyHostToDevice, c->stream));
            dks[f] = dk + (size_t)f * nk;
        }
    }
    unsigned *amax = nullptr;
    PYL_TRY(pk_amax_words(c, nfields, false, &amax));
    std::vector<const unsigned *> amf(nfields);
    for (int f = 0; f < nfields; ++f) {
        PYL_TRY(complex_absmax(c, dks[f], dims, 0, 1, nk, amax + 64 * f));
        amf[f] = amax + 64 * f;
    }
    PYL_TRY(pk_bin_device(c, dks.data(), 0, 0, 1, nfields, mas, dims, BoxSize, axis, flags, out,
                          amf.data()));
    return finish(c, flags);
}

int pyl_pos_redshift_space(pyl_ctx *ctx, float *pos, const float *vel, int64_t n, float BoxSize,
                           float Hubble, float redshift, int axis, int flags) {
    PYL_CHECK(ctx && pos && vel, PYL_EINVAL, "NULL argument");
    PYL_CHECK(axis >= 0 && axis <= 2, PYL_EINVAL, "axis must be 0, 1 or 2");
    Ctx *c = &ctx->c;
    PYL_HIP(hipSetDevice(c->device));
    if (n <= 0) return PYL_OK;
    const float factor = (float)((1.0 + (double)redshift) / (double)Hubble);
    float *dpos = pos;
    const float *dvel = vel;
    if (!(flags & PYL_PTR_DEVICE)) {
        PYL_TRY(ensure(c, BUF_POS, (size_t)n * 3 * sizeof(float)));
        PYL_TRY(ensure(c, BUF_VEL, (size_t)n * 3 * sizeof(float)));
        dpos = (float *)c->bufs[BUF_POS].ptr;
        dvel = (const float *)c->bufs[BUF_VEL].ptr;
        PYL_HIP(hipMemcpyAsync(dpos, pos, (size_t)n * 3 * sizeof(float), hipMemcpyHostToDevice, c->stream));
        PYL_HIP(hipMemcpyAsync((void *)dvel, vel, (size_t)n * 3 * sizeof(float), hipMemcpyHostToDevice,
                               c->stream));
    }
    const int nb = (int)std::min<long long>((n + 255) / 256, 65536);
    rsd_kernel<<<nb, 256, 0, c->stream>>>(dpos, dvel, n, BoxSize, factor, axis);
    PYL_HIP(hipGetLastError());
    if (!(flags & PYL_PTR_DEVICE))
        PYL_HIP(hipMemcpyAsync(pos, dpos, (size_t)n * 3 * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    return finish(c, flags);
}

}  // extern "C"
