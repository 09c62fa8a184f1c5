// k_sites.hip -- electric-field projection fused with the site records, and
// the exciton Hamiltonian build (gfx950).
//
// Field + sites (calcIR.cu:1020-1168 and the per-row part of get_kappa_GPU,
// calcIR.cu:1245-1304): one wave per chromophore.  Its lanes test 64 molecules
// at a time against the cutoff (oxygens in LDS) and collect the ones inside in
// a list; the field of the listed molecules is then summed 64 at a time.  With
// a lane per chromophore and the field evaluated where a molecule lies inside,
// nearly every molecule lies inside some lane's sphere, so each wave evaluated
// the field of all of them with 7% of its lanes (32 frames of 2048 OH: 1.72
// ms, against 0.15 ms here).  Field sums are FP64 for FP32 sites and
// Neumaier-compensated for FP64 ones.
//
// Hamiltonian (calcIR.cu:1306-1404): a 64x64 tile on or below the diagonal per
// workgroup over the site records; every element is computed once and written
// to both triangles, lanes along the rows of each (the mirrored tile through
// LDS), so H(i,j) == H(j,i) bit for bit.  Bound by its arithmetic (an IEEE root
// and two quotients an element among it).  32 frames of 2048 OH in FP32: 0.44
// ms with every element of both triangles computed, 0.37 ms here, against 0.105
// ms for writing H at the rate of a large copy.

#include <algorithm>
#include <cfloat>
#include <cmath>

#include "common.hpp"
#include "sites.hpp"
#include "spectra.hpp"

namespace cir {

constexpr int kFieldBlock = 256;
constexpr int kFieldWaves = kFieldBlock / 64;
constexpr int kFieldChrom = 16;    // chromophores per workgroup
constexpr int kFieldTile = 4096;   // molecules whose oxygens are staged in LDS at a time (48 KB)

// The discrete cutoff decision (calcIR.cu:1106-1113), always in FP32 with
// the reference's operation order, identical in every precision form:
// !(sqrt(r2) > cutoff) with the correctly rounded root, as a comparison of r2
// with the largest value whose root does not exceed the cutoff
// (cutoff_square, on the host: the rounded root is monotonic).
__device__ __forceinline__ bool within_cutoff(float ox, float oy, float oz, float hx, float hy,
                                              float hz, const PBox<float>& B, float cut2) {
#pragma clang fp contract(off)
    float d0 = ox - hx, d1 = oy - hy, d2 = oz - hz;
    minimage3<float>(d0, d1, d2, B);
    return !(d0 * d0 + d1 * d1 + d2 * d2 > cut2);
}

float cutoff_square(float cutoff) {
    if (std::isnan(cutoff) || std::isinf(cutoff)) return cutoff;
    if (cutoff < 0.f) return -1.f;  // no separation is below a negative cutoff
    float t = cutoff * cutoff;
    if (std::isinf(t)) t = FLT_MAX;
    while (t > 0.f && std::sqrt(t) > cutoff) t = std::nextafter(t, 0.f);
    for (;;) {
        const float u = std::nextafter(t, INFINITY);
        if (std::isinf(u) || std::sqrt(u) > cutoff) return t;
        t = u;
    }
}

// Sum over a wave's lanes of a field component: FP64 for FP32 sites, whose
// terms carry FP32 rounding; compensated pairs for FP64 sites.
template <typename T>
struct FieldSum;
template <>
struct FieldSum<float> {
    double s = 0.0;
    __device__ __forceinline__ void add(float v) { s += double(v); }
    __device__ __forceinline__ float total() const { return float(wave_sum(s)); }
};
template <>
struct FieldSum<double> {
    Compensated<double> s;
    __device__ __forceinline__ void add(double v) { s.add(v); }
    __device__ __forceinline__ double total() const {
        Compensated<double> t = s;
        for (int off = 32; off > 0; off >>= 1) {
            const double os = __shfl_xor(t.sum, off, 64), oc = __shfl_xor(t.c, off, 64);
            t.add(os);
            t.c += oc;
        }
        return t.value();
    }
};

template <typename T>
__global__ void __launch_bounds__(kFieldBlock)
eproj_sites_kernel(int natoms, int natom_mol, int nchrom_mol, int imodel, int rules, float cut2,
                   const float* __restrict__ xyz, const float* __restrict__ box, int boxk, MapT<T> mc,
                   T* __restrict__ sites) {
    extern __shared__ float sO[];  // x, y, z of min(nmol, kFieldTile) oxygens
    __shared__ int list[kFieldWaves][128];
    __shared__ T sE[kFieldChrom][3];

    const int f = blockIdx.y;
    const int nmol = natoms / natom_mol;
    const int N = nmol * nchrom_mol;
    const float* x = xyz + size_t(f) * natoms * 3;
    const PBox<float> Bf = load_box<float>(box, boxk, f);
    const PBox<T> Bt = load_box<T>(box, boxk, f);
    // calcIR.cu:1117-1160: the charged sites of molecule m are its atoms
    // 1..natom_mol-1, +0.52 on atoms 1 and 2 and -1.04 on atom 3 (later atoms
    // carry nothing), so three-site water has no negative site.  The
    // msite_bisector rule builds one for it instead.
    const bool built_m = (rules & kRuleMsiteBisector) && natom_mol == 3;
    const bool have_m = natom_mol >= 4 || built_m;
    // calcIR.cu:1061-1070 picks H1 or H2 by chrom % 2 whatever nchrom_mol is
    // (with nchrom_mol 1, even molecules use H1 and odd ones H2); the
    // oh_per_molecule rule takes H(1 + chrom % nchrom_mol).
    auto hatom_of = [&](int chrom) {
        return 1 + ((rules & kRuleOhPerMolecule) ? chrom % nchrom_mol : chrom % 2);
    };
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c0 = blockIdx.x * kFieldChrom;
    const int ts = min(nmol, kFieldTile);  // pitch of the staged coordinates
    const T bohr = T(kBohrPerNm);
    auto stage = [&](int m0) {
        const int cnt = min(ts, nmol - m0);
        for (int t = tid; t < cnt; t += kFieldBlock) {
            const float* mx = x + 3 * size_t(m0 + t) * natom_mol;
            sO[t] = mx[0];
            sO[ts + t] = mx[1];
            sO[2 * ts + t] = mx[2];
        }
    };
    if (nmol <= kFieldTile) {
        stage(0);
        __syncthreads();
    }
    // every wave of a workgroup runs the same number of chromophores, so the
    // barriers of the staged tiles are reached by all of them
#pragma unroll 1
    for (int q = wave; q < kFieldChrom; q += kFieldWaves) {
        const int chrom = c0 + q;
        const bool active = chrom < N;
        const int n = active ? chrom / nchrom_mol : 0;
        const float* xh = x + 3 * (size_t(n) * natom_mol + hatom_of(active ? chrom : 0));
        const float hxf = xh[0], hyf = xh[1], hzf = xh[2];
        const T hx = T(hxf), hy = T(hyf), hz = T(hzf);
        FieldSum<T> ex, ey, ez;
        // the field of molecule m's charged sites at this chromophore's H
        auto field = [&](int m) {
            const float* mx = x + 3 * size_t(m) * natom_mol;
            T a[9];
#pragma unroll
            for (int c = 0; c < 6; ++c) a[c] = T(mx[3 + c]);
            const T o[3] = {T(mx[0]), T(mx[1]), T(mx[2])};
            T ms[3] = {T(0), T(0), T(0)};
            if (built_m) {
                // the TIP4P negative site on the HOH bisector, 0.015 nm from O
                T h1[3] = {a[0] - o[0], a[1] - o[1], a[2] - o[2]};
                T h2[3] = {a[3] - o[0], a[4] - o[1], a[5] - o[2]};
                minimage3<T>(h1[0], h1[1], h1[2], Bt);
                minimage3<T>(h2[0], h2[1], h2[2], Bt);
                const T r1 = sqrt(image_square<T>(h1[0], h1[1], h1[2]));
                const T r2 = sqrt(image_square<T>(h2[0], h2[1], h2[2]));
                T bi[3];
                for (int c = 0; c < 3; ++c) bi[c] = h1[c] / r1 + h2[c] / r2;
                const T rb = sqrt(bi[0] * bi[0] + bi[1] * bi[1] + bi[2] * bi[2]);
                for (int c = 0; c < 3; ++c) ms[c] = o[c] + T(kOMTip4p) * bi[c] / rb;
            } else if (have_m) {
                for (int c = 0; c < 3; ++c) ms[c] = T(mx[9 + c]);
                if (imodel != 0) {
                    // calcIR.cu:1124-1140: M moved to 0.015 nm along O->M
                    T om[3] = {ms[0] - o[0], ms[1] - o[1], ms[2] - o[2]};
                    minimage3<T>(om[0], om[1], om[2], Bt);
                    const T rom = sqrt(image_square<T>(om[0], om[1], om[2]));
                    for (int c = 0; c < 3; ++c) ms[c] = o[c] + T(kOMTip4p) * om[c] / rom;
                }
            }
            for (int c = 0; c < 3; ++c) a[6 + c] = ms[c];
#pragma unroll
            for (int s = 0; s < 3; ++s) {
                if (s == 2 && !have_m) break;
                T dx = hx - a[3 * s + 0], dy = hy - a[3 * s + 1], dz = hz - a[3 * s + 2];
                minimage3<T>(dx, dy, dz, Bt);
                dx = dx * bohr;
                dy = dy * bohr;
                dz = dz * bohr;
                const T r = sqrt(image_square<T>(dx, dy, dz));
                const T qc = (s < 2) ? T(kQH) : T(-kQM);
                const T qr3 = qc / (r * r * r);
                ex.add(qr3 * dx);
                ey.add(qr3 * dy);
                ez.add(qr3 * dz);
            }
        };
        int cnt = 0;  // molecules in the wave's list
        int* const lw = list[wave];
        for (int m0 = 0; m0 < nmol; m0 += kFieldTile) {
            if (nmol > kFieldTile) {
                __syncthreads();
                stage(m0);
                __syncthreads();
            }
            const int tc = min(ts, nmol - m0);
            for (int t0 = 0; t0 < tc; t0 += 64) {
                const int t = t0 + lane, ti = min(t, tc - 1);
                const bool in = within_cutoff(sO[ti], sO[ts + ti], sO[2 * ts + ti], hxf, hyf, hzf, Bf, cut2) &&
                                t < tc && active && m0 + t != n;  // calcIR.cu:1099
                const unsigned long long mask = __ballot(in);
                if (mask == 0) continue;
                if (in) lw[cnt + __popcll(mask & ((1ull << lane) - 1))] = m0 + t;
                cnt += __popcll(mask);
                if (cnt >= 64) {
                    wave_lds_sync();
                    field(lw[lane]);
                    cnt -= 64;
                    const int left = lw[64 + lane];
                    wave_lds_sync();
                    if (lane < cnt) lw[lane] = left;
                    wave_lds_sync();
                }
            }
        }
        wave_lds_sync();
        if (lane < cnt) field(lw[lane]);
        const T tx = ex.total(), ty = ey.total(), tz = ez.total();
        if (lane == 0) {
            sE[q][0] = tx;
            sE[q][1] = ty;
            sE[q][2] = tz;
        }
    }
    __syncthreads();
    const int chrom = c0 + tid;
    if (tid >= kFieldChrom || chrom >= N) return;

    // own OH unit vector, TDM position and maps (calcIR.cu:1047-1080, 1253-1304)
    const float* no = x + 3 * size_t(chrom / nchrom_mol) * natom_mol;
    const float* nh = no + 3 * hatom_of(chrom);
    const T ox = T(no[0]), oy = T(no[1]), oz = T(no[2]);
    T ux = T(nh[0]) - ox, uy = T(nh[1]) - oy, uz = T(nh[2]) - oz;
    minimage3<T>(ux, uy, uz, Bt);
    const T r = sqrt(image_square<T>(ux, uy, uz));
    ux /= r;
    uy /= r;
    uz /= r;
    const T E = sE[tid][0] * ux + sE[tid][1] * uy + sE[tid][2] * uz;
    const T w = mc.w0 + mc.w1 * E + mc.w2 * E * E;
    const T xx = mc.x0 + mc.x1 * w;
    const T p = mc.p0 + mc.p1 * w;
    const T mup = mc.m0 + mc.m1 * E + mc.m2 * E * E;
    const T A = T(kRamanAniso);
    T* S = sites + size_t(f) * CIR_NSITE * N;
    S[CIR_SITE_E * N + chrom] = E;
    S[CIR_SITE_W * N + chrom] = w;
    S[CIR_SITE_X * N + chrom] = xx;
    S[CIR_SITE_P * N + chrom] = p;
    S[CIR_SITE_MUP * N + chrom] = mup;
    S[(CIR_SITE_U + 0) * N + chrom] = ux;
    S[(CIR_SITE_U + 1) * N + chrom] = uy;
    S[(CIR_SITE_U + 2) * N + chrom] = uz;
    T rx = ox + T(kTdmOffset) * ux, ry = oy + T(kTdmOffset) * uy, rz = oz + T(kTdmOffset) * uz;
    minimage3<T>(rx, ry, rz, Bt);  // calcIR.cu:1289-1291 (wrapped; only differences are used)
    S[(CIR_SITE_R + 0) * N + chrom] = rx;
    S[(CIR_SITE_R + 1) * N + chrom] = ry;
    S[(CIR_SITE_R + 2) * N + chrom] = rz;
    S[(CIR_SITE_MU + 0) * N + chrom] = ux * mup * xx;
    S[(CIR_SITE_MU + 1) * N + chrom] = uy * mup * xx;
    S[(CIR_SITE_MU + 2) * N + chrom] = uz * mup * xx;
    S[(CIR_SITE_A + 0) * N + chrom] = (A * ux * ux + T(1)) * xx;
    S[(CIR_SITE_A + 1) * N + chrom] = (A * uy * uy + T(1)) * xx;
    S[(CIR_SITE_A + 2) * N + chrom] = (A * uz * uz + T(1)) * xx;
    S[(CIR_SITE_A + 3) * N + chrom] = A * ux * uy * xx;
    S[(CIR_SITE_A + 4) * N + chrom] = A * uy * uz * xx;
    S[(CIR_SITE_A + 5) * N + chrom] = A * uz * ux * xx;
}

constexpr int kHTile = 64;

template <typename T>
__global__ void __launch_bounds__(256)
hamiltonian_kernel(int N, int ld, int nchrom_mol, int hod, T avef, T wi0, T wi1, T wi2,
                   const float* __restrict__ box, int boxk, const T* __restrict__ sites, T* __restrict__ H) {
    // per-tile site data: E, w, x, p, s = x*mup, u(3), r(3)
    __shared__ T rs[11][kHTile];
    __shared__ T cs[11][kHTile];
    __shared__ T mir[kHTile][kHTile + 1];
    // tiles on or below the diagonal (with the padding rows below N)
    if (blockIdx.x < blockIdx.y) return;
    const int f = blockIdx.z;
    const int i0 = blockIdx.x * kHTile, j0 = blockIdx.y * kHTile;
    const T* S = sites + size_t(f) * CIR_NSITE * N;
    const int tid = threadIdx.x;
    if (tid < 2 * kHTile) {
        const bool row = tid < kHTile;
        const int l = row ? tid : tid - kHTile;
        const int g = (row ? i0 : j0) + l;
        T(*d)[kHTile] = row ? rs : cs;
        if (g < N) {
            d[0][l] = S[CIR_SITE_E * N + g];
            d[1][l] = S[CIR_SITE_W * N + g];
            d[2][l] = S[CIR_SITE_X * N + g];
            d[3][l] = S[CIR_SITE_P * N + g];
            d[4][l] = S[CIR_SITE_X * N + g] * S[CIR_SITE_MUP * N + g];
            for (int c = 0; c < 3; ++c) {
                d[5 + c][l] = S[(CIR_SITE_U + c) * N + g];
                d[8 + c][l] = S[(CIR_SITE_R + c) * N + g];
            }
        } else {
            for (int c = 0; c < 11; ++c) d[c][l] = T(0);
        }
    }
    __syncthreads();
    const PBox<T> bb = load_box<T>(box, boxk, f);
    const int tx = tid % kHTile, ty = tid / kHTile;
    const int i = i0 + tx;
    T* Hf = H + size_t(f) * N * ld;
    const bool mirror = i0 != j0;
    for (int q = 0; q < kHTile / 4; ++q) {
        const int jl = ty + 4 * q;
        const int j = j0 + jl;
        if (j >= N) break;
        T h;
        if (i >= N) {
            h = T(0);  // padding rows of the leading dimension
        } else if (i == j) {
            h = rs[1][tx] - avef;  // calcIR.cu:1322-1327
        } else if (hod) {
            h = T(0);  // calcIR.cu:1334-1336, 1348-1350
        } else if (i / nchrom_mol == j / nchrom_mol) {
            // calcIR.cu:1330-1341
            h = (wi0 + wi1 * (rs[0][tx] + cs[0][jl])) * (rs[2][tx] * cs[2][jl]) +
                wi2 * (rs[3][tx] * cs[3][jl]);
        } else {
            // calcIR.cu:1353-1401, symmetric operation order
            const T g = tdc_geometry<T>(rs[5][tx], rs[6][tx], rs[7][tx], rs[8][tx], rs[9][tx], rs[10][tx],
                                        cs[5][jl], cs[6][jl], cs[7][jl], cs[8][jl], cs[9][jl], cs[10][jl], bb);
            h = g * (rs[4][tx] * cs[4][jl]) * T(kCmPerHartree);
        }
        if (i < ld) Hf[size_t(j) * ld + i] = h;
        if (mirror) mir[jl][tx] = h;
    }
    if (!mirror) return;
    // the same elements above the diagonal: column i0 + c, rows j0 + lane
    __syncthreads();
    const int j = j0 + tx;
    for (int q = 0; q < kHTile / 4; ++q) {
        const int c = ty + 4 * q;
        if (i0 + c < N && j < N) Hf[size_t(i0 + c) * ld + j] = mir[tx][c];
    }
}

template <typename T>
int launch_eproj_sites(int nframes, int natoms, int natom_mol, int nchrom_mol, int imodel, int rules,
                       float cutoff, const float* xyz, const float* box, int boxk, const MapCoef& mc,
                       void* sites, hipStream_t s) {
    const int N = (natoms / natom_mol) * nchrom_mol;
    dim3 grid(unsigned(ceil_div(N, kFieldChrom)), unsigned(nframes));
    const size_t sm = size_t(std::min(natoms / natom_mol, kFieldTile)) * 3 * sizeof(float);
    hipLaunchKernelGGL(eproj_sites_kernel<T>, grid, dim3(kFieldBlock), sm, s, natoms, natom_mol,
                       nchrom_mol, imodel, rules, cutoff_square(cutoff), xyz, box, boxk, map_t<T>(mc),
                       static_cast<T*>(sites));
    CIR_CHECK_LAUNCH();
    return CIR_OK;
}

template <typename T>
int launch_hamiltonian(int nframes, int N, int ld, int nchrom_mol, int ispecies, const MapCoef& mc,
                       float avef, const float* box, int boxk, const void* sites, void* H, hipStream_t s) {
    dim3 grid(unsigned(ceil_div(ld, kHTile)), unsigned(ceil_div(N, kHTile)), unsigned(nframes));
    const int hod = (ispecies == 1 || ispecies == 2) ? 1 : 0;
    hipLaunchKernelGGL(hamiltonian_kernel<T>, grid, dim3(256), 0, s, N, ld, nchrom_mol, hod, T(avef),
                       T(mc.wi[0]), T(mc.wi[1]), T(mc.wi[2]), box, boxk, static_cast<const T*>(sites),
                       static_cast<T*>(H));
    CIR_CHECK_LAUNCH();
    return CIR_OK;
}

int eproj_sites(int prec, int nframes, int natoms, int natom_mol, int nchrom_mol, int imodel, int rules,
                const MapCoef& mc, float cutoff, const float* xyz_d, const float* box_d, int boxk, void* sites_d,
                hipStream_t s) {
    // atoms 1 and 2 of a molecule are its hydrogens (calcIR.cu:1061-1070)
    if (nframes <= 0 || natom_mol < 3 || nchrom_mol < 1 || natoms <= 0 || natoms % natom_mol || !xyz_d ||
        !box_d || !sites_d || (boxk != 0 && boxk != 1) || (rules & ~(kRuleOhPerMolecule | kRuleMsiteBisector)))
        return fail(CIR_ERR_ARG, "cir_eproj_sites: bad sizes or null pointer");
    if ((rules & kRuleOhPerMolecule) && nchrom_mol > 2)
        return fail(CIR_ERR_ARG, "cir_eproj_sites: one or two OH stretches per molecule with oh_per_molecule");
    if (int64_t(nframes) > 65535) return fail(CIR_ERR_ARG, "cir_eproj_sites: nframes > 65535");
    if (int64_t(natoms / natom_mol) * nchrom_mol > (int64_t(1) << 30))
        return fail(CIR_ERR_ARG, "cir_eproj_sites: too many chromophores");
    if (prec == CIR_PREC_FP64)
        return launch_eproj_sites<double>(nframes, natoms, natom_mol, nchrom_mol, imodel, rules, cutoff, xyz_d,
                                          box_d, boxk, mc, sites_d, s);
    return launch_eproj_sites<float>(nframes, natoms, natom_mol, nchrom_mol, imodel, rules, cutoff, xyz_d, box_d,
                                     boxk, mc, sites_d, s);
}

int hamiltonian(int prec, int nframes, int n, int ld, int nchrom_mol, int ispecies, const MapCoef& mc, float avef,
                const float* box_d, int boxk, const void* sites_d, void* H_d, hipStream_t s) {
    if (nframes <= 0 || n <= 0 || ld < n || nchrom_mol <= 0 || !box_d || !sites_d || !H_d ||
        (boxk != 0 && boxk != 1))
        return fail(CIR_ERR_ARG, "cir_hamiltonian: bad sizes or null pointer");
    if (nframes > 65535) return fail(CIR_ERR_ARG, "cir_hamiltonian: nframes > 65535");
    if (prec == CIR_PREC_FP64)
        return launch_hamiltonian<double>(nframes, n, ld, nchrom_mol, ispecies, mc, avef, box_d, boxk, sites_d, H_d,
                                          s);
    return launch_hamiltonian<float>(nframes, n, ld, nchrom_mol, ispecies, mc, avef, box_d, boxk, sites_d, H_d, s);
}

}  // namespace cir

using namespace cir;

extern "C" int cir_eproj_sites(int prec, int nframes, int natoms, int natom_mol, int nchrom_mol,
                               int imodel, int ispecies, int imap, float cutoff,
                               const float* xyz_d, const float* box_d, void* sites_d,
                               void* stream) {
    MapCoef mc;
    if (!map_coef(imap, ispecies, &mc)) return fail(CIR_ERR_MAP, "map/species not in the map table");
    return eproj_sites(prec, nframes, natoms, natom_mol, nchrom_mol, imodel, 0, mc, cutoff, xyz_d, box_d, 0,
                       sites_d, as_stream(stream));
}

extern "C" int cir_hamiltonian(int prec, int nframes, int n, int ld, int nchrom_mol, int ispecies,
                               int imap, float avef, const float* box_d, const void* sites_d,
                               void* H_d, void* stream) {
    MapCoef mc;
    if (!map_coef(imap, ispecies, &mc)) return fail(CIR_ERR_MAP, "map/species not in the map table");
    return hamiltonian(prec, nframes, n, ld, nchrom_mol, ispecies, mc, avef, box_d, 0, sites_d, H_d,
                       as_stream(stream));
}
