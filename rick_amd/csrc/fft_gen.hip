// Backward C2C FFT of w-planes for axis lengths the power-of-two engine
// (fft.hip) does not take: FFTW plans any Ny x Nx (fourier_transform.c:
// 34-36), so the fftw_data stage must too.
//
// Each axis of the 2-D transform is planned on its own:
//   * direct     -- one pass over lines of length L <= 4096 whose prime
//                   factors are <= 13: a mixed-radix Stockham transform held
//                   in LDS (every radix from 2 to 16), one workgroup per G
//                   lines;
//   * four-step  -- N = N1 * N2 (both direct lengths, N1 closest to sqrt(N)):
//                   pass A does the N1-point DFTs with the twiddle W_N^(k1 n2)
//                   into a one-plane scratch, pass B the N2-point DFTs back,
//                   in natural order.  Used for long rows (N > 4096) and for
//                   columns longer than 256 (G >= 16 adjacent columns per
//                   workgroup keeps the strided reads in whole 256-byte runs);
//   * Bluestein  -- lengths with a prime factor above 13: X[k] = b[k] *
//                   sum_n (x[n] b[n]) conj(b[k-n]), b[n] = exp(+i pi n^2/N),
//                   as a cyclic convolution of power-of-two length
//                   M >= 2N-1 done with two M-point transforms of the
//                   engine above and the precomputed transform of the chirp.
// Twiddles are tables exp(+2 pi i m/N) of the axis length (computed on the
// host in long double); a pass of length L | N uses them with stride N/L.
#include <algorithm>
#include <cmath>
#include <vector>

#include "fft_kernels.h"
#include "rick_internal.h"
#include "rick_math.h"
#include "rick_tables.h"

namespace rick {
namespace {

using namespace fftk;

constexpr int kGenThreads = 512;      // most threads of a workgroup
constexpr int kGenValues = 16;        // most complex values a thread holds (its largest radix)
constexpr int kPhaseValues = 10;      // ... in the fused phase pass
constexpr int kGenElems = 4096;       // longest line of one pass
constexpr int kGenDirectCols = 256;   // longest column transform done in one pass
constexpr size_t kBlueChunk = size_t(1) << 25;   // Bluestein scratch: elements per chunk

constexpr int kGenLdsBytes = 80 * 1024;          // dynamic LDS of a workgroup, at most

// Butterflies of radix R a thread of V values takes in one pass.
__host__ __device__ constexpr int gen_bpt(int R, int V) { return V / R > 1 ? V / R : 1; }

// floor(x / d) for x * d < 2^32, from m = ceil(2^32 / d) (d > 1; 0 stands for 1).
__host__ __device__ inline uint32_t gen_magic(uint32_t d)
{
    return d > 1 ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u;
}
__device__ __forceinline__ int gen_div(int x, uint32_t m)
{
    return m ? (int)__umulhi((uint32_t)x, m) : x;
}

// Occupancy of the first axis transformed (rows of a sparse grid, see
// Occupancy in fft.hip), or the row flags of the axis after it (columns).
struct GenOcc {
    const uint32_t *offsets;        // rows: the gridder's bucket offsets (null: dense)
    const unsigned char *rows;      // [planes * ny] row flags (null: dense)
    int tu_shift, tv, tiles_u, tiles_v, ny;
};

// Line addressing of one launch.  Workgroup (group, set, plane) transforms
// lines g0 .. g0+G-1 of that set; element n of line g is read at
//   z*pz + s*ps_in  + g*pg_in  + n*pe_in
// and written at
//   z*pz + s*ps_out + g*pg_out + n*pe_out,
// after the optional four-step twiddle W_N^(n*s) (tw_by 1) or W_N^(n*g)
// (tw_by 2), N the table length, and the scale.
struct GenAddr {
    int nl, G, ngroups, sets;
    uint32_t mG;      // gen_magic(G)
    long long pz, ps_in, pg_in, pe_in, ps_out, pg_out, pe_out;
    int tw_by;
    int line_major;   // butterflies along a line are consecutive threads (contiguous lines)
    int row_mul;      // columns: input row of element n of set s is s * set_mul + n * row_mul
    int set_mul;
};

// LDS slot of element n of line g: line-major lines are padded by one slot
// per 16 elements (the first pass writes with the stride of its radix).
__host__ __device__ constexpr int gen_pad(int n) { return n + (n >> 4); }
__device__ __forceinline__ int gen_lds(int g, int n, int L, int G, int line_major)
{
    return line_major ? g * (gen_pad(L) + 1) + gen_pad(n) : n * G + g;
}

// exp(+2 pi i k/R) constants of the odd prime radices: cosines and sines of
// 2 pi m / R for m = 1 .. (R-1)/2.
template <int R>
struct OddRoots;
template <>
struct OddRoots<7> {
    static constexpr double c[3] = {0.62348980185873353053, -0.22252093395631440429,
                                    -0.90096886790241912624};
    static constexpr double s[3] = {0.78183148246802980871, 0.97492791218182360702,
                                    0.43388373911755812048};
};
template <>
struct OddRoots<11> {
    static constexpr double c[5] = {0.84125353283118116886, 0.41541501300188642553,
                                    -0.14231483827328514044, -0.65486073394528506406,
                                    -0.95949297361449738989};
    static constexpr double s[5] = {0.54064081745559758211, 0.90963199535451837141,
                                    0.98982144188093273238, 0.75574957435425828377,
                                    0.28173255684142969771};
};
template <>
struct OddRoots<13> {
    static constexpr double c[6] = {0.88545602565320989590, 0.56806474673115580251,
                                    0.12053668025532305335, -0.35460488704253562597,
                                    -0.74851074817110109863, -0.97094181742605202716};
    static constexpr double s[6] = {0.46472317204376854566, 0.82298386589365639458,
                                    0.99270887409805399280, 0.93501624268541482344,
                                    0.66312265824079520238, 0.23931566428755776715};
};

// Odd prime radix: with a_m = x_m + x_(R-m) and b_m = x_m - x_(R-m),
// X_k, X_(R-k) = x_0 + sum_m cos(2 pi k m/R) a_m +- i sum_m sin(2 pi k m/R) b_m.
template <typename T, int R>
__device__ __forceinline__ void dft_odd(C2<T> *v)
{
    constexpr int H = (R - 1) / 2;
    C2<T> a[H], b[H];
#pragma unroll
    for (int m = 0; m < H; ++m) {
        a[m] = cadd(v[m + 1], v[R - 1 - m]);
        b[m] = csub(v[m + 1], v[R - 1 - m]);
    }
    const C2<T> x0 = v[0];
    C2<T> sum = x0;
#pragma unroll
    for (int m = 0; m < H; ++m) sum = cadd(sum, a[m]);
    v[0] = sum;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        C2<T> re = x0, im = {T(0), T(0)};
#pragma unroll
        for (int m = 1; m <= H; ++m) {
            const int e = (k * m) % R, f = e > H ? R - e : e;
            const T c = (T)OddRoots<R>::c[f - 1];
            const T s = e > H ? -(T)OddRoots<R>::s[f - 1] : (T)OddRoots<R>::s[f - 1];
            re.x += c * a[m - 1].x;
            re.y += c * a[m - 1].y;
            im.x += s * b[m - 1].x;
            im.y += s * b[m - 1].y;
        }
        v[k] = {re.x - im.y, re.y + im.x};
        v[R - k] = {re.x + im.y, re.y - im.x};
    }
}

template <typename T, int R>
__device__ __forceinline__ void dft_mix(C2<T> *v);

constexpr int inv_mod(int a, int m)
{
    for (int x = 1; x < m; ++x)
        if (a * x % m == 1) return x;
    return 0;
}

// R = A * B with coprime factors (the prime-factor algorithm): inputs
// n = (B n1 + A n2) mod R, outputs k with k mod A = k1, k mod B = k2, no
// twiddles between the two.
template <typename T, int A, int B>
__device__ __forceinline__ void dft_coprime(C2<T> *v)
{
    constexpr int R = A * B, U = B * inv_mod(B % A, A), V = A * inv_mod(A % B, B);
    C2<T> y[B][A];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) y[n2][n1] = v[(B * n1 + A * n2) % R];
        dft_mix<T, A>(y[n2]);
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        C2<T> t[B];
#pragma unroll
        for (int n2 = 0; n2 < B; ++n2) t[n2] = y[n2][k1];
        dft_mix<T, B>(t);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2) v[(U * k1 + V * k2) % R] = t[k2];
    }
}

// Radix 9 as 3 x 3 with the twiddles exp(2 pi i m/9), m = 1, 2, 4.
template <typename T>
__device__ __forceinline__ void dft9(C2<T> *v)
{
    constexpr double c1 = 0.76604444311897803520, s1 = 0.64278760968653932632,
                     c2 = 0.17364817766693034885, s2 = 0.98480775301220805937,
                     c4 = -0.93969262078590838405, s4 = 0.34202014332566873304;
    C2<T> y[3][3];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
        for (int n1 = 0; n1 < 3; ++n1) y[n2][n1] = v[3 * n1 + n2];
        dft3(y[n2]);
    }
    y[1][1] = cmul(y[1][1], C2<T>{(T)c1, (T)s1});
    y[1][2] = cmul(y[1][2], C2<T>{(T)c2, (T)s2});
    y[2][1] = cmul(y[2][1], C2<T>{(T)c2, (T)s2});
    y[2][2] = cmul(y[2][2], C2<T>{(T)c4, (T)s4});
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
        C2<T> t[3] = {y[0][k1], y[1][k1], y[2][k1]};
        dft3(t);
#pragma unroll
        for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = t[k2];
    }
}

template <typename T, int R>
__device__ __forceinline__ void dft_mix(C2<T> *v)
{
    if constexpr (R == 2 || R == 4 || R == 8 || R == 16) dftR<T, R>(v);
    else if constexpr (R == 3) dft3(v);
    else if constexpr (R == 5) dft5(v);
    else if constexpr (R == 9) dft9(v);
    else if constexpr (R == 6) dft_coprime<T, 3, 2>(v);
    else if constexpr (R == 10) dft_coprime<T, 5, 2>(v);
    else if constexpr (R == 12) dft_coprime<T, 4, 3>(v);
    else if constexpr (R == 14) dft_coprime<T, 7, 2>(v);
    else if constexpr (R == 15) dft_coprime<T, 5, 3>(v);
    else dft_odd<T, R>(v);
}

// v[q] *= w^q for q = 1 .. R-1.  Every power comes from the table, rounded once: formed
// as products of w, w^2, w^4 and w^8 they carry up to three roundings more (FP32 error
// of 2053 points 2.09e-7, of 4099 2.16e-7; here 1.72e-7 and 1.83e-7).  The eleven
// loads more that a radix-16 butterfly makes cost 1 % of a 3000^2 x 8 FP64 image (1701
// -> 1723 us) and 11 % of an FP32 one (949 -> 1050).
template <typename T, int R>
__device__ __forceinline__ void gen_twiddle(C2<T> *v, int at, const C2<T> *__restrict__ tw)
{
#pragma unroll
    for (int q = 1; q < R; ++q) v[q] = cmul(v[q], tw[q * at]);
}

template <typename T>
struct GenCtx {
    const GenAddr *a;
    const C2<T> *tw;
    const C2<T> *in;
    C2<T> *out;
    C2<T> *lds;
    const unsigned char *occ;       // LDS: [g * tiles + tile] or [element], null: dense
    int occ_stride, occ_shift;
    int L, s, g0, nvalid;
    T scale;
};

// The last column pass of the FP64 image chain: instead of the transformed planes,
// their phase-rotated sum, kept per pixel by the thread that transforms it.  Element n
// of set s is image row s + n * row_mul (k1 + N1 * k2).
struct GenPhase {
    static constexpr bool kOn = true;
    static constexpr int kValues = kPhaseValues;
    PhaseGeom g;
    double *ore, *oim;
    int iw, row_mul;
    bool phase;
    double are[kValues], aim[kValues], nf[kValues];
    __device__ __forceinline__ void add(C2<double> o, int idx, int iu, int iv)
    {
        if (iw == 0) {
            are[idx] = aim[idx] = 0.0;
            nf[idx] = phase ? pixel_n(g.ltab[iu], g.mtab[iv]) : 1.0;
        }
        if (phase) {
            double wterm;   // the plane's w as the separate pass forms it
            {
#pragma clang fp contract(off)
                wterm = g.wmin + iw * g.dw;
            }
            phase_add_f64(o.x, o.y, wterm, nf[idx], g.dwnorm, are[idx], aim[idx]);
        } else {
            are[idx] += o.x;
            aim[idx] += o.y;
        }
        if (iw == g.planes - 1) {
            const size_t pix = (size_t)iv * g.nx + iu;
            store_stream(are[idx], &ore[pix]);
            store_stream(aim[idx], &oim[pix]);
        }
    }
};
struct GenStore {
    static constexpr bool kOn = false;
    static constexpr int kValues = kGenValues;
};

// One radix-R pass (Stockham: Ns = product of the earlier radices).  The
// first pass reads global memory, later ones LDS; the last writes global
// memory, or hands its values to the phase sum.  Reads of a pass all complete (barrier) before its writes, so the
// LDS buffer is used in place.
template <typename T, int R, typename Sink>
__device__ __forceinline__ void gen_pass(const GenCtx<T> &c, const GenPass &ps, bool first,
                                         bool last, Sink &sink)
{
    constexpr int BPT = gen_bpt(R, Sink::kValues);
    const GenAddr &a = *c.a;
    const int L = c.L, G = a.G, Lr = ps.Lr, Ns = ps.Ns, nb = G * Lr;
    C2<T> v[BPT][R];
    int gi[BPT], ji[BPT];
#pragma unroll
    for (int i = 0; i < BPT; ++i) {
        const int b = threadIdx.x + i * blockDim.x;
        gi[i] = -1;
        ji[i] = 0;
        if (b < nb) {
            int g, j;
            if (a.line_major) {
                g = gen_div(b, ps.mLr);
                j = b - g * Lr;
            } else {
                j = gen_div(b, a.mG);
                g = b - j * G;
            }
            gi[i] = g;
            ji[i] = j;
            if (first) {
                const C2<T> *p = c.in + (size_t)g * a.pg_in + (size_t)j * a.pe_in;
                const size_t step = (size_t)Lr * a.pe_in;
                const unsigned char *oc = c.occ ? c.occ + g * c.occ_stride : nullptr;
                const bool there = g < c.nvalid;
#pragma unroll
                for (int q = 0; q < R; ++q) {
                    const bool live =
                        there && (oc == nullptr || oc[(j + q * Lr) >> c.occ_shift]);
                    v[i][q] = live ? load_stream2(p + q * step) : C2<T>{T(0), T(0)};
                }
            } else {
#pragma unroll
                for (int q = 0; q < R; ++q)
                    v[i][q] = c.lds[gen_lds(g, j + q * Lr, L, G, a.line_major)];
            }
        }
    }
    if (!first) __syncthreads();
#pragma unroll
    for (int i = 0; i < BPT; ++i) {
        const int g = gi[i];
        if (g < 0) continue;
        const int j = ji[i];
        int dbase = j * R;
        if (!first) {
            const int jq = gen_div(j, ps.mNs), k = j - jq * Ns;
            gen_twiddle<T, R>(v[i], k * ps.tstep, c.tw);
            dbase = jq * (Ns * R) + k;
        }
        dft_mix<T, R>(v[i]);
        if (!last) {
#pragma unroll
            for (int q = 0; q < R; ++q)
                c.lds[gen_lds(g, dbase + q * Ns, L, G, a.line_major)] = v[i][q];
            continue;
        }
        if (g >= c.nvalid) continue;   // (its twiddle index would pass the table)
        if constexpr (Sink::kOn) {
#pragma unroll
            for (int q = 0; q < R; ++q)
                sink.add(v[i][q], i * R + q, c.g0 + g, c.s + (dbase + q * Ns) * sink.row_mul);
            continue;
        }
        C2<T> *p = c.out + (size_t)g * a.pg_out + (size_t)dbase * a.pe_out;
        const size_t step = (size_t)Ns * a.pe_out;
        const int e = a.tw_by == 1 ? c.s : c.g0 + g;
#pragma unroll
        for (int q = 0; q < R; ++q) {
            C2<T> o = v[i][q];
            if (a.tw_by) o = cmul(o, c.tw[(dbase + q * Ns) * e]);
            o.x *= c.scale;
            o.y *= c.scale;
            store_stream2(o, p + q * step);
        }
    }
    if (!last) __syncthreads();
}

// All passes of a workgroup's lines.
template <typename T, bool HARD, typename Sink>
__device__ __forceinline__ void gen_lines_of(const GenCtx<T> &c, const GenPassDesc &gp, Sink &sink)
{
    for (int p = 0; p < gp.np; ++p) {
        const bool first = p == 0, last = p == gp.np - 1;
        const GenPass &ps = gp.pass[p];
        switch (ps.R) {
            case 10: gen_pass<T, 10>(c, ps, first, last, sink); break;
            case 9: gen_pass<T, 9>(c, ps, first, last, sink); break;
            case 8: gen_pass<T, 8>(c, ps, first, last, sink); break;
            case 7: gen_pass<T, 7>(c, ps, first, last, sink); break;
            case 6: gen_pass<T, 6>(c, ps, first, last, sink); break;
            case 5: gen_pass<T, 5>(c, ps, first, last, sink); break;
            case 4: gen_pass<T, 4>(c, ps, first, last, sink); break;
            case 3: gen_pass<T, 3>(c, ps, first, last, sink); break;
            case 2: gen_pass<T, 2>(c, ps, first, last, sink); break;
            default:
                if constexpr (!Sink::kOn) {
                    if (ps.R == 16) gen_pass<T, 16>(c, ps, first, last, sink);
                    else if (ps.R == 15) gen_pass<T, 15>(c, ps, first, last, sink);
                    else if (ps.R == 14) gen_pass<T, 14>(c, ps, first, last, sink);
                    else if (ps.R == 12) gen_pass<T, 12>(c, ps, first, last, sink);
                }
                if constexpr (HARD) {
                    if (ps.R == 11) gen_pass<T, 11>(c, ps, first, last, sink);
                    else if (ps.R == 13) gen_pass<T, 13>(c, ps, first, last, sink);
                }
                break;
        }
    }}

// Passes of one workgroup.  A thread holds one butterfly of a radix above 8 (16
// values at most) or as many smaller ones as make 16 values, so a pass needs no
// more registers than its largest radix (132 VGPRs in FP64, 3 waves per SIMD;
// 243 and 2 when each thread held up to 4096 / R / 256 butterflies), and all
// index divisions are by constants formed on the host.  Bound by memory now:
// column pass A of 8 planes of 3000^2 FP64 moves 2.3 GB in 0.51 ms where half
// its rows are live, rows 0.37 ms over the live ones (before, dense: 2.0 ms the
// columns, 1.33 ms the rows).  HARD: the instance with radices 11 and 13, whose
// registers the lengths without them do not pay for.
template <typename T, bool HARD>
__global__ void __launch_bounds__(kGenThreads)
k_fft_gen(GenPassDesc gp, GenAddr a, const C2<T> *__restrict__ tw, const C2<T> *in, C2<T> *out,
          T scale, GenOcc oc, int occ_off)
{
    extern __shared__ double gen_smem[];
    const unsigned bid = blockIdx.x;
    const int grp = (int)(bid % (unsigned)a.ngroups);
    const unsigned rest = bid / (unsigned)a.ngroups;
    const int s = (int)(rest % (unsigned)a.sets);
    const size_t z = rest / (unsigned)a.sets;
    GenCtx<T> c;
    c.a = &a;
    c.tw = tw;
    c.lds = reinterpret_cast<C2<T> *>(gen_smem);
    c.L = gp.L;
    c.s = s;
    c.g0 = grp * a.G;
    c.nvalid = min(a.G, a.nl - c.g0);
    c.in = in + z * (size_t)a.pz + (size_t)s * (size_t)a.ps_in + (size_t)c.g0 * (size_t)a.pg_in;
    c.out = out + z * (size_t)a.pz + (size_t)s * (size_t)a.ps_out + (size_t)c.g0 * (size_t)a.pg_out;
    c.scale = scale;
    c.occ = nullptr;
    c.occ_stride = c.occ_shift = 0;
    if (oc.rows) {
        unsigned char *occ = reinterpret_cast<unsigned char *>(gen_smem) + occ_off;
        const unsigned char *rows = oc.rows + z * (size_t)oc.ny;
        if (oc.offsets) {
            // Rows g0 .. of plane z: none live -> their transforms are zero,
            // neither computed nor written; else the tiles of the live ones.
            int live = 0;
            for (int g = threadIdx.x; g < c.nvalid; g += blockDim.x) live |= rows[c.g0 + g];
            if (!__syncthreads_or(live)) return;
            for (int i = threadIdx.x; i < c.nvalid * oc.tiles_u; i += blockDim.x) {
                const int g = i / oc.tiles_u, t = i - g * oc.tiles_u, v = c.g0 + g;
                const size_t b = (z * oc.tiles_v + v / oc.tv) * oc.tiles_u + t;
                occ[i] = rows[v] && oc.offsets[b] != oc.offsets[b + 1];
            }
            c.occ_stride = oc.tiles_u;
            c.occ_shift = oc.tu_shift;
        } else {
            // Columns: the flags of this set's input rows.
            for (int n = threadIdx.x; n < gp.L; n += blockDim.x)
                occ[n] = rows[s * a.set_mul + n * a.row_mul];
        }
        c.occ = occ;
        __syncthreads();
    }
    GenStore sink;
    gen_lines_of<T, HARD>(c, gp, sink);
}

// Last pass of a four-step column axis, the phase correction and the plane sum in
// one: each plane is read once, and not written and read again.  A thread holds 10
// values (with 16, and their sums, 776 registers spill), so radices above 10 are not
// used here.  Bound by the vector units now, half of it the sines, at 2 waves per
// SIMD: last pass and phase of 8 planes of 3000^2 752 -> 663 us, of 10 of 1920 x 2560
// 462 -> 370, of 16 of 960 x 3000 480 -> 400, of 30 of 2400 x 1280 819 -> 811.
__global__ void __launch_bounds__(kGenThreads)
k_fft_gen_phase(GenPassDesc gp, GenAddr a, const C2<double> *__restrict__ tw,
                const C2<double> *in, PhaseGeom pg, double *ore, double *oim)
{
    extern __shared__ double gen_smem[];
    const int grp = (int)(blockIdx.x % (unsigned)a.ngroups);
    const int s = (int)(blockIdx.x / (unsigned)a.ngroups);
    GenCtx<double> c;
    c.a = &a;
    c.tw = tw;
    c.lds = reinterpret_cast<C2<double> *>(gen_smem);
    c.L = gp.L;
    c.s = s;
    c.g0 = grp * a.G;
    c.nvalid = min(a.G, a.nl - c.g0);
    c.in = in + (size_t)s * (size_t)a.ps_in + (size_t)c.g0 * (size_t)a.pg_in;
    c.out = nullptr;
    c.scale = 1.0;
    c.occ = nullptr;
    c.occ_stride = c.occ_shift = 0;
    GenPhase sink;
    sink.g = pg;
    sink.ore = ore;
    sink.oim = oim;
    sink.row_mul = a.sets;
    sink.phase = pg.phase_on && pg.planes > 1;
    for (int iw = 0; iw < pg.planes; ++iw, c.in += a.pz) {
        sink.iw = iw;
        gen_lines_of<double, false>(c, gp, sink);
    }
}

// Bluestein pre-multiply: w[c*M + m] = x[line l0+c][m] * b[m] for m < N, else 0.
template <typename T>
__global__ void __launch_bounds__(256)
k_blue_pre(const C2<T> *__restrict__ x, size_t base, long long ls, long long es, int l0, int cl,
           int N, int M, const C2<T> *__restrict__ chirp, C2<T> *__restrict__ w)
{
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)cl * M) return;
    int cc, m;
    if (es == 1) { cc = (int)(idx / M); m = (int)(idx % M); }
    else { m = (int)(idx / cl); cc = (int)(idx % cl); }
    C2<T> v{T(0), T(0)};
    if (m < N) v = cmul(x[base + (size_t)(l0 + cc) * ls + (size_t)m * es], chirp[m]);
    w[(size_t)cc * M + m] = v;
}

// w *= H (the M-point transform of the wrapped conjugate chirp), per line.
template <typename T>
__global__ void __launch_bounds__(256)
k_blue_mul(C2<T> *__restrict__ w, const C2<T> *__restrict__ h, int cl, int M)
{
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)cl * M) return;
    w[idx] = cmul(w[idx], h[idx % M]);
}

// Bluestein post-multiply: X[k] = b[k] * scale/M * F(w)[(M-k) mod M], k < N.
template <typename T>
__global__ void __launch_bounds__(256)
k_blue_post(const C2<T> *__restrict__ w, int cl, int N, int M, const C2<T> *__restrict__ chirp,
            T scale, C2<T> *__restrict__ y, size_t base, long long ls, long long es, int l0)
{
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)cl * N) return;
    int cc, k;
    if (es == 1) { cc = (int)(idx / N); k = (int)(idx % N); }
    else { k = (int)(idx / cl); cc = (int)(idx % cl); }
    C2<T> v = cmul(w[(size_t)cc * M + (size_t)((M - k) % M)], chirp[k]);
    v.x *= scale;
    v.y *= scale;
    y[base + (size_t)(l0 + cc) * ls + (size_t)k * es] = v;
}

// ---------------------------------------------------------------------------
// Host side.

// Radices of a direct length: the fewest passes, then the most of radix 16, then
// the largest smallest radix (a small radix leaves lanes idle between the larger
// ones).  Radix 16 first keeps the error of powers of two and their small multiples
// down: 1024 points as 16 x 8 x 8 are off by up to 8 % more than as 16 x 16 x 4.  False
// if L has a prime factor above 13.
void gen_search(int rest, int max_r, std::vector<int> &cur, std::vector<int> &best)
{
    if (rest == 1) {
        const auto n16 = [](const std::vector<int> &r) { return std::count(r.begin(), r.end(), 16); };
        if (best.empty() || cur.size() < best.size() ||
            (cur.size() == best.size() && n16(cur) == n16(best) && cur.back() > best.back()))
            best = cur;   // (the search tries more 16s first)
        return;
    }
    if (!best.empty() && cur.size() >= best.size()) return;
    for (int r = std::min(max_r, rest); r >= 2; --r)
        if (rest % r == 0) {
            cur.push_back(r);
            gen_search(rest / r, r, cur, best);
            cur.pop_back();
        }
}

bool gen_radices(int L, GenPassDesc &gp, int values = kGenValues)
{
    gp = GenPassDesc{};
    gp.L = L;
    if (L < 2 || L > kGenElems) return false;
    std::vector<int> cur, best;
    gen_search(L, values, cur, best);
    if (best.empty() || (int)best.size() > kGenMaxPasses) return false;
    int Ns = 1;
    for (int r : best) {
        GenPass &ps = gp.pass[gp.np++];
        ps.R = r;
        ps.Ns = Ns;
        ps.Lr = L / r;
        ps.mNs = gen_magic((uint32_t)Ns);
        ps.mLr = gen_magic((uint32_t)ps.Lr);
        Ns *= r;
    }
    return true;
}

// Threads that G lines of this plan take (0: more than a workgroup has).
int gen_threads(const GenPassDesc &gp, int G, int values = kGenValues)
{
    int need = 1;
    for (int p = 0; p < gp.np; ++p) {
        const int nb = G * gp.pass[p].Lr, bpt = gen_bpt(gp.pass[p].R, values);
        need = std::max(need, (nb + bpt - 1) / bpt);
    }
    return need > kGenThreads ? 0 : (need + 63) / 64 * 64;
}

// Lines per workgroup: as many as the threads and `elems` LDS elements take,
// whole groups of 8 lines where lines are adjacent in memory (128-byte runs).
int gen_lines(const GenPassDesc &gp, int nl, int elems, bool adjacent, int values = kGenValues)
{
    int G = std::max(1, std::min(nl, elems / gp.L));
    while (G > 1 && !gen_threads(gp, G, values)) --G;
    if (adjacent && G > 8 && G < nl) G = G / 8 * 8;
    return G;
}

bool smooth(long long n)
{
    for (int p : {2, 3, 5, 7, 11, 13})
        while (n % p == 0) n /= p;
    return n == 1;
}

// Split n = n1 * n2 with both direct lengths, n1 closest to sqrt(n); false if none.
bool gen_split(int n, int &n1, int &n2)
{
    int best = 0;
    double bestd = 1e300;
    for (int d = 2; d <= kGenElems && d <= n / 2; ++d) {
        if (n % d) continue;
        const int e = n / d;
        if (e < 2 || e > kGenElems || !smooth(d) || !smooth(e)) continue;
        const double dist = std::fabs(std::log((double)d) - 0.5 * std::log((double)n));
        if (dist < bestd) {
            bestd = dist;
            best = d;
        }
    }
    if (!best) return false;
    n1 = best;
    n2 = n / best;
    return true;
}

// Direct (0) or four-step (1) plan of a smooth length on a given axis kind.
bool plan_smooth(int n, bool rows, int &mode, int &n1, int &n2, GenPassDesc &a, GenPassDesc &b)
{
    const int direct_max = rows ? kGenElems : kGenDirectCols;
    if (n <= direct_max && gen_radices(n, a)) {
        mode = 0;
        n1 = n;
        n2 = 1;
        return true;
    }
    if (!gen_split(n, n1, n2)) {
        // A short smooth column with no split (a prime <= 13 times little):
        // one pass even if narrower than the coalescing target.
        if (n <= kGenElems && gen_radices(n, a)) {
            mode = 0;
            n1 = n;
            n2 = 1;
            return true;
        }
        return false;
    }
    mode = 1;
    return gen_radices(n1, a) && gen_radices(n2, b);
}

// exp(+2 pi i m/n) and the Bluestein tables, in long double.
void host_twiddles(long long n, std::vector<long double> &re_im)
{
    re_im.resize(2 * (size_t)n);
    const long double pi = 3.141592653589793238462643383279502884L;
    for (long long m = 0; m < n; ++m) {
        const long double a = 2.0L * pi * (long double)m / (long double)n;
        re_im[2 * m] = cosl(a);
        re_im[2 * m + 1] = sinl(a);
    }
}

// In-place sign +1 DFT of a power-of-two length (host, long double; radix 2).
void host_fft_pow2(std::vector<long double> &x, long long n)
{
    for (long long i = 1, j = 0; i < n; ++i) {
        long long bit = n >> 1;
        for (; j & bit; bit >>= 1) j ^= bit;
        j ^= bit;
        if (i < j) {
            std::swap(x[2 * i], x[2 * j]);
            std::swap(x[2 * i + 1], x[2 * j + 1]);
        }
    }
    std::vector<long double> tw;
    host_twiddles(n, tw);
    for (long long len = 2; len <= n; len <<= 1) {
        const long long half = len >> 1, step = n / len;
        for (long long s = 0; s < n; s += len)
            for (long long k = 0; k < half; ++k) {
                const long double wr = tw[2 * (k * step)], wi = tw[2 * (k * step) + 1];
                long double *pa = &x[2 * (s + k)], *pb = &x[2 * (s + k + half)];
                const long double br = pb[0] * wr - pb[1] * wi, bi = pb[0] * wi + pb[1] * wr;
                pb[0] = pa[0] - br;
                pb[1] = pa[1] - bi;
                pa[0] += br;
                pa[1] += bi;
            }
    }
}

// Lines of one axis per plane: rows (axis 0) are ny lines of nx contiguous
// elements; columns (axis 1) are nx lines of ny elements at stride nx.
struct AxisGeom {
    int n, nl;
    long long es, ls;
};

AxisGeom axis_geom(int axis, int nx, int ny)
{
    if (axis == 0) return AxisGeom{nx, ny, 1, nx};
    return AxisGeom{ny, nx, nx, 1};
}

size_t csize(int precision) { return precision == RICK_FP64 ? 16 : 8; }

// LDS elements of a workgroup's lines: two workgroups per CU in FP64, and as
// many bytes in FP32 (longer runs of adjacent columns).
template <typename T>
constexpr int gen_elems() { return sizeof(T) == 8 ? 4096 : 8192; }

// Lines of a workgroup of the fused last column pass, or 0 where the pass is not
// used: it walks the planes one after another, so images that fill the chip less
// than four times over are faster apart (1000^2 x 8 88 us, fused 119; 1500^2 x 8 200
// and 218), the larger among them not always (2000^2 x 8 347 and 291).  FP32 is faster
// apart too, the plain pass having six waves per SIMD (3000^2 x 8, before every twiddle
// came from the table: 375 us, fused 463; apart now 411).
int gen_phase_lines(const GenPassDesc &gp, int nl, int sets)
{
    if (gp.np == 0) return 0;
    const int G = gen_lines(gp, nl, gen_elems<double>(), true, kPhaseValues);
    if (!gen_threads(gp, G, kPhaseValues)) return 0;   // radix 6 or 7 of a line above 3072
    return (long long)((nl + G - 1) / G) * sets >= 1024 ? G : 0;
}

hipError_t launch_gen_phase(GenPassDesc gp, GenAddr a, int G, const void *tw, long long ntab,
                            const void *in, const PhaseGeom &pg, double *re, double *im,
                            hipStream_t s)
{
    a.G = G;
    a.mG = gen_magic((uint32_t)G);
    a.ngroups = (a.nl + G - 1) / G;
    const int nt = gen_threads(gp, G, kPhaseValues);
    const size_t lds = gp.np == 1 ? 0 : (size_t)G * gp.L * sizeof(C2<double>);
    const unsigned long long blocks = (unsigned long long)a.ngroups * a.sets;
    if (!nt || blocks > 0x7fffffffull || lds > (size_t)kGenLdsBytes)
        return hipErrorInvalidConfiguration;
    for (int p = 0; p < gp.np; ++p)
        gp.pass[p].tstep = (int)(ntab / ((long long)gp.pass[p].Ns * gp.pass[p].R));
    hipLaunchKernelGGL(k_fft_gen_phase, dim3((unsigned)blocks), dim3(nt), lds, s, gp, a,
                       static_cast<const C2<double> *>(tw), static_cast<const C2<double> *>(in),
                       pg, re, im);
    return hipGetLastError();
}

template <typename T>
hipError_t launch_gen(GenPassDesc gp, GenAddr a, long long planes, const void *tw,
                      long long ntab, const void *in, void *out, double scale, hipStream_t s,
                      const GenOcc &oc = GenOcc{})
{
    a.G = gen_lines(gp, a.nl, gen_elems<T>(), !a.line_major);
    a.mG = gen_magic((uint32_t)a.G);
    a.ngroups = (a.nl + a.G - 1) / a.G;
    const int nt = gen_threads(gp, a.G);
    if (!nt) return hipErrorInvalidConfiguration;
    bool hard = false;
    for (int p = 0; p < gp.np; ++p) {
        gp.pass[p].tstep = (int)(ntab / ((long long)gp.pass[p].Ns * gp.pass[p].R));
        hard |= gp.pass[p].R == 11 || gp.pass[p].R == 13;
    }
    const unsigned long long blocks = (unsigned long long)a.ngroups * a.sets * planes;
    if (blocks == 0) return hipSuccess;
    if (blocks > 0x7fffffffull) return hipErrorInvalidConfiguration;
    size_t lds = a.line_major ? (size_t)a.G * (gen_pad(gp.L) + 1) : (size_t)a.G * gp.L;
    if (gp.np == 1) lds = 0;   // no exchange
    lds *= sizeof(C2<T>);
    const int occ_off = (int)lds;
    if (oc.rows) lds += (size_t)(oc.offsets ? a.G * oc.tiles_u : gp.L) + 16;
    if (lds > (size_t)kGenLdsBytes) return hipErrorInvalidConfiguration;
    auto kernel = hard ? k_fft_gen<T, true> : k_fft_gen<T, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(nt), lds, s, gp, a,
                       static_cast<const C2<T> *>(tw), static_cast<const C2<T> *>(in),
                       static_cast<C2<T> *>(out), (T)scale, oc, occ_off);
    return hipGetLastError();
}

// Addresses of a direct axis, and of the two passes of a four-step axis
// (n = n1 * n2): A reads elements n2 + N2*n1 and writes them, times
// W_N^(k1*n2), at n2 + N2*k1; B reads N2*k1 + n2 and writes X[k1 + N1*k2] at
// that element, or (in_place) at N2*k1 + k2.
GenAddr direct_addr(const AxisGeom &ag, bool rows, long long plane_elems)
{
    GenAddr a{};
    a.nl = ag.nl;
    a.sets = 1;
    a.pz = plane_elems;
    a.pg_in = a.pg_out = ag.ls;
    a.pe_in = a.pe_out = ag.es;
    a.line_major = rows ? 1 : 0;
    a.row_mul = 1;
    return a;
}

GenAddr step_a_addr(const GenAxis &ax, const AxisGeom &ag, bool rows, long long plane_elems)
{
    GenAddr A{};
    const int N2 = ax.n2;
    A.pz = plane_elems;
    if (rows) {
        A.nl = N2; A.sets = ag.nl;
        A.pg_in = A.pg_out = 1;
        A.ps_in = A.ps_out = ag.ls;
        A.pe_in = A.pe_out = (long long)N2;
        A.tw_by = 2;
    } else {
        A.nl = ag.nl; A.sets = N2;
        A.pg_in = A.pg_out = ag.ls;
        A.ps_in = A.ps_out = ag.es;
        A.pe_in = A.pe_out = (long long)N2 * ag.es;
        A.tw_by = 1;
        A.row_mul = N2;
        A.set_mul = 1;
    }
    return A;
}

GenAddr step_b_addr(const GenAxis &ax, const AxisGeom &ag, bool rows, long long plane_elems,
                    bool in_place)
{
    GenAddr B{};
    const int N1 = ax.n1, N2 = ax.n2;
    B.pz = plane_elems;
    if (rows) {
        B.nl = N1; B.sets = ag.nl;
        B.pg_in = N2; B.pe_in = 1; B.ps_in = ag.ls;
        B.pg_out = 1; B.pe_out = N1; B.ps_out = ag.ls;
        B.line_major = 1;
    } else {
        B.nl = ag.nl; B.sets = N1;
        B.pg_in = B.pg_out = ag.ls;
        B.ps_in = (long long)N2 * ag.es; B.pe_in = ag.es;
        B.ps_out = in_place ? B.ps_in : ag.es;
        B.pe_out = in_place ? B.pe_in : (long long)N1 * ag.es;
    }
    return B;
}

// One smooth axis transform of `planes` planes (direct: all planes in one
// launch; four-step: per plane through the scratch plane `tmp`).
template <typename T>
hipError_t smooth_axis(const GenAxis &ax, const AxisGeom &ag, bool rows, int planes,
                       long long plane_elems, const void *tw, const C2<T> *in, C2<T> *out,
                       C2<T> *tmp, double scale, hipStream_t s)
{
    const int n = ag.n;
    if (ax.mode == 0)
        return launch_gen<T>(ax.a, direct_addr(ag, rows, plane_elems), planes, tw, n, in, out,
                             scale, s);
    const GenAddr A = step_a_addr(ax, ag, rows, 0), B = step_b_addr(ax, ag, rows, 0, false);
    for (int z = 0; z < planes; ++z) {
        const size_t at = (size_t)z * plane_elems;
        hipError_t e = launch_gen<T>(ax.a, A, 1, tw, n, in + at, tmp, 1.0, s);
        if (e != hipSuccess) return e;
        e = launch_gen<T>(ax.b, B, 1, tw, n, tmp, out + at, scale, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// The transform of the image chain on a sparse grid, in place: live rows over
// their occupied tiles, then the columns reading the other rows as zero.  A
// four-step column axis leaves X[k1 + N1*k2] in row N2*k1 + k2.
template <typename T>
hipError_t gen_chain(const GenFft &g, int planes, int nx, int ny, void *grid_v, double scale,
                     hipStream_t s, Timing *tm, const GridGeom &geom, const uint32_t *offsets,
                     const unsigned char *rowlive, const PhaseGeom &pg, double *re, double *im)
{
    C2<T> *grid = static_cast<C2<T> *>(grid_v);
    const long long plane = (long long)nx * ny;
    const AxisGeom ag0 = axis_geom(0, nx, ny), ag1 = axis_geom(1, nx, ny);
    const GenAxis &ay = g.ax[1];
    GenOcc oc{offsets, rowlive, geom.tu_shift, geom.tv, geom.tiles_u, geom.tiles_v, ny};
    tm->begin(RICK_STAGE_FFT_ROWS, s);
    hipError_t e = launch_gen<T>(g.ax[0].a, direct_addr(ag0, true, plane), planes, g.ax[0].tw, nx,
                                 grid, grid, scale, s, oc);
    tm->end(RICK_STAGE_FFT_ROWS, s);
    if (e != hipSuccess) return e;
    oc.offsets = nullptr;
    tm->begin(RICK_STAGE_FFT_COLS, s);
    if (ay.mode == 0)
        e = launch_gen<T>(ay.a, direct_addr(ag1, false, plane), planes, ay.tw, ny, grid, grid,
                          1.0, s, oc);
    else
        e = launch_gen<T>(ay.a, step_a_addr(ay, ag1, false, plane), planes, ay.tw, ny, grid, grid,
                          1.0, s, oc);
    tm->end(RICK_STAGE_FFT_COLS, s);
    if (e != hipSuccess) return e;
    const int prec = sizeof(T) == 8 ? RICK_FP64 : RICK_FP32;
    if (ay.mode == 0) return launch_phase(pg, prec, grid, re, im, 0, s, tm);
    const GenAddr B = step_b_addr(ay, ag1, false, plane, true);
    const int G = prec == RICK_FP64 ? gen_phase_lines(ay.p, B.nl, B.sets) : 0;
    if (G) {
        tm->begin(RICK_STAGE_PHASE, s);
        e = launch_gen_phase(ay.p, B, G, ay.tw, ny, grid, pg, re, im, s);
        tm->end(RICK_STAGE_PHASE, s);
        return e;
    }
    tm->begin(RICK_STAGE_FFT_COLS_B, s);
    e = launch_gen<T>(ay.b, B, planes, ay.tw, ny, grid, grid, 1.0, s);
    tm->end(RICK_STAGE_FFT_COLS_B, s);
    if (e != hipSuccess) return e;
    return launch_phase(pg, prec, grid, re, im, 0, s, tm, ay.n1, ay.n2);
}

template <typename T>
hipError_t blue_axis(const GenAxis &ax, const AxisGeom &ag, int planes, long long plane_elems,
                     const C2<T> *in, C2<T> *out, void *work, double scale, hipStream_t s)
{
    const int N = ag.n, M = ax.m;
    const int chunk = (int)std::max<size_t>(1, std::min<size_t>((size_t)ag.nl, kBlueChunk / M));
    C2<T> *w1 = static_cast<C2<T> *>(work);
    C2<T> *w2 = w1 + (size_t)chunk * M;
    // The conv FFT's own plan: rows of length M, direct or four-step.
    GenAxis conv{};
    conv.mode = ax.mmode;
    conv.n1 = ax.m1;
    conv.n2 = ax.m2;
    conv.a = ax.ma;
    conv.b = ax.mb;
    for (int z = 0; z < planes; ++z) {
        const size_t pbase = (size_t)z * plane_elems;
        for (int l0 = 0; l0 < ag.nl; l0 += chunk) {
            const int cl = std::min(chunk, ag.nl - l0);
            const size_t nw = (size_t)cl * M;
            hipLaunchKernelGGL(k_blue_pre<T>, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, s,
                               in, pbase, ag.ls, ag.es, l0, cl, N, M,
                               static_cast<const C2<T> *>(ax.chirp), w1);
            hipError_t e = hipGetLastError();
            if (e != hipSuccess) return e;
            const AxisGeom cg{M, cl, 1, M};
            e = smooth_axis<T>(conv, cg, true, 1, 0, ax.tw, w1, w1, w2, 1.0, s);
            if (e != hipSuccess) return e;
            hipLaunchKernelGGL(k_blue_mul<T>, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, s,
                               w1, static_cast<const C2<T> *>(ax.hf), cl, M);
            e = hipGetLastError();
            if (e != hipSuccess) return e;
            e = smooth_axis<T>(conv, cg, true, 1, 0, ax.tw, w1, w1, w2, 1.0, s);
            if (e != hipSuccess) return e;
            const size_t ny_ = (size_t)cl * N;
            hipLaunchKernelGGL(k_blue_post<T>, dim3((unsigned)((ny_ + 255) / 256)), dim3(256), 0,
                               s, w1, cl, N, M, static_cast<const C2<T> *>(ax.chirp),
                               (T)(scale / (double)M), out, pbase, ag.ls, ag.es, l0);
            e = hipGetLastError();
            if (e != hipSuccess) return e;
        }
    }
    return hipSuccess;
}

template <typename T>
hipError_t gen_impl(const GenFft &g, int planes, int nx, int ny, const void *in_v, void *out_v,
                    double scale, hipStream_t s, Timing *tm)
{
    const C2<T> *in = static_cast<const C2<T> *>(in_v);
    C2<T> *out = static_cast<C2<T> *>(out_v);
    const long long plane = (long long)nx * ny;
    // Columns first (reading `in`), then rows in place on `out`, scaled.
    for (int axis = 1; axis >= 0; --axis) {
        const GenAxis &ax = g.ax[axis];
        const AxisGeom ag = axis_geom(axis, nx, ny);
        const C2<T> *src = axis == 1 ? in : out;
        const double sc = axis == 0 ? scale : 1.0;
        const int st = axis == 0 ? RICK_STAGE_FFT_ROWS : RICK_STAGE_FFT_COLS;
        tm->begin(st, s);
        hipError_t e;
        if (ax.mode == 2)
            e = blue_axis<T>(ax, ag, planes, plane, src, out, g.work, sc, s);
        else
            e = smooth_axis<T>(ax, ag, axis == 0, planes, plane, ax.tw, src, out,
                               static_cast<C2<T> *>(g.work), sc, s);
        tm->end(st, s);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace

bool gen_fft_prepare(int nx, int ny, int precision, GenFft *g)
{
    *g = GenFft{};
    const size_t cs = csize(precision);
    size_t tables = 0, work = 0;
    for (int axis = 0; axis < 2; ++axis) {
        GenAxis &ax = g->ax[axis];
        const AxisGeom ag = axis_geom(axis, nx, ny);
        ax.n = ag.n;
        if (ag.n < 2) return false;
        if (smooth(ag.n) && plan_smooth(ag.n, axis == 0, ax.mode, ax.n1, ax.n2, ax.a, ax.b)) {
            if (axis == 1 && ax.mode == 1) gen_radices(ax.n2, ax.p, kPhaseValues);
            tables += (cs * (size_t)ag.n + 255) / 256 * 256;
            if (ax.mode == 1) work = std::max(work, cs * (size_t)nx * ny);
            continue;
        }
        // Bluestein.
        long long M = 1;
        while (M < 2LL * ag.n - 1) M <<= 1;
        if (M > (1LL << 24)) return false;
        ax.mode = 2;
        ax.m = (int)M;
        if (!plan_smooth(ax.m, true, ax.mmode, ax.m1, ax.m2, ax.ma, ax.mb)) return false;
        tables += 2 * ((cs * (size_t)M + 255) / 256 * 256) + (cs * (size_t)ag.n + 255) / 256 * 256;
        const size_t chunk = std::max<size_t>(1, std::min<size_t>((size_t)ag.nl, kBlueChunk / M));
        work = std::max(work, cs * chunk * (size_t)M * (ax.mmode == 1 ? 2 : 1));
    }
    g->table_bytes = tables;
    g->work_bytes = work;
    return true;
}

hipError_t gen_fft_upload(GenFft *g, int precision, void *tables, void *work)
{
    // Padded lines of 4096 FP64 elements take 69 KB of LDS.
    for (const void *k : {reinterpret_cast<const void *>(&k_fft_gen<double, false>),
                          reinterpret_cast<const void *>(&k_fft_gen<double, true>),
                          reinterpret_cast<const void *>(&k_fft_gen<float, false>),
                          reinterpret_cast<const void *>(&k_fft_gen<float, true>)}) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 kGenLdsBytes);
        if (e != hipSuccess) return e;
    }
    char *p = static_cast<char *>(tables);
    const size_t cs = csize(precision);
    auto put = [&](const std::vector<long double> &v, size_t n) -> const void * {
        void *dst = p;
        p += (cs * n + 255) / 256 * 256;
        if (precision == RICK_FP64) {
            std::vector<double> d(v.begin(), v.begin() + 2 * n);
            return hipMemcpy(dst, d.data(), 16 * n, hipMemcpyHostToDevice) == hipSuccess ? dst
                                                                                         : nullptr;
        }
        std::vector<float> f(v.begin(), v.begin() + 2 * n);
        return hipMemcpy(dst, f.data(), 8 * n, hipMemcpyHostToDevice) == hipSuccess ? dst
                                                                                    : nullptr;
    };
    std::vector<long double> t;
    for (int axis = 0; axis < 2; ++axis) {
        GenAxis &ax = g->ax[axis];
        if (ax.mode != 2) {
            host_twiddles(ax.n, t);
            if (!(ax.tw = put(t, ax.n))) return hipErrorUnknown;
            continue;
        }
        const long long N = ax.n, M = ax.m;
        host_twiddles(M, t);
        if (!(ax.tw = put(t, M))) return hipErrorUnknown;
        // b[n] = exp(+i pi n^2 / N), with n^2 reduced mod 2N.
        const long double pi = 3.141592653589793238462643383279502884L;
        std::vector<long double> b(2 * N);
        for (long long k = 0; k < N; ++k) {
            const long long q = (long long)((unsigned long long)k * (unsigned long long)k %
                                            (unsigned long long)(2 * N));
            const long double a = pi * (long double)q / (long double)N;
            b[2 * k] = cosl(a);
            b[2 * k + 1] = sinl(a);
        }
        if (!(ax.chirp = put(b, N))) return hipErrorUnknown;
        // H = F_M(h), h[d mod M] = conj(b[|d|]) for |d| < N.
        std::vector<long double> h(2 * M, 0.0L);
        for (long long k = 0; k < N; ++k) {
            h[2 * k] = b[2 * k];
            h[2 * k + 1] = -b[2 * k + 1];
            if (k) {
                h[2 * (M - k)] = b[2 * k];
                h[2 * (M - k) + 1] = -b[2 * k + 1];
            }
        }
        host_fft_pow2(h, M);
        if (!(ax.hf = put(h, M))) return hipErrorUnknown;
    }
    g->work = work;
    return hipSuccess;
}

bool gen_chain_ok(const GenFft &g)
{
    return g.ax[0].mode == 0 && g.ax[1].mode != 2;
}

hipError_t launch_gen_chain(const GenFft &g, int precision, int planes, int nx, int ny, void *grid,
                            double scale, hipStream_t s, Timing *tm, const GridGeom &geom,
                            const uint32_t *offsets, const unsigned char *rowlive,
                            const PhaseGeom &pg, double *re, double *im)
{
    Timing off;
    if (tm == nullptr) tm = &off;
    if (precision == RICK_FP64)
        return gen_chain<double>(g, planes, nx, ny, grid, scale, s, tm, geom, offsets, rowlive, pg,
                                 re, im);
    return gen_chain<float>(g, planes, nx, ny, grid, scale, s, tm, geom, offsets, rowlive, pg, re,
                            im);
}

hipError_t launch_fft_gen(const GenFft &g, int precision, int planes, int nx, int ny,
                          const void *in, void *out, double scale, hipStream_t s, Timing *tm)
{
    Timing off;
    if (tm == nullptr) tm = &off;
    if (precision == RICK_FP64)
        return gen_impl<double>(g, planes, nx, ny, in, out, scale, s, tm);
    return gen_impl<float>(g, planes, nx, ny, in, out, scale, s, tm);
}

}  // namespace rick
