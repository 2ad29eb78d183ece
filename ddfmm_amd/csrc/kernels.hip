// HIP kernels of the directional-FMM evaluation for gfx950 (CDNA4, wave64).
//
//   kapply_kernel  generated-kernel block apply: out(t_i) (+)= sum_j G(t_i, s_j) v_j with
//                  LDS-staged source tiles; serves the near field (U list), S2M, L2T,
//                  W/X lists (Kernel3d::kernel + zgemv, kernel3d.cpp:26-107,
//                  wave3d_eval.cpp:441-451, 550-560, 585-718)
//   gemm_kernel    grouped complex GEMM on MFMA (16x16x4, f64 or f32) over (box, rhs)
//                  columns with gather/scatter and store/add epilogues: every translation
//                  the reference applies as a per-box zgemv (vecmatop.cpp:102-125)
//   reduce_kernel  fixed-order sum of per-contribution slots: the HF M2L/L2L targets
//                  (the reference's zgemv accumulations into one vector) and the
//                  near-field mirror products of pairs evaluated once
//   fft_fwd_kernel / vlist_acc_kernel / vlist_inv_kernel
//                  FFT-diagonal LF M2L on the (2P)^3 grid
//                  (wave3d_eval.cpp:602-661)
//   kgen_kernel    setup-time translation-matrix generation (mlib3d.cpp:106-280 and the
//                  per-offset HF M2L matrices of wave3d_eval.cpp:876-928)
//
// Vectors are double2 (FP64 mode) or float2 (mixed mode).  In the mixed mode the
// kernel G is evaluated from FP64 coordinate differences with FP32 sqrt/rcp and the
// hardware sin/cos on the phase reduced to [0, 1) revolutions (k = 2*pi, so
// exp(ikr) = exp(2*pi*i*fract(r))).
#include <hip/hip_runtime.h>

#include <mutex>
#include <vector>

#include "device.hpp"

// No implicit FP contraction: a + b * c is fused only where the code says fma.  Kernels
// that serve different right-hand-side counts (1-RHS and multi-RHS instances) then round
// every operation the same way, which keeps each right-hand side's bits independent of
// the batch it is evaluated in.
#pragma clang fp contract(off)

namespace ddfmm {

namespace {

template <class V> struct Real;
template <> struct Real<double2> { using T = double; };
template <> struct Real<float2> { using T = float; };

template <class V>
__device__ __forceinline__ V mk(double x, double y) {
    V v;
    v.x = (typename Real<V>::T)x;
    v.y = (typename Real<V>::T)y;
    return v;
}

template <class V>
__device__ __forceinline__ void cfma(V& acc, V a, V b) {
    acc.x = fma(a.x, b.x, fma(-a.y, b.y, acc.x));
    acc.y = fma(a.x, b.y, fma(a.y, b.x, acc.y));
}

// FP64 G(r), k = 2*pi: e^{ikr}/r (type 0) or e^{ikr} (type 1); r^2 < 1e-16 => r := 1.
// Library functions: the operator tables, generated once, keep these roundings (their FP32
// copies decide the last bits of every mixed evaluation).
__device__ __forceinline__ double2 green64_table(double dx, double dy, double dz, int ktype) {
    double r2 = fma(dz, dz, fma(dy, dy, dx * dx));
    r2 = r2 < 1e-16 ? 1.0 : r2;
    double r = sqrt(r2);
    double s, c;
    sincospi(2.0 * r, &s, &c);
    if (ktype == 0) {
        double ir = 1.0 / r;
        return make_double2(c * ir, s * ir);
    }
    return make_double2(c, s);
}

// The same for the pair loops (direct sum, FP64 near field), which its instructions bound:
// about 50 a pair where the library functions take about 130.  r and 1/r by Goldschmidt's
// iteration from one v_rsq_f64, each corrected by its residual; sin and cos of the phase,
// r revolutions, on the eighth of a turn around the nearest quarter (the reduction is
// exact), by polynomials that interpolate sin(2 pi f) / f and cos(2 pi f) at Chebyshev
// points of f^2 in [0, 1/64] (within 4e-17 and 2e-17 of them; f in quarter turns below).
// The largest errors against long double are those of the library functions (r from 1e-6
// to 1e7: G r within 2.1 (2 pi r + 1) 2^-53 where r's own rounding dominates).
// Direct sum at 1000 targets of 1M sources 3.19 -> 2.02 ms, FP64 near field of 60k points
// 0.242 -> 0.166 ms.
template <int KT>
__device__ __forceinline__ double2 green64(double dx, double dy, double dz) {
    double r2 = fma(dz, dz, fma(dy, dy, dx * dx));
    r2 = r2 < 1e-16 ? 1.0 : r2;
    const double y = __builtin_amdgcn_rsq(r2);
    double r = r2 * y, h = 0.5 * y;          // -> sqrt(r2), 1 / (2 sqrt(r2))
    const double e = fma(-r, h, 0.5);
    r = fma(r, e, r);
    h = fma(h, e, h);
    r = fma(fma(-r, r, r2), h, r);
    const double t = __builtin_amdgcn_fract(r);
    const double big = 6755399441055744.0;   // 1.5 * 2^52: rounds 4 t to an integer, in its low bits
    const double m = fma(4.0, t, big);
    const double f = fma(4.0, t, big - m), u = f * f;      // [-1/2, 1/2] quarter turns
    const int q = __double2loint(m);
    // coefficients of sin(pi f / 2) / f and cos(pi f / 2) in u: those of the revolution's
    // polynomials over 4^(2 i + 1) and 4^(2 i)
    double s = 5.6339337815378543e-08, c = -6.3212568696285881e-09;
    c = fma(c, u, 4.7106097267578228e-07);
    s = fma(s, u, -3.5986433529823099e-06);
    c = fma(c, u, -2.520203677046026e-05);
    s = fma(s, u, 0.00016044115074219091);
    c = fma(c, u, 0.00091926027418315576);
    s = fma(s, u, -0.0046817541323409756);
    c = fma(c, u, -0.02086348076331121);
    s = fma(s, u, 0.079692626246043008);
    c = fma(c, u, 0.2536695079010467);
    s = fma(s, u, -0.64596409750624428);
    c = fma(c, u, -1.2337005501361697);
    s = fma(s, u, 1.5707963267948966) * f;
    c = fma(c, u, 1.0);
    // the turn by q quarters: swapped for odd q, signs by its second bit
    const double sn = q & 1 ? c : s, cs = q & 1 ? s : c;
    s = __hiloint2double(__double2hiint(sn) ^ ((q & 2) << 30), __double2loint(sn));
    c = __hiloint2double(__double2hiint(cs) ^ (((q + 1) & 2) << 30), __double2loint(cs));
    if (KT == 0) {
        double ir = h + h;
        ir = fma(ir, fma(-r, ir, 1.0), ir);
        return make_double2(c * ir, s * ir);
    }
    return make_double2(c, s);
}

// FP32 G(r) from FP64 differences: r^2 in FP64 (full-rate FMAs, one conversion), 1/r from
// v_rsq_f32, r = r^2 / r, and v_sin_f32 / v_cos_f32 on the phase fract(r) in revolutions
// (three transcendental operations).
__device__ __forceinline__ float2 green32(double dx, double dy, double dz, int ktype) {
    float r2 = (float)fma(dz, dz, fma(dy, dy, dx * dx));
    r2 = r2 < 1e-16f ? 1.0f : r2;
    const float ir = __builtin_amdgcn_rsqf(r2);
    // phase in [0, 1) revolutions, the argument range of the hardware sin/cos: v_fract_f32
    // of the rounded r (its rounding, at most 2^-23 revolution for r < 4, is below that of
    // the rsq approximation in r)
    const float t = __builtin_amdgcn_fractf(r2 * ir);
    float s = __builtin_amdgcn_sinf(t), c = __builtin_amdgcn_cosf(t);
    if (ktype == 0) return make_float2(c * ir, s * ir);
    return make_float2(c, s);
}

template <class V, int KT>
__device__ __forceinline__ V green(double dx, double dy, double dz) {
    if constexpr (sizeof(V) == 16) return green64<KT>(dx, dy, dz);
    else return green32(dx, dy, dz, KT);
}

template <class V>
__device__ __forceinline__ V* bufp(const BufTable& bt, int b) { return (V*)bt.p[b]; }

// Workgroups are dispatched round-robin over the 8 XCDs (each with its own L2): give
// XCD x the contiguous chunk [x*q + min(x, r), ...) of the n work items (q = n/8, r = n%8)
// so that neighbouring items (Morton-ordered boxes, tiles of one operator) share an L2.
__device__ __forceinline__ int xcd_item(int b, int n) {
    const int x = b & 7, k = b >> 3;
    const int q = n >> 3, r = n & 7;
    return x * q + min(x, r) + k;
}

// The same in chunks of C consecutive items, dealt to the XCDs in turn: neighbours still share
// an L2, and items whose cost drifts along the list (GEMM groups in order of rank) spread
// over the XCDs, where eighths of the list left the XCDs with up to a fifth more or less work
// than the mean (W = 1 L2L of 4M points x 8 RHS: 8.1 -> 7.0 ms by this mapping alone).
template <int C>
__device__ __forceinline__ int xcd_chunk(int b, int n) {
    const int full = n / (8 * C) * (8 * C);
    if (b >= full) return full + xcd_item(b - full, n - full);
    const int x = b & 7, k = b >> 3;
    return (k / C) * 8 * C + x * C + k % C;
}
// 64-column tiles per chunk; 64 to 512 measured within 1% of each other, 8 and 32 up to 25%
// slower at 64 RHS, where one planned tile alone becomes 64 tiles of the same operator
constexpr int GEMM_XCD_CHUNK = 128;

// ---------------------------------------------------------------- kernel apply
constexpr int KA_THREADS = 256;

// One block per task.  A pass covers nt = min(count, 256) targets; when nt < 256 the
// 256 threads split into G = 256 / nt source groups (thread = target x group) that
// stride through each LDS source tile, and the partial sums are reduced through LDS.
template <class V, int RC, int KT>
__global__ __launch_bounds__(KA_THREADS) void kapply_kernel(
    const KTask* __restrict__ tasks, const KSrc* __restrict__ srcs,
    const double* __restrict__ px, const double* __restrict__ py, const double* __restrict__ pz,
    BufTable bt, int task0, int ntask, int nrhs) {
    const int r0 = blockIdx.y * RC;
    const int nr = min(RC, nrhs - r0);
    __shared__ double sx[KA_THREADS], sy[KA_THREADS], sz[KA_THREADS];
    __shared__ V sv[RC][KA_THREADS];
    __shared__ V red[RC][KA_THREADS];
    // grid-stride over the tasks (a grid smaller than the task count keeps a launch on the
    // second stream to a few blocks per CU); gridDim.x is a multiple of 8 or >= ntask
    for (int bi = blockIdx.x; bi < ntask; bi += gridDim.x) {
    const KTask t = tasks[task0 + bi];   // tasks are ordered by cost, longest first
    for (int tb = 0; tb < t.count; tb += KA_THREADS) {
        const int nt = min(KA_THREADS, t.count - tb);
        const int G = KA_THREADS / nt;
        const int ti = threadIdx.x % nt, gi = threadIdx.x / nt;
        const bool act = gi < G;
        const int i = tb + ti;
        double tx = 0, ty = 0, tz = 0;
        if (act) {
            tx = px[t.off + i] * t.scale + t.c[0];
            ty = py[t.off + i] * t.scale + t.c[1];
            tz = pz[t.off + i] * t.scale + t.c[2];
        }
        V acc[RC];
#pragma unroll
        for (int q = 0; q < RC; ++q) acc[q] = mk<V>(0, 0);
        for (int si = t.s0; si < t.s1; ++si) {
            const KSrc s = srcs[si];
            const V* vb = bufp<V>(bt, s.vbuf) + s.voff;
            const int64_t vs = bt.stride[s.vbuf];
            for (int sb = 0; sb < s.count; sb += KA_THREADS) {
                const int n = min(KA_THREADS, s.count - sb);
                __syncthreads();
                if ((int)threadIdx.x < n) {
                    const int64_t j = s.off + sb + threadIdx.x;
                    sx[threadIdx.x] = px[j] * s.scale + s.c[0];
                    sy[threadIdx.x] = py[j] * s.scale + s.c[1];
                    sz[threadIdx.x] = pz[j] * s.scale + s.c[2];
#pragma unroll
                    for (int q = 0; q < RC; ++q)
                        sv[q][threadIdx.x] = q < nr ? vb[(int64_t)(r0 + q) * vs + sb + threadIdx.x] : mk<V>(0, 0);
                }
                __syncthreads();
                if (act) {
                    for (int j = gi; j < n; j += G) {
                        const V g = green<V, KT>(tx - sx[j], ty - sy[j], tz - sz[j]);
#pragma unroll
                        for (int q = 0; q < RC; ++q) cfma(acc[q], g, sv[q][j]);
                    }
                }
            }
        }
        if (G > 1) {                      // reduce the source groups of each target
            __syncthreads();
#pragma unroll
            for (int q = 0; q < RC; ++q) red[q][threadIdx.x] = acc[q];
            __syncthreads();
            if (gi == 0) {
                for (int h = 1; h < G; ++h)
#pragma unroll
                    for (int q = 0; q < RC; ++q) {
                        const V o = red[q][ti + h * nt];
                        acc[q].x += o.x;
                        acc[q].y += o.y;
                    }
            }
        }
        if (gi == 0) {
            V* ob = bufp<V>(bt, t.obuf) + t.ooff + i;
            const int64_t os = bt.stride[t.obuf];
#pragma unroll
            for (int q = 0; q < RC; ++q) {
                if (q >= nr) break;
                V* o = ob + (int64_t)(r0 + q) * os;
                if (t.mode == 0) {
                    *o = acc[q];
                } else {
                    V v = *o;
                    v.x += acc[q].x;
                    v.y += acc[q].y;
                    *o = v;
                }
            }
        }
        __syncthreads();
    }
    }
}

// Kernel apply on the matrix cores (mixed precision): out_q(t) = sum_s G(t, s) v_q(s) for
// 8 * NB right-hand sides, per block of 16 targets x 4 sources as two real products on
// v_mfma_f32_16x16x4f32 whose 16 columns are n = (rhs q, re/im):
//   C += Re G . B1,   B1[s][(q, 0)] = Re v_q(s),   B1[s][(q, 1)] = Im v_q(s)
//   C += Im G . B2,   B2[s][(q, 0)] = -Im v_q(s),  B2[s][(q, 1)] = Re v_q(s)
// so that C[t][(q, 0)] = Re out_q(t) and C[t][(q, 1)] = Im out_q(t).  Lane i + 16 k holds
// A[i][k] and B[k][i]: it evaluates G for its own pair (target i, source k) on the VALU
// (FP64 differences, FP32 G, the formula of the VALU path) and feeds Re G and Im G to the
// two products unchanged; its B entries come from the density of source k for right-hand
// side i / 2.  A block owns one task; targets go in passes of 256 (16 row tiles of 16),
// the four waves split the row tiles (up to 4 each, every source step serving all of
// them) and, for up to 8 row tiles, the sources, with a fixed-order reduction through
// LDS.  Every column's k order is the same for any right-hand-side count, so each
// right-hand side keeps its bits in any batch.
constexpr int KM_ST = 256;    // sources per LDS tile

typedef float kacc4 __attribute__((ext_vector_type(4)));

// One wave's pass over the source groups gs = g0, g0 + gstep, ... < ng of an LDS tile for
// its NM row tiles.  The next group's coordinates and densities are read from LDS while
// the current group is evaluated.
template <int NM, int NB, int KT>
__device__ __forceinline__ void kmfma_steps(kacc4 (&acc)[4][NB], const double (&tx)[4], const double (&ty)[4],
                                            const double (&tz)[4], const double* sx, const double* sy,
                                            const double* sz, const float2 (*sv)[8 * NB + 1], int g0, int gstep,
                                            int ng, int g, int li) {
    const bool imcol = li & 1;
    if (g0 >= ng) return;
    int j = 4 * g0 + g;
    double xs = sx[j], ys = sy[j], zs = sz[j];
    float2 v[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) v[c] = sv[j][8 * c + (li >> 1)];
    for (int gs = g0; gs < ng; gs += gstep) {
        const int jn = gs + gstep < ng ? 4 * (gs + gstep) + g : j;
        const double xn = sx[jn], yn = sy[jn], zn = sz[jn];
        float2 vn[NB];
#pragma unroll
        for (int c = 0; c < NB; ++c) vn[c] = sv[jn][8 * c + (li >> 1)];
        float b1[NB], b2[NB];
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            b1[c] = imcol ? v[c].y : v[c].x;
            b2[c] = imcol ? v[c].x : -v[c].y;
        }
        float gr[NM], gi[NM];
#pragma unroll
        for (int m = 0; m < NM; ++m) {
            const float2 gv = green32(tx[m] - xs, ty[m] - ys, tz[m] - zs, KT);
            gr[m] = gv.x;
            gi[m] = gv.y;
        }
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int c = 0; c < NB; ++c) acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(gr[m], b1[c], acc[m][c], 0, 0, 0);
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
            for (int c = 0; c < NB; ++c) acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(gi[m], b2[c], acc[m][c], 0, 0, 0);
        j = jn;
        xs = xn;
        ys = yn;
        zs = zn;
#pragma unroll
        for (int c = 0; c < NB; ++c) v[c] = vn[c];
    }
}

// Orders one wave's LDS writes before its later LDS reads (and those reads before later
// writes): LDS executes a wave's instructions in order, so only the compiler must not move
// the accesses across.
__device__ __forceinline__ void wave_lds_order() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Near-field pairs evaluated once for both directions.  For a mirrored source leaf s of the
// task's leaf k (KSrc::moff >= 0) one wave takes 16-source tiles st = st0, st0 + 4, ...,
// each lane reading its four sources from memory (no block staging: the waves share no
// sources, so they run without barriers), and evaluates G over its row tiles m x the
// tile's 16 sources, four values per lane and row tile in the forward operand layout
// (lane i + 16 g: target i, sources 4 jj + g):
//   forward  acc[m] += G v_s                      (as kmfma_steps, groups 4 st + jj)
//   mirror   macc   += G^T den_k over the targets (K = targets 4 j + g of row tile m)
// The mirror's A operand is the transposed tile (lane i + 16 g: source i, targets 4 j + g),
// taken from per-wave LDS copies of two row tiles at a time.  G of all row tiles comes
// first and the products of different row tiles interleave (independent accumulators;
// the mirror sums even and odd row tiles apart and adds the two at the end).  The task has
// at most four row tiles and this wave holds them all (the waves split the sources), so
// macc is the tile's whole mirror: stored into the source's slot.
template <int NM, int NB, int KT>
__device__ __forceinline__ void kmfma_mirror(kacc4 (&acc)[4][NB], const double (&tx)[4], const double (&ty)[4],
                                             const double (&tz)[4], const double* px, const double* py,
                                             const double* pz, const float2* vb, int64_t vs,
                                             const float2 (*tv)[8 * NB + 1], float2* gt, int n, int st0, int g,
                                             int li, float* mslot, int64_t ms, int r0, int nr) {
    const bool imcol = li & 1;
    const int nst = (n + 15) >> 4;
    for (int st = st0; st < nst; st += 4) {
        float gr[NM][4], gi[NM][4];
        float b1[4][NB], b2[4][NB];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
            // sources past n: coordinates 0 (a finite G) and zero densities
            const int j = 16 * st + 4 * jj + g;
            const bool in = j < n;
            const double xs = in ? px[j] : 0.0, ys = in ? py[j] : 0.0, zs = in ? pz[j] : 0.0;
#pragma unroll
            for (int c = 0; c < NB; ++c) {
                const int q = 8 * c + (li >> 1);
                const float2 v = in && q < nr ? vb[(int64_t)(r0 + q) * vs + j] : make_float2(0.f, 0.f);
                b1[jj][c] = imcol ? v.y : v.x;
                b2[jj][c] = imcol ? v.x : -v.y;
            }
#pragma unroll
            for (int m = 0; m < NM; ++m) {
                const float2 gv = green32(tx[m] - xs, ty[m] - ys, tz[m] - zs, KT);
                gr[m][jj] = gv.x;
                gi[m][jj] = gv.y;
            }
        }
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int c = 0; c < NB; ++c) acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(gr[m][jj], b1[jj][c], acc[m][c], 0, 0, 0);
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
#pragma unroll
            for (int m = 0; m < NM; ++m)
#pragma unroll
                for (int c = 0; c < NB; ++c) acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(gi[m][jj], b2[jj][c], acc[m][c], 0, 0, 0);
        kacc4 macc[2][NB];
#pragma unroll
        for (int p = 0; p < 2; ++p)
#pragma unroll
            for (int c = 0; c < NB; ++c) macc[p][c] = kacc4{0, 0, 0, 0};
#pragma unroll
        for (int h = 0; h < (NM + 1) / 2; ++h) {
            constexpr int T = 16 * 17;       // one tile [source][target], rows padded to 17
            const int mh = NM - 2 * h < 2 ? NM - 2 * h : 2;
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                if (p >= mh) break;
#pragma unroll
                for (int jj = 0; jj < 4; ++jj)
                    gt[p * T + (4 * jj + g) * 17 + li] = make_float2(gr[2 * h + p][jj], gi[2 * h + p][jj]);
            }
            wave_lds_order();
            float hr[2][4], hi[2][4], d1[2][4][NB], d2[2][4][NB];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                if (p >= mh) break;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float2 e = gt[p * T + li * 17 + 4 * j + g];
                    hr[p][j] = e.x;
                    hi[p][j] = e.y;
#pragma unroll
                    for (int c = 0; c < NB; ++c) {
                        const float2 w = tv[16 * (2 * h + p) + 4 * j + g][8 * c + (li >> 1)];
                        d1[p][j][c] = imcol ? w.y : w.x;
                        d2[p][j][c] = imcol ? w.x : -w.y;
                    }
                }
            }
            wave_lds_order();
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    if (p >= mh) break;
#pragma unroll
                    for (int c = 0; c < NB; ++c)
                        macc[p][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(hr[p][j], d1[p][j][c], macc[p][c], 0, 0, 0);
                }
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    if (p >= mh) break;
#pragma unroll
                    for (int c = 0; c < NB; ++c)
                        macc[p][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(hi[p][j], d2[p][j][c], macc[p][c], 0, 0, 0);
                }
        }
        // rows 4 g + v: sources 16 st + 4 g + v; column li: (rhs 8 c + li / 2, re/im)
#pragma unroll
        for (int c = 0; c < NB; ++c) {
            const int q = 8 * c + (li >> 1);
            if (q >= nr) continue;
            float* o = mslot + 2 * ((int64_t)(r0 + q) * ms) + (li & 1);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int jx = 16 * st + 4 * g + v;
                if (jx >= n) continue;
                o[2 * jx] = macc[0][c][v] + macc[1][c][v];
            }
        }
    }
}

// Waves per SIMD the register allocation targets: the 8-RHS instance at five (96 VGPRs, a
// few spilled: G on the vector ALU needs more waves in flight than the 111 VGPRs of a
// free allocation allow; config 3 near field 16.5 -> 15.3 ms), its mirror instance at
// three (168 VGPRs without spills); the 16-RHS instances are held by LDS to three and two
// blocks per CU and keep their free allocation.
template <int NB, bool MIR> struct KmfmaOcc { static constexpr int waves = NB == 1 ? (MIR ? 3 : 5) : 1; };

template <int NB, int KT, bool MIR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(KmfmaOcc<NB, MIR>::waves))) void kapply_mfma_kernel(
    const KTask* __restrict__ tasks, const KSrc* __restrict__ srcs,
    const double* __restrict__ px, const double* __restrict__ py, const double* __restrict__ pz,
    BufTable bt, int task0, int ntask, int nrhs) {
    constexpr int NR = 8 * NB;                       // right-hand sides of the block
    __shared__ double sx[KM_ST], sy[KM_ST], sz[KM_ST];
    // densities, right-hand side fastest, rows padded by one entry (the staging stores of
    // consecutive sources then spread over the banks); after the last source tile, the
    // partial sums of waves that split the sources (4 waves x 4 row tiles x 64 lanes x 4 NB)
    __shared__ __align__(16) float2 sv[KM_ST][NR + 1];
    static_assert(sizeof(float2) * KM_ST * (NR + 1) >= sizeof(float) * 4 * 4 * 64 * 4 * NB, "reduction fits the tile");
    float* red = (float*)&sv[0][0];
    // mirror mode: the densities of a task that evaluates mirrored sources (at most 64
    // targets, one pass: every wave holds all its row tiles; rows past the task zero), the
    // mirror's operand, and one transposition tile per wave
    __shared__ __align__(16) float2 tv[MIR ? MIRROR_MAX_TARGETS : 1][NR + 1];
    __shared__ float2 gts[MIR ? 4 : 1][2 * 16 * 17];
    const int r0 = blockIdx.y * NR;
    const int nr = min(NR, nrhs - r0);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, li = lane & 15;
    for (int bi = blockIdx.x; bi < ntask; bi += gridDim.x) {
    const KTask t = tasks[task0 + bi];   // tasks are ordered by cost, longest first
    for (int tb = 0; tb < t.count; tb += 256) {
        const int nt = min(256, t.count - tb);
        const int nT = (nt + 15) >> 4;
        // up to 4 row tiles: every wave takes all of them and a quarter of the sources;
        // up to 8: two waves per row tile set; beyond: the waves split the row tiles
        const int wrt = nT > 8 ? 4 : nT > 4 ? 2 : 1, wsrc = 4 / wrt;
        const int myrt0 = wave % wrt, mysrc = wave / wrt;
        // this wave's row tiles: myrt0 + wrt * m < nT, m < nm
        const int nm = min(4, (nT - myrt0 + wrt - 1) / wrt);
        double tx[4], ty[4], tz[4];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            const int i = (myrt0 + wrt * m) * 16 + li;
            tx[m] = ty[m] = tz[m] = 0;
            if (m < nm && i < nt) {
                tx[m] = px[t.off + tb + i] * t.scale + t.c[0];
                ty[m] = py[t.off + tb + i] * t.scale + t.c[1];
                tz[m] = pz[t.off + tb + i] * t.scale + t.c[2];
            }
        }
        kacc4 acc[4][NB];
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int c = 0; c < NB; ++c) acc[m][c] = kacc4{0, 0, 0, 0};
        if (MIR && t.count <= MIRROR_MAX_TARGETS) {    // block-uniform
            const float2* den = bufp<float2>(bt, BUF_DEN) + t.off;
            const int64_t ds = bt.stride[BUF_DEN];
            for (int e = tid; e < MIRROR_MAX_TARGETS * NR; e += 256) {
                const int i = e / NR, q = e % NR;
                tv[i][q] = (i < nt && q < nr) ? den[(int64_t)(r0 + q) * ds + i] : make_float2(0.f, 0.f);
            }
            __syncthreads();
        }
        for (int si = t.s0; si < t.s1; ++si) {
            const KSrc s = srcs[si];
            const float2* vb = bufp<float2>(bt, s.vbuf) + s.voff;
            const int64_t vs = bt.stride[s.vbuf];
            if (MIR && s.moff >= 0) {
                // the first tile rotates with the source, which spreads the tiles evenly
                // over the waves
                const int st0 = (wave + si) & 3;
                float* ms = (float*)(bufp<float2>(bt, BUF_NMIR) + s.moff);
                const int64_t mst = bt.stride[BUF_NMIR];
                float2* gt = gts[MIR ? wave : 0];
                const double *qx = px + s.off, *qy = py + s.off, *qz = pz + s.off;
                switch (nm) {      // wave-uniform; every wave holds the task's row tiles
                case 4: kmfma_mirror<4, NB, KT>(acc, tx, ty, tz, qx, qy, qz, vb, vs, tv, gt, s.count, st0, g, li, ms, mst, r0, nr); break;
                case 3: kmfma_mirror<3, NB, KT>(acc, tx, ty, tz, qx, qy, qz, vb, vs, tv, gt, s.count, st0, g, li, ms, mst, r0, nr); break;
                case 2: kmfma_mirror<2, NB, KT>(acc, tx, ty, tz, qx, qy, qz, vb, vs, tv, gt, s.count, st0, g, li, ms, mst, r0, nr); break;
                case 1: kmfma_mirror<1, NB, KT>(acc, tx, ty, tz, qx, qy, qz, vb, vs, tv, gt, s.count, st0, g, li, ms, mst, r0, nr); break;
                default: break;
                }
                continue;
            }
            for (int sb = 0; sb < s.count; sb += KM_ST) {
                const int n = min(KM_ST, s.count - sb);
                __syncthreads();
                {   // sources past n: coordinates 0 (a finite G) and zero densities
                    const int j = tid;
                    double x = 0, y = 0, z = 0;
                    if (j < n) {
                        x = px[s.off + sb + j] * s.scale + s.c[0];
                        y = py[s.off + sb + j] * s.scale + s.c[1];
                        z = pz[s.off + sb + j] * s.scale + s.c[2];
                    }
                    sx[j] = x;
                    sy[j] = y;
                    sz[j] = z;
#pragma unroll
                    for (int q = 0; q < NR; ++q)
                        sv[j][q] = (j < n && q < nr) ? vb[(int64_t)(r0 + q) * vs + sb + j] : make_float2(0.f, 0.f);
                }
                __syncthreads();
                // groups of 4 sources: this wave takes groups mysrc, mysrc + wsrc, ...; the
                // staged rows past n hold zero densities
                const int ng = (n + 3) >> 2;
                switch (nm) {      // wave-uniform
                case 4: kmfma_steps<4, NB, KT>(acc, tx, ty, tz, sx, sy, sz, sv, mysrc, wsrc, ng, g, li); break;
                case 3: kmfma_steps<3, NB, KT>(acc, tx, ty, tz, sx, sy, sz, sv, mysrc, wsrc, ng, g, li); break;
                case 2: kmfma_steps<2, NB, KT>(acc, tx, ty, tz, sx, sy, sz, sv, mysrc, wsrc, ng, g, li); break;
                case 1: kmfma_steps<1, NB, KT>(acc, tx, ty, tz, sx, sy, sz, sv, mysrc, wsrc, ng, g, li); break;
                default: break;    // a wave with no row tile in this pass
                }
            }
        }
        // waves that split the sources of one row tile: sum their partials (fixed order)
        if (wsrc > 1) {
            __syncthreads();
            auto slot = [&](int w, int m, int c, int v) { return ((w * 4 + m) * 64 + lane) * 4 * NB + 4 * c + v; };
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                if (m >= nm) break;
#pragma unroll
                for (int c = 0; c < NB; ++c)
#pragma unroll
                    for (int v = 0; v < 4; ++v) red[slot(wave, m, c, v)] = acc[m][c][v];
            }
            __syncthreads();
            if (mysrc == 0) {
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    if (m >= nm) break;
#pragma unroll
                    for (int c = 0; c < NB; ++c)
#pragma unroll
                        for (int v = 0; v < 4; ++v) {
                            float a = red[slot(wave, m, c, v)];
                            for (int h = 1; h < wsrc; ++h) a += red[slot(wave + h * wrt, m, c, v)];
                            acc[m][c][v] = a;
                        }
                }
            }
        }
        // D[row][col] of a 16x16 f32 MFMA: lane holds rows 4 * (lane / 16) + v, column lane % 16
        if (mysrc == 0) {
            float* ob = (float*)(bufp<float2>(bt, t.obuf) + t.ooff + tb);
            const int64_t os = bt.stride[t.obuf];
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                if (m >= nm) break;
                const int rt = myrt0 + wrt * m;
#pragma unroll
                for (int c = 0; c < NB; ++c) {
                    const int q = 8 * c + (li >> 1);
                    if (q >= nr) continue;
                    float* oq = ob + 2 * ((int64_t)(r0 + q) * os) + (li & 1);
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int i = rt * 16 + 4 * g + v;
                        if (i >= nt) continue;
                        if (t.mode == 0) oq[2 * i] = acc[m][c][v];
                        else oq[2 * i] += acc[m][c][v];
                    }
                }
            }
        }
        __syncthreads();
    }
    }
}

// ---------------------------------------------------------------- grouped complex GEMM (MFMA)
template <class R> struct Mfma;
// Operand layouts (both): A lane l holds A[l%16][l/16], B lane l holds B[l/16][l%16].
// Output register v of lane l holds D[row(l/16, v)][l%16]; the row mapping differs
// between the f32 and the f64 instruction (checked on gfx950).
template <> struct Mfma<float> {
    typedef float acc4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc4 op(float a, float b, acc4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int v) { return 4 * lk + v; }
};
template <> struct Mfma<double> {
    typedef double acc4 __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc4 op(double a, double b, acc4 c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int lk, int v) { return lk + 4 * v; }
};

constexpr int MAXKB = 8;           // at most 8 K blocks (children of a box)

// Two adjacent FP32 complex values by one 16-byte load (global loads need dword alignment
// only).
struct CPair {
    float2 e[2];
};
__device__ __forceinline__ CPair load_pair(const float2* p) {
    typedef float f4u __attribute__((ext_vector_type(4), aligned(8)));
    const f4u r = *(const f4u*)p;
    return {{make_float2(r.x, r.y), make_float2(r.z, r.w)}};
}

// Units (8 k in FP32, 4 in FP64) per pipeline step: short tiles run few MFMAs per unit, so
// they load further ahead.  U2U of 6k points in FP64 (858 waves of one row block) 0.123 -> 0.104
// ms, of 60k 0.39 -> 0.35; twice as many units at one and two row blocks: 0.103 and 0.37.
constexpr int gemm_units(int mb, int cb) { return cb > 1 || mb > 3 ? 1 : mb > 1 ? 2 : 4; }

// C[:, ccol] (=|+=) diag(scale) * A * B[:, bcol] on MFMA 16x16x4 (f32 or f64).
// A block covers MB row blocks of 16 (the group's rows split evenly over its tiles; tiles
// are launched per MB) and 64 CB columns; each of its four waves owns 16 CB columns and
// works alone: operands go straight from memory (A from L2 and L1, where the block's waves
// meet) into the MFMA registers, one pipeline step of KQ k steps ahead, with no LDS staging
// and no barriers.  K runs over segments: the whole K, or the K blocks present in at least
// one of the wave's columns.
//
// What bounds it: loads first, then the ends of segments and launches.  4M points x 8 RHS on
// one stream: the translations take 23.2 ms, the matrix cores busy 65% of it (101 TF/s, padding
// included, of the 155 that they sustain); with the operands of a wave's first step in place
// of all later loads 18.8 ms (125 TF/s).  250k x 64 RHS 42.9 and 34.7 ms, 1M x 1 RHS 4.41 and 3.57.
// A in the stored order (ten 8-byte loads per 30 MFMAs, each over four half-filled line groups,
// where packed A takes five 16-byte loads of a contiguous KiB) reached 0.82 of this rate.
// Staged through LDS (two buffers, one barrier per 16 k), the waves stall together at the
// barriers; LDS form -> this one: 4M x 8 28.9 -> 23.4 ms, 250k x 64 58.9 -> 43.7, 1M x 1 5.9 -> 4.5.
//
// Launches of a wave or less per SIMD are bound by that wave's own instructions: beside the
// MFMAs of a k step of one row block (106 ns in FP64, 40 in FP32) stands its address
// arithmetic, which only other waves can hide.  So little of that is left in a step: absent
// blocks and columns point to a block of zeros, and the loads run up to a step past a segment's
// end, at constant offsets from one pointer per column block.  With clamps and selects in place
// of that -> now: FP64 U2U of 6k points 0.105 -> 0.084 ms, of 60k 0.35 -> 0.30, 1M x 1 RHS 2.04 ->
// 1.95.
//
// Bounds of the loads: B up to GEMM_AHEAD k past the segment, in the slack behind each
// buffer at its end (BUF_SLACK; the zeros behind the operator table, the setup window's
// slack), and replaced by zeros from the segment's end on; packed A up to the step's end, in
// the slack behind the packed tables, A as stored inside its block (what a zero of B
// multiplies is the block's own); row blocks past the group's last one are never read, rows
// past it not stored.  A column's order of k depends on G3M alone, so neither MB nor CB changes a
// bit (the instruction itself sums its k in order by fma).
//
// PACK: A packed (PackA in plan.hpp) in the order the lanes take it; else as stored in the
// operator table (the setup's products, FP64 contexts whose budget holds no packed copy).
template <class TA, class V, class R, int MB, int CB, bool PACK, bool G3M>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void gemm_kernel(
    const GGroup* __restrict__ groups, const GTile* __restrict__ tiles,
    const int64_t* __restrict__ colB, const int64_t* __restrict__ colC, const int64_t* __restrict__ colA,
    const TA* __restrict__ opm, const double2* __restrict__ scl, const void* __restrict__ zeros, BufTable bt,
    int tile0, int nr) {
    using M = Mfma<R>;
    using T = typename Real<V>::T;
    constexpr int TN = GEMM_TN * CB;
    constexpr int UQ = sizeof(R) == 4 ? 2 : 1, UK = 4 * UQ;          // k steps and k per unit
    constexpr int NU = gemm_units(MB, CB), KQ = NU * UQ, KS = NU * UK;   // per pipeline step
    static_assert(KS <= GEMM_AHEAD, "a step's loads stay in the slack");
    // k order of a unit: with three products lane group lk takes k = 2 lk + q in k step q (one
    // 16-byte load of B; a last unit of at most 4 k runs k = lk alone), with four k = lk + 4 q
    constexpr bool PAIR = G3M;
    // columns are (box, rhs) pairs, rhs fastest: column n is box n / nr of the group in
    // right-hand side n % nr (that rhs slab of the buffer).  A planned tile (GEMM_TN boxes)
    // becomes ceil(nr / CB) launched tiles of TN such columns; waves past its boxes or the
    // group's last column exit at once.
    const int per = (nr + CB - 1) / CB;
    const bool one = blockDim.x == 64;                 // a block per wave (launch_gemm_form)
    constexpr int CH = GEMM_XCD_CHUNK / CB;
    const int it = one ? xcd_chunk<4 * CH>(blockIdx.x, gridDim.x) : 4 * xcd_chunk<CH>(blockIdx.x, gridDim.x);
    const int bx = it >> 2;
    const GTile tl = tiles[tile0 + bx / per];
    const GGroup g = groups[tl.g];
    const int ncx = min(g.ncols, tl.n0 + GEMM_TN) * nr;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int li = lane & 15, lk = lane >> 4;
    const int n0 = tl.n0 * nr + TN * (bx % per) + 16 * CB * (one ? it & 3 : wave);   // the wave's first column
    if (n0 >= ncx) return;
    const V* B = bufp<V>(bt, g.bbuf);
    V* C = bufp<V>(bt, g.cbuf);
    const int64_t sB = bt.stride[g.bbuf], sC = bt.stride[g.cbuf];
    const int kb = g.kb ? g.kb : g.K;                   // segment length
    const int nkb = g.kb ? g.K / g.kb : 1;
    // B offsets of the wave's columns per K block, -1 = absent (no block there, or past the
    // group's last column: read as zeros): written and read by this wave
    __shared__ int64_t bo[4][MAXKB][16 * CB];

    int64_t coff[CB];                                   // this lane's output columns
    unsigned act = 0;                                   // segments with a present column
    {
        int64_t base[CB], rs[CB];
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            const int n = n0 + 16 * c + li;
            const int box = n / nr, r = n - box * nr;
            base[c] = n < ncx ? g.bcol0 + (int64_t)box * nkb : -1;
            rs[c] = r * sB;
            coff[c] = n < ncx ? colC[g.col0 + box] + r * sC : -1;
        }
#pragma unroll
        for (int t = 0; t < MAXKB / 4; ++t) {
            const int h = 4 * t + lk;
            bool any = false;
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                int64_t v = base[c] >= 0 && h < nkb ? colB[base[c] + h] : -1;
                any |= v >= 0;
                bo[wave][h][16 * c + li] = v >= 0 ? v + rs[c] : -1;
            }
            const uint64_t m = __ballot(any);
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if ((m >> (16 * q)) & 0xffff) act |= 1u << (4 * t + q);
        }
        wave_lds_order();
    }
    // A elements of this lane within a unit, per row block and per unit.  As stored (either
    // order), rows past the group's last repeat that one, and k past the segment's end its
    // first.
    static_assert(PACK || sizeof(R) == 8, "operators as stored in FP64 only");
    constexpr unsigned ROWS = 64 * UQ;
    const unsigned lda = g.lda;
    const unsigned kst = g.transA == 1 ? 1 : lda, ustep = PACK ? ROWS * lda : UK * kst;
    unsigned ao[PACK ? 1 : MB];
    if constexpr (PACK) {
        ao[0] = UQ * lane;
    } else {
#pragma unroll
        for (int a = 0; a < MB; ++a) ao[a] = min(tl.m0 + 16 * a + li, g.M - 1) * (g.transA == 1 ? lda : 1);
    }

    // G3M (FP32 contexts of the e^{ikr}/r kernel): three real products per complex one,
    // summed over k apart: k1 = (Ar + Ai) Br, k2 = Ar (Bi - Br), k3 = Ai (Br + Bi); Re C =
    // k1 - k3 and Im C = k1 + k2 in the epilogue.  Where |Ar| and |Ai| (or |Br| and |Bi|)
    // differ widely, k1 and k3 are both about Ai Br and cancel: the e^{ikr} kernel's larger
    // equivalent densities then lose accuracy, so it keeps four products (Re C in cr, Im C
    // in ci), as FP64 does.
    static_assert(!G3M || sizeof(R) == 4, "three products in FP32 only");
    typename M::acc4 cr[CB][MB], ci[CB][MB], c3[CB][G3M ? MB : 1];
#pragma unroll
    for (int c = 0; c < CB; ++c)
#pragma unroll
        for (int a = 0; a < MB; ++a)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                cr[c][a][v] = 0;
                ci[c][a][v] = 0;
                if constexpr (G3M) c3[c][a][v] = 0;
            }

    struct Step {                  // operands of one pipeline step
        TA a[KQ][MB];
        V b[KQ][CB];
        int kl;                    // k left in the segment
    };
    // loader: A and, at this lane's k, B of the step, and the k left in the segment
    const TA* Ap = nullptr;
    const V* Bp[CB];
    int kl = 0;
    auto segment = [&]() {
        const int h = __builtin_ctz(act);
        act &= act - 1;
        Ap = opm + (g.kb ? colA[g.acol0 + h] : g.aoff) + (PACK ? ROWS / 16 * tl.m0 : 0);
        kl = kb;
#pragma unroll
        for (int c = 0; c < CB; ++c) {
            const int64_t v = bo[wave][h][16 * c + li];
            Bp[c] = (v >= 0 ? B + v : (const V*)zeros) + lk;
        }
    };
    auto advance = [&]() {         // false: there is no further step (the loader stays)
        if (kl > KS) {
            kl -= KS;
            Ap += NU * ustep;
#pragma unroll
            for (int c = 0; c < CB; ++c) Bp[c] += KS;
            return true;
        }
        if (!act) return false;
        segment();
        return true;
    };
    // The loads of a step are unconditional and in one block (past the last step they repeat
    // it), so that the waits before their use count the next step's loads as outstanding.
    auto fetch = [&](Step& s) {
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            if constexpr (PAIR) {
                const int o = u * UK + (kl - u * UK <= 4 ? 0 : lk);
#pragma unroll
                for (int c = 0; c < CB; ++c) {
                    const CPair b = load_pair(Bp[c] + o);
                    s.b[u * UQ][c] = b.e[0];
                    s.b[u * UQ + UQ - 1][c] = b.e[1];
                }
            } else {
#pragma unroll
                for (int q = 0; q < UQ; ++q)
#pragma unroll
                    for (int c = 0; c < CB; ++c) s.b[u * UQ + q][c] = Bp[c][u * UK + 4 * q];
            }
            const int left = kl - u * UK;          // k left from the unit's first
            const TA* ap = PACK ? Ap + u * ustep + ao[0]
                                : Ap + ((left > 0 ? u * ustep : 0) + (lk < left ? lk * kst : 0));
#pragma unroll
            for (int a = 0; a < MB; ++a) {
                if constexpr (PACK && sizeof(R) == 4) {
                    const float4 v = *(const float4*)(ap + ROWS * a);
                    s.a[u * UQ][a] = make_float2(v.x, v.y);
                    s.a[u * UQ + UQ - 1][a] = make_float2(v.z, v.w);
                } else {
                    s.a[u * UQ][a] = ap[PACK ? ROWS * a : ao[PACK ? 0 : a]];
                }
            }
        }
        s.kl = kl;
    };
    // sweeps over the row blocks, so consecutive MFMAs never accumulate into the same
    // registers; one row fragment serves the wave's CB column blocks
    auto compute = [&](Step& s) {
        if (s.kl < KS) {           // zeros past the segment's end
#pragma unroll
            for (int q = 0; q < KQ; ++q) {
                const int kl = s.kl - q / UQ * UK;     // k left from the unit's first
                const int kq = PAIR && kl > 4 ? 2 * lk + q % UQ : 4 * (q % UQ) + lk;
#pragma unroll
                for (int c = 0; c < CB; ++c)
                    if (kq >= kl) s.b[q][c] = mk<V>(0, 0);
            }
        }
#pragma unroll
        for (int q = 0; q < KQ; ++q) {
            if (q > 0 && s.kl <= 4 * q) break;
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                const R br = (R)s.b[q][c].x, bi = (R)s.b[q][c].y;
                if constexpr (G3M) {   // cr = sum k1, ci = sum k2, c3 = sum k3
                    const R bd = bi - br, bs = br + bi;
#pragma unroll
                    for (int a = 0; a < MB; ++a) ci[c][a] = M::op((R)s.a[q][a].x, bd, ci[c][a]);
#pragma unroll
                    for (int a = 0; a < MB; ++a) c3[c][a] = M::op((R)s.a[q][a].y, bs, c3[c][a]);
#pragma unroll
                    for (int a = 0; a < MB; ++a) cr[c][a] = M::op((R)s.a[q][a].x + (R)s.a[q][a].y, br, cr[c][a]);
                } else {
                    const R mbi = -bi;
#pragma unroll
                    for (int a = 0; a < MB; ++a) cr[c][a] = M::op((R)s.a[q][a].x, br, cr[c][a]);
#pragma unroll
                    for (int a = 0; a < MB; ++a) ci[c][a] = M::op((R)s.a[q][a].x, bi, ci[c][a]);
#pragma unroll
                    for (int a = 0; a < MB; ++a) cr[c][a] = M::op((R)s.a[q][a].y, mbi, cr[c][a]);
#pragma unroll
                    for (int a = 0; a < MB; ++a) ci[c][a] = M::op((R)s.a[q][a].y, br, ci[c][a]);
                }
            }
        }
    };
    if (act) {
        Step s0, s1;
        segment();
        fetch(s0);
        while (true) {             // the next step's loads are in flight during this one's MFMAs
            const bool second = advance();
            fetch(s1);
            __builtin_amdgcn_sched_barrier(0);
            compute(s0);
            const bool more = second && advance();
            fetch(s0);
            __builtin_amdgcn_sched_barrier(0);
            if (second) compute(s1);
            if (!more) break;
        }
    }
    // D layout of a 16x16 MFMA tile: lane holds rows M::row(lane/16, v), column lane%16
#pragma unroll
    for (int c = 0; c < CB; ++c) {
        if (coff[c] < 0) continue;
        V* Cc = C + coff[c];
#pragma unroll
        for (int a = 0; a < MB; ++a) {
            R re[4], im[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                re[v] = cr[c][a][v];
                im[v] = ci[c][a][v];
                if constexpr (G3M) {
                    re[v] = cr[c][a][v] - c3[c][a][v];
                    im[v] = cr[c][a][v] + ci[c][a][v];
                }
            }
            if constexpr (sizeof(R) == 4) {      // four adjacent rows: two 16-byte stores
                typedef float f4u __attribute__((ext_vector_type(4), aligned(8)));
                const int m = tl.m0 + 16 * a + 4 * lk;
                if (g.mode == 0 && m + 3 < g.M) {
                    f4u lo = {re[0], im[0], re[1], im[1]}, hi = {re[2], im[2], re[3], im[3]};
                    *(f4u*)(Cc + m) = lo;
                    *(f4u*)(Cc + m + 2) = hi;
                    continue;
                }
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int m = tl.m0 + 16 * a + M::row(lk, v);
                if (m >= g.M) continue;
                R x = re[v], y = im[v];
                if constexpr (sizeof(R) == 8) {        // row scales: FP64 groups only
                    if (g.soff >= 0) {
                        const double2 s = scl[g.soff + m];
                        const R t = x * s.x - y * s.y;
                        y = x * s.y + y * s.x;
                        x = t;
                    }
                }
                if (g.mode == 0) {
                    Cc[m] = mk<V>(x, y);
                } else {
                    V o = Cc[m];
                    o.x += (T)x;
                    o.y += (T)y;
                    Cc[m] = o;
                }
            }
        }
    }
}

// Tallest tiles of a form: with two column blocks, seven row blocks take all 256 registers and
// spill.
constexpr int gemm_max_mb(int cb) { return cb > 1 ? GEMM_MB - 1 : GEMM_MB; }

// From 16 right-hand sides up, where a wave's 16 columns are one box's and tiles fill whole
// waves, each FP32 wave is a block of its own: the waves share nothing but cache lines, and a
// block of four is not placed before a slot is free on every SIMD, nor its slots reused before
// its last wave ends (e^{ikr} 250k x 16 RHS 29.6 -> 28.6 ms, 250k x 64 66.7 -> 66.4).  Below,
// blocks of one gain nothing (4M x 8: the same) or lose: FP64 200k x 5 17.1 -> 17.7, as they leave
// the other stream's large blocks no room, and with most tiles filling one wave of four
// the waves with work fall on a quarter of the CUs (1M x 1 6.6 -> 7.4).
template <class TA, class V, class R, int CB, bool PACK, bool G3M>
void launch_gemm_form(const Stage& s, int nrhs, hipStream_t st, const DevPlan& d, const TA* opm) {
    const bool one = sizeof(R) == 4 && nrhs >= 16;
    const dim3 grid((s.end - s.begin) * ((nrhs + CB - 1) / CB) * (one ? 4 : 1), 1), block(one ? 64 : 256);
#define DDFMM_GEMM_MB(X)                                                                                            \
    case X:                                                                                                         \
        if constexpr (X <= gemm_max_mb(CB))                                                                         \
            gemm_kernel<TA, V, R, X, CB, PACK, G3M><<<grid, block, 0, st>>>(d.groups, d.tiles, d.colB, d.colC,      \
                                                                            d.colA, opm, d.opmat, d.zeros, d.bt,    \
                                                                            s.begin, nrhs);                         \
        break;
    switch (s.mb) {
        DDFMM_GEMM_MB(1) DDFMM_GEMM_MB(2) DDFMM_GEMM_MB(3) DDFMM_GEMM_MB(4) DDFMM_GEMM_MB(5)
        DDFMM_GEMM_MB(6) DDFMM_GEMM_MB(7)
    }
#undef DDFMM_GEMM_MB
}

// FP64 products, on packed operators or, where the context holds none, as stored.
void launch_gemm64(const Stage& s, int nrhs, hipStream_t st, const DevPlan& d) {
    if (d.oppack64) launch_gemm_form<double2, double2, double, 1, true, false>(s, nrhs, st, d, d.oppack64);
    else launch_gemm_form<double2, double2, double, 1, false, false>(s, nrhs, st, d, d.opmat);
}

// FP32 products on packed operators.  Two column blocks per wave (CB = 2) halve the operator
// traffic per product but leave two waves per SIMD and take the union of twice the columns'
// K blocks.  They pay with three products per complex one, where K is not blocked and the
// columns of a box fill a wave, and the launch still has four blocks per CU: all translations
// of 250k points at 24, 32, 48 and 64 RHS, one block -> two, 17.3 -> 17.15, 22.75 -> 22.4, 34.6 -> 34.0
// and 44.9 -> 44.0 ms; at 8 and 16 RHS the same or slower, K-blocked U2U at 64 RHS 17.3 -> 18.1.  With
// four products the matrix cores are the longer part: 35.3 -> 35.6, 46.1 -> 46.6, 69.4 -> 69.8 and 91.2 ->
// 91.7 ms, so those keep one.
template <bool G3M>
void launch_gemm32(const Stage& s, int nrhs, hipStream_t st, const DevPlan& d) {
    if constexpr (G3M) {
        if (nrhs >= 32 && !s.kblocked && (int64_t)(s.end - s.begin) * nrhs / 2 >= 1024 && s.mb <= gemm_max_mb(2)) {
            launch_gemm_form<float2, float2, float, 2, true, G3M>(s, nrhs, st, d, d.oppack);
            return;
        }
    }
    launch_gemm_form<float2, float2, float, 1, true, G3M>(s, nrhs, st, d, d.oppack);
}

// Blocks per kernel matrix or packed operator block at setup: a setup window holds a few
// hundred of them, and one block each takes 20-90 dependent rounds for every window (6k points
// in FP64, 7 windows: 0.3 ms for generation and packing, 0.65 with one block).
constexpr int SETUP_SPLIT = 8;

// One packed operator block per job (PackA): zeros past the block's edges.
template <class T>
__global__ __launch_bounds__(256) void pack_kernel(const PackA* __restrict__ jobs, const double2* __restrict__ opmat,
                                                   T* __restrict__ out, int pair) {
    constexpr int UQ = 16 / (int)sizeof(T), UK = 4 * UQ;
    const PackA p = jobs[blockIdx.x];
    const int nrb = (p.M + 15) / 16, nk = (p.K + UK - 1) / UK;
    for (int e = blockIdx.y * 256 + threadIdx.x; e < nrb * nk * 64 * UQ; e += SETUP_SPLIT * 256) {
        const int q = e % UQ, lane = e / UQ & 63, rb = e / (64 * UQ) % nrb, o = e / (64 * UQ) / nrb;
        const int m = 16 * rb + (lane & 15), lk = lane >> 4;
        const int k = UK * o + (pair && p.K - UK * o > 4 ? 2 * lk + q : lk + 4 * q);
        T v = mk<T>(0, 0);
        if (m < p.M && k < p.K) {
            const double2 a = opmat[p.src + (p.trans ? k + (int64_t)m * p.lda : m + (int64_t)k * p.lda)];
            v = mk<T>(a.x, a.y);
        }
        out[p.dst + e] = v;
    }
}

// ---------------------------------------------------------------- split-BF16 complex GEMM (MFMA)
// The translation GEMM of the mixed mode with every FP32 operand written as the sum of
// three bf16 terms (x = x1 + x2 + x3, exact for FP32 x) and the products of
// v_mfma_f32_16x16x32_bf16 kept down to the third order (x1y1, x1y2, x2y1, x1y3, x2y2,
// x3y1; the dropped terms are below 2^-32 |x||y|), accumulated in FP32: FP32 accuracy at
// 2.7x the FP32 matrix-core rate.  The operator table is split once at setup (Bf16s
// entries); the vectors are split when a slab is staged.  A complex product is one real
// product with K' = 32 per 16 complex k:
//   Re C = [Ar, -Ai] [Br; Bi],   Im C = [Ai, Ar] [Br; Bi],
// lane i + 16 g of a 16x16x32 block holding A[i][8g..8g+7] and B[8g..8g+7][i], so lanes
// g < 2 take the real parts of k-octet g and lanes g >= 2 the imaginary parts of octet
// g - 2.  Tiles, K segments, column gathers, wave skips and epilogue as in gemm_kernel.
struct Bf16s {
    unsigned short v[8];    // re1, im1, re2, im2, re3, im3, 0, 0
};
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ unsigned short bf16_rne(float x) { return __builtin_bit_cast(unsigned short, (__bf16)x); }
__device__ __forceinline__ float bf16_val(unsigned short h) { return __uint_as_float((unsigned)h << 16); }
// x = h1 + h2 + h3 (each bf16, round to nearest even; the remainders are exact in FP32)
__device__ __forceinline__ void split3(float x, unsigned short& h1, unsigned short& h2, unsigned short& h3) {
    h1 = bf16_rne(x);
    const float r1 = x - bf16_val(h1);
    h2 = bf16_rne(r1);
    h3 = bf16_rne(r1 - bf16_val(h2));
}

__global__ void to_bf16s_kernel(const double2* __restrict__ in, Bf16s* __restrict__ out, int64_t n) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        Bf16s e;
        split3((float)in[i].x, e.v[0], e.v[2], e.v[4]);
        split3((float)in[i].y, e.v[1], e.v[3], e.v[5]);
        e.v[6] = e.v[7] = 0;
        out[i] = e;
    }
}

union Oct {                   // 8 bf16 of one plane and k-octet
    uint4 u;
    unsigned short h[8];
    bf16x8 v;
};

template <int MB>
__global__ __launch_bounds__(256) void gemm_bf16s_kernel(
    const GGroup* __restrict__ groups, const GTile* __restrict__ tiles,
    const int64_t* __restrict__ colB, const int64_t* __restrict__ colC, const int64_t* __restrict__ colA,
    const Bf16s* __restrict__ opb, const float2* __restrict__ opm32, BufTable bt, int tile0, int nr) {
    typedef float acc4 __attribute__((ext_vector_type(4)));
    constexpr int KS = 16, TM = 16 * MB;
    const int bx = xcd_item(blockIdx.x, gridDim.x);
    GTile tl = tiles[tile0 + bx / nr];
    const GGroup g = groups[tl.g];
    const int ncx = g.ncols * nr;
    tl.n0 = tl.n0 * nr + GEMM_TN * (bx % nr);
    if (tl.n0 >= ncx) return;
    const float2* B = bufp<float2>(bt, g.bbuf);
    float2* C = bufp<float2>(bt, g.cbuf);
    const int64_t sB = bt.stride[g.bbuf], sC = bt.stride[g.cbuf];
    // [buffer][term][plane re/im][row or column][k-octet]: k-octet h of row r is stored
    // at h ^ ((r >> 3) & 1), so the 16 lanes of a fragment read (16 rows, one octet) and
    // the 16 lanes of a staging store cover all banks once
    __shared__ uint4 As[2][3][2][TM][2];
    __shared__ uint4 Bs[2][3][2][GEMM_TN][2];
    __shared__ int64_t bo[MAXKB][GEMM_TN];
    __shared__ int64_t ao[MAXKB];
    __shared__ int used[MAXKB][4], act[MAXKB], wm[MAXKB], nact_s;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const int kb = g.kb ? g.kb : g.K;
    const int nkb = g.kb ? g.K / g.kb : 1;

    // staging units: A (row am, k-octet ah) for tid < 2 TM; B (column bn, k-octet bh) for
    // tid < 128
    const int mrows = g.M - tl.m0;
    const int64_t kstride = g.transA ? 1 : g.lda;
    const bool hasA = tid < 2 * TM, hasB = tid < 2 * GEMM_TN;
    const int am = tid % TM, ah = tid / TM;
    const int64_t aoff = g.transA ? (int64_t)(tl.m0 + am) * g.lda : (int64_t)(tl.m0 + am);
    const bool arow = hasA && am < mrows;
    const int bn = tid & (GEMM_TN - 1), bh = tid >> 6;
    int64_t bcol = -1;
    const int ncol = tl.n0 + wave * 16 + li;
    const int64_t coff = ncol < ncx ? colC[g.col0 + ncol / nr] + (int64_t)(ncol % nr) * sC : -1;

    int nact = 1, wm0 = 0;
    if (g.kb == 0) {
        const int nv = ncx - tl.n0;
        wm0 = nv >= GEMM_TN ? 15 : (1 << ((nv + 15) >> 4)) - 1;
        const int n = tl.n0 + bn;
        bcol = (hasB && n < ncx) ? colB[g.bcol0 + n / nr] + (int64_t)(n % nr) * sB : -1;
    } else {
        if (tid < MAXKB * 4) used[tid >> 2][tid & 3] = 0;
        __syncthreads();
        for (int e = tid; e < nkb * GEMM_TN; e += 256) {
            const int h = e / GEMM_TN, j = e % GEMM_TN;
            const int n = tl.n0 + j;
            int64_t v = n < ncx ? colB[g.bcol0 + (int64_t)(n / nr) * nkb + h] : -1;
            if (v >= 0) v += (int64_t)(n % nr) * sB;
            bo[h][j] = v;
            if (v >= 0) used[h][j >> 4] = 1;
        }
        __syncthreads();
        if (tid == 0) {
            int c = 0;
            for (int h = 0; h < nkb; ++h) {
                const int w = used[h][0] | (used[h][1] << 1) | (used[h][2] << 2) | (used[h][3] << 3);
                if (w) {
                    act[c] = h;
                    wm[c] = w;
                    ++c;
                }
            }
            nact_s = c;
        }
        __syncthreads();
        nact = nact_s;
        if (tid < nact) ao[tid] = colA[g.acol0 + act[tid]];
        __syncthreads();
    }
    Bf16s ra[8];
    float2 rb[8];
    auto load = [&](int i, int k0, bool newseg) {
        const int kl = kb - k0;
        if (newseg && hasB) bcol = bo[act[i]][bn];
        if (hasA) {
            const Bf16s* Ab = opb + (g.kb ? ao[i] : g.aoff) + k0 * kstride + aoff;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int k = 8 * ah + j;
                Bf16s a = {};
                if (arow && k < kl) a = Ab[k * kstride];
                ra[j] = a;
            }
        }
        if (hasB) {
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int k = 8 * bh + j;
                float2 b = make_float2(0.f, 0.f);
                if (bcol >= 0 && k < kl) b = B[bcol + k0 + k];
                rb[j] = b;
            }
        }
    };
    auto store = [&](int q) {
        if (hasA) {
            const int sl = ah ^ ((am >> 3) & 1);
#pragma unroll
            for (int t = 0; t < 3; ++t)
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    Oct o;
#pragma unroll
                    for (int j = 0; j < 8; ++j) o.h[j] = ra[j].v[2 * t + c];
                    As[q][t][c][am][sl] = o.u;
                }
        }
        if (hasB) {
            Oct o[3][2];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                split3(rb[j].x, o[0][0].h[j], o[1][0].h[j], o[2][0].h[j]);
                split3(rb[j].y, o[0][1].h[j], o[1][1].h[j], o[2][1].h[j]);
            }
            const int sl = bh ^ ((bn >> 3) & 1);
#pragma unroll
            for (int t = 0; t < 3; ++t)
#pragma unroll
                for (int c = 0; c < 2; ++c) Bs[q][t][c][bn][sl] = o[t][c].u;
        }
    };

    acc4 cr[MB], ci[MB];
#pragma unroll
    for (int a = 0; a < MB; ++a)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            cr[a][v] = 0;
            ci[a][v] = 0;
        }
    // fragment addressing of this lane: octet lk & 1 (swizzled by row/column bit 3), plane
    // re for lanes lk < 2 and im for lk >= 2 (B and the Re-C operand of A), im/re for the
    // Im-C operand of A; the Re-C operand of lanes lk >= 2 is negated (-Ai)
    const int oct = (lk & 1) ^ ((li >> 3) & 1);
    const int px = lk >> 1, py = px ^ 1;
    const unsigned neg = lk >= 2 ? 0x80008000u : 0u;
    auto mfma_slab = [&](int i, int q) {
        if (!(((g.kb ? wm[i] : wm0) >> wave) & 1)) return;
        Oct bf[3];
#pragma unroll
        for (int t = 0; t < 3; ++t) bf[t].u = Bs[q][t][px][wave * 16 + li][oct];
#pragma unroll
        for (int a = 0; a < MB; ++a) {
            Oct xr[3], yi[3];
#pragma unroll
            for (int t = 0; t < 3; ++t) {
                xr[t].u = As[q][t][px][16 * a + li][oct];
                xr[t].u.x ^= neg;
                xr[t].u.y ^= neg;
                xr[t].u.z ^= neg;
                xr[t].u.w ^= neg;
                yi[t].u = As[q][t][py][16 * a + li][oct];
            }
            // smallest terms first
            cr[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xr[2].v, bf[0].v, cr[a], 0, 0, 0);
            ci[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yi[2].v, bf[0].v, ci[a], 0, 0, 0);
            cr[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xr[1].v, bf[1].v, cr[a], 0, 0, 0);
            ci[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yi[1].v, bf[1].v, ci[a], 0, 0, 0);
            cr[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xr[0].v, bf[2].v, cr[a], 0, 0, 0);
            ci[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yi[0].v, bf[2].v, ci[a], 0, 0, 0);
            cr[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xr[1].v, bf[0].v, cr[a], 0, 0, 0);
            ci[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yi[1].v, bf[0].v, ci[a], 0, 0, 0);
            cr[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xr[0].v, bf[1].v, cr[a], 0, 0, 0);
            ci[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yi[0].v, bf[1].v, ci[a], 0, 0, 0);
            cr[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xr[0].v, bf[0].v, cr[a], 0, 0, 0);
            ci[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(yi[0].v, bf[0].v, ci[a], 0, 0, 0);
        }
    };
    auto next = [&](int i, int k0, int& ni, int& nk0) {
        ni = i;
        nk0 = k0 + KS;
        if (nk0 >= kb) {
            ni = i + 1;
            nk0 = 0;
        }
    };
    if (nact > 0) {
        load(0, 0, g.kb != 0);
        store(0);
    }
    // slab s+1 waits in registers while slab s runs; one barrier per slab
    int i = 0, k0 = 0, ni, nk0;
    next(i, k0, ni, nk0);
    bool more = ni < nact;
    if (more) load(ni, nk0, ni != i);
    __syncthreads();
    int q = 0;
    while (i < nact) {
        mfma_slab(i, q);
        int n2i = nact, n2k0 = 0;
        bool more2 = false;
        if (more) {
            store(q ^ 1);
            next(ni, nk0, n2i, n2k0);
            more2 = n2i < nact;
            if (more2) load(n2i, n2k0, n2i != ni);
        }
        __syncthreads();
        i = ni;
        k0 = nk0;
        ni = n2i;
        nk0 = n2k0;
        more = more2;
        q ^= 1;
    }
    // D layout of the 16x16 output: lane holds rows 4 (lane / 16) + v, column lane % 16
    if (coff < 0) return;
    float2* Cc = C + coff;
#pragma unroll
    for (int a = 0; a < MB; ++a) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int m = tl.m0 + 16 * a + 4 * lk + v;
            if (m >= g.M) continue;
            float re = cr[a][v], im = ci[a][v];
            if (g.soff >= 0) {
                const float2 s = opm32[g.soff + m];
                const float t = re * s.x - im * s.y;
                im = re * s.y + im * s.x;
                re = t;
            }
            if (g.mode == 0) {
                Cc[m] = make_float2(re, im);
            } else {
                float2 o = Cc[m];
                o.x += re;
                o.y += im;
                Cc[m] = o;
            }
        }
    }
}

void launch_gemm_bf16s(int mb, int n, int nrhs, hipStream_t st, const DevPlan& d, int t0) {
    const dim3 grid(n * nrhs, 1);
#define DDFMM_GEMM_MB(X)                                                                                      \
    case X:                                                                                                   \
        gemm_bf16s_kernel<X><<<grid, 256, 0, st>>>(d.groups, d.tiles, d.colB, d.colC, d.colA,                 \
                                                   (const Bf16s*)d.opmatbf, d.opmat32, d.bt, t0, nrhs);       \
        break;
    switch (mb) {
        DDFMM_GEMM_MB(1) DDFMM_GEMM_MB(2) DDFMM_GEMM_MB(3) DDFMM_GEMM_MB(4) DDFMM_GEMM_MB(5)
        DDFMM_GEMM_MB(6) DDFMM_GEMM_MB(7)
    }
#undef DDFMM_GEMM_MB
}

// ---------------------------------------------------------------- pruned (2P)^3 DFT, P = 6
// The equivalent surface of a box sits on the 6^3 sub-cube [6, 12)^3 of the 12^3 grid
// (grid index = round((x + W/2)/step) + P), so the forward transform has non-zero input
// only there and the inverse transform is sampled only there: each 1-D pass runs on the
// lines that carry data and produces the outputs later passes use (18144 complex MACs
// per 3-D transform instead of 62208).  One thread per line, twiddles as constants.
struct Tw12 {
    static constexpr double c[12] = {1.0, 0.86602540378443865, 0.5, 0.0, -0.5, -0.86602540378443865,
                                     -1.0, -0.86602540378443865, -0.5, 0.0, 0.5, 0.86602540378443865};
    static constexpr double s[12] = {0.0, 0.5, 0.86602540378443865, 1.0, 0.86602540378443865, 0.5,
                                     0.0, -0.5, -0.86602540378443865, -1.0, -0.86602540378443865, -0.5};
};

// out[o * os] = sum_{q < NI} in[q * is] * exp(SGN * 2 pi i (q + QOFF)(o + OOFF) / 12), o < NO
template <class V, int NI, int NO, int QOFF, int OOFF, int SGN>
__device__ __forceinline__ void dft12_line(const V* in, int is, V* out, int os) {
    using T = typename Real<V>::T;
    V x[NI];
#pragma unroll
    for (int q = 0; q < NI; ++q) x[q] = in[q * is];
#pragma unroll
    for (int o = 0; o < NO; ++o) {
        V acc = mk<V>(0, 0);
#pragma unroll
        for (int q = 0; q < NI; ++q) {
            const int m = ((q + QOFF) * (o + OOFF)) % 12;
            const V w = mk<V>((T)Tw12::c[m], (T)(SGN * Tw12::s[m]));
            cfma(acc, x[q], w);
        }
        out[o * os] = acc;
    }
}

template <class V>
__global__ __launch_bounds__(256) void fft_fwd_kernel(const FftSrc* __restrict__ fs, const int* __restrict__ grid,
                                                      int NL, BufTable bt, int f0, int nf, int nrhs) {
    __shared__ V sub[216], A[432], B[864];
    const int rhs = blockIdx.y;
    const int t = threadIdx.x;
    for (int bi = blockIdx.x; bi < nf; bi += gridDim.x) {
    const FftSrc f = fs[f0 + xcd_item(bi, nf)];
    __syncthreads();
    const V* in = bufp<V>(bt, BUF_LF_UPEQ) + (int64_t)rhs * bt.stride[BUF_LF_UPEQ] + f.in_off;
    // spectra right-hand side fastest: frequency k of this source at (spec_off + k) * nrhs + rhs
    V* out = bufp<V>(bt, BUF_SPEC) + f.spec_off * nrhs + rhs;
    if (t < 216) sub[t] = mk<V>(0, 0);
    __syncthreads();
    for (int k = t; k < NL; k += blockDim.x) {
        const int g = grid[f.grid + k];
        sub[(g % 12 - 6) + 6 * ((g / 12) % 12 - 6) + 36 * (g / 144 - 6)] = in[k];
    }
    __syncthreads();
    if (t < 36)          // x lines (y', z'): 6 inputs -> 12 outputs, A[z'][y'][kx]
        dft12_line<V, 6, 12, 6, 0, -1>(sub + 6 * t, 1, A + 12 * t, 1);
    __syncthreads();
    if (t < 72)          // y lines (kx, z'): A -> B[z'][ky][kx]
        dft12_line<V, 6, 12, 6, 0, -1>(A + (t % 12) + 72 * (t / 12), 12, B + (t % 12) + 144 * (t / 12), 12);
    __syncthreads();
    if (t < 144)         // z lines (kx, ky): B -> spectrum [kz][ky][kx]
        dft12_line<V, 6, 12, 6, 0, -1>(B + t, 144, out + (int64_t)t * nrhs, 144 * nrhs);
    }
}

// Forward transforms of R right-hand sides of one source per block (nrhs > 1).  The
// scatter into the 6^3 sub-grids and the x and y passes run H right-hand sides at a time
// (H x 36 and H x 72 line transforms per pass over the block's threads) into each one's
// slab of B; the z pass then runs over (line, rhs) with the right-hand side fastest, so the
// spectra, stored right-hand side fastest, are written in runs of R consecutive values
// (64 bytes: whole write sectors).
template <class V, int R, int H>
__global__ __launch_bounds__(256) void fft_fwd_multi_kernel(const FftSrc* __restrict__ fs,
                                                            const int* __restrict__ grid, int NL, BufTable bt,
                                                            int f0, int nf, int nrhs) {
    __shared__ V sub[H][216], A[H][432], B[R][864];
    const int t = threadIdx.x;
    const int r0 = blockIdx.y * R, nr = min(R, nrhs - r0);
    const int64_t is = bt.stride[BUF_LF_UPEQ];
    for (int bi = blockIdx.x; bi < nf; bi += gridDim.x) {
        const FftSrc f = fs[f0 + xcd_item(bi, nf)];
        for (int h0 = 0; h0 < nr; h0 += H) {
            const int hn = min(H, nr - h0);
            const V* in = bufp<V>(bt, BUF_LF_UPEQ) + (int64_t)(r0 + h0) * is + f.in_off;
            __syncthreads();
            for (int e = t; e < H * 216; e += blockDim.x) sub[e / 216][e % 216] = mk<V>(0, 0);
            __syncthreads();
            for (int e = t; e < hn * NL; e += blockDim.x) {
                const int r = e / NL, k = e % NL;
                const int g = grid[f.grid + k];
                sub[r][(g % 12 - 6) + 6 * ((g / 12) % 12 - 6) + 36 * (g / 144 - 6)] = in[(int64_t)r * is + k];
            }
            __syncthreads();
            for (int e = t; e < hn * 36; e += blockDim.x) {    // x lines (y', z'): 6 inputs -> 12 outputs
                const int r = e / 36, l = e % 36;
                dft12_line<V, 6, 12, 6, 0, -1>(sub[r] + 6 * l, 1, A[r] + 12 * l, 1);
            }
            __syncthreads();
            for (int e = t; e < hn * 72; e += blockDim.x) {    // y lines (kx, z'): A -> B[rhs][z'][ky][kx]
                const int r = e / 72, l = e % 72;
                dft12_line<V, 6, 12, 6, 0, -1>(A[r] + (l % 12) + 72 * (l / 12), 12,
                                               B[h0 + r] + (l % 12) + 144 * (l / 12), 12);
            }
        }
        __syncthreads();
        V* out = bufp<V>(bt, BUF_SPEC) + f.spec_off * nrhs + r0;
        for (int q = t; q < 144 * nr; q += blockDim.x) {   // z lines (kx, ky) x rhs, rhs fastest
            const int line = q / nr, r = q % nr;
            dft12_line<V, 6, 12, 6, 0, -1>(B[r] + line, 144, out + (int64_t)line * nrhs + r, 144 * nrhs);
        }
    }
}

// V list, accumulation: T_t[f] = sum_{(t, s) in V} Tab[offidx(t, s)][f] * S_s[f] over the
// (2P)^3 frequencies.  A block owns one slice of VSlice<V>::F frequencies (64 B of one
// spectrum) of one chunk of Morton-consecutive targets.  It stages in LDS the slice of the
// level's translation tensor (343 offsets) and the slice of every source in the chunk's
// union (at most VCH_SRC), with independent loads only; the pair loop then reads both
// operands from LDS.  Items are numbered slice-major and given to the XCDs in contiguous
// ranges (xcd_item), so an XCD works through a few slices at a time and the source
// slices it stages come from its own L2.  Threads: F frequencies x 256 / F targets.
template <class V> struct VSlice {
    static constexpr int F = 64 / (int)sizeof(V);          // frequencies per slice
    // LDS row stride, unpadded: the two targets' 64-byte rows that a 16-lane read group
    // takes then sit in aligned bank halves (with a 72-byte pitch their bank windows nearly
    // always overlap), and the 1-RHS block's LDS (51 KB instead of 56) lets three blocks
    // share a CU instead of two; together 12% faster than the padded pitch
    static constexpr int SE = F;
};

constexpr int VL_THREADS = 512;

// Stage the chunk's packed pair words (vpk[k0, k1), a multiple of 8 words, 16-byte
// aligned) into LDS with int4 loads.
__device__ __forceinline__ void stage_pairs(const int* __restrict__ vpk, const VChunk& ch, int* pkl, int t) {
    const int4* src = (const int4*)(vpk + ch.k0);
    int4* dst = (int4*)pkl;
    const int n4 = (ch.k1 - ch.k0) >> 2;
    for (int e = t; e < n4; e += VL_THREADS) dst[e] = src[e];
}

// A block walks VL_SLICES consecutive frequency slices of one chunk: the chunk's packed
// pairs are staged once, and the tensor and source slices of the next frequency slice
// are loaded into registers while the current one is accumulated.
constexpr int VL_GROUPS = 108;    // slice groups per chunk: 1728 / (F * slices per group)

template <class V>
__global__ __launch_bounds__(VL_THREADS) void vlist_acc_kernel(const VTarget* __restrict__ vt,
                                                               const VChunk* __restrict__ vc,
                                                               const int* __restrict__ vsrc,
                                                               const int* __restrict__ vpk,
                                                               const V* __restrict__ opm, BufTable bt, int v0,
                                                               int c0, int nchunk) {
    constexpr int G3 = 1728, F = VSlice<V>::F, SE = VSlice<V>::SE, TPP = VL_THREADS / F;
    constexpr int NSL = G3 / F / VL_GROUPS;
    constexpr int NT = (343 * F + VL_THREADS - 1) / VL_THREADS, NS = (VCH_SRC * F + VL_THREADS - 1) / VL_THREADS;
    __shared__ V tab[343 * SE], src[VCH_SRC * SE];
    __shared__ __align__(16) int pkl[VCH_PK];
    const int t = threadIdx.x, fl = t % F;
    const int item = xcd_item(blockIdx.x, VL_GROUPS * nchunk);
    const int fg = (item / nchunk) * NSL * F;
    const VChunk ch = vc[c0 + item % nchunk];
    const V* T = opm + vt[v0].tab_off;
    const V* spec = bufp<V>(bt, BUF_SPEC);
    const int nu = (ch.u1 - ch.u0) * F;
    int64_t si[NS];                          // source row offsets, fixed for the block
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int e = t + VL_THREADS * k;
        si[k] = (e >= F && e < nu) ? (int64_t)vsrc[ch.u0 + e / F] * G3 + e % F : -1;
    }
    V a[NT], b[NS];
    auto fetch = [&](int f0) {
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            const int e = t + VL_THREADS * k;
            a[k] = e < 343 * F ? T[(int64_t)(e / F) * G3 + f0 + e % F] : mk<V>(0, 0);
        }
#pragma unroll
        for (int k = 0; k < NS; ++k) b[k] = si[k] >= 0 ? spec[si[k] + f0] : mk<V>(0, 0);
    };
    fetch(fg);
    stage_pairs(vpk, ch, pkl, t);
    const V* srcl = src + fl;
    const V* tabl = tab + fl;
    for (int sl = 0; sl < NSL; ++sl) {
        const int f0 = fg + sl * F;
        __syncthreads();                     // the previous slice's reads of tab / src are done
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            const int e = t + VL_THREADS * k;
            if (e < 343 * F) tab[(e / F) * SE + e % F] = a[k];
        }
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const int e = t + VL_THREADS * k;
            if (e < nu) src[(e / F) * SE + e % F] = b[k];     // row 0 stays zero (si = -1)
        }
        __syncthreads();
        if (sl + 1 < NSL) fetch(f0 + F);     // in flight during the pair loop below
        V* out = bufp<V>(bt, BUF_TSPEC) + f0 + fl;
        for (int i = ch.t0 + t / F; i < ch.t1; i += TPP) {
            const VTarget tg = vt[i];
            V acc = mk<V>(0, 0);
            // the target's packed pairs (zero pairs pad to a multiple of 8; row 0 is zero),
            // read from LDS by every lane of its group (one address: a broadcast)
            const int n = (tg.p1 - tg.p0 + 7) & ~7;
            const int4* pk = (const int4*)(pkl + (tg.k0 - ch.k0));
            for (int j = 0; j < n; j += F) {
                V sv[F], tv[F];
#pragma unroll
                for (int u = 0; u < F; ++u) {
                    const int4 q = pk[(j + u) / 4];
                    const int w = (u % 4 == 0) ? q.x : (u % 4 == 1) ? q.y : (u % 4 == 2) ? q.z : q.w;
                    sv[u] = srcl[(w & 0xffff) * SE];
                    tv[u] = tabl[(w >> 16) * SE];
                }
#pragma unroll
                for (int u = 0; u < F; ++u) cfma(acc, sv[u], tv[u]);
            }
            out[(int64_t)(i - v0) * G3] = acc;
        }
    }
}

// V list, accumulation for several right-hand sides (nrhs > 1).  The source spectra are
// stored right-hand side fastest, SPEC[(row * (2P)^3 + f) * nrhs + r], so the values of
// one source for F frequencies and RC = R1 * R2 right-hand sides of a block are one
// 128-byte run per frequency.  A block owns (chunk, group of frequency slices of F
// frequencies, group of RC right-hand sides) and stages the slice of the translation
// tensor (343 offsets, shared by the group) and the union's source rows (128 bytes each).
// Eight lanes work on one target: lane l takes frequency l / R1 and the R2 right-hand
// sides (l % R1) * R2 + q, so the eight lanes read one whole source row per pair (all 32
// banks) and one tensor value serves R2 complex FMAs.  The accumulated target spectra go
// to TSPEC right-hand side fastest too: the eight lanes of a target write one 128-byte run
// (with a slab per right-hand side they were pieces of 8 or 16 bytes, written back to HBM as
// partial lines: V list with its inverse 12.9 -> 8.7 ms at 250k points x 64 RHS, 6.3 -> 4.9 ms at
// 4M x 8, 3.3 -> 2.2 ms at 250k x 16).
template <class V> struct VMulti { static constexpr int R2 = 16 / (int)sizeof(V); };   // float2: 2, double2: 1

template <class V, int F, int R1>
__global__ __launch_bounds__(VL_THREADS) void vlist_acc_multi_kernel(const VTarget* __restrict__ vt,
                                                                     const VChunk* __restrict__ vc,
                                                                     const int* __restrict__ vsrc,
                                                                     const int* __restrict__ vpk,
                                                                     const V* __restrict__ opm, BufTable bt, int v0,
                                                                     int c0, int nchunk, int nrhs) {
    constexpr int G3 = 1728, R2 = VMulti<V>::R2, RC = R1 * R2, ROW = F * RC;
    constexpr int NSL = G3 / F / VL_GROUPS;
    constexpr int NT = (343 * F + VL_THREADS - 1) / VL_THREADS, NS = (VCH_SRC * ROW + VL_THREADS - 1) / VL_THREADS;
    static_assert(F * R1 == 8, "eight lanes per target");
    static_assert(ROW * (int)sizeof(V) == 128, "128-byte source rows");
    __shared__ V tab[343 * F];
    __shared__ __align__(16) V src[VCH_SRC * ROW];
    __shared__ __align__(16) int pkl[VCH_PK];
    const int t = threadIdx.x, l = t & 7;
    const int fl = l / R1, rq = (l % R1) * R2;
    const int item = xcd_item(blockIdx.x, VL_GROUPS * nchunk);
    const int fg = (item / nchunk) * NSL * F;
    const int rg = blockIdx.y * RC;
    const VChunk ch = vc[c0 + item % nchunk];
    const V* T = opm + vt[v0].tab_off;
    const V* spec = bufp<V>(bt, BUF_SPEC);
    const int nu = (ch.u1 - ch.u0) * ROW;
    int64_t si[NS];                          // element offsets at frequency 0, fixed for the block
#pragma unroll
    for (int k = 0; k < NS; ++k) {
        const int e = t + VL_THREADS * k;
        const int u = e / ROW, w = e % ROW, f = w / RC, r = rg + w % RC;
        si[k] = (e >= ROW && e < nu && r < nrhs) ? ((int64_t)vsrc[ch.u0 + u] * G3 + f) * nrhs + r : -1;
    }
    V a[NT], b[NS];
    auto fetch = [&](int f0) {
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            const int e = t + VL_THREADS * k;
            a[k] = e < 343 * F ? T[(int64_t)(e / F) * G3 + f0 + e % F] : mk<V>(0, 0);
        }
#pragma unroll
        for (int k = 0; k < NS; ++k) b[k] = si[k] >= 0 ? spec[si[k] + (int64_t)f0 * nrhs] : mk<V>(0, 0);
    };
    fetch(fg);
    stage_pairs(vpk, ch, pkl, t);
    const V* tabl = tab + fl;
    const V* srcl = src + l * R2;
    V* out = bufp<V>(bt, BUF_TSPEC);
    for (int sl = 0; sl < NSL; ++sl) {
        const int f0 = fg + sl * F;
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            const int e = t + VL_THREADS * k;
            if (e < 343 * F) tab[e] = a[k];
        }
#pragma unroll
        for (int k = 0; k < NS; ++k) {
            const int e = t + VL_THREADS * k;
            if (e < nu) src[e] = b[k];       // row 0 and right-hand sides past nrhs are zero
        }
        __syncthreads();
        if (sl + 1 < NSL) fetch(f0 + F);     // in flight during the pair loop below
        for (int i = ch.t0 + t / 8; i < ch.t1; i += VL_THREADS / 8) {
            const VTarget tg = vt[i];
            V acc[R2];
#pragma unroll
            for (int q = 0; q < R2; ++q) acc[q] = mk<V>(0, 0);
            const int n = (tg.p1 - tg.p0 + 7) & ~7;
            const int4* pk = (const int4*)(pkl + (tg.k0 - ch.k0));
            for (int j = 0; j < n; j += 8) {
                V tv[8], sv[8][R2];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const int4 q = pk[(j + u) / 4];
                    const int w = (u % 4 == 0) ? q.x : (u % 4 == 1) ? q.y : (u % 4 == 2) ? q.z : q.w;
                    tv[u] = tabl[(w >> 16) * F];
                    const V* sp = srcl + (w & 0xffff) * ROW;
                    if constexpr (R2 == 2) {
                        const float4 x = *(const float4*)sp;
                        sv[u][0] = mk<V>(x.x, x.y);
                        sv[u][R2 - 1] = mk<V>(x.z, x.w);
                    } else {
                        sv[u][0] = sp[0];
                    }
                }
#pragma unroll
                for (int u = 0; u < 8; ++u)
#pragma unroll
                    for (int q = 0; q < R2; ++q) cfma(acc[q], sv[u][q], tv[u]);   // operand order of the 1-RHS kernel
            }
            V* o = out + ((int64_t)(i - v0) * G3 + f0 + fl) * nrhs + rg + rq;
            if constexpr (R2 == 2) {
                typedef float f4u __attribute__((ext_vector_type(4), aligned(8)));
                if (rg + rq + 1 < nrhs) *(f4u*)o = f4u{acc[0].x, acc[0].y, acc[R2 - 1].x, acc[R2 - 1].y};
                else if (rg + rq < nrhs) o[0] = acc[0];
            } else {
                if (rg + rq < nrhs) o[0] = acc[0];
            }
        }
    }
}

// V list, inverse: one block per target and group of R right-hand sides, the accumulated
// spectra (right-hand side fastest, as the source spectra) back to the 6^3 sub-cube (pruned
// inverse DFT, 1/(2P)^3 scaling) and added into the target's check values.  Each pass runs
// the R right-hand sides' lines together (R x 144 x lines read straight from the spectra,
// adjacent lanes on adjacent right-hand sides; R x 72 y lines, R x 36 z lines over the
// block's threads).  The groups of one target are adjacent items, so they share the spectra's
// lines in one L2.  LDS: R x 1298 values (41 KB for R = 4 in FP32 or 2 in FP64), each
// right-hand side's slab padded by one value against the x pass's bank conflicts.
template <class V, int R>
__global__ __launch_bounds__(256) void vlist_inv_kernel(const VTarget* __restrict__ vt, const int* __restrict__ grid,
                                                        int NL, BufTable bt, int v0, int nrhs) {
    constexpr int G3 = 1728;
    __shared__ V A[R][865], B[R][433];
    const int groups = (nrhs + R - 1) / R;
    const int item = xcd_item(blockIdx.x, gridDim.x);
    const int i = item / groups, r0 = (item - i * groups) * R, nr = min(R, nrhs - r0);
    const int t = threadIdx.x;
    const int64_t os = bt.stride[BUF_LF_CHK];
    const VTarget tg = vt[v0 + i];
    const V* in = bufp<V>(bt, BUF_TSPEC) + (int64_t)i * G3 * nrhs + r0;
    for (int e = t; e < nr * 144; e += blockDim.x) {   // x lines (ky, kz): 12 inputs -> x' in [6, 12)
        const int l = e / nr, r = e - l * nr;
        dft12_line<V, 12, 6, 0, 6, 1>(in + (int64_t)(12 * l) * nrhs + r, nrhs, A[r] + 6 * l, 1);
    }
    __syncthreads();
    for (int e = t; e < nr * 72; e += blockDim.x) {    // y lines (x', kz): A -> B[kz][y'][x']
        const int r = e / 72, l = e % 72;
        dft12_line<V, 12, 6, 0, 6, 1>(A[r] + (l % 6) + 72 * (l / 6), 6, B[r] + (l % 6) + 36 * (l / 6), 6);
    }
    __syncthreads();
    for (int e = t; e < nr * 36; e += blockDim.x) {    // z lines (x', y'): B -> C[z'][y'][x'] (reuses A)
        const int r = e / 36, l = e % 36;
        dft12_line<V, 12, 6, 0, 6, 1>(B[r] + l, 36, A[r] + l, 36);
    }
    __syncthreads();
    V* out = bufp<V>(bt, BUF_LF_CHK) + (int64_t)r0 * os + tg.out_off;
    const typename Real<V>::T coef = (typename Real<V>::T)(1.0 / G3);
    for (int e = t; e < nr * NL; e += blockDim.x) {
        const int r = e / NL, k = e % NL;
        const int g = grid[tg.grid + k];
        const V v = A[r][(g % 12 - 6) + 6 * ((g / 12) % 12 - 6) + 36 * (g / 144 - 6)];
        V* o = out + (int64_t)r * os + k;
        V w = *o;
        w.x += v.x * coef;
        w.y += v.y * coef;
        *o = w;
    }
}

// ---------------------------------------------------------------- setup-time generation
__global__ __launch_bounds__(256) void kgen_kernel(const KGen* __restrict__ jobs, const double* __restrict__ gp,
                                                   double2* __restrict__ gen, int j0, int ktype) {
    const KGen k = jobs[j0 + blockIdx.x];
    const double sg = k.tneg ? -1.0 : 1.0;
    const int64_t mn = (int64_t)k.m * k.n;
    for (int64_t e = blockIdx.y * 256 + threadIdx.x; e < mn; e += SETUP_SPLIT * 256) {
        const int i = (int)(e % k.m), j = (int)(e / k.m);
        const double* t = gp + 3 * (k.toff + i);
        const double* s = gp + 3 * (k.soff + j);
        double d[3];
        for (int q = 0; q < 3; ++q) d[q] = (sg * t[q] + k.tshift[q]) - (s[q] + k.sshift[q]);
        gen[k.out + e] = green64_table(d[0], d[1], d[2], ktype);
    }
}

__global__ void to_f32_kernel(const double2* __restrict__ in, float2* __restrict__ out, int64_t n) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x)
        out[e] = make_float2((float)in[e].x, (float)in[e].y);
}

template <class V>
__global__ void zero_kernel(V* p, int64_t n) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x)
        p[e] = mk<V>(0, 0);
}

// The caller's densities are read in input order (coalesced: random 16-byte reads would
// fetch a whole line each) and written to their leaf-sorted positions.
template <class V>
__global__ void gather_kernel(const IoPtrs* __restrict__ io, V* __restrict__ out, const int* __restrict__ iperm,
                              int64_t N, int nrhs) {
    const double2* __restrict__ in = io->den;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < N * nrhs; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = e / N, j = e % N;
        const double2 v = in[e];
        out[r * N + iperm[j]] = mk<V>(v.x, v.y);
    }
}

template <class V>
__global__ void scatter_kernel(const V* __restrict__ in, const IoPtrs* __restrict__ io, const int* __restrict__ perm,
                               int64_t N, int nrhs) {
    double2* __restrict__ out = io->val;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < N * nrhs; e += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = e / N, i = e % N;
        const V v = in[e];
        out[r * N + perm[i]] = make_double2(v.x, v.y);
    }
}

// direct sum u(t_i) = sum_j G(t_i, s_j) f_j (Wave3d::check, wave3d_check.cpp:66-76).
// Block (target tile x, source range y, right-hand-side group z): 256 targets, one thread
// each, over the sources [y * chunk, (y + 1) * chunk) staged through LDS in tiles of 256;
// G is evaluated once per pair for the RC right-hand sides of the group.  With one source
// range the sums go straight to out, otherwise to part[y][rhs][target] for the fixed-order
// reduction below.
template <int RC, int KT>
__global__ __launch_bounds__(256) void direct_kernel(const double* __restrict__ trg, int M,
                                                     const double* __restrict__ src, int Ns,
                                                     const double2* __restrict__ den, int nrhs,
                                                     double2* __restrict__ out, int chunk) {
    __shared__ double s3[256 * 3];
    __shared__ double2 sd[RC][256];
    const int i = blockIdx.x * 256 + threadIdx.x;
    const int r0 = blockIdx.z * RC, nr = min(RC, nrhs - r0);
    const bool ok = i < M;
    double tx = 0, ty = 0, tz = 0;
    if (ok) { tx = trg[3 * i]; ty = trg[3 * i + 1]; tz = trg[3 * i + 2]; }
    double2 acc[RC];
#pragma unroll
    for (int q = 0; q < RC; ++q) acc[q] = make_double2(0, 0);
    const int j0 = blockIdx.y * chunk, j1 = min(Ns, j0 + chunk);
    for (int sb = j0; sb < j1; sb += 256) {
        const int n = min(256, j1 - sb);
        __syncthreads();
        if ((int)threadIdx.x < n) {
            const int j = sb + threadIdx.x;
            s3[3 * threadIdx.x] = src[3 * j];
            s3[3 * threadIdx.x + 1] = src[3 * j + 1];
            s3[3 * threadIdx.x + 2] = src[3 * j + 2];
#pragma unroll
            for (int q = 0; q < RC; ++q)
                sd[q][threadIdx.x] = q < nr ? den[(int64_t)(r0 + q) * Ns + j] : make_double2(0, 0);
        }
        __syncthreads();
        if (ok)
            for (int j = 0; j < n; ++j) {
                const double2 g = green64<KT>(tx - s3[3 * j], ty - s3[3 * j + 1], tz - s3[3 * j + 2]);
#pragma unroll
                for (int q = 0; q < RC; ++q) cfma(acc[q], g, sd[q][j]);
            }
    }
    if (!ok) return;
    double2* o = out + (int64_t)blockIdx.y * nrhs * M + i;
#pragma unroll
    for (int q = 0; q < RC; ++q)
        if (q < nr) o[(int64_t)(r0 + q) * M] = acc[q];
}

// out[e] = sum_{y < S} part[y][e] in the order y = 0, 1, ... (deterministic)
__global__ void direct_reduce_kernel(const double2* __restrict__ part, int64_t n, int S, double2* __restrict__ out) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
        double2 a = part[e];
        for (int y = 1; y < S; ++y) {
            const double2 b = part[(int64_t)y * n + e];
            a.x += b.x;
            a.y += b.y;
        }
        out[e] = a;
    }
}

// dense Kernel3d::kernel block: out(i,j) = G(trg_i, src_j), column-major M x N
template <class V>
__global__ void kmatrix_kernel(const double* __restrict__ trg, int M, const double* __restrict__ src, int Ns,
                               V* __restrict__ out, int ktype) {
    const int64_t mn = (int64_t)M * Ns;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < mn; e += (int64_t)gridDim.x * blockDim.x) {
        const int i = (int)(e % M), j = (int)(e / M);
        const double x = trg[3 * i] - src[3 * j], y = trg[3 * i + 1] - src[3 * j + 1], z = trg[3 * i + 2] - src[3 * j + 2];
        out[e] = ktype == 0 ? green<V, 0>(x, y, z) : green<V, 1>(x, y, z);
    }
}

// segmented reduction: target t gets the sum of its cnt adjacent contribution slots
// (M elements each) in a fixed order; one wave per target, four targets per block.  A lane
// owns rows lane + 64 r (r < R, R = 2 for M <= 128, 3 for M <= 192) and walks the slots
// once, all R loads of a slot in flight together; lanes past M read row M - 1 (in bounds)
// and store nothing.
template <class V, int R>
__device__ __forceinline__ void reduce_rows(const V* __restrict__ in, V* __restrict__ out, int M, int cnt, int mode,
                                            int m0, int lane) {
    using T = typename Real<V>::T;
    int idx[R];
    T sx[R], sy[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        idx[r] = min(m0 + lane + 64 * r, M - 1);
        sx[r] = 0;
        sy[r] = 0;
    }
#pragma unroll 4
    for (int j = 0; j < cnt; ++j) {
        const V* s = in + (int64_t)j * M;
        V v[R];
#pragma unroll
        for (int r = 0; r < R; ++r) v[r] = s[idx[r]];
#pragma unroll
        for (int r = 0; r < R; ++r) {
            sx[r] += v[r].x;
            sy[r] += v[r].y;
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int m = m0 + lane + 64 * r;
        if (m < M) {
            if (mode) {
                const V o = out[m];
                sx[r] += o.x;
                sy[r] += o.y;
            }
            out[m] = mk<V>(sx[r], sy[r]);
        }
    }
}

template <class V>
__global__ __launch_bounds__(256) void reduce_kernel(const RTarget* __restrict__ rtrg, int n, BufTable bt, int t0,
                                                     const V* __restrict__ inb, int64_t ins) {
    const int ti = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (ti >= n) return;
    const RTarget r = rtrg[t0 + ti];
    const int rhs = blockIdx.y;
    const V* in = inb + (int64_t)rhs * ins + r.red_off;
    V* out = bufp<V>(bt, r.obuf) + (int64_t)rhs * bt.stride[r.obuf] + r.out_off;
    if (r.M <= 128) {
        reduce_rows<V, 2>(in, out, r.M, r.cnt, r.mode, 0, lane);
    } else {
        for (int m0 = 0; m0 < r.M; m0 += 192) reduce_rows<V, 3>(in, out, r.M, r.cnt, r.mode, m0, lane);
    }
}

int grid_for(int64_t n, int threads) {
    int64_t b = (n + threads - 1) / threads;
    return (int)std::min<int64_t>(std::max<int64_t>(b, 1), 65536);
}

template <class V>
hipError_t launch_stage_t(const DevPlan& d, const Stage& s, int nrhs, hipStream_t st) {
    const int n = s.end - s.begin;
    switch (s.kind) {
    case ST_ZERO: {
        int64_t cnt = s.count * nrhs;   // rhs slabs are contiguous with stride = count
        if (cnt > 0) zero_kernel<V><<<grid_for(cnt, 256), 256, 0, st>>>((V*)d.bt.p[s.buf], cnt);
        break;
    }
    case ST_GATHER:
        gather_kernel<V><<<grid_for(d.N * nrhs, 256), 256, 0, st>>>(d.io, (V*)d.bt.p[BUF_DEN], d.iperm, d.N, nrhs);
        break;
    case ST_SCATTER:
        scatter_kernel<V><<<grid_for(d.N * nrhs, 256), 256, 0, st>>>((const V*)d.bt.p[BUF_VAL], d.io, d.perm, d.N,
                                                                     nrhs);
        break;
    case ST_KAPPLY: {
        if constexpr (sizeof(V) == 8) if (d.kmfma) {   // mixed precision: the products on the matrix cores
            const int nb = nrhs > 8 ? 2 : 1;
            const dim3 grid(n, (nrhs + 8 * nb - 1) / (8 * nb));
#define DDFMM_KMFMA(NB, KT, MIR) \
    kapply_mfma_kernel<NB, KT, MIR><<<grid, 256, 0, st>>>(d.ktasks, d.ksrcs, d.px, d.py, d.pz, d.bt, s.begin, n, nrhs)
            const int sel = (nb == 2 ? 4 : 0) + (d.ktype ? 2 : 0) + (s.mb == 1 ? 1 : 0);
            switch (sel) {
            case 0: DDFMM_KMFMA(1, 0, false); break;
            case 1: DDFMM_KMFMA(1, 0, true); break;
            case 2: DDFMM_KMFMA(1, 1, false); break;
            case 3: DDFMM_KMFMA(1, 1, true); break;
            case 4: DDFMM_KMFMA(2, 0, false); break;
            case 5: DDFMM_KMFMA(2, 0, true); break;
            case 6: DDFMM_KMFMA(2, 1, false); break;
            case 7: DDFMM_KMFMA(2, 1, true); break;
            }
#undef DDFMM_KMFMA
            break;
        }
        if (s.mb == 1) return hipErrorInvalidValue;    // mirror slots need the matrix-core kernel
#define DDFMM_KAPPLY(RC, KT) \
    kapply_kernel<V, RC, KT><<<dim3(n, (nrhs + RC - 1) / RC), KA_THREADS, 0, st>>>(d.ktasks, d.ksrcs, d.px, d.py, \
                                                                                   d.pz, d.bt, s.begin, n, nrhs)
        // G(t, s) evaluated once for up to 1, 4 or 8 right-hand sides
        switch ((nrhs == 1 ? 0 : nrhs <= 4 ? 2 : 4) + (d.ktype ? 1 : 0)) {
        case 0: DDFMM_KAPPLY(1, 0); break;
        case 1: DDFMM_KAPPLY(1, 1); break;
        case 2: DDFMM_KAPPLY(4, 0); break;
        case 3: DDFMM_KAPPLY(4, 1); break;
        case 4: DDFMM_KAPPLY(8, 0); break;
        case 5: DDFMM_KAPPLY(8, 1); break;
        }
#undef DDFMM_KAPPLY
        break;
    }
    case ST_GEMM:
        if (s.mb < 1 || s.mb > GEMM_MB) return hipErrorInvalidValue;
        if (d.mixed && s.prec == PREC_SOLVE)
            launch_gemm_form<double2, float2, double, 1, true, false>(s, nrhs, st, d, d.oppack64);
        else if (d.mixed && d.opmatbf)
            launch_gemm_bf16s(s.mb, n, nrhs, st, d, s.begin);
        else if (d.mixed && d.ktype == 0)    // e^{ikr}/r: three real products per complex one
            launch_gemm32<true>(s, nrhs, st, d);
        else if (d.mixed)
            launch_gemm32<false>(s, nrhs, st, d);
        else
            launch_gemm64(s, nrhs, st, d);
        break;
    case ST_FFTFWD:
        if (d.P != 6) return hipErrorInvalidValue;
        if (nrhs == 1) {
            fft_fwd_kernel<V><<<dim3(n, 1), 256, 0, st>>>(d.fsrc, d.grid, d.NL, d.bt, s.begin, n, 1);
        } else {    // 8 (FP32) or 4 (FP64) right-hand sides per block, two at a time: 66 or 76 KB of
            // LDS.  One and four at a time: 250k x 64 alone 2.64 and 1.98 ms (two 2.39), the pass
            // 66.4 and 66.0 (66.05); 1M x 2 0.29 and 0.244 (0.239).  Beside the GEMMs the FFT is
            // hidden, so the block that takes less LDS stays.
            constexpr int R = sizeof(V) == 8 ? 8 : 4;
            fft_fwd_multi_kernel<V, R, 2><<<dim3(n, (nrhs + R - 1) / R), 256, 0, st>>>(d.fsrc, d.grid, d.NL, d.bt,
                                                                                 s.begin, n, nrhs);
        }
        break;
    case ST_VLIST: {
        if (d.P != 6) return hipErrorInvalidValue;
        if (n == 0) break;
        const int nchunk = (int)s.count;
        const V* opm = d.mixed ? (const V*)d.opmat32 : (const V*)d.opmat;
        if (nrhs == 1) {
            vlist_acc_kernel<V><<<dim3(VL_GROUPS * nchunk, 1), VL_THREADS, 0, st>>>(d.vtrg, d.vchunk, d.vsrc, d.vpk, opm,
                                                                              d.bt, s.begin, s.buf, nchunk);
        } else {
            // right-hand sides per block: 16 / 8 / 4 (FP32) or 8 / 4 / 2 (FP64) by nrhs
            constexpr int R2 = VMulti<V>::R2;
            if (nrhs >= 8 * R2) {
                vlist_acc_multi_kernel<V, 1, 8><<<dim3(VL_GROUPS * nchunk, (nrhs + 8 * R2 - 1) / (8 * R2)), VL_THREADS, 0, st>>>(
                    d.vtrg, d.vchunk, d.vsrc, d.vpk, opm, d.bt, s.begin, s.buf, nchunk, nrhs);
            } else if (nrhs >= 4 * R2) {
                vlist_acc_multi_kernel<V, 2, 4><<<dim3(VL_GROUPS * nchunk, (nrhs + 4 * R2 - 1) / (4 * R2)), VL_THREADS, 0, st>>>(
                    d.vtrg, d.vchunk, d.vsrc, d.vpk, opm, d.bt, s.begin, s.buf, nchunk, nrhs);
            } else {
                vlist_acc_multi_kernel<V, 4, 2><<<dim3(VL_GROUPS * nchunk, (nrhs + 2 * R2 - 1) / (2 * R2)), VL_THREADS, 0, st>>>(
                    d.vtrg, d.vchunk, d.vsrc, d.vpk, opm, d.bt, s.begin, s.buf, nchunk, nrhs);
            }
        }
        {
            constexpr int R = sizeof(V) == 8 ? 4 : 2;      // right-hand sides per block
            vlist_inv_kernel<V, R><<<n * ((nrhs + R - 1) / R), 256, 0, st>>>(d.vtrg, d.grid, d.NL, d.bt, s.begin, nrhs);
        }
        break;
    }
    case ST_REDUCE:
        if (s.buf != BUF_RED && s.buf != BUF_NMIR) return hipErrorInvalidValue;
        reduce_kernel<V><<<dim3((n + 3) / 4, nrhs), 256, 0, st>>>(d.rtrg, n, d.bt, s.begin, (const V*)d.bt.p[s.buf],
                                                                  d.bt.stride[s.buf]);
        break;
    default:
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

__global__ void set_io_kernel(IoPtrs* io, const double2* den, double2* val) {
    io->den = den;
    io->val = val;
}

}  // namespace

// ---------------------------------------------------------------- launchers
hipError_t launch_set_io(IoPtrs* io, const double2* den, double2* val, hipStream_t st) {
    set_io_kernel<<<1, 1, 0, st>>>(io, den, val);
    return hipGetLastError();
}

hipError_t launch_stage(const DevPlan& d, const Stage& s, int nrhs, hipStream_t st) {
    return d.mixed ? launch_stage_t<float2>(d, s, nrhs, st) : launch_stage_t<double2>(d, s, nrhs, st);
}

hipError_t launch_setup_gemm(const DevPlan& d, const Stage& s, hipStream_t st) {
    if (s.kind != ST_GEMM || s.mb < 1 || s.mb > GEMM_MB || s.buf < BUF_OPMAT || s.buf >= BUF_ALL)
        return hipErrorInvalidValue;
    launch_gemm_form<double2, double2, double, 1, false, false>(s, 1, st, d, (const double2*)d.bt.p[s.buf]);
    return hipGetLastError();
}

hipError_t launch_kgen(const KGen* jobs, int njobs, const double* gp, double2* gen, int ktype, hipStream_t st) {
    for (int j0 = 0; j0 < njobs; j0 += 65536) {
        int n = std::min(65536, njobs - j0);
        kgen_kernel<<<dim3(n, SETUP_SPLIT), 256, 0, st>>>(jobs, gp, gen, j0, ktype);
    }
    return hipGetLastError();
}

hipError_t launch_pack(const PackA* jobs, int njobs, const double2* opmat, void* out, int f32, int pair, hipStream_t st) {
    for (int j0 = 0; j0 < njobs; j0 += 65536) {
        const int n = std::min(65536, njobs - j0);
        const dim3 grid(n, SETUP_SPLIT);
        if (f32) pack_kernel<float2><<<grid, 256, 0, st>>>(jobs + j0, opmat, (float2*)out, pair);
        else pack_kernel<double2><<<grid, 256, 0, st>>>(jobs + j0, opmat, (double2*)out, 0);
    }
    return hipGetLastError();
}

hipError_t launch_to_bf16s(const double2* in, void* out, int64_t n, hipStream_t st) {
    if (n > 0) to_bf16s_kernel<<<grid_for(n, 256), 256, 0, st>>>(in, (Bf16s*)out, n);
    return hipGetLastError();
}

hipError_t launch_to_f32(const double2* in, float2* out, int64_t n, hipStream_t st) {
    if (n > 0) to_f32_kernel<<<grid_for(n, 256), 256, 0, st>>>(in, out, n);
    return hipGetLastError();
}

DirectSplit direct_split(int M, int Ns, int nrhs) {
    DirectSplit d;
    d.rc = nrhs == 1 ? 1 : nrhs <= 4 ? 4 : 8;
    const int mb = (M + 255) / 256, rg = (nrhs + d.rc - 1) / d.rc;
    const int tiles = std::max(1, (Ns + 255) / 256);
    // about 1024 blocks: source ranges until the target tiles and groups alone fill that;
    // S * nrhs * M <= 1024 * 256 * 8 elements, so the partial sums fit in DIRECT_SCRATCH_BYTES
    int S = std::max(1, std::min(tiles, 1024 / std::max(1, mb * rg)));
    const int per = (tiles + S - 1) / S;
    d.chunk = per * 256;
    d.S = (std::max(Ns, 1) + d.chunk - 1) / d.chunk;
    d.part_elems = d.S > 1 ? (int64_t)d.S * nrhs * M : 0;
    return d;
}

hipError_t launch_direct(const double* trg, int M, const double* src, int Ns, const double2* den, int nrhs,
                         double2* out, double2* part, int ktype, hipStream_t st) {
    const DirectSplit d = direct_split(M, Ns, nrhs);
    if (d.S > 1 && !part) return hipErrorInvalidValue;
    double2* dst = d.S > 1 ? part : out;
    const dim3 grid((M + 255) / 256, d.S, (nrhs + d.rc - 1) / d.rc);
#define DDFMM_DIRECT(RC)                                                                          \
    (ktype == 0 ? direct_kernel<RC, 0> : direct_kernel<RC, 1>)<<<grid, 256, 0, st>>>(trg, M, src, Ns, den, nrhs, dst, \
                                                                                     d.chunk)
    if (d.rc == 1) DDFMM_DIRECT(1);
    else if (d.rc == 4) DDFMM_DIRECT(4);
    else DDFMM_DIRECT(8);
#undef DDFMM_DIRECT
    if (d.S > 1) {
        const int64_t n = (int64_t)nrhs * M;
        direct_reduce_kernel<<<grid_for(n, 256), 256, 0, st>>>(part, n, d.S, out);
    }
    return hipGetLastError();
}

hipError_t launch_kmatrix(const double* trg, int M, const double* src, int Ns, void* out, int ktype, int f32,
                          hipStream_t st) {
    if (f32)
        kmatrix_kernel<float2><<<grid_for((int64_t)M * Ns, 256), 256, 0, st>>>(trg, M, src, Ns, (float2*)out, ktype);
    else
        kmatrix_kernel<double2><<<grid_for((int64_t)M * Ns, 256), 256, 0, st>>>(trg, M, src, Ns, (double2*)out, ktype);
    return hipGetLastError();
}

// ---------------------------------------------------------------- no-allocation direct sum
// Partial sums of the direct sum for callers that cannot allocate: one static array per
// GPU, its device address taken once per device with that device current.  Calls on one
// GPU share the array, so calls that overlap on one GPU race.
static __device__ __align__(256) double2 scratch[DIRECT_SCRATCH_BYTES / sizeof(double2)];

hipError_t direct_static_scratch(double2** out) {
    static std::mutex mu;
    static std::vector<double2*> ptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    std::lock_guard<std::mutex> lock(mu);
    if ((int)ptr.size() <= dev) ptr.resize(dev + 1, nullptr);
    if (!ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        ptr[dev] = (double2*)p;
    }
    *out = ptr[dev];
    return hipSuccess;
}

}  // namespace ddfmm
