// Rotation + range decimation for filters longer than the bfloat16 x 3 forms take (more than 128 taps: small images from
// wide-band histories), in float32 on v_mfma_f32_16x16x4_f32 (the stage of fastsar/ffbp_cpu.cpp:147-255). With k_j = D j
// - pl,
//   y_c[j] = rho_c(j) sum_r x[k_j + r] g_c[r],   g_c[r] = h[r] exp(2 pi i sl_c r),
//   rho_c(j) = exp(2 pi i (c0_c + (k_j - kc) sl_c)),
// per row the real product Y^T [2C x Ko] = G [2C x 2L] X [2L x Ko]: rows (Re y_c, Im y_c), contraction over (tap, Re or
// Im of x), tap r = D u + ph taken in (ph, u) order two phases at a time: contraction index k of a step is component
// k % 2 of phase ph + k / 2.
//
// Work: block (row p, parent n, N-group and M-chunk), four waves. The row's window goes to LDS as D planes (plane ph
// holds x[D m + ph - pl], m = 0, 1, ...): the operand of output j at tap D u + ph is word j + u of plane ph, planes 16
// mod 32 samples apart, so a wave's read (16 outputs, two planes, two components) falls on 64 different banks. The
// children's taps go to LDS once a block, [child][ph][u], each tap's phasor from float64 (runs of a phase's taps stepped in
// float32 from one seed took as long, 256 us of the image below for 251, and their steps' rounding adds up: 141 taps at D 9
// -128.2 dB from float64 against the VALU form's -130.6, -131.2 so); a lane reads the component its row and index need and
// flips its sign for (Re, Im x). Wave w takes N-tile (8 children) w mod NTG and runs up to four M-tiles (16 outputs) a time
// against them, a step's operands read ahead of the step before. Result: lane (output j = lane % 16, q = lane / 16) holds
// (Re, Im) of children 2 q and 2 q + 1, rotated by rho from float64 and stored, 16 consecutive outputs of a child a time.
//
// Bound by the float32 matrix rate (the VALU's; no operand is rounded) and, at two waves a SIMD, by the reads of a step.
// 534 x 534 image from 1,400 x 4,088 samples (D 16, 134 taps, 25 children): 1,395 us on the VALU kernel, which read two
// LDS words a tap and output, 257 us here (10 GFLOP of real products, 39 TFLOP/s). Two waves a SIMD are all that LDS leaves,
// and declared, so that the sums stay in VGPRs: in AGPRs the compiler moved 12 of them a step (262 us).
#include "fsh_common.h"
#include "fsh_kernels.h"

#include <algorithm>

namespace fsh {

namespace {

typedef float floatx4_t __attribute__((ext_vector_type(4)));

// Contraction steps of one chain of sums (four products each); the chains' results are added. One chain of all 2 L products
// rounds above the VALU form, which deals an output's taps to several threads where a block has few outputs: -127.8 dB from
// float64 against -130.2 at 261 taps, -134.2 in chains of 32 steps, -136.5 of 11. First level of the 534 x 534 image above:
// 251 us in one chain, 257 in chains of 32 steps, 255 of 64.
constexpr int SUM_STEPS = 32;

struct F32Shape {
    int U, Up, D2, CS, PS, NTG, MC, chunks, ngroups;
    size_t lds;
};

}  // namespace

__global__ __launch_bounds__(256, 2) void k_rot_fir_k_f32(const float2* __restrict__ x, int P, int K,
                                                          const float* __restrict__ c0, const float* __restrict__ sl, int Cn,
                                                          const float* __restrict__ taps, int L, int pl, int D, int Ko,
                                                          double kc, int U, int Up, int D2, int CS, int PS, int NTG, int MC,
                                                          int chunks, float2* __restrict__ y)
{
    extern __shared__ float lds_f[];
    float2* X = reinterpret_cast<float2*>(lds_f);          // [D2][PS]
    float* G = lds_f + 2 * (size_t)D2 * PS;                // [8 NTG][CS]
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int p = blockIdx.x, n = blockIdx.y, chunk = blockIdx.z % chunks, cb = blockIdx.z / chunks * 8 * NTG;
    const int MT = (Ko + 15) / 16;
    const int m0 = chunk * MC, m1 = min(m0 + MC, MT);
    const int WM = 16 * (m1 - m0) + U;                     // words a plane
    const int ks = D * 16 * m0 - pl;                       // sample of word 0 of plane 0
    const float2* xrow = x + ((size_t)n * P + p) * K;
    {
        // sample ks + i is word i / D of plane i mod D; eight loads in flight
        constexpr int XB = 8;
        const int total = D * WM, dm = 256 / D, dph = 256 - dm * D;
        int m = tid / D, ph = tid - m * D;
        for (int i0 = tid; i0 < total; i0 += 256 * XB) {
            float2 v[XB];
            int dst[XB];
            #pragma unroll
            for (int e = 0; e < XB; ++e) {
                const int i = i0 + 256 * e, kk = ks + i;
                v[e] = make_float2(0.f, 0.f);
                if (i < total && kk >= 0 && kk < K) v[e] = xrow[kk];
                dst[e] = i < total ? ph * PS + m : -1;
                m += dm;
                ph += dph;
                if (ph >= D) { ph -= D; ++m; }
            }
            #pragma unroll
            for (int e = 0; e < XB; ++e)
                if (dst[e] >= 0) X[dst[e]] = v[e];
        }
        if (D2 > D)                                        // an odd count of phases: a plane of zeros
            for (int i = tid; i < WM; i += 256) X[(size_t)D * PS + i] = make_float2(0.f, 0.f);
    }
    // taps: run (child, ph), every tap's phasor from float64
    for (int e = tid; e < 8 * NTG * D2; e += 256) {
        const int c = e / D2, ph = e - c * D2;
        float2* g = reinterpret_cast<float2*>(G + (size_t)c * CS) + ph * Up;
        const bool ok = cb + c < Cn && ph < D;
        const double b = ok ? (double)sl[((size_t)n * Cn + cb + c) * P + p] : 0.0;
        for (int u = 0; u < U; ++u) {
            const int r = D * u + ph;
            float2 v = make_float2(0.f, 0.f);
            if (ok && r < L) {
                float cs, sn;
                cis_cyc((double)r * b, cs, sn);
                v = make_float2(taps[r] * cs, taps[r] * sn);
            }
            g[u] = v;
        }
    }
    __syncthreads();
    const int wps = 4 / NTG, nt = wv / wps, ws = wv - nt * wps;    // N-tile, and this wave's share of its M-tiles
    const int i = lane & 15, k = lane >> 4, t = i & 1, comp = k & 1;
    const unsigned flip = (!t && comp) ? 0x80000000u : 0u;
    const float* ga = G + (size_t)(8 * nt + (i >> 1)) * CS + (k >> 1) * 2 * Up + (t ^ comp);
    const float* xa = reinterpret_cast<const float*>(X) + 2 * ((size_t)(k >> 1) * PS + i) + comp;
    const int steps = (D2 / 2) * U;
    const int j2 = i;                                      // result role: output column
    for (int mg = m0 + 4 * ws; mg < m1; mg += 4 * wps) {
        floatx4_t acc[4] = {};
        const float* xm = xa + 2 * 16 * (mg - m0);
        // tiles past the last read the last tile's words again (in bounds) and are not stored
        int off[4];
        #pragma unroll
        for (int m = 0; m < 4; ++m) off[m] = 32 * min(m, m1 - 1 - mg);
        int u = 0, go = 0, xo = 0;                         // offsets (floats) of the step to read next
        float gn = ga[0], xn[4];
        #pragma unroll
        for (int m = 0; m < 4; ++m) xn[m] = xm[off[m]];
        for (int s0 = 0; s0 < steps; s0 += SUM_STEPS) {
            floatx4_t part[4] = {};
            for (int s = s0; s < min(s0 + SUM_STEPS, steps); ++s) {
                const float g = __uint_as_float(__float_as_uint(gn) ^ flip);
                float xv[4];
                #pragma unroll
                for (int m = 0; m < 4; ++m) xv[m] = xn[m];
                const bool wrap = ++u == U;
                go += wrap ? 4 * Up - 2 * U + 2 : 2;
                xo += wrap ? 4 * PS - 2 * U + 2 : 2;
                u = wrap ? 0 : u;
                if (s + 1 == steps) go = xo = 0;           // (read, not used)
                gn = ga[go];
                #pragma unroll
                for (int m = 0; m < 4; ++m) xn[m] = xm[xo + off[m]];
                #pragma unroll
                for (int m = 0; m < 4; ++m) part[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(g, xv[m], part[m], 0, 0, 0);
            }
            #pragma unroll
            for (int m = 0; m < 4; ++m) acc[m] += part[m];
        }
        #pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int c = cb + 8 * nt + 2 * k + e;
            if (c >= Cn) continue;
            const size_t rc = ((size_t)n * Cn + c) * P + p;
            const double a = (double)c0[rc], b = (double)sl[rc];
            #pragma unroll
            for (int m = 0; m < 4; ++m) {
                const int j = 16 * (mg + m) + j2;
                if (mg + m < m1 && j < Ko) {
                    float cs, sn;
                    cis_cyc(fma((double)(D * j - pl) - kc, b, a), cs, sn);
                    const float ar = acc[m][2 * e], ai = acc[m][2 * e + 1];
                    y[rc * Ko + j] = make_float2(fmaf(ar, cs, -(ai * sn)), fmaf(ar, sn, ai * cs));
                }
            }
        }
    }
}

// the launch's shape: as many N-tiles a block as its waves (four) and as few M-chunks as fit 80 KB of LDS (two blocks a
// CU), else 156 KB; false where not even one N-tile and M-tile fit, or a phase has more than 16 taps
static bool f32_shape(int L, int D, int Ko, int Cn, F32Shape& s)
{
    if (D < 2) return false;
    s.U = (L + D - 1) / D;
    if (s.U > 16) return false;
    s.Up = s.U | 1;
    s.D2 = D + (D & 1);
    s.CS = (2 * s.D2 * s.Up + 7) / 16 * 16 + 8;            // 8 mod 16 words: eight children on different banks
    const int MT = (Ko + 15) / 16, NT = (Cn + 7) / 8;
    for (size_t budget : {80, 156})
        for (int ntg : {4, 2, 1}) {
            if (ntg > 1 && NT <= ntg / 2) continue;
            for (int chunks = 1; chunks <= MT; ++chunks) {
                s.NTG = ntg;
                s.MC = (MT + chunks - 1) / chunks;
                s.chunks = (MT + s.MC - 1) / s.MC;
                s.PS = (16 * s.MC + s.U - 16 + 31) / 32 * 32 + 16;
                s.lds = (size_t)8 * s.D2 * s.PS + (size_t)4 * 8 * ntg * s.CS;
                s.ngroups = (NT + ntg - 1) / ntg;
                if (s.lds <= budget * 1024) return true;
                if (budget == 80 && s.MC <= 4) break;      // shorter chunks only where nothing else fits
            }
        }
    return false;
}

int launch_rot_fir_k_f32(const float2* x, int Np, int P, int K, const float* c0, const float* sl, int Cn, const float* taps,
                         int L, int pl, int D, int Ko, double kc, float2* y, hipStream_t s)
{
    F32Shape h;
    if (!f32_shape(L, D, Ko, Cn, h) || (long)h.chunks * h.ngroups > 65535) return E_INVALID;
    for (int n0 = 0; n0 < Np; n0 += 65535) {
        const dim3 grid((unsigned)P, (unsigned)std::min(65535, Np - n0), (unsigned)(h.chunks * h.ngroups));
        hipLaunchKernelGGL(k_rot_fir_k_f32, grid, dim3(256), h.lds, s, x + (size_t)n0 * P * K, P, K, c0 + (size_t)n0 * Cn * P,
                           sl + (size_t)n0 * Cn * P, Cn, taps, L, pl, D, Ko, kc, h.U, h.Up, h.D2, h.CS, h.PS, h.NTG, h.MC,
                           h.chunks, y + (size_t)n0 * Cn * P * Ko);
        FSH_TRY(hipGetLastError());
    }
    return OK;
}

}  // namespace fsh
