// The one-pass VALU level's kernel template, shared by the translation units that instantiate it
// (fused_kernels.hip: the decimation factors read at run time; fused_kernels_k<Dk>p<Dp>.hip: both fixed).
#pragma once
#include "fsh_common.h"

#include <type_traits>

namespace fsh {

constexpr int DMAX = 4;                        // the largest decimation factor of the fused form, on either axis

// Taps (uniform values) are moved to vector registers where a filter's fit VTAPS of them: a float32 fma whose operands
// are all VGPRs issues in about 2.5 cycles a wave, one with a scalar operand in 4.4 (both at two or more waves a SIMD). Not
// where the form with its factors read at run time, which keeps room for DMAX phases, would pass the 128 registers of four
// waves a SIMD: with the rows' addresses kept for every period of its unrolled loop as well it took 140 to 211, and levels
// that fill the device ran up to 1.8 times as long as with 70 to 112 (4,000 parents of 4 x 30 columns, 2 x 1, 85 -> 152 us)
constexpr int VTAPS = 32;
__device__ __forceinline__ void in_vgpr(float& v) { asm volatile("" : "+v"(v)); }

// f(std::integral_constant<int, I>) for I = B .. E - 1, unrolled at compile time
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f)
{
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// the row stride of x in LDS (float2): the samples and Dk - 1 zeros on either side, odd
__host__ __device__ inline int fused_row(int K, int Dk) { return (K + 2 * (Dk - 1)) | 1; }

// DK, DP: the range and pulse decimation factors fixed at compile time (the loops over phases exact, half the taps
// or fewer in scalar registers), or 0: read at run time, the loops running to DMAX with the phases past it skipped
template <int NWK, int NWP, int DK = 0, int DP = 0>
__global__ __launch_bounds__(256) void k_level_fused(const float2* __restrict__ x, int P, int K, const float* __restrict__ c0,
                                                      const float* __restrict__ sl, int C, const float* __restrict__ hk_t,
                                                      int Dk, int plk, int Ko, const float* __restrict__ hp_t, int Dp, int plp,
                                                      int Po, double kc, int Np, int CB, int R, float2* __restrict__ z)
{
    extern __shared__ float2 lds_f2[];
    const int nCB = (C + CB - 1) / CB;
    const int G = Np * nCB;
    // blocks are dispatched round-robin over the 8 XCDs; renumber so that each XCD runs a contiguous range of
    // (parent, child block) pairs and the blocks of one parent share that XCD's L2
    int wg = blockIdx.x;
    {
        const int q = G >> 3, rem = G & 7, xcd = wg & 7;
        wg = xcd * q + min(xcd, rem) + (wg >> 3);
    }
    const int n = wg / nCB, cb = wg - n * nCB;
    const int cbeg = cb * CB, cn = min(CB, C - cbeg);
    // a row of x in LDS: Dk - 1 zeros, its K samples, Dk - 1 zeros, so that a period partly outside [0, K) reads zeros and
    // no read is checked or clamped
    const int pad = (DK ? DK : Dk) - 1, KS = fused_row(K, DK ? DK : Dk), KoS = Ko | 1;
    float2* xs = lds_f2;                       // [R][KS]
    float2* ys = xs + (size_t)R * KS;          // [cn][R][KoS]
    const int tid = threadIdx.x, BT = blockDim.x;
    const float2* xn = x + (size_t)n * P * K;
    for (int i = tid; i < R * 2 * pad; i += BT) {
        const int r = i / (2 * pad), e = i - r * 2 * pad;
        xs[r * KS + (e < pad ? e : K + e)] = make_float2(0.f, 0.f);
    }

    // pulse-filter column of this thread and its streaming state
    const bool colok = tid < cn * Ko;
    const int pc = colok ? tid / Ko : 0, pj = colok ? tid - pc * Ko : 0;
    float2* zc = z + ((size_t)(n * C + cbeg + pc) * Po) * Ko + pj;
    float2 pacc[NWP];
    #pragma unroll
    for (int s = 0; s < NWP; ++s) pacc[s] = make_float2(0.f, 0.f);
    // rows are numbered p = Dp m - plp + ph (period m, phase ph); slot s holds output m - NWP + 1 + s in period m;
    // the stream starts at the virtual row -plp (m = 0, ph = 0), rows before 0 being zero. The slots move down by one
    // from a period to the next with the sums of its first row (acc[s] = h v + acc[s + 1]), not by moves of their own
    int pm = plp / Dp, pph = plp - pm * Dp;    // row 0: the zero rows before it leave every slot zero
    for (int d = 0; d <= pm - NWP && d < Po; ++d)      // (outputs that read no other rows)
        if (colok) zc[(size_t)d * Ko] = make_float2(0.f, 0.f);
    auto end_period = [&]() {
        const int done = pm - NWP + 1;
        if (colok && done >= 0 && done < Po) zc[(size_t)done * Ko] = pacc[0];
        ++pm;
    };

    // the first XPF samples per thread of each chunk are loaded a chunk ahead into registers (their latency hidden
    // behind the chunk before), the rest when the chunk is staged
    constexpr int XPF = 4;
    float2 xpf[XPF];
    // (every thread makes the same XPF reads, past the chunk clamped to its last sample, so that the number of
    // reads in flight does not depend on the path and a wait for an earlier read leaves these in flight)
    auto prefetch = [&](int p0) {
        const float2* src = xn + (size_t)p0 * K;
        const int cnt = min(R, P - p0) * K;
        #pragma unroll
        for (int k = 0; k < XPF; ++k) xpf[k] = load_ahead(src + min(tid + BT * k, cnt - 1));
    };
    prefetch(0);
    for (int p0 = 0; p0 < P; p0 += R) {
        const int rn = min(R, P - p0);
        {
            const float2* src = xn + (size_t)p0 * K;
            const int cnt = rn * K;
            #pragma unroll
            for (int k = 0; k < XPF; ++k) {
                const int i = tid + BT * k;
                if (i < cnt) {
                    const int r = i / K;
                    xs[r * KS + pad + (i - r * K)] = xpf[k];
                }
            }
            for (int i = tid + BT * XPF; i < cnt; i += BT) {
                const int r = i / K;
                xs[r * KS + pad + (i - r * K)] = src[i];
            }
        }
        __syncthreads();
        // this thread's range-filter row phase terms, read before the next chunk's prefetch so that waiting for
        // them leaves the prefetch in flight (both are ordered reads)
        float ra0, rb0;
        {
            const int c = min(tid / R, cn - 1), r = min(tid - (tid / R) * R, rn - 1);   // clamped: every thread reads
            const size_t ci = ((size_t)n * C + cbeg + c) * P + p0 + r;
            ra0 = load_ahead(c0 + ci);
            rb0 = load_ahead(sl + ci);
        }
        prefetch(p0 + R < P ? p0 + R : p0);             // the last chunk reads its own rows again, unused

        // range filter: thread (c, r)
        if (tid < cn * R) {
            const int c = tid / R, r = tid - c * R;
            if (r < rn) {
                constexpr int DL = DK ? DK : DMAX;    // phases the loops run over
                float hk[DL][NWK];                    // the taps of every phase
                #pragma unroll
                for (int ph = 0; ph < DL; ++ph) {
                    #pragma unroll
                    for (int s = 0; s < NWK; ++s) {
                        hk[ph][s] = (DK || ph < Dk) ? hk_t[ph * NWK + s] : 0.f;
                        if (DL * NWK <= VTAPS && (DK || NWK + NWP <= 18)) in_vgpr(hk[ph][s]);
                    }
                }
                const double a = (double)ra0, b = (double)rb0;
                float er, ei, wr = 0.f, wi = 0.f;
                cis_cyc(b, er, ei);
                const float2* xr = xs + r * KS + pad;
                float2* yr = ys + ((size_t)c * R + r) * KoS;
                // ring of accumulators: output o lives in slot o mod NWK; the period loop is unrolled NWK times so
                // that every slot index is a constant
                float2 acc[NWK];
                #pragma unroll
                for (int s = 0; s < NWK; ++s) acc[s] = make_float2(0.f, 0.f);
                const int mend = Ko + NWK - 1;
                int mseed = -(1 << 30);
                for (int m0 = 0; m0 < mend; m0 += NWK) {
                    static_for<0, NWK>([&](auto qc) {
                        constexpr int q = decltype(qc)::value;
                        const int m = m0 + q;
                        if (m < mend) {
                            int kb = (DK ? DK : Dk) * m - plk;
                            // opaque, so that the run-time form keeps no address a period and phase in registers (VTAPS)
                            if (!DK) asm volatile("" : "+s"(kb));
                            if (kb + (DK ? DK : Dk) > 0 && kb < K) {  // a period with samples in [0, K)
                                float2 v[DL];
                                #pragma unroll
                                for (int ph = 0; ph < DL; ++ph) v[ph] = xr[kb + (DK ? ph : min(ph, Dk - 1))];
                                if (m - mseed >= 16) {        // reseed in float64 every 16 periods
                                    cis_cyc(fma((double)kb - kc, b, a), wr, wi);
                                    mseed = m;
                                }
                                #pragma unroll
                                for (int ph = 0; ph < DL; ++ph) {
                                    if (DK || ph < Dk) {
                                        const float vr = fmaf(v[ph].x, wr, -(v[ph].y * wi));
                                        const float vi = fmaf(v[ph].x, wi, v[ph].y * wr);
                                        const float nr = fmaf(wr, er, -(wi * ei));
                                        wi = fmaf(wr, ei, wi * er);
                                        wr = nr;
                                        #pragma unroll
                                        for (int s = 0; s < NWK; ++s) {
                                            float2& o = acc[(q + 1 + s) % NWK];
                                            o.x = fmaf(hk[ph][s], vr, o.x);
                                            o.y = fmaf(hk[ph][s], vi, o.y);
                                        }
                                    }
                                }
                            } else {
                                mseed = -(1 << 30);           // the rotation restarts at the next period in range
                            }
                            // output m - NWK + 1 (slot (q + 1) mod NWK) is complete; the slot starts output m + 1
                            float2& o = acc[(q + 1) % NWK];
                            const int done = m - NWK + 1;
                            if (done >= 0) yr[done] = o;
                            o = make_float2(0.f, 0.f);
                        }
                    });
                }
            }
        }
        __syncthreads();

        // pulse filter: thread (c, j) over the chunk's rows
        constexpr int PL = DP ? DP : DMAX;
        float hp[PL][NWP];
        #pragma unroll
        for (int ph = 0; ph < PL; ++ph) {
            #pragma unroll
            for (int s = 0; s < NWP; ++s) {
                hp[ph][s] = (DP || ph < Dp) ? hp_t[ph * NWP + s] : 0.f;
                if (PL * NWP <= VTAPS) in_vgpr(hp[ph][s]);
            }
        }
        const float2* yc = ys + (size_t)pc * R * KoS + pj;
        for (int r = 0; r < rn; ++r) {
            const float2 v = colok ? yc[r * KoS] : make_float2(0.f, 0.f);
            #pragma unroll
            for (int ph = 0; ph < PL; ++ph) {
                if (ph == pph) {
                    #pragma unroll
                    for (int s = 0; s < NWP; ++s) {
                        const float2 o = ph ? pacc[s] : s + 1 < NWP ? pacc[s + 1 < NWP ? s + 1 : s] : make_float2(0.f, 0.f);
                        pacc[s].x = fmaf(hp[ph][s], v.x, o.x);
                        pacc[s].y = fmaf(hp[ph][s], v.y, o.y);
                    }
                }
            }
            if (++pph == (DP ? DP : Dp)) { end_period(); pph = 0; }
        }
        // the next chunk's x load writes only xs, which no thread reads after the barrier above; its range filter
        // writes ys, which the barrier after that load orders after every thread's pulse filter of this chunk
    }
    // the zero rows after the last: finish the open period, then every period until the last output is stored
    if (pph != 0) end_period();
    while (pm - NWP + 1 < Po) {
        #pragma unroll
        for (int s = 0; s < NWP - 1; ++s) pacc[s] = pacc[s + 1];
        pacc[NWP - 1] = make_float2(0.f, 0.f);
        end_period();
    }
}

}  // namespace fsh
