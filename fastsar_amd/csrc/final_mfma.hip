// The final stage of 16 x 16 and 32 x 32 tiles of images with few tiles, on the float32 matrix instructions: per tile
//   out[i, j] = sum_{p, q} A[i; p, q] B[p, q; j],   A = d[p, q] exp(-2 pi i ux_p dlx_i (a0 + a1 q)) (w0 + gx dlx_i),
//                                                 B =         exp(-2 pi i uy_p dly_j (a0 + a1 q)) (1 + gyr dly_j),
// then the quadratic phase of each pixel and the cropped write (fastsar/ffbp_cpu.cpp:302-469).
//
// A workgroup forms an FB x FB block of a tile (FB 16, or 32 where there are tiles enough), each wave taking PC = 256 /
// FB subapertures at a time and walking their samples q. A lane builds one run of 8 table entries (rows 8 c .. 8 c + 7
// of A or B) of one subaperture: the run's first entry and its ratio seeded in float64 at q = 0 and advanced over q by
// their own ratios, the entries by repeated products with the ratio (k_final_tiles_reg's tables, bit for bit). The
// entries go through the wave's own LDS into the operand layout of v_mfma_f32_16x16x4_f32 (lane l: row or column l % 16,
// contraction index l / 16, here the subaperture), four products a 16 x 16 block (Re Re, Im Im, Re Im, Im Re) into
// independent accumulators. Waves' sums meet in LDS at the end, in wave order; images do not depend on the launch's
// tile range.
//
// The float32 matrix instructions do the VALU's float32 rate (154 TFLOP/s) and take turns with its instructions. What
// they change is that a pixel block no longer lives in one lane's registers: 64 lanes share 256 or 1,024 pixels' tables
// and sums, so that an image of few tiles runs four or more waves a SIMD where one 8 x 8 block a lane ran a quarter to
// one wave (final stage of 64 tiles of 32 x 32 with 103 x 72 samples 351 -> 60 us, of 768 with 102 x 91 994 -> 560 us,
// of 576 of 16 x 16 with 113 x 64 and weights 512 -> 140 us). Bound by the two pipes' sum: 512 matrix cycles a step of
// PC samples (1,024 at FB 32) and about 240 for the tables and their passage.
#include "fsh_common.h"
#include "fsh_kernels.h"

#include <algorithm>

namespace fsh {

namespace {

typedef float floatx4_t __attribute__((ext_vector_type(4)));
constexpr int FW_MAX = 8;                  // waves a workgroup

// Samples of one chain of sums of a 16 x 16 block (16 subapertures each), the chains' sums added. One chain over all samples
// is four times as long as the register form's, which deals the subapertures to 16 lanes, and rounds by up to 0.1 dB above
// it (24 subapertures of 30 samples: -113.7 dB from float64 for -113.8; so -113.8). 2 % of the stage's time; 32 x 32 blocks,
// whose chains were the register form's eight lanes', keep one
constexpr int QC = 8;

template <int FB>
struct FinalShape {
    static constexpr int PC = 256 / FB;            // subapertures a wave takes at a time
    static constexpr int RS = PC + (FB == 16 ? 2 : 1);    // row stride of the tables (float2), spread over the banks
    static constexpr int ESZ = 2 * FB * RS;        // table entries (float2) a wave
};

}  // namespace

template <int T, int FB, bool W>
__global__ __launch_bounds__(64 * FW_MAX) void k_final_tiles_mfma(const float2* __restrict__ data, int Pf, int Qf,
                                                                  const double* __restrict__ ux, const double* __restrict__ uy,
                                                                  const double* __restrict__ tgeo, double spx, double spy,
                                                                  double a0, double a1, double fc2, const float* __restrict__ w0,
                                                                  const float* __restrict__ gx, const float* __restrict__ gyr,
                                                                  const int* __restrict__ tile_xy, int ox, int oy, int nx, int ny,
                                                                  float2* __restrict__ out)
{
    typedef FinalShape<FB> S;
    constexpr int PC = S::PC, RS = S::RS, NB = FB / 16, NS = T / FB;
    extern __shared__ float2 lds[];                          // tables [waves][2 FB][RS], then sums [waves][FB][FB]
    const int nw = blockDim.x >> 6;
    const int tid = threadIdx.x, wv = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    // blocks are dispatched round-robin over the 8 XCDs: renumbered so that the blocks of one tile share an XCD's L2
    int wg = blockIdx.x;
    {
        const int G = gridDim.x, q = G >> 3, rem = G & 7, xcd = wg & 7;
        wg = xcd * q + min(xcd, rem) + (wg >> 3);
    }
    const int b = wg / (NS * NS), blk = wg - b * (NS * NS), bx = blk / NS, by = blk - bx * NS;
    const double hc = 0.5 * (T - 1);
    // table role: subaperture pl of the wave's PC, run ch; runs 0 .. FB / 8 - 1 are A's rows, the rest B's columns
    const int pl = lane % PC, ch = lane / PC;
    const bool isA = ch < FB / 8;
    const int e0 = isA ? FB * bx + 8 * ch : FB * by + 8 * (ch - FB / 8);      // the run's first row or column of the tile
    const double sp = isA ? spx : spy, dl0 = (e0 - hc) * sp;
    float2* E = lds + wv * S::ESZ;
    float2* ew = E + 8 * ch * RS + pl;
    // product role: row or column i, contraction index k
    const int i = lane & 15, k = lane >> 4;
    const float2* ea = E + i * RS + k;
    const float2* eb = ea + FB * RS;
    floatx4_t rr[NB][NB], ii[NB][NB], ri[NB][NB], ir[NB][NB];
    #pragma unroll
    for (int m = 0; m < NB; ++m)
        #pragma unroll
        for (int n = 0; n < NB; ++n) rr[m][n] = ii[m][n] = ri[m][n] = ir[m][n] = floatx4_t{};

    floatx4_t tre = {}, tim = {};                            // FB 16: sums of chains of QC samples
    auto flush = [&]() {
        if (FB == 16) {
            tre += rr[0][0] - ii[0][0];
            tim += ri[0][0] + ir[0][0];
            rr[0][0] = ii[0][0] = ri[0][0] = ir[0][0] = floatx4_t{};
        }
    };
    for (int p0 = PC * wv; p0 < Pf; p0 += PC * nw) {
        const bool pok = p0 + pl < Pf;
        const size_t bp = (size_t)b * Pf + min(p0 + pl, Pf - 1);
        const float2* dq = data + bp * Qf;
        float2 dn = load_ahead(dq);                    // the next sample, read one ahead
        const double g = (isA ? ux : uy)[bp];
        float2 r, sr, ba, sb;
        cis_cyc(-(g * sp) * a0, r.x, r.y);             // ratio along the run at q = 0
        cis_cyc(-(g * sp) * a1, sr.x, sr.y);           // its step over q
        cis_cyc(-(g * dl0) * a0, ba.x, ba.y);          // the run's first entry, q = 0
        cis_cyc(-(g * dl0) * a1, sb.x, sb.y);
        float wt[8];
        if (W) {
            const float c0 = isA ? w0[bp] : 1.f, c1 = (isA ? gx : gyr)[bp];
            #pragma unroll
            for (int e = 0; e < 8; ++e) wt[e] = c0 + c1 * (float)(dl0 + e * sp);
        }
        const int steps = min(PC, Pf - p0 + 3) >> 2;   // contraction steps of four subapertures that hold one
        for (int qc = 0; qc < Qf; qc += FB == 16 ? QC : Qf) {
            for (int q = qc; q < (FB == 16 ? min(qc + QC, Qf) : Qf); ++q) {
                // B's lanes take 1 in the sample's place, subapertures past the last 0
                float2 v = cmul(isA ? (pok ? dn : make_float2(0.f, 0.f)) : make_float2(1.f, 0.f), ba);
                dn = load_ahead(dq + min(q + 1, Qf - 1));
                #pragma unroll
                for (int e = 0; e < 8; ++e) {
                    ew[e * RS] = W ? make_float2(v.x * wt[e], v.y * wt[e]) : v;
                    if (e < 7) v = cmul(v, r);
                }
                r = cmul(r, sr);
                ba = cmul(ba, sb);
                wave_lds_sync();
                #pragma unroll
                for (int s = 0; s < PC / 4; ++s) {
                    if (s < steps) {
                        float2 a[NB], c[NB];
                        #pragma unroll
                        for (int m = 0; m < NB; ++m) { a[m] = ea[16 * m * RS + 4 * s]; c[m] = eb[16 * m * RS + 4 * s]; }
                        #pragma unroll
                        for (int m = 0; m < NB; ++m)
                            #pragma unroll
                            for (int n = 0; n < NB; ++n) {
                                rr[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m].x, c[n].x, rr[m][n], 0, 0, 0);
                                ii[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m].y, c[n].y, ii[m][n], 0, 0, 0);
                                ri[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m].x, c[n].y, ri[m][n], 0, 0, 0);
                                ir[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m].y, c[n].x, ir[m][n], 0, 0, 0);
                            }
                    }
                }
                wave_lds_sync();
            }
            flush();
        }
    }
    if (FB == 16) {
        rr[0][0] = tre;
        ri[0][0] = tim;
    }
    __syncthreads();                                   // every wave is done with its tables
    // result element r of a lane: row 4 k + r, column i of its 16 x 16 block
    #pragma unroll
    for (int m = 0; m < NB; ++m)
        #pragma unroll
        for (int n = 0; n < NB; ++n)
            #pragma unroll
            for (int r = 0; r < 4; ++r)
                lds[(wv * FB + 16 * m + 4 * k + r) * FB + 16 * n + i] =
                    make_float2(rr[m][n][r] - ii[m][n][r], ri[m][n][r] + ir[m][n][r]);
    __syncthreads();
    const double cx = tgeo[3 * b], cy = tgeo[3 * b + 1], f = fc2 / (2.0 * tgeo[3 * b + 2]);
    const int X0 = tile_xy[2 * b] - ox, Y0 = tile_xy[2 * b + 1] - oy;
    for (int t = tid; t < FB * FB; t += blockDim.x) {
        float2 v = lds[t];
        for (int w = 1; w < nw; ++w) {
            const float2 u = lds[w * FB * FB + t];
            v.x += u.x;
            v.y += u.y;
        }
        const int pi = FB * bx + t / FB, pj = FB * by + t % FB, X = X0 + pi, Y = Y0 + pj;
        if (X < 0 || X >= nx || Y < 0 || Y >= ny) continue;
        const double dx = (pi - hc) * spx, dy = (pj - hc) * spy;
        const double los = cx * dx + cy * dy;
        float cs, sn;
        cis_cyc((dx * dx + dy * dy - los * los) * f, cs, sn);
        out[(size_t)X * ny + Y] = cmul(v, make_float2(cs, sn));
    }
}

int launch_final_tiles_mfma(const float2* data, int B, int Pf, int Qf, int T, const double* ux, const double* uy,
                            const double* tgeo, double spx, double spy, double a0, double a1, double fc2, const float* w0,
                            const float* gx, const float* gyr, const int* tile_xy, int ox, int oy, int nx, int ny, float2* out,
                            hipStream_t s, int split)
{
    // split 8: an image of 512 to 1,023 tiles of 32 x 32 (final_split), whose 32 x 32 blocks fill the device; 16: fewer
    const int FB = T == 32 && split < 16 ? 32 : 16, PC = FinalShape<16>::PC;
    // four waves, a SIMD each (5 or 7 leave the SIMDs uneven: the 768 tiles above took 712 and 642 us); eight of 16 x 16
    // blocks with the runs to share
    const int nw = FB == 16 && Pf > 4 * PC ? FW_MAX : 4;
    const long G = (long)B * (T / FB) * (T / FB);
    if (G > 2147483647L) { set_error("final_tiles: too many tiles"); return E_INVALID; }
    const dim3 grid((unsigned)G), block(64 * nw);
    const size_t lds = nw * sizeof(float2) * std::max<size_t>(FB == 32 ? FinalShape<32>::ESZ : FinalShape<16>::ESZ, FB * FB);
#define FSH_FM(TT, BB, WW) hipLaunchKernelGGL((k_final_tiles_mfma<TT, BB, WW>), grid, block, lds, s, data, Pf, Qf, ux, uy, tgeo, \
                                              spx, spy, a0, a1, fc2, w0, gx, gyr, tile_xy, ox, oy, nx, ny, out)
    if (T == 16) { if (w0) FSH_FM(16, 16, true); else FSH_FM(16, 16, false); }
    else if (FB == 16) { if (w0) FSH_FM(32, 16, true); else FSH_FM(32, 16, false); }
    else { if (w0) FSH_FM(32, 32, true); else FSH_FM(32, 32, false); }
#undef FSH_FM
    FSH_TRY(hipGetLastError());
    return OK;
}

// 32 x 32 tiles with each pixel's terms in the order of k_final_tiles_reg, bit for bit: a wave holds a tile's sums over the
// subapertures p = sp, sp + SP, ... and adds two samples' terms an instruction (contraction index: sample, then real and
// imaginary part; the instruction is an ascending chain of fused multiply-adds). The wave's lanes build eight samples'
// tables of one subaperture at a time, eight runs x eight samples, each lane from its own sample's ratio and first entry,
// advanced eight products a chunk; seeds for eight subapertures at once.
//
// One 8 x 8 block a lane took 337 instructions for 256 multiply-adds and, at 1.1 to 2 waves a SIMD, waited for half of
// them; here 1,024 pixels share tables of 64 entries a sample and the launch runs 4.5 waves a SIMD at 2,304 tiles with
// two waves each. Final stage of 1,536 x 1,536 pixels (116 x 78 samples a tile) 3.50 -> 1.88 ms, 2,048 x 2,048 (118 x 77)
// 5.69 -> 3.14, 3,000 x 2,500 8.9 -> 6.3, 8,192 x 8,192 59 -> 44 (101 TFLOP/s of the float32 rate's 154): faster at every
// size, so no 32 x 32 tile takes the register form. Bound by the matrix pipe (1,120 cycles a chunk) and the tables'
// VALU instructions (about 500) in turn (FSH_FINAL_KERNEL=reg takes the register form, for comparison). v_mfma_f32_32x32x2_f32, a sample an instruction: 1.95 ms, 44.5.
namespace {
struct OrderShape {
    static constexpr int RS = 65;                            // row stride of the tables (float2): writes free of conflicts
    static constexpr int TAB = 8 * RS;                       // [8 samples][32 rows of A, 32 columns of B]
    static constexpr int SEED = 4 * 64;                      // seeds of 8 subapertures x 8 runs
    static constexpr int ESZ = 1024;                         // float2 a wave: tables and seeds, then the sums
    static_assert(TAB + SEED <= ESZ, "a wave's tables and seeds fit its sums' room");
};
}  // namespace

template <bool W>
__global__ __launch_bounds__(256) void k_final_tiles_order(const float2* __restrict__ data, int B, int Pf, int Qf,
                                                            const double* __restrict__ ux, const double* __restrict__ uy,
                                                            const double* __restrict__ tgeo, double spx, double spy, double a0,
                                                            double a1, double fc2, const float* __restrict__ w0,
                                                            const float* __restrict__ gx, const float* __restrict__ gyr,
                                                            const int* __restrict__ tile_xy, int ox, int oy, int nx, int ny,
                                                            float2* __restrict__ out, int SP)
{
    typedef OrderShape S;
    constexpr int T = 32;
    __shared__ float2 lds[4 * S::ESZ];
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int sp = wv & (SP - 1);                            // SP 1, 2 or 4 waves a tile
    const long bt = (long)blockIdx.x * (4 / SP) + wv / SP;
    const bool live = bt < B;
    const int b = (int)(live ? bt : B - 1);
    const double hc = 0.5 * (T - 1);
    // table role: run of 8 entries (0 .. 3 A's rows, 4 .. 7 B's columns), sample qi of the chunk's 8
    const int run = lane >> 3, qi = lane & 7;
    const bool isA = run < 4;
    const double spc = isA ? spx : spy, dl0 = (8 * (run & 3) - hc) * spc;
    const double* gp = (isA ? ux : uy) + (size_t)b * Pf;
    float2* E = lds + wv * S::ESZ;
    float2* sd = E + S::TAB;
    float2* ew = E + qi * S::RS + 8 * run;
    // product role: row or column i; contraction index k: sample k / 2 of the two, component k % 2
    const int i = lane & 15, k = lane >> 4, comp = k & 1;
    const float* ea = (const float*)(E + (k >> 1) * S::RS + i) + comp;
    const float* er = (const float*)(E + (k >> 1) * S::RS + 32 + i) + comp;
    const float* ei = (const float*)(E + (k >> 1) * S::RS + 32 + i) + (comp ^ 1);
    const unsigned neg = comp ? 0x80000000u : 0u;            // re: Ax Bx - Ay By
    floatx4_t re[2][2], im[2][2];
    #pragma unroll
    for (int m = 0; m < 2; ++m)
        #pragma unroll
        for (int n = 0; n < 2; ++n) re[m][n] = im[m][n] = floatx4_t{};

    for (int pg = sp; pg < Pf; pg += 8 * SP) {
        {   // seeds of the group's eight subapertures, one a lane and run
            const double g = gp[min(pg + qi * SP, Pf - 1)];
            float2 v;
            wave_lds_sync();
            cis_cyc(-(g * spc) * a0, v.x, v.y);              // ratio along the run at q = 0
            sd[4 * lane] = v;
            cis_cyc(-(g * spc) * a1, v.x, v.y);              // its step over q
            sd[4 * lane + 1] = v;
            cis_cyc(-(g * dl0) * a0, v.x, v.y);              // the run's first entry, q = 0
            sd[4 * lane + 2] = v;
            cis_cyc(-(g * dl0) * a1, v.x, v.y);
            sd[4 * lane + 3] = v;
            wave_lds_sync();
        }
        for (int j = 0; j < 8 && pg + j * SP < Pf; ++j) {
            const size_t bp = (size_t)b * Pf + pg + j * SP;
            const float2* dq = data + bp * Qf;
            float2 dn = load_ahead(dq + min(qi, Qf - 1));    // the lane's sample, read one chunk ahead
            const float2* sj = sd + 4 * (8 * run + j);
            float2 r = sj[0], ba = sj[2];
            const float2 sr = sj[1], sb = sj[3];
            float wt[8];
            if (W) {
                const float c0 = isA ? w0[bp] : 1.f, c1 = (isA ? gx : gyr)[bp];
                #pragma unroll
                for (int e = 0; e < 8; ++e) wt[e] = c0 + c1 * (float)(dl0 + e * spc);
            }
            #pragma unroll
            for (int t = 0; t < 7; ++t) {                    // to the lane's sample, by the same products
                const float2 r1 = cmul(r, sr), b1 = cmul(ba, sb);
                r.x = t < qi ? r1.x : r.x;
                r.y = t < qi ? r1.y : r.y;
                ba.x = t < qi ? b1.x : ba.x;
                ba.y = t < qi ? b1.y : ba.y;
            }
            for (int q0 = 0; q0 < Qf; q0 += 8) {
                // B's lanes take 1 in the sample's place; A's entries past the last sample are 0
                const float2 z = q0 + qi < Qf ? dn : make_float2(0.f, 0.f);
                float2 v = cmul(isA ? z : make_float2(1.f, 0.f), ba);
                dn = load_ahead(dq + min(q0 + 8 + qi, Qf - 1));
                #pragma unroll
                for (int e = 0; e < 8; ++e) {
                    ew[e] = W ? make_float2(v.x * wt[e], v.y * wt[e]) : v;
                    if (e < 7) v = cmul(v, r);
                }
                if (q0 + 8 < Qf) {
                    #pragma unroll
                    for (int t = 0; t < 8; ++t) {
                        r = cmul(r, sr);
                        ba = cmul(ba, sb);
                    }
                }
                wave_lds_sync();
                #pragma unroll
                for (int s = 0; s < 4; ++s) {
                    if (q0 + 2 * s < Qf) {
                        float a[2], cr[2], ci[2];
                        #pragma unroll
                        for (int m = 0; m < 2; ++m) {
                            a[m] = ea[4 * s * S::RS + 32 * m];
                            cr[m] = __uint_as_float(__float_as_uint(er[4 * s * S::RS + 32 * m]) ^ neg);
                            ci[m] = ei[4 * s * S::RS + 32 * m];
                        }
                        #pragma unroll
                        for (int m = 0; m < 2; ++m)
                            #pragma unroll
                            for (int n = 0; n < 2; ++n) {
                                re[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m], cr[n], re[m][n], 0, 0, 0);
                                im[m][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[m], ci[n], im[m][n], 0, 0, 0);
                            }
                    }
                }
                wave_lds_sync();
            }
        }
    }
    // the waves of a tile add their sums in k_final_tiles_reg's order (neighbours first)
    for (int m = 1; m < SP; m <<= 1) {
        __syncthreads();
        float2* mine = lds + wv * S::ESZ + lane;
        if (sp & m) {
            #pragma unroll
            for (int u = 0; u < 16; ++u)
                mine[64 * u] = make_float2(re[u >> 3][u >> 2 & 1][u & 3], im[u >> 3][u >> 2 & 1][u & 3]);
        }
        __syncthreads();
        if (!(sp & m)) {
            const float2* o = mine + m * S::ESZ;
            #pragma unroll
            for (int u = 0; u < 16; ++u) {
                re[u >> 3][u >> 2 & 1][u & 3] += o[64 * u].x;
                im[u >> 3][u >> 2 & 1][u & 3] += o[64 * u].y;
            }
        }
    }
    if (sp || !live) return;
    const double cx = tgeo[3 * b], cy = tgeo[3 * b + 1], f = fc2 / (2.0 * tgeo[3 * b + 2]);
    const int X0 = tile_xy[2 * b] - ox, Y0 = tile_xy[2 * b + 1] - oy;
    #pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int pi = 16 * (u >> 3) + 4 * k + (u & 3), pj = 16 * (u >> 2 & 1) + i, X = X0 + pi, Y = Y0 + pj;
        if (X < 0 || X >= nx || Y < 0 || Y >= ny) continue;
        const double dx = (8 * (pi >> 3) - hc) * spx + (pi & 7) * spx, dy = (8 * (pj >> 3) - hc) * spy + (pj & 7) * spy;
        const double los = cx * dx + cy * dy;
        float cs, sn;
        cis_cyc((dx * dx + dy * dy - los * los) * f, cs, sn);
        out[(size_t)X * ny + Y] = cmul(make_float2(re[u >> 3][u >> 2 & 1][u & 3], im[u >> 3][u >> 2 & 1][u & 3]),
                                       make_float2(cs, sn));
    }
}

int launch_final_tiles_order(const float2* data, int B, int Pf, int Qf, const double* ux, const double* uy, const double* tgeo,
                             double spx, double spy, double a0, double a1, double fc2, const float* w0, const float* gx,
                             const float* gyr, const int* tile_xy, int ox, int oy, int nx, int ny, float2* out, hipStream_t s,
                             int split)
{
    if (split < 1 || split > 4) { set_error("final_tiles: one, two or four waves a tile"); return E_INVALID; }
    const long G = ((long)B * split + 3) / 4;
    if (w0)
        hipLaunchKernelGGL(k_final_tiles_order<true>, dim3((unsigned)G), dim3(256), 0, s, data, B, Pf, Qf, ux, uy, tgeo, spx, spy,
                           a0, a1, fc2, w0, gx, gyr, tile_xy, ox, oy, nx, ny, out, split);
    else
        hipLaunchKernelGGL(k_final_tiles_order<false>, dim3((unsigned)G), dim3(256), 0, s, data, B, Pf, Qf, ux, uy, tgeo, spx, spy,
                           a0, a1, fc2, w0, gx, gyr, tile_xy, ox, oy, nx, ny, out, split);
    FSH_TRY(hipGetLastError());
    return OK;
}

}  // namespace fsh
