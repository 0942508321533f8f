// NUFFT readout runs in the reverse sweep, beside it (no counterpart in the reference, whose NUFFT readouts are forward
// only, src/blochparty/engines/gpu/driver.py:221-225).
//
// The forward takes a run's samples s_ic = sum over spins of K_ic S_c m0 (the spreading, the grid's DFT, the decay terms,
// the demodulation; m0 the spin's Mxy at the run's start). What the samples add to the adjoint at the run's start,
//     sum_c conj(S_c) A_c,  A_c = e^{2 pi i ph} Y_c,  Y_c = sum_m e^{-R2 tau_m} sum_u psi(z_u) G[m][u][c]
// (G from hb_nufft_adjoint_grid), depends on neither the adjoint nor the state, and the coil gradients conj(m0) A_c and
// the gradients along R2 (through -tau_m e^{-R2 tau_m}) and the phase per sample (through ph and psi'(z_u)) need only m0.
// So all of it is taken out of the sweep: one lane per spin walks the interval's runs, and leaves per run the two values
// that the sweep adds to lambda.
//
// A run is three matrix products per wave of 64 spins: with the weights w = psi e^{-R2 tau} on the workgroup's window of at
// most kColsB columns (cell x term) and their derivative along z, both the same for every run of a kind and so formed
// once and held as matrix-core operands (rows: spins), against the window's G (columns: Re, Im of the coils) and tau G:
// Y = w G, R = w (tau G), X = (dw/dz) G on v_mfma_f32_16x16x32_f16, three products of float16 hi and lo parts each, 36
// instructions; each lane gets its spin's values back through LDS (one wave's block, no barrier) and contracts them with
// its sensitivities. G is scaled by a power of two per column (a coil's Re or Im, by its largest value in the window), so
// that the pairs hold each coil's values to 2^-24, or to 2^-33 of that coil's largest, whatever the others' residuals: with
// one scale for all coils, a coil with a residual 2^-17 of the largest had gradients 2.6e-5 off and one with 2^-34 of it
// 80 %. (In float32 on v_mfma_f32_16x16x4_f32 the products take four times as long: the backward at 64^3 264.8 -> 273.5 ms.)
// That is about 350 VALU instructions a run; taken column by column in the sweep it was 2,300, at two waves per SIMD.
// Measured at 64^3 spins, 8 coils, 16 runs of 64 samples an interval: the sweep 1,086 -> 682 us, with 120 us here and 109 us
// for the replay on its own; the whole backward of 4,096 runs 341 -> 295 ms (now 549, 113 and 103 us; forward and backward
// 254 ms). Where it is not taken: engines/adjoint.py, runs_beside.
#include "nufft_back.h"

#include "bloch_device.h"
#include "contract_device.h"

namespace hb {

constexpr int kColsB = 32;        // K of one instruction
constexpr int kStrideB = 36;      // floats per spin in the LDS block: 16-byte rows, 36 = 4 mod 32 banks apart
constexpr float kLiftW = 1024.0f, kLiftD = 64.0f, kLiftG = 256.0f;  // off float16's subnormals (w <= 1, |dw/dz| < 200)

__device__ __forceinline__ void fence_wave() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// NC: coils (nc of hb_adjoint: 1, 2, 4, 8, 16); CT: tiles of 16 columns that hold their Re and Im.
template <int NC>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(NC <= 8 ? 2 : 1))) void nufft_back_kernel(
    NufftBack a, const float* __restrict__ spins, const float* __restrict__ pos_lo, const hb_segment* __restrict__ segs,
    const float* __restrict__ sens, const float* __restrict__ par, const int32_t* __restrict__ win,
    const float* __restrict__ G, const int32_t* __restrict__ heads, const float* __restrict__ m0) {
    constexpr int CT = NC > 8 ? 2 : 1;
    __shared__ __align__(16) float block[kWaves][64 * kStrideB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, jj = lane & 15;
    const int j = blockIdx.x * kBlock + tid, np = a.n_pad;
    float* mine = block[wave];
    const Spin p = load_spin(spins, pos_lo, np, j);
    const Pos64 r64 = pos64(p);
    const int ng = (int)par[0], terms = (int)par[2], shift = (int)par[4];
    const float hz = par[6 + HB_NUFFT_MAX_TERMS], bl2 = par[7 + HB_NUFFT_MAX_TERMS];
    const float beta = bl2 * 0.6931471805599453f;
    float tau_max = 0.0f;
    for (int m = 0; m < terms; ++m) tau_max = fmaxf(tau_max, par[6 + m]);
    const float tau_inv = tau_max > 0.0f ? 1.0f / tau_max : 0.0f;
    float sr[NC], si[NC];
    double gc[2 * NC], ga[5];  // coil gradients; R2, px, py, pz, db0
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        sr[c] = sens[(2 * c) * (size_t)np + j];
        si[c] = sens[(2 * c + 1) * (size_t)np + j];
        gc[2 * c] = gc[2 * c + 1] = 0.0;
    }
#pragma unroll
    for (int i = 0; i < 5; ++i) ga[i] = a.g[(size_t)i * np + j];
    if (a.coil_grads) {
#pragma unroll
        for (int c = 0; c < 2 * NC; ++c) gc[c] = a.g[(size_t)(5 + c) * np + j];
    }
    h8 wh[4], wl[4], dh[4], dl[4];  // weights and their z derivatives of spins 16 t + jj, columns 8 g .. 8 g + 7
#pragma unroll
    for (int t = 0; t < 4; ++t) wh[t] = wl[t] = dh[t] = dl[t] = (h8){};
    int at[8];       // G's offsets of this lane's columns 8 g .. 8 g + 7 within a run (< 0: past the window)
    float tau_w[8];  // their decay times over the largest
#pragma unroll
    for (int i = 0; i < 8; ++i) at[i] = -1, tau_w[i] = 0.0f;
    float cp = 1.0f, sp = 0.0f;
    int r = a.r1 - 1;
    while (r >= a.r0) {
        // the weights of the run's kind (uniform)
        const int kind = segs[heads[r]].pad[2];
        {
            const hb_segment& q = segs[heads[r]];
            const double cyc = free_cycles64(r64, p, q), fr = cyc - floor(cyc), xg = fr * ng;
            double ph = fr * shift;
            ph -= rint(ph);
            sincospi(2.0f * (float)ph, &sp, &cp);  // e^{+2 pi i ph}
            const int* w = win + ((size_t)kind * gridDim.x + blockIdx.x) * 2;
            const int wb = w[0], cols = min(w[1] * terms, kColsB);
            const float z0 = (float)(((double)wb - xg) * (double)hz);
#pragma unroll
            for (int pass = 0; pass < 2; ++pass) {
                int m = 0;
                float lcf = 0.0f;
#pragma unroll 1
                for (int c = 0; c < kColsB; ++c) {
                    const float z = fmaf(lcf, hz, z0), u = fmaf(-z, z, 1.0f);
                    const bool in = u > 0.0f && c < cols;
                    const float su = __builtin_amdgcn_sqrtf(in ? u : 1.0f);
                    const float kv = in ? __builtin_amdgcn_exp2f(fmaf(bl2, su, -bl2)) : 0.0f;
                    const float e = __builtin_amdgcn_exp2f(-(par[6 + m] * 1.4426950408889634f) * p.r2);
                    mine[lane * kStrideB + c] = pass ? -kv * beta * z / su * e * kLiftD : kv * e * kLiftW;
                    if (++m == terms) m = 0, lcf += 1.0f;
                }
                fence_wave();
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    const f4* src = reinterpret_cast<const f4*>(mine + (16 * t + jj) * kStrideB + 8 * g);
                    float x[8];
#pragma unroll
                    for (int v = 0; v < 2; ++v) {
                        const f4 y = src[v];
                        x[4 * v] = y[0], x[4 * v + 1] = y[1], x[4 * v + 2] = y[2], x[4 * v + 3] = y[3];
                    }
                    if (pass)
                        split8(x, dh[t], dl[t]);
                    else
                        split8(x, wh[t], wl[t]);
                }
                fence_wave();
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int c = 8 * g + i, m = c % terms;
                int cell = (wb + c / terms) % ng;
                if (cell < 0) cell += ng;
                at[i] = c < cols ? (m * ng + cell) * 2 * NC : -1;
                tau_w[i] = par[6 + m] * tau_inv;
            }
        }
        for (; r >= a.r0; --r) {
            const hb_segment& q = segs[heads[r]];
            if (q.pad[2] != kind) break;
            const float* Gr = G + (size_t)r * terms * ng * (2 * NC);
            // this lane's part of the window: columns 8 g .. 8 g + 7, values jj (and 16 + jj)
            float x[CT][8];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const int v = 16 * ct + jj;
                    x[ct][i] = at[i] >= 0 && v < 2 * NC ? Gr[at[i] + v] : 0.0f;
                }
            h8 bh[CT], bl[CT], th[CT], tl[CT];
            float unscale[CT];
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                // the power of two that brings the column's largest value to [1/2, 1) times the lift
                float big = 0.0f;
#pragma unroll
                for (int i = 0; i < 8; ++i) big = fmaxf(big, fabsf(x[ct][i]));
                big = fmaxf(big, __shfl_xor(big, 16, 64));
                big = fmaxf(big, __shfl_xor(big, 32, 64));
                const int ex = (__float_as_int(big) >> 23) & 255;  // 0: zero or subnormal, 255: not finite
                const int up = min(max(253 - ex, 1), 245);
                const float scale = __int_as_float(up << 23) * kLiftG;
                unscale[ct] = __int_as_float((254 - up) << 23) / kLiftG;
                float y[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) x[ct][i] *= scale, y[i] = x[ct][i] * tau_w[i];
                split8(x[ct], bh[ct], bl[ct]);
                split8(y, th[ct], tl[ct]);
            }
            const float mx = m0[(size_t)(2 * (r - a.r0)) * np + j], my = m0[(size_t)(2 * (r - a.r0) + 1) * np + j];
            const float fre = mx * cp + my * sp, fim = mx * sp - my * cp;  // conj(m0) e^{2 pi i ph}
            float S[3][2];                                                  // sums over the coils: Q, R, X (Re, Im)
#pragma unroll
            for (int set = 0; set < 3; ++set) {
                // D[spin 16 t + 4 g + r][value] of the set into the wave's block, then this lane's spin's values
                float s[CT];  // undoes the column's scale and the lifts
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
                    s[ct] = unscale[ct] * (set == 0 ? 1.0f / kLiftW : set == 1 ? -tau_max / kLiftW : 1.0f / kLiftD);
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int ct = 0; ct < CT; ++ct) {
                        const h8 ah = set == 2 ? dh[t] : wh[t], al = set == 2 ? dl[t] : wl[t];
                        const h8 vh = set == 1 ? th[ct] : bh[ct], vl = set == 1 ? tl[ct] : bl[ct];
                        f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, vh, acc, 0, 0, 0);
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, vl, acc, 0, 0, 0);
                        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah, vh, acc, 0, 0, 0);
#pragma unroll
                        for (int i = 0; i < 4; ++i) mine[(16 * t + 4 * g + i) * kStrideB + 16 * ct + jj] = acc[i] * s[ct];
                    }
                fence_wave();
                float yr_s = 0.0f, yi_s = 0.0f;
                constexpr int kQuads = (2 * NC + 3) / 4;
#pragma unroll
                for (int v = 0; v < kQuads; ++v) {
                    const f4 y = reinterpret_cast<const f4*>(mine + lane * kStrideB)[v];
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int c = 2 * v + e;
                        if (c < NC) {
                            const float yr = y[2 * e], yi = y[2 * e + 1];
                            yr_s += sr[c] * yr + si[c] * yi;  // conj(S_c) Y_c
                            yi_s += sr[c] * yi - si[c] * yr;
                            if (set == 0) {  // coil gradients conj(m0) A_c
                                gc[2 * c] += (double)(fre * yr - fim * yi);
                                gc[2 * c + 1] += (double)(fre * yi + fim * yr);
                            }
                        }
                    }
                }
                fence_wave();
                S[set][0] = yr_s, S[set][1] = yi_s;
            }
            const float Qr = S[0][0], Qi = S[0][1], Rr = S[1][0], Ri = S[1][1], Xr = S[2][0], Xi = S[2][1];
            a.q[(size_t)(2 * (r - a.r0)) * np + j] = cp * Qr - sp * Qi;
            a.q[(size_t)(2 * (r - a.r0) + 1) * np + j] = cp * Qi + sp * Qr;
            ga[0] += (double)(mx * (cp * Rr - sp * Ri) + my * (cp * Ri + sp * Rr));
            const float a2 = HB_TWO_PI * (float)shift, b2 = -(float)ng * hz;  // d/dfr: 2 pi i shift Q + (-ng hz) X
            const float Fr = -a2 * Qi + b2 * Xr, Fi = a2 * Qr + b2 * Xi;
            const float gb = (mx * (cp * Fr - sp * Fi) + my * (cp * Fi + sp * Fr)) * (float)q.dt64;  // dL/dbz
            ga[1] += (double)(gb * q.g_x);
            ga[2] += (double)(gb * q.g_y);
            ga[3] += (double)(gb * q.g_z);
            ga[4] += (double)gb;
        }
    }
#pragma unroll
    for (int i = 0; i < 5; ++i) a.g[(size_t)i * np + j] = ga[i];
    if (a.coil_grads) {
#pragma unroll
        for (int c = 0; c < 2 * NC; ++c) a.g[(size_t)(5 + c) * np + j] = gc[c];
    }
}

bool nufft_back_takes(int nc, int cols) {
    return (nc == 1 || nc == 2 || nc == 4 || nc == 8 || nc == 16) && cols >= 1 && cols <= kColsB;
}

template <int NC>
static void launch(const NufftBack& a, const hb_case& cs, const hb_adjoint& ad, const int32_t* heads, hipStream_t st) {
    hipLaunchKernelGGL((nufft_back_kernel<NC>), dim3(a.n_pad / kBlock), dim3(kBlock), 0, st, a, cs.spins, cs.pos_lo,
                       cs.segs, ad.sens, ad.nu_params, ad.nu_win, ad.nu_grid, heads, a.m0);
}

void launch_nufft_back(const NufftBack& a, const hb_case& cs, const hb_adjoint& ad, const int32_t* heads,
                       hipStream_t st) {
    switch (ad.nc) {
        case 1: launch<1>(a, cs, ad, heads, st); break;
        case 2: launch<2>(a, cs, ad, heads, st); break;
        case 4: launch<4>(a, cs, ad, heads, st); break;
        case 8: launch<8>(a, cs, ad, heads, st); break;
        default: launch<16>(a, cs, ad, heads, st); break;
    }
}

}  // namespace hb
