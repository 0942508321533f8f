// Forward kernels: the event loop with the coil contraction on the matrix cores, and the deterministic cross-block
// signal sum. Replaces the reference's bloch_chunk_mma (src/blochparty/engines/gpu/cuda/kernels.cu.in:2-185) and
// its float atomicAdd flush (cuda/common.cuh:77-117).
//
// Launch: one lane per isochromat, workgroups of 256 lanes (4 waves of 64). Every lane walks the same segments
// [s0, s1), so segment records are uniform loads (scalar cache) and the control flow never diverges.
//
// Coil contraction: contract_device.h.
#include <mutex>

#include "bloch_device.h"
#include "contract_device.h"

namespace hb {

// A flush of nb staged columns of which the first `pending` are samples (rows [row, row + pending) of the partial
// rows, row advanced) and the rest grid columns (from grid_out).
template <int NT>
__device__ __forceinline__ void flush_cols(float* stg, float* wred, int& par, const Sens<NT>& S, int nt, int nb,
                                           int pending, int& row, int rows, float* __restrict__ partial,
                                           float* __restrict__ grid_out) {
    const int vals = 16 * nt;
    if (pending == 0) {
        flush_to(stg, wred, par, S, nt, nb, grid_out);
        return;
    }
    const int keep = row + pending <= rows ? pending : (rows > row ? rows - row : 0);  // never past the rows
    flush_to(stg, wred, par, S, nt, nb, partial + ((size_t)blockIdx.x * rows + row) * vals, keep, grid_out,
                 pending - keep);
    row += pending;
}

// One NUFFT readout run of L samples (record q, the run's first segment; pad[1] its slot in the dispatch, pad[2] its
// kind, pad[3] L). The spin's weight (mx + i my) e^{-2 pi i q (L // 2 + 1)} times the kernel psi at each cell of the
// workgroup's window and e^{-R2 tau_m} for each decay term is staged column by column (column = local cell * terms +
// term) and contracted with the coils like samples; the workgroup's window of columns goes to its slot of the grid
// partials. Then the run is one exact free step of L dt (phase L q, relaxation over L dt), and a spoil at its end.
// Samples still staged (nb of them, rows [row, row + nb)) share the first flush with the grid columns.
template <int NT, int NUT>
__device__ __forceinline__ void nufft_run(const hb_case& cs, const hb_nufft& nu, const hb_segment& q, const Spin& p,
                                          const Pos64& r64, const float (&em)[NUT], float& e1_run, State& m,
                                          float* stg, float* wred, int& par, const Sens<NT>& S, int nt, int lane,
                                          int& nb_io, int& row, int rows, float* __restrict__ partial) {
    const int L = q.pad[3], slot = q.pad[1], kind = q.pad[2];
    const int ng = (int)nu.params[0], terms = (int)nu.params[2], shift = (int)nu.params[4];
    const float h = nu.params[6 + HB_NUFFT_MAX_TERMS];       // 2 / width: z per grid cell
    const float bl2 = nu.params[7 + HB_NUFFT_MAX_TERMS];     // beta log2(e)
    const int vals = 16 * nt;
    const double cyc = free_cycles64(r64, p, q);
    const double fr = cyc - floor(cyc);
    const double xg = fr * ng;  // float64: at x ~ ng a float32 position is 1e-5 of a cycle off at the last sample
    double ph = fr * shift;
    ph -= rint(ph);
    float sp, cp;
    sincospi(-2.0f * (float)ph, &sp, &cp);
    const float cr = (m.mx * cp - m.my * sp) * S.x_scale, ci = (m.mx * sp + m.my * cp) * S.x_scale;
    // the weight (times the staged values' scale) times each decay term e^{-R2 tau_m}
    float wr[NUT], wi[NUT];
#pragma unroll
    for (int t = 0; t < NUT; ++t) wr[t] = em[t] * cr, wi[t] = em[t] * ci;
    const int* win = nu.win + ((size_t)kind * gridDim.x + blockIdx.x) * 2;
    const int wb = win[0], W = win[1];
    float* out = nu.part + ((size_t)slot * gridDim.x + blockIdx.x) * nu.cols * vals;
    int nb = nb_io, col = 0, pending = nb_io;  // the staged samples come first in the first flush
    nb_io = 0;
    // z = (cell - x) 2 / width: at the window's first cell from the float64 position (x ~ ng would leave a float32
    // z 1e-6 off), then by float32 steps (|z| error under 3e-7 over a 32-cell window)
    const float z0 = (float)(((double)wb - xg) * (double)h);
    float lcf = 0.0f;  // lc as a float
    for (int lc = 0; lc < W; ++lc, lcf += 1.0f) {
        const float z = fmaf(lcf, h, z0);
        const float u = fmaf(-z, z, 1.0f);
        // the ES kernel e^{beta (sqrt(1 - z^2) - 1)} = 2^{beta log2(e) (sqrt(u) - 1)}, zero outside |z| < 1, on the
        // hardware square root and exp2 (about 1 ulp each; the argument's rounding, |arg| < 20, leaves the
        // kernel value within 2e-6 relative)
        const float kv = u > 0.0f ? __builtin_amdgcn_exp2f(fmaf(bl2, __builtin_amdgcn_sqrtf(u), -bl2)) : 0.0f;
#pragma unroll
        for (int t = 0; t < NUT; ++t) {
            if (t < terms) {
                stg[nb * kStgStride + lane] = kv * wr[t];
                stg[(8 + nb) * kStgStride + lane] = kv * wi[t];
                if (++nb == 8) {
                    flush_cols<NT>(stg, wred, par, S, nt, 8, pending, row, rows, partial, out + (size_t)col * vals);
                    col += 8 - pending;
                    pending = 0;
                    nb = 0;
                }
            }
        }
    }
    if (nb > 0) {
        flush_cols<NT>(stg, wred, par, S, nt, nb, pending, row, rows, partial, out + (size_t)col * vals);
        pending = 0;
    }
    // the jump over the run: phase L cyc, relaxation over L dt (Mz only when the run's Mxy is never read)
    if (!(q.flags & HB_SAME_RUN)) e1_run = expm1x(-((float)L * q.dt) * p.r1);
    run_jump(q, p, cyc, e1_run, m);
}

// ---- NUFFT runs whose windows hold at most kCols columns (cells x terms): the spreading as one matrix product.
//
// A spin's weight on each column, psi(cell) e^{-R2 tau_m}, is real and the same for every run of a kind (one phase per
// sample), so it is formed once per kind and kept in registers as matrix-core operands (kCols x 64 spins per wave, as
// float16 hi and lo parts); so is the start's phase factor. Per run the lanes then only form S_c c (c = Mxy times that
// factor) for every coil: lane (g, jj) the value jj (Re S_0 c, Im S_0 c, ...) of spins 16 g .. 16 g + 15, from the
// sensitivities it and its neighbour lane keep for those spins and c broadcast through LDS, so that the products come
// out in the operand layout. D[value][column] = sum over spins (S_c c) w on v_mfma_f32_16x16x32_f16 (three products
// of hi and lo parts, as the samples'), 12 per coil tile; the waves' sums are added in LDS in a fixed order. Where a
// run's window was staged column by column (nufft_run: three flushes, each splitting 16 values per lane anew, and the
// window's kernel values and two sines of a float64 phase per run), a run costs about 95 VALU instructions instead of
// 430 (SQ counters of the whole
// kernel: 330 VALU instructions per wave and repetition of the 64^3 GRE, 512 staged). A single reused pulse's map is
// held too (12 registers, some of them spilled: still faster than reading it from the L2 at every occurrence, 83.2 ->
// 72.9 ms). 64^3 x 4 spins, 8 coils: 83.5 -> 70.9 ms a pass; 96^3, 16 coils: 219.3 -> 188 ms. Four waves per SIMD
// (128 registers) and three (168, no spills) measured the same at a million spins; four keep 262,144 spins in one
// round of workgroups. Only for dispatches without stepped RF: the RF loop is faster with five waves than this is with
// four. Reading the next record ahead costs 32 scalar moves a record and measured 8 % slower.
constexpr int kCols = 32;
// S_c c is an operand itself: with S lifted by kLift and c by this, a product of values at their bounds (|Re S|, |Im S|,
// |M| scaled to 1) is at most sqrt(2) 2^14 = 23,170 of float16's 65,504, and its pair holds it to 2^-39 of the bound
// (both lifted by kLift it would reach 92,681). The signal's error against 64 bits is 1.6e-6 with either lift, at 64^3 x 4
// spins and 8 coils and at 96^3 and 16.
constexpr float kProductLift = 64.0f;
constexpr float kWeightLift = 1024.0f;  // the weights (<= 1) in float16's range, as kLift
constexpr int kColTiles = kCols / 16;

// LDS of these kernels: the samples' staging block, then two buffers of the waves' sums (kCols columns each; also the
// weights' scratch while they are formed), then c of every wave (64 Re, 64 -Im, 64 Im).
__host__ __device__ constexpr int lds_floats_cols(int nt) {
    return kWaves * kStgFloats + 2 * kWaves * kCols * 16 * nt + kWaves * 192;
}

__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int NT>
struct Spread {
    float a[NT][16];                         // value jj of spins 16 g + u: Re S_0, Im S_0, Re S_1, ... scaled
    h8 wh[kColTiles][2], wl[kColTiles][2];   // the weights of column 16 tile + jj, spins 16 g + u (u < 8, u >= 8)
    float cp, sp;                            // cos, sin of the start's phase factor times the case's x_scale, lifted
    int kind, cols;                          // the kind they belong to (-1: none yet), its window's columns

    // sens_scale: Sens::scales' (lifted)
    __device__ __forceinline__ void load(const float* __restrict__ sa, float sens_scale) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int u = 0; u < 16; ++u) a[t][u] = sa[t * 1024 + u * 64] * sens_scale;
        kind = -1, cols = 0, cp = sp = 0.0f;
    }
};

// x of lane ^ 1 (DPP quad permutation; folded into the instruction that uses it).
__device__ __forceinline__ float dpp_xor1(float x) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0xB1, 0xf, 0xf, true));
}

// The staged samples' sums (flush_to's, from Spread's values: eight spins per lane are split at a time, anew per flush,
// which costs 32 instructions per eight samples and holds no operand in registers).
template <int NT>
__device__ __forceinline__ void flush_spread(const float* stg, float* wred2, int& par, const Spread<NT>& W,
                                             float out_scale, int nb, int row, int rows, float* __restrict__ partial) {
    constexpr int vals = 16 * NT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, jj = lane & 15;
    float* wred = wred2 + par * (kWaves * kCols * vals);
    par ^= 1;
    wave_fence();
    float* mine = wred + wave * kCols * vals;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        h8 ah[2], bh[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float x[8];
            h8 al, bl;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                x[e] = W.a[t][8 * i + e];
                asm volatile("" : "+v"(x[e]));  // keeps the compiler from hoisting the split out of the event loop
            }
            split8(x, ah[i], al);
            *reinterpret_cast<f4*>(x) = *reinterpret_cast<const f4*>(stg + jj * kStgStride + 16 * g + 8 * i);
            *reinterpret_cast<f4*>(x + 4) = *reinterpret_cast<const f4*>(stg + jj * kStgStride + 16 * g + 8 * i + 4);
            split8(x, bh[i], bl);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(al, bh[i], acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], bl, acc, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(ah[i], bh[i], acc, 0, 0, 0);
        store_pq(mine, vals, t, lane, acc);
    }
    __syncthreads();
    const int keep = row + nb <= rows ? nb : (rows > row ? rows - row : 0);  // never past the rows
    float* out = partial + ((size_t)blockIdx.x * rows + row) * vals;
    for (int v = tid; v < keep * vals; v += kBlock) {
        float s = wred[v];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) s += wred[w * kCols * vals + v];
        out[v] = s * out_scale;
    }
}

__device__ __forceinline__ void load16(float (&x)[16], const float* src) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const f4 y = reinterpret_cast<const f4*>(src)[v];
        x[4 * v] = y[0], x[4 * v + 1] = y[1], x[4 * v + 2] = y[2], x[4 * v + 3] = y[3];
    }
}

// The weights and phase factor of a run's kind. Every lane of the workgroup calls it (the kind is uniform).
template <int NT>
__device__ __forceinline__ void make_weights(Spread<NT>& W, const hb_nufft& nu, const hb_segment& q, const Spin& p,
                                             const Pos64& r64, float* wred, float x_scale, int lane, int wave) {
    const int kind = q.pad[2];
    const int ng = (int)nu.params[0], terms = (int)nu.params[2], shift = (int)nu.params[4];
    const float h = nu.params[6 + HB_NUFFT_MAX_TERMS];       // 2 / width: z per grid cell
    const float bl2 = nu.params[7 + HB_NUFFT_MAX_TERMS];     // beta log2(e)
    const double cyc = free_cycles64(r64, p, q);
    const double fr = cyc - floor(cyc);
    const double xg = fr * ng;  // float64: at x ~ ng a float32 position is 1e-5 of a cycle off at the last sample
    double ph = fr * shift;
    ph -= rint(ph);
    float sp, cp;
    sincospi(-2.0f * (float)ph, &sp, &cp);
    W.cp = cp * x_scale, W.sp = sp * x_scale;
    const int* win = nu.win + ((size_t)kind * gridDim.x + blockIdx.x) * 2;
    W.kind = kind;
    W.cols = min(win[1] * terms, kCols);
    // z = (cell - x) 2 / width: at the window's first cell from the float64 position (x ~ ng would leave a float32
    // z 1e-6 off), then by float32 steps (|z| error under 3e-7 over a 32-cell window)
    const float z0 = (float)(((double)win[0] - xg) * (double)h);
    float* scr = wred + wave * 1024;  // 16 columns x 64 spins
    const int g = lane >> 4, jj = lane & 15;
    __syncthreads();  // the sums' buffers are free
    int m = 0;
    float lcf = 0.0f;
#pragma unroll
    for (int t = 0; t < kColTiles; ++t) {
#pragma unroll 1
        for (int r = 0; r < 16; ++r) {
            const float z = fmaf(lcf, h, z0);
            const float u = fmaf(-z, z, 1.0f);
            // the ES kernel e^{beta (sqrt(1 - z^2) - 1)} = 2^{beta log2(e) (sqrt(u) - 1)}, zero outside |z| < 1, on the
            // hardware square root and exp2 (about 1 ulp each; the argument's rounding, |arg| < 20, leaves the
            // kernel value within 2e-6 relative)
            const float kv =
                u > 0.0f ? __builtin_amdgcn_exp2f(fmaf(bl2, __builtin_amdgcn_sqrtf(u), -bl2)) : 0.0f;
            const float em = __builtin_amdgcn_exp2f(-(nu.params[6 + m] * 1.4426950408889634f) * p.r2);
            scr[r * 64 + lane] = 16 * t + r < W.cols ? kv * em * kWeightLift : 0.0f;
            if (++m == terms) m = 0, lcf += 1.0f;
        }
        wave_fence();
        float x[16];
        load16(x, scr + jj * 64 + 16 * g);
        split8(x, W.wh[t][0], W.wl[t][0]);
        split8(x + 8, W.wh[t][1], W.wl[t][1]);
        wave_fence();
    }
    __syncthreads();
}

// One NUFFT readout run (record q: pad[1] its slot, pad[2] its kind, pad[3] its length): its window's columns into its
// slot of the grid partials, then the exact jump over it.
template <int NT>
__device__ __forceinline__ void spread_run(const Spread<NT>& W, const hb_nufft& nu, const hb_segment& q, const Spin& p,
                                           const Pos64& r64, float& e1_run, State& m, float* wred, float* cbuf, int& par,
                                           float out_scale, int tid) {
    constexpr int vals = 16 * NT;
    const int lane = tid & 63, wave = tid >> 6, g = lane >> 4, jj = lane & 15;
    const float ci_ = m.mx * W.sp + m.my * W.cp;
    cbuf[lane] = m.mx * W.cp - m.my * W.sp;
    cbuf[64 + lane] = -ci_;
    cbuf[128 + lane] = ci_;
    wave_fence();
    float* buf = wred + par * (kWaves * kCols * vals);
    par ^= 1;
    float* mine = buf + wave * (kCols * vals);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        f4 acc[kColTiles];
        h8 vh[2];
#pragma unroll
        for (int k = 0; k < kColTiles; ++k) acc[k] = (f4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < 2; ++i) {  // eight spins per lane at a time, the small products first
            h8 vl;
            float x[8];
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const f4 cr = *reinterpret_cast<const f4*>(cbuf + 16 * g + 8 * i + 4 * v);
                // values Re S c = Sr cr - Si ci (even jj), Im S c = Si cr + Sr ci (odd): the partner lane's S
                const f4 ci = *reinterpret_cast<const f4*>(cbuf + 64 + 64 * (jj & 1) + 16 * g + 8 * i + 4 * v);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int u = 8 * i + 4 * v + e;
                    x[4 * v + e] = fmaf(dpp_xor1(W.a[t][u]), ci[e], W.a[t][u] * cr[e]);
                }
            }
            split8(x, vh[i], vl);
#pragma unroll
            for (int k = 0; k < kColTiles; ++k) {
                if (16 * k < W.cols) {  // uniform
                    acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vl, W.wh[k][i], acc[k], 0, 0, 0);
                    acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh[i], W.wl[k][i], acc[k], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int k = 0; k < kColTiles; ++k) {
            if (16 * k < W.cols) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vh[i], W.wh[k][i], acc[k], 0, 0, 0);
                // values 4 g .. 4 g + 3 of column 16 k + jj
                *reinterpret_cast<f4*>(mine + (16 * k + jj) * vals + 16 * t + 4 * g) = acc[k];
            }
        }
    }
    __syncthreads();
    if (4 * tid < W.cols * vals) {
        f4 s = reinterpret_cast<const f4*>(buf)[tid];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) s += reinterpret_cast<const f4*>(buf + w * (kCols * vals))[tid];
        float* out = nu.part + ((size_t)q.pad[1] * gridDim.x + blockIdx.x) * nu.cols * vals;
        reinterpret_cast<f4*>(out)[tid] = s * (out_scale * (kLift / kProductLift / kWeightLift));
    }
    if (!(q.flags & HB_SAME_RUN)) e1_run = expm1x(-((float)q.pad[3] * q.dt) * p.r1);
    double cyc = 0.0;
    if (!(q.flags & (HB_XY_DEAD | HB_PULSE_SPOIL))) cyc = free_cycles64(r64, p, q);
    run_jump(q, p, cyc, e1_run, m);
}

// NT: coil tiles (0: any, the sensitivities read from memory per flush); NUT: NUFFT runs: 0 none, 1 by spread_run
// (hb_forward_product), 4 and 8 by nufft_run with up to NUT decay terms (their weights in registers); RF: RF segments are
// stepped (false when every pulse of the dispatch is applied as a map: the RF step is then left out, and its registers).
// The read-only inputs and the NUFFT partials come in again as noalias parameters (the same pointers as in cs_in and
// nu_in): no store of the kernel can change the records, so they load through the scalar cache instead of one vector
// load per wave and a readfirstlane per value.
template <int NT, int NUT, bool RF>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(NT == 2 ? 3 : NUT == 1 ? 4 : 5))) void forward_kernel(
    hb_case cs_in, int s0, int s1, float* __restrict__ partial, int rows, hb_nufft nu_in,
    const hb_segment* __restrict__ segs, const float* __restrict__ spins, const float* __restrict__ pos_lo,
    const float* __restrict__ sens_a, const float* __restrict__ maps, const float* __restrict__ nu_params,
    const int32_t* __restrict__ nu_win, float* __restrict__ nu_part) {
    hb_case cs = cs_in;
    cs.segs = segs, cs.spins = spins, cs.pos_lo = pos_lo, cs.sens_a = sens_a, cs.maps = maps;
    hb_nufft nu = nu_in;
    nu.params = nu_params, nu.win = nu_win, nu.part = nu_part;
    extern __shared__ float lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j = blockIdx.x * kBlock + tid;
    const int np = cs.n_pad;
    const int nt = NT > 0 ? NT : cs.n_tiles;
    float* stg = lds + wave * kStgFloats;
    float* wred = lds + kWaves * kStgFloats;
    const Spin p = load_spin(cs.spins, cs.pos_lo, np, j);
    const Pos64 r64 = pos64(p);
    const float b1sq = p.b1 * p.b1;
    State m = load_state(cs.state, np, j);
    // The dispatch's records into the L2s, 256 a workgroup: each XCD's first workgroups (workgroups go round robin over
    // the 8 XCDs) touch them all, so that no wave waits for memory at a record's first use. A dispatch of 17,000 records
    // takes 2 MB of an XCD's 4 MB; 32^3 x 4 spins, every RF substep: 78.4 -> 61.3 ms; 96^3, maps and NUFFT runs, 16 coils:
    // 196.5 -> 189.1 ms.
    {
        const int first = blockIdx.x >> 3, stride = max(1, min((int)gridDim.x >> 3, 64));
        if (first < stride) {
            float touched = 0.0f;
            for (int r = s0 + first * kBlock + tid; r < s1; r += stride * kBlock) touched += segs[r].dt;
            asm volatile("" ::"v"(touched));
        }
    }
    Sens<NT> S;
    S.sa = cs.sens_a + (size_t)(blockIdx.x * kWaves + wave) * nt * 1024 + lane;
    S.st = 1024, S.su = 64;
    int nb = 0, row = 0, par = 0;
    constexpr bool MAT = NUT == 1;
    constexpr int NS = NT > 0 ? NT : 1;
    Spread<NS> W;
    float* cbuf = wred + 2 * kWaves * kCols * 16 * NS + wave * 192;
    if constexpr (MAT) {
        float scale = cs.sens_scale;
        S.scales(cs.x_scale, scale);
        W.load(S.sa, scale);
    } else {
        S.load(cs.x_scale, cs.sens_scale, lane);
    }
    // the staged samples (all of them, or at the end the nb left) into the partial rows
    auto flush_samples = [&](int count, int at) {
        if constexpr (MAT) {
            flush_spread<NS>(stg, wred, par, W, S.out_scale, count, at, rows, partial);
        } else {
            flush(stg, wred, par, S, nt, count, at, rows, partial);
        }
    };
    // records of an RF train in flight: where the NUFFT runs' or many coils' scalars are live, three spill scalar registers
    // in the walk itself (200 repetitions of two RF substeps and a NUFFT run, 340,736 spins, 8 coils: 2.59 ms with three,
    // 2.25 with two)
    constexpr int kAhead = NUT == 0 && NT > 0 ? kTrain : 2;
    Cache k = {1.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    float e1_run = 0.0f;  // expm1(-L dt R1) of the last readout run (per sample or NUFFT)
    // the NUFFT decay terms e^{-R2 tau_m}: the spin's, the same for every run
    float em[NUT > 1 ? NUT : 1];
    if constexpr (NUT > 1) {
        const int terms = (int)nu.params[2];
#pragma unroll
        for (int t = 0; t < NUT; ++t)
            em[t] = t < terms ? __builtin_amdgcn_exp2f(-(nu.params[6 + t] * 1.4426950408889634f) * p.r2) : 0.0f;
    }
    // a single reused pulse's map in registers (more pulses: read per occurrence)
    constexpr bool MAP = MAT;
    const bool one_map = MAP && cs.n_pulses == 1;  // uniform
    float U[MAP ? 12 : 1];
    if constexpr (MAP) {
        if (one_map) {
#pragma unroll
            for (int i = 0; i < 12; ++i) U[i] = cs.maps[(size_t)i * np + j];
        }
    }
    // a dispatch that starts inside a reused pulse's occurrence or a NUFFT run (checkpoint intervals do not avoid
    // them): the record was applied at its first segment, in the dispatch before
    int s_start = s0;
    if (cs.segs[s0].flags & HB_PULSE_BODY) {
        const int head = cs.segs[s0].pad[3];
        const hb_segment& hq = cs.segs[head];
        s_start = head + ((hq.flags & HB_PULSE) ? hq.pad[2] : hq.pad[3]);
    }
    // (With spread_run the loop runs from one change of the runs' kind to the next: the weights, formed between, do not
    // change inside it and stay in their registers.)
    for (int s = s_start; s < s1;) {
        if constexpr (MAT) {
            const hb_segment q = cs.segs[s];
            if ((q.flags & HB_NUFFT) && q.pad[2] != W.kind)
                make_weights<NS>(W, nu, q, p, r64, wred, S.x_scale * (kProductLift / kLift), lane, wave);
        }
        for (; s < s1; ++s) {
            const hb_segment q = cs.segs[s];
            const int f = q.flags;
            if constexpr (NUT > 0) {
                if (f & HB_NUFFT) {  // a readout run as a type-1 NUFFT: spread onto the grid window, jump the run
                    if constexpr (MAT) {
                        if (q.pad[2] != W.kind) break;
                        spread_run<NS>(W, nu, q, p, r64, e1_run, m, wred, cbuf, par, S.out_scale, tid);
                    } else {
                        nufft_run<NT, NUT>(cs, nu, q, p, r64, em, e1_run, m, stg, wred, par, S, nt, lane, nb, row, rows,
                                           partial);
                    }
                    s += q.pad[3] - 1;
                    continue;
                }
            }
            if (RF && (f & HB_TRAIN)) {  // RF substeps of a shaped pulse, in a loop of their own (only RF state live)
                const int L = q.pad[3];
                const hb_segment* first = cs.segs + s;
                if (!(f & HB_SAME_RF_DT)) half_relax(q.dt, p, k);
                rf_records<kAhead>(
                    L, [&](int i) { return first + i; },
                    [&](int i, const RfRec& r) {
                        if (i > 0 && !(r.flags & HB_SAME_RF_DT)) half_relax(first[i].dt, p, k);
                        rf_step(r, p, b1sq, m, k);
                    });
                s += L - 1;
                continue;
            }
            if (f & HB_RUN) {  // L identical free ADC segments: Mxy stepped and sampled per segment, Mz relaxed once
                const int L = q.pad[3];
                if (!(f & HB_SAME_FREE)) {
                    sincospi(-2.0f * free_cycles(r64, p, q), &k.s, &k.c);
                    if (!(f & HB_SAME_FREE_DT)) {
                        k.e1 = expm1x(-q.dt * p.r1);
                        k.e2 = expm1x(-q.dt * p.r2);
                    }
                }
                if (!(f & HB_SAME_RUN)) e1_run = expm1x(-(float)L * q.dt * p.r1);
                for (int i = 0; i < L; ++i) {
                    precess(k.c, k.s, k.e2, m);
                    stg[nb * kStgStride + lane] = m.mx * S.x_scale;
                    stg[(8 + nb) * kStgStride + lane] = m.my * S.x_scale;
                    if (++nb == 8) {
                        flush_samples(8, row);
                        row += 8;
                        nb = 0;
                    }
                }
                two_sum(m.mz, m.lz, (m.mz - p.pd) * e1_run);
                s += L - 1;
                continue;
            }
            if (f & HB_PULSE) {  // a reused pulse: m += Rz(psi) (D Rz(-psi) m + v), then skip its segments
                // cos, sin of the occurrence's RF phase (host float64)
                if (MAP && one_map)
                    apply_map(U, 1, q.w_rf_x, q.w_rf_y, m);
                else
                    apply_map(cs.maps + (size_t)q.pad[1] * 12 * np + j, np, q.w_rf_x, q.w_rf_y, m);
                if (f & HB_PULSE_SPOIL) m.mx = m.my = 0.0f;
                s += q.pad[2] - 1;
                continue;
            }
            if (f & HB_SPOILED_FREE) {  // only Mz survives the spoil: relax it, zero Mxy
                two_sum(m.mz, m.lz, (m.mz - p.pd) * expm1x(-q.dt * p.r1));
                m.mx = m.my = 0.0f;
                if (f & HB_MERGED) s += q.pad[3] - 1;
                continue;
            }
            if constexpr (RF)
                step(q, f, p, r64, b1sq, m, k);
            else
                free_step(q, f, p, r64, m, k);
            if (f & HB_MERGED) s += q.pad[3] - 1;
            if (f & HB_ADC) {
                stg[nb * kStgStride + lane] = m.mx * S.x_scale;
                stg[(8 + nb) * kStgStride + lane] = m.my * S.x_scale;
                if (++nb == 8) {
                    flush_samples(8, row);
                    row += 8;
                    nb = 0;
                }
            }
            if (f & HB_SPOIL) m.mx = m.my = 0.0f;
        }
    }
    if (nb > 0) flush_samples(nb, row);
    store_state(cs.state, np, j, m);
}

// The cross-block sum in two passes, both in a fixed order (deterministic): the blocks in chunks of kRedChunk,
// summed in float64 in block order by one lane per partial value (consecutive lanes read consecutive floats); then
// the chunks in order, demodulated: sig[row0 + r][c] = exp(-i psi) sum_chunks sum_b partial[b][r][c].
constexpr int kRedChunk = 256;

__global__ __launch_bounds__(256) void reduce_chunks_kernel(const float* __restrict__ partial, int n_blocks,
                                                            int per_block, double* __restrict__ work) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= per_block) return;
    const int b0 = blockIdx.y * kRedChunk, b1 = min(n_blocks, b0 + kRedChunk);
    const float* src = partial + i;
    double acc = 0.0;
#pragma unroll 16
    for (int b = b0; b < b1; ++b) acc += (double)src[(size_t)b * per_block];
    work[(size_t)blockIdx.y * per_block + i] = acc;
}

__global__ __launch_bounds__(256) void reduce_final_kernel(const double* __restrict__ work, int chunks, int rows,
                                                           int vals, int n_coils, const double* __restrict__ psi,
                                                           int row0, const int* __restrict__ row_map,
                                                           double* __restrict__ sig) {
    const int idx = blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= rows * n_coils) return;
    const int r = idx / n_coils, c = idx - r * n_coils;
    const size_t stride = (size_t)rows * vals;
    const double* src = work + (size_t)r * vals + 2 * c;
    double re = 0.0, im = 0.0;
    for (int k = 0; k < chunks; ++k) {
        re += src[k * stride];
        im += src[k * stride + 1];
    }
    const int dst = row_map ? row_map[row0 + r] : row0 + r;
    double sp, cp;
    sincos(psi[dst], &sp, &cp);
    double* out = sig + ((size_t)dst * n_coils + c) * 2;
    out[0] = re * cp + im * sp;
    out[1] = im * cp - re * sp;
}

}  // namespace hb

namespace hb {
template <int NUT, bool RF>
static void launch_nt(const hb_case& cs, int s0, int s1, float* partial, int rows, const hb_nufft& nu, dim3 grid,
                      dim3 block, size_t lds, hipStream_t st) {
    auto kernel = cs.n_tiles == 1 ? forward_kernel<1, NUT, RF> : forward_kernel<2, NUT, RF>;
    if constexpr (NUT != 1) {
        if (cs.n_tiles > 2) kernel = forward_kernel<0, NUT, RF>;
    }
    hipLaunchKernelGGL(kernel, grid, block, lds, st, cs, s0, s1, partial, rows, nu, cs.segs, cs.spins, cs.pos_lo,
                       cs.sens_a, cs.maps, nu.params, nu.win, nu.part);
}

template <int NUT>
static void launch_forward(const hb_case& cs, int s0, int s1, float* partial, int rows, const hb_nufft& nu,
                           dim3 grid, dim3 block, size_t lds, hipStream_t st) {
    if (NUT == 1 || cs.rf_free)
        launch_nt<NUT, false>(cs, s0, s1, partial, rows, nu, grid, block, lds, st);
    else
        launch_nt<NUT == 1 ? 0 : NUT, true>(cs, s0, s1, partial, rows, nu, grid, block, lds, st);
}
}  // namespace hb

// spread_run against nufft_run. A run gains with its columns, and two tiles' products lose where the windows are narrow; a
// change of kind costs the weights formed anew. 1,024 runs of 64 samples, 262,144 spins, product against columns staged, one
// kind: 8 coils 3.81 against 3.91 ms with 5 columns, 3.81 / 4.21 with 7, 4.17 / 5.72 with 21, 4.19 / 6.50 with 28; 16 coils
// 5.74 / 4.02 with 5, 5.91 / 5.56 with 14, 6.74 / 6.86 with 21, 7.04 / 8.15 with 28. Two kinds in turn (bipolar readouts), 21
// columns: 10.29 / 5.75 and 14.38 / 6.89. So a column is worth a change in 64 runs, from 4 columns (one tile) or 20 (two).
extern "C" int32_t hb_forward_product(int32_t cols, int32_t n_tiles, int32_t kind_changes) {
    using namespace hb;
    return cols <= kCols && n_tiles <= 2 && kind_changes <= 16 * (cols - (n_tiles == 1 ? 4 : 20));
}

extern "C" int hb_forward(const hb_case* cs, int32_t s0, int32_t s1, float* partial, int32_t rows,
                          const hb_nufft* nu, void* stream) {
    using namespace hb;
    if (!cs || cs->n_pad <= 0 || cs->n_pad % kBlock || cs->n < 0 || cs->n > cs->n_pad) return hipErrorInvalidValue;
    if (cs->n_tiles < 1 || cs->n_tiles > kMaxTiles || 8 * cs->n_tiles < cs->n_coils) return hipErrorInvalidValue;
    if (s0 < 0 || s1 < s0 || s1 > cs->n_segments || rows < 0) return hipErrorInvalidValue;
    if (cs->n_pulses < 0 || (cs->n_pulses > 0 && !cs->maps)) return hipErrorInvalidValue;
    if (nu && (!nu->params || !nu->win || !nu->part || nu->runs_max < 1 || nu->cols < 1 || nu->terms < 1 ||
               nu->terms > HB_NUFFT_MAX_TERMS))
        return hipErrorInvalidValue;
    if (s1 == s0) return hipSuccess;
    const dim3 grid(cs->n_pad / kBlock), block(kBlock);
    const size_t lds = sizeof(float) * lds_floats(cs->n_tiles);
    hipStream_t st = (hipStream_t)stream;
    const hb_nufft none = {nullptr, nullptr, nullptr, 0, 0, 0, 0};
    const hb_nufft arg = nu ? *nu : none;
    if (!nu)
        launch_forward<0>(*cs, s0, s1, partial, rows, arg, grid, block, lds, st);
    else if (cs->rf_free && hb_forward_product(nu->cols, cs->n_tiles, nu->kind_changes))
        launch_forward<1>(*cs, s0, s1, partial, rows, arg, grid, block, sizeof(float) * lds_floats_cols(cs->n_tiles),
                          st);
    else if (nu->terms <= 4)
        launch_forward<4>(*cs, s0, s1, partial, rows, arg, grid, block, lds, st);
    else
        launch_forward<8>(*cs, s0, s1, partial, rows, arg, grid, block, lds, st);
    return hipGetLastError();
}

extern "C" int64_t hb_signal_reduce_workspace(int32_t n_blocks, int32_t rows, int32_t n_tiles) {
    if (n_blocks < 1 || rows < 0 || n_tiles < 1) return 0;
    return (int64_t)((n_blocks + hb::kRedChunk - 1) / hb::kRedChunk) * rows * 16 * n_tiles;
}

extern "C" int hb_signal_reduce(const float* partial, int32_t n_blocks, int32_t rows, int32_t n_tiles,
                                int32_t n_coils, const double* psi, int32_t row0, const int32_t* row_map,
                                double* work, double* sig, void* stream) {
    using namespace hb;
    if (rows < 0 || n_blocks < 1 || n_tiles < 1 || n_tiles > kMaxTiles || n_coils < 1 || 8 * n_tiles < n_coils ||
        row0 < 0 || !work)
        return hipErrorInvalidValue;
    if (rows == 0) return hipSuccess;
    const int vals = 16 * n_tiles, per_block = rows * vals, chunks = (n_blocks + kRedChunk - 1) / kRedChunk;
    hipLaunchKernelGGL(reduce_chunks_kernel, dim3((per_block + 255) / 256, chunks), dim3(256), 0,
                       (hipStream_t)stream, partial, n_blocks, per_block, work);
    const int total = rows * n_coils;
    hipLaunchKernelGGL(reduce_final_kernel, dim3((total + 255) / 256), dim3(256), 0, (hipStream_t)stream, work, chunks,
                       rows, vals, n_coils, psi, row0, row_map, sig);
    return hipGetLastError();
}

// ---- hb_signal_reduce_noalloc: hb_signal_reduce with its float64 chunk sums in a fixed device array.
//
// `scratch` is a file-scope device array that each GPU the library runs on holds until the process ends. Host code
// never passes its name to a kernel (in host code the name is a host-side stand-in, not a device address): the
// first call on a device resolves the array's address on that device with hipGetSymbolAddress, and every launch
// uses that address. Calls on one GPU share its array; the chunk sums are written in full before they are read,
// so nothing needs clearing, but calls that overlap on one GPU (other streams, other threads) race.
static __device__ __align__(256) double scratch[HB_NOALLOC_SCRATCH_DOUBLES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex scratch_mutex;
double* scratch_ptr[kMaxDevices] = {};

// The current device's address of `scratch` (resolved once per device), or nullptr with *err set.
double* device_scratch(hipError_t* err) {
    int dev = 0;
    *err = hipGetDevice(&dev);
    if (*err != hipSuccess) return nullptr;
    if (dev < 0 || dev >= kMaxDevices) {
        *err = hipErrorInvalidDevice;
        return nullptr;
    }
    std::lock_guard<std::mutex> lock(scratch_mutex);
    if (!scratch_ptr[dev]) {
        void* p = nullptr;
        *err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (*err != hipSuccess) return nullptr;
        scratch_ptr[dev] = static_cast<double*>(p);
    }
    return scratch_ptr[dev];
}
}  // namespace

extern "C" int hb_signal_reduce_noalloc(const float* partial, int32_t n_blocks, int32_t rows, int32_t n_tiles,
                                        int32_t n_coils, const double* psi, int32_t row0, const int32_t* row_map,
                                        double* sig, void* stream) {
    using namespace hb;
    if (rows < 0 || n_blocks < 1 || n_tiles < 1 || n_tiles > kMaxTiles || n_coils < 1 || 8 * n_tiles < n_coils ||
        row0 < 0)
        return hipErrorInvalidValue;
    if (hb_signal_reduce_workspace(n_blocks, rows, n_tiles) > HB_NOALLOC_SCRATCH_DOUBLES)
        return hipErrorInvalidValue;  // beyond the fixed array: use hb_signal_reduce with a workspace
    hipError_t err = hipSuccess;
    double* work = device_scratch(&err);
    if (!work) return err;
    return hb_signal_reduce(partial, n_blocks, rows, n_tiles, n_coils, psi, row0, row_map, work, sig, stream);
}

extern "C" const char* hb_error_string(int code) { return hipGetErrorString((hipError_t)code); }

extern "C" int hb_abi_version(void) { return 26; }
