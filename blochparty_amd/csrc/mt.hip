// The full-variant forward kernel: a rate bound pool (magnetization transfer) and / or a scanner's concomitant fields.
// Replaces the reference's V = 1 variant of bloch_chunk_mma (src/blochparty/engines/gpu/shaders/common.metal:113-208:
// lineshape, the exchange step, step_mt; :563-601 the field model; engines/core.py:115-121, 190-217).
//
// One lane per isochromat, workgroups of 256 (4 waves of 64), every lane walking the same plain segment records. Per
// spin the free pool's (Mx, My, Mz) and, with a bound pool, its Mzb; Mz and Mzb carry low parts. Without a bound pool
// the longitudinal step is plain T1 recovery.
// - Concomitant field f_c [Hz] of a segment with gradient g: leading order c . (gx^2, gy^2, gz^2, gx gy, gx gz,
//   gy gz), or exact |B| - f0 - lin = t^2 / (sqrt(u^2 + t^2) + u) (t^2 = (ax . g)^2 + (ay . g)^2, u = f0 + lin, lin the
//   rest of the offset); it adds to an RF segment's offset (and so to the bound pool's saturation offset) and, times
//   the segment's length, to a free segment's float64 phase.
// - RF segment: Strang split. Half a segment of transverse decay and of longitudinal exchange, with the bound pool
//   saturated at W = (2 pi b1 |rf|)^2 G(f_rf - bz - dw); the water's rotation (only the precession about z for RF
//   that only the bound pool feels); the other half.
// - Free segment: exact precession (float64 phase, as the plain kernels') and transverse decay; the unsaturated
//   exchange over the segment.
// - The exchange over t is exact, in increment form from the rates of change d = A z + c (A the 2 x 2 generator of
//   (Mz, Mzb), c its source): (exp(A t) - I)(z - z_ss) = t phi1(A t) d, phi1(x) = (e^x - 1) / x, as alpha d +
//   beta (A - m I) d with m the mean eigenvalue. d is formed from differences (PD - Mz, Mzb - f Mz, f PD - Mzb) that
//   vanish at equilibrium, so that its rounding vanishes there too, and no steady state (two divisions) is needed.
//   Short steps (an RF substep: eigenvalues times t under 0.03) take alpha and beta from their series: no square root,
//   exponential or division; longer ones from the eigenvalues' expm1.
// - ADC: eight samples at a time are staged in LDS and contracted with the coils on the matrix cores in float32
//   (contract_device.h), one barrier per eight; the workgroup's sums go to the partial rows that hb_signal_reduce sums
//   in a fixed order: no atomics. (float16 pairs took 0.2 ms less, but lost a coil 2^-17 of another, or spins
//   beside one 2^24 as bright that no coil sees, most of their bits.)
//
// What bounds it: with 65,536 spins every SIMD has one wave, so nothing hides a wave's latency, and a segment costs its
// chain of dependent instructions. What only depends on a segment's offset (its concomitant field, the saturation's
// lineshape with its table lookup, the rotation's z component) is kept while HB_SAME_RF_OFFSET says that the next RF
// segment's is the same, a free segment's phase factors while HB_SAME_FREE does, factors of the length while it stays;
// an RF train is stepped in a loop of its own that reads four values per substep, a readout run in one that reads none
// and relaxes the longitudinal components once. The next record is loaded while the current one is stepped, and the
// lanes touch the records 64 ahead, so that they are in the L2 when their turn comes. 65,536 spins with a bound pool and
// leading-order fields, 8 coils, 32,256 segments (12,800 RF, 16,384 samples): 9.9 ms, against 34.8 ms with a barrier and
// a shuffle tree per sample, steady states by division and every factor formed per segment. Of its 5.75 million issue
// slots a wave uses 2.3 for VALU and 1.0 for scalar instructions and waits in 1.8 (SQ counters).
#include "bloch_device.h"
#include "contract_device.h"

#include "../../include/blochparty_amd_mt.h"

namespace hb {
namespace {

// A spin's bound pool: f, the exchange rates k and k f, R1b, T2b, dw, and f PD.
struct Pool {
    float f, k, kf, r1b, t2b, dw, fpd;
};

// The exchange step over t of the generator A = [[-(R1 + k f), k], [k f, -(R1b + k + W)]]: the increment of (Mz, Mzb)
// is alpha d + beta (h d1 + k d2, k f d1 - h d2) with d the rates of change, A - m I = [[h, k], [k f, -h]].
struct XStep {
    float alpha, beta, h;
};

__device__ __forceinline__ XStep xstep(float t, float r1, const Pool& b, float w) {
    const float a11 = -(r1 + b.kf), a22 = -(b.r1b + b.k + w);
    const float m = 0.5f * (a11 + a22), h = 0.5f * (a11 - a22);
    const float Q = fmaf(h, h, b.k * b.kf);
    XStep x;
    x.h = h;
    const float mt = m * t;
    if (mt > -0.015f) {  // both eigenvalues are in [2 m, 0]: |lambda t| < 0.03
        // phi1(z) = 1 + z/2 + z^2/6 + z^3/24 + z^4/120 at z = m t +- sqrt(Q) t: the mean and the divided difference
        // (the next terms are under 1e-8 of the first)
        const float y = Q * t * t, m2 = mt * mt;
        x.alpha = t * (1.0f + 0.5f * mt + (m2 + y) * (1.0f / 6.0f) + mt * fmaf(3.0f, y, m2) * (1.0f / 24.0f));
        x.beta = t * t * (0.5f + mt * (1.0f / 3.0f) + fmaf(3.0f, m2, y) * (1.0f / 24.0f) +
                          mt * (m2 + y) * (1.0f / 30.0f));
        return x;
    }
    const float q = sqrtf(Q);
    const float lm = m - q;                                          // no cancellation: m < 0
    const float det = r1 * (b.r1b + b.k + w) + b.kf * (b.r1b + w);   // lp lm, without cancellation
    const float lp = det / lm;
    const float fp = lp != 0.0f ? expm1x(lp * t) / lp : t, fm = expm1x(lm * t) / lm;
    x.alpha = 0.5f * (fp + fm);
    if (q * t > 1e-3f) {
        x.beta = 0.5f * (fp - fm) / q;
    } else {  // a (nearly) double eigenvalue: t^2 phi1'(m t), by its series for small m t
        const float small =
            0.5f + mt * (1.0f / 3.0f + mt * (0.125f + mt * (1.0f / 30.0f + mt * (1.0f / 144.0f + mt * (1.0f / 840.0f)))));
        x.beta = t * t * (mt > -0.25f ? small : (__expf(mt) * (mt - 1.0f) + 1.0f) / (mt * mt));
    }
    return x;
}

// The increments of (Mz, Mzb) over the step x from (z, b) with the rates of change (d1, d2).
__device__ __forceinline__ void increments(const XStep& x, const Pool& p, float d1, float d2, float& dz, float& db) {
    dz = x.alpha * d1 + x.beta * fmaf(x.h, d1, p.k * d2);
    db = x.alpha * d2 + x.beta * fmaf(p.kf, d1, -(x.h * d2));
}

// An RF half step from (z, b), the bound pool saturated at w (the low parts, under half an ulp, change nothing over a
// substep).
__device__ __forceinline__ void exchange_rf(const XStep& x, const Pool& p, float pd, float r1, float w, float z,
                                            float b, float& dz, float& db) {
    const float ex = p.k * fmaf(-p.f, z, b);
    increments(x, p, fmaf(r1, pd - z, ex), fmaf(p.r1b, p.fpd - b, -fmaf(w, b, ex)), dz, db);
}

// A free step of the state (unsaturated), from the whole values with their low parts.
__device__ __forceinline__ void exchange_free(const XStep& x, const Pool& p, float pd, float r1, State& m, float& mb,
                                              float& lb) {
    const float ex = p.k * (fmaf(-p.f, m.mz, mb) + fmaf(-p.f, m.lz, lb));
    float dz, db;
    increments(x, p, fmaf(r1, (pd - m.mz) - m.lz, ex), fmaf(p.r1b, (p.fpd - mb) - lb, -ex), dz, db);
    two_sum(m.mz, m.lz, dz);
    two_sum(mb, lb, db);
}

// G(2 pi delta) [s]: the Lorentzian, or T2b F(x) from the table of ln F (held at the cut, 0 past the table's end).
__device__ __forceinline__ float lineshape_g(const hb_mt& mt, float delta, float t2b) {
    if (mt.lineshape == HB_LINE_LORENTZIAN) {
        const float x = HB_TWO_PI * delta * t2b;
        return t2b / fmaf(x, x, 1.0f);
    }
    const float x = HB_TWO_PI * fmaxf(fabsf(delta), mt.cutoff) * t2b;
    const float pos = (logf(x) - mt.lx0) / mt.dlx;
    if (!(pos <= (float)(mt.n_table - 1))) return 0.0f;
    const float pc = fmaxf(pos, 0.0f);
    const int i = min((int)pc, mt.n_table - 2);
    const float a = pc - (float)i;
    return t2b * expf(mt.table[i] * (1.0f - a) + mt.table[i + 1] * a);
}

// The spin's concomitant field in segment q, lin the rest of its offset there [Hz]; cc the spin's coefficients.
__device__ __forceinline__ float conc_field(int mode, const float (&cc)[7], const hb_segment& q, float lin) {
    const float gx = q.g_x, gy = q.g_y, gz = q.g_z;
    if (mode == HB_CONC_LEADING)
        return cc[0] * gx * gx + cc[1] * gy * gy + cc[2] * gz * gz + cc[3] * gx * gy + cc[4] * gx * gz +
               cc[5] * gy * gz;
    const float tx = cc[0] * gx + cc[1] * gy + cc[2] * gz, ty = cc[3] * gx + cc[4] * gy + cc[5] * gz;
    const float t2 = tx * tx + ty * ty, u = cc[6] + lin;
    const float den = sqrtf(u * u + t2) + u;  // > 0 for any real field (u = f0 + lin > 0)
    return den > 0.0f ? t2 / den : 0.0f;
}

__device__ __forceinline__ int bits_differ(float a, float b) { return __float_as_int(a) ^ __float_as_int(b); }

// NT: coil tiles as forward_kernel's (1, 2: the sensitivities in registers; 0: any, read per flush). segs, sens_r,
// rf_freq and table are the pointers of cs_in and mt_in again, as noalias parameters: no store of the kernel can change
// what they point to, so the records load through the scalar cache.
template <int NT>
__global__ __launch_bounds__(kBlock) void forward_mt_kernel(hb_case cs, hb_mt mt_in, int s0, int s1,
                                                            float* __restrict__ partial, int rows, int row0,
                                                            const hb_segment* __restrict__ segs,
                                                            const float* __restrict__ sens_r,
                                                            const float* __restrict__ rf_freq,
                                                            const float* __restrict__ table) {
    hb_mt mt = mt_in;
    mt.table = table;
    extern __shared__ float lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j = blockIdx.x * kBlock + tid;
    const int np = cs.n_pad;
    const int nt = NT > 0 ? NT : cs.n_tiles;
    float* stg = lds + wave * kStgFloats;
    float* wred = lds + kWaves * kStgFloats;
    float warm = segs[min(s0 + lane, s1 - 1)].dt;
    const Spin p = load_spin(cs.spins, cs.pos_lo, np, j);
    const Pos64 r64 = pos64(p);
    const float b1sq = p.b1 * p.b1;
    const bool pool = mt.pool != nullptr;  // uniform
    Pool b;
    b.f = pool ? mt.pool[j] : 0.0f, b.k = pool ? mt.pool[np + j] : 0.0f;
    b.r1b = pool ? mt.pool[2 * np + j] : 1.0f, b.t2b = pool ? mt.pool[3 * np + j] : 1.0f;
    b.dw = pool ? mt.pool[4 * np + j] : 0.0f;
    b.kf = b.k * b.f, b.fpd = b.f * p.pd;
    State m = load_state(cs.state, np, j);
    float mb = pool ? mt.mb[j] : 0.0f, lb = pool ? mt.mb[np + j] : 0.0f;
    const int cmode = mt.conc_mode;
    float cc[7] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    if (cmode != HB_CONC_NONE) {
#pragma unroll
        for (int i = 0; i < 7; ++i) cc[i] = mt.conc[(size_t)i * np + j];
    }
    Sens<NT, true> S;
    S.sa0 = sens_r + blockIdx.x * kBlock + wave * 64 + 16 * (lane >> 4);
    S.sa = S.sa0 + (size_t)(lane & 15) * np;
    S.st = 16 * (size_t)np, S.su = 1, S.n_rows = 2 * cs.n_coils;
    S.load_f32(lane);
    int nb = 0, row = 0, par = 0;   // staged samples, the first one's partial row, the flush's buffer
    XStep xf = {0.0f, 0.0f, 0.0f};  // free segments: the unsaturated exchange over dt (with a bound pool)
    XStep xl = {0.0f, 0.0f, 0.0f};  // and over the last readout run
    float e1f = 0.0f, e2f = 0.0f;   // free segments: expm1 of -dt R1 (without a bound pool), -dt R2
    float e1l = 0.0f;               // the last readout run's expm1 of -L dt R1 (without a bound pool)
    float cs_ = 1.0f, sn = 0.0f;    // free segments: cos, sin of the precession
    float e1r = 0.0f, e2r = 0.0f;   // RF segments: expm1 of -dt/2 R1 (without a bound pool), -dt/2 R2
    float wG = 0.0f, wz = 0.0f;     // RF segments: W over |w_rf|^2, the rotation vector's z
    float run_dt = -1.0f;
    int run_len = 0;
    bool free_ok = false, rf_ok = false;

    // what an RF segment's offset, length and RF frequency give: decays, the saturation's lineshape, w_z
    auto rf_offset = [&](const hb_segment& q, float frf) {
        e2r = expm1x(-0.5f * q.dt * p.r2);
        if (!pool) e1r = expm1x(-0.5f * q.dt * p.r1);
        float bz = offset(p, q);
        const float fc = cmode != HB_CONC_NONE ? conc_field(cmode, cc, q, bz) : 0.0f;
        bz += fc;
        if (pool) {  // W = (2 pi b1 |rf|)^2 G, |w_rf| = 2 pi dt |rf|
            const float t = q.dt > 0.0f ? p.b1 / q.dt : 0.0f;
            wG = t * t * lineshape_g(mt, frf - bz - b.dw, b.t2b);
        }
        wz = p.px * q.w_g_x + p.py * q.w_g_y + p.pz * q.w_g_z + (p.db0 * q.w + q.w_b0) + q.w * fc;
        rf_ok = true;
    };
    // the Strang step with the transverse rotation vector factors (wrx, wry), wr2 = |w_rf|^2; water: the water feels it
    auto rf_segment = [&](float t, float wrx, float wry, float wr2, bool water) {
        XStep x = {0.0f, 0.0f, 0.0f};
        float w = 0.0f, dz1, db1 = 0.0f;
        if (pool) {
            w = wr2 * wG;
            x = xstep(t, p.r1, b, w);
            exchange_rf(x, b, p.pd, p.r1, w, m.mz, mb, dz1, db1);
        } else {
            dz1 = (m.mz - p.pd) * e1r;
        }
        const float dx1 = m.mx * e2r, dy1 = m.my * e2r;
        const float x1 = m.mx + dx1, y1 = m.my + dy1, z1 = m.mz + dz1, b1 = mb + db1;
        const float wx = water ? p.b1 * wrx : 0.0f, wy = water ? p.b1 * wry : 0.0f;
        float ra, rb;
        rot_ab((water ? b1sq * wr2 : 0.0f) + wz * wz, ra, rb);
        const float cx = wy * z1 - wz * y1, cy = wz * x1 - wx * z1, cz = wx * y1 - wy * x1;
        const float ex = wy * cz - wz * cy, ey = wz * cx - wx * cz, ez = wx * cy - wy * cx;
        const float drx = ra * cx + rb * ex, dry = ra * cy + rb * ey, drz = ra * cz + rb * ez;
        m.mx += dx1 + drx + (x1 + drx) * e2r;
        m.my += dy1 + dry + (y1 + dry) * e2r;
        const float z2 = z1 + drz;
        if (pool) {
            float dz2, db2;
            exchange_rf(x, b, p.pd, p.r1, w, z2, b1, dz2, db2);
            two_sum(m.mz, m.lz, dz1 + drz + dz2);
            two_sum(mb, lb, db1 + db2);
        } else {
            two_sum(m.mz, m.lz, dz1 + drz + (z2 - p.pd) * e1r);
        }
    };
    // the free segment's factors (hints in f, honoured once factors are held)
    auto free_factors = [&](const hb_segment& q, int f) {
        if (!free_ok) f &= ~(HB_SAME_FREE | HB_SAME_FREE_DT);
        if (!(f & HB_SAME_FREE)) {
            double cyc = free_cycles64(r64, p, q);
            if (cmode != HB_CONC_NONE) cyc += (double)(conc_field(cmode, cc, q, offset(p, q)) * q.dt);
            cyc -= rint(cyc);
            sincospi(-2.0f * (float)cyc, &sn, &cs_);
            if (!(f & HB_SAME_FREE_DT)) {
                e2f = expm1x(-q.dt * p.r2);
                if (pool)
                    xf = xstep(q.dt, p.r1, b, 0.0f);
                else
                    e1f = expm1x(-q.dt * p.r1);
            }
            free_ok = true;
        }
    };
    auto precess = [&]() {
        const float nx = cs_ * m.mx - sn * m.my, ny = sn * m.mx + cs_ * m.my;
        m.mx = nx + nx * e2f;
        m.my = ny + ny * e2f;
    };
    auto stage = [&](int r) {  // uniform: every lane takes it
        if (r < 0 || r >= rows) return;
        if (nb == 0) row = r;
        stg[nb * kStgStride + lane] = m.mx;
        stg[(8 + nb) * kStgStride + lane] = m.my;
        if (++nb == 8) {
            flush(stg, wred, par, S, nt, 8, row, rows, partial);
            nb = 0;
        }
    };

    int warm_at = s0;
    hb_segment nq = segs[s0];
    for (int s = s0; s < s1;) {
        const hb_segment q = nq;
        const int fl = q.flags;
        int len = 1;
        if (fl & (HB_RUN | HB_TRAIN)) len = max(1, min(q.pad[3], s1 - s));
        nq = segs[min(s + len, s1 - 1)];  // in flight while this record is stepped
        if (s >= warm_at) {  // the records up to 128 ahead into the L2 (the value itself is not used)
            asm volatile("" ::"v"(warm));
            warm = segs[min(s + 64 + lane, s1 - 1)].dt;
            warm_at = s + 64;
        }
        if (fl & HB_RF) {
            if (!(fl & HB_SAME_RF_OFFSET) || !rf_ok) rf_offset(q, pool ? rf_freq[s] : 0.0f);
            float wrx = q.w_rf_x, wry = q.w_rf_y, wr2 = q.w_rf2;
            const float t = 0.5f * q.dt;
            if (!(fl & HB_TRAIN)) {
                rf_segment(t, wrx, wry, wr2, !(fl & HB_BOUND_ONLY));
            } else {
                // a train: the next segment's flags and rotation factors are in flight while one is stepped
                int f = fl;
                float tt = t;
                for (int i = 1; i <= len; ++i) {
                    const hb_segment* nx = segs + s + (i < len ? i : 0);
                    const int nf = nx->flags;
                    const float nwx = nx->w_rf_x, nwy = nx->w_rf_y, nw2 = nx->w_rf2;
                    rf_segment(tt, wrx, wry, wr2, !(f & HB_BOUND_ONLY));
                    if (i < len && !(nf & HB_SAME_RF_OFFSET)) {
                        const hb_segment qi = *nx;
                        rf_offset(qi, pool ? rf_freq[s + i] : 0.0f);
                        tt = 0.5f * qi.dt;
                    }
                    f = nf, wrx = nwx, wry = nwy, wr2 = nw2;
                }
            }
        } else {
            free_factors(q, fl);
            if (fl & HB_RUN) {  // len identical samples: Mxy stepped per sample, the longitudinal step once
                const float T = (float)len * q.dt;
                if (bits_differ(q.dt, run_dt) | (len ^ run_len)) {
                    if (pool)
                        xl = xstep(T, p.r1, b, 0.0f);
                    else
                        e1l = expm1x(-T * p.r1);
                    run_dt = q.dt, run_len = len;
                }
                const int r0 = q.pad[0] - row0;
                for (int i = 0; i < len; ++i) {
                    precess();
                    stage(r0 + i);
                }
                if (pool)
                    exchange_free(xl, b, p.pd, p.r1, m, mb, lb);
                else
                    two_sum(m.mz, m.lz, (m.mz - p.pd) * e1l);
                s += len;
                continue;
            }
            precess();
            if (pool)
                exchange_free(xf, b, p.pd, p.r1, m, mb, lb);
            else
                two_sum(m.mz, m.lz, (m.mz - p.pd) * e1f);
        }
        if (fl & HB_ADC) stage(q.pad[0] - row0);
        if (fl & HB_SPOIL) m.mx = m.my = 0.0f;
        s += len;
    }
    if (nb > 0) flush(stg, wred, par, S, nt, nb, row, rows, partial);
    store_state(cs.state, np, j, m);
    if (pool) mt.mb[j] = mb, mt.mb[np + j] = lb;
}

}  // namespace
}  // namespace hb

extern "C" int hb_forward_mt(const hb_case* cs, const hb_mt* mt, int32_t s0, int32_t s1, float* partial,
                             int32_t rows, int32_t row0, void* stream) {
    using namespace hb;
    if (!cs || !mt || !mt->sens) return hipErrorInvalidValue;
    if (mt->pool && (!mt->mb || !mt->rf_freq)) return hipErrorInvalidValue;
    if (mt->conc_mode < HB_CONC_NONE || mt->conc_mode > HB_CONC_EXACT || (mt->conc_mode && !mt->conc))
        return hipErrorInvalidValue;
    if (cs->n_pad <= 0 || cs->n_pad % kBlock || cs->n < 0 || cs->n > cs->n_pad) return hipErrorInvalidValue;
    if (cs->n_coils < 1 || cs->n_coils > 8 * kMaxTiles || cs->n_tiles < 1 || 8 * cs->n_tiles < cs->n_coils)
        return hipErrorInvalidValue;
    if (s0 < 0 || s1 < s0 || s1 > cs->n_segments || rows < 0 || row0 < 0) return hipErrorInvalidValue;
    if (mt->pool && mt->lineshape == HB_LINE_SUPERLORENTZIAN && (!mt->table || mt->n_table < 2 || !(mt->dlx > 0.0f)))
        return hipErrorInvalidValue;
    if (mt->pool && mt->lineshape != HB_LINE_SUPERLORENTZIAN && mt->lineshape != HB_LINE_LORENTZIAN)
        return hipErrorInvalidValue;
    if (s1 == s0) return hipSuccess;
    if (cs->n_tiles > kMaxTiles) return hipErrorInvalidValue;
    const dim3 grid(cs->n_pad / kBlock), block(kBlock);
    const size_t lds = sizeof(float) * lds_floats(cs->n_tiles);
    auto kernel = cs->n_tiles == 1   ? forward_mt_kernel<1>
                  : cs->n_tiles == 2 ? forward_mt_kernel<2>
                                     : forward_mt_kernel<0>;
    hipLaunchKernelGGL(kernel, grid, block, lds, (hipStream_t)stream, *cs, *mt, s0, s1, partial, rows, row0, cs->segs,
                       mt->sens, mt->rf_freq, mt->table);
    return hipGetLastError();
}
