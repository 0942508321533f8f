// The full variant's adjoint: the reverse sweep of one checkpoint interval with a rate bound pool, a scanner's
// concomitant fields and / or bound-only RF. Replaces the reference's V = 1 replay and adjoint kernels
// (src/blochparty/engines/gpu/shaders/adjoint_common.metal:66-203, driven per interval by engines/gpu/adjoint.py:
// 179-220).
//
// One lane per isochromat, float64 throughout (the physics and its reverse mode in full_device.h), in up to three
// launches per interval [s0, s1):
//   1. sweep_kernel: the interval replayed from its checkpoint, the state before every segment into traj (float32, 16 B
//      per spin and segment); in other workgroups of the same launch, where the reverse is split into chunks of
//      segments, the adjoint alone taken back over the interval (the transpose of every step needs no state), its
//      value at the end of every chunk kept in float64.
//   2. reverse_kernel, a workgroup per 256 spins and chunk: last segment first, zero the transverse adjoint at a spoil,
//      add an ADC sample's source sum_c h_c conj(S_c) and its coil gradients h_c conj(Mxy), then reverse the step from
//      its state before (recomputed intermediates), its spin gradients summed in float64 registers. Per-segment
//      gradients (dt, rf, g, b0_offset, the RF frequency) are summed over each wave by a float64 reduce-scatter and over
//      the workgroup's 4 waves in LDS in a fixed order, one partial per workgroup and segment, for hb_seg_reduce.
//   3. with chunks, chunk_sums_kernel adds their spin and coil gradients in a fixed order, last chunk first.
// What bounds it: the chain of float64 instructions of one lane. 16,384 spins are 256 waves on 1,024 SIMDs, so a reverse
// that walks the interval segment by segment leaves three quarters of the chip idle; chunks fill it, and the serial
// part shrinks to the replay and the bare adjoint, side by side: 16,384 spins, 12,032 segments, 8 coils in 94 intervals
// take 26 ms here, 54 ms in one walk per interval (with the exchange's exponentials and the lineshape at every segment).
// chunk_for: chunks until every CU has a workgroup, at least kMinChunk segments each. From there on splitting only adds
// the bare adjoint: 65,536 spins (256 workgroups) take 127 ms in one chunk and 170 ms in four.
// Factors that depend only on a segment's length (decays, the unsaturated exchange) are kept while consecutive segments
// of the kind have the same dt, the saturation's lineshape while consecutive RF segments have the same offset.
// Coil gradients sit in LDS (each lane its own slots).
#include <algorithm>

#include "bloch_device.h"
#include "full_device.h"

#include "../../include/blochparty_amd_mt.h"

namespace hb {
namespace {

constexpr int kBlockF = 256;
constexpr int kWavesF = kBlockF / 64;
constexpr int kMaxCoilsF = 16;
constexpr int kMinChunk = 8;      // segments per chunk at least
constexpr int kFillBlocks = 256;   // workgroups that fill the chip (one per CU: a wave takes the registers of a SIMD)
static_assert(full::N_G == HB_FULL_GRADS, "per-spin gradient rows");

// The wave's sums of the N_S = 8 per-segment gradients in a fixed order: over lane bits 5, 4, 3 each step keeps half
// the values (a lane with the bit set the upper half) and adds the partner's copy of them, then lane bits 2, 1, 0 by a
// butterfly; gradient i ends on lanes 8 i .. 8 i + 7 (10 shuffles instead of 48).
__device__ __forceinline__ double seg_scatter_sums(double (&v)[full::N_S], int lane) {
    static_assert(full::N_S == 8, "three halving steps");
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const bool up = lane & 32;
        const double send = up ? v[k] : v[k + 4], keep = up ? v[k + 4] : v[k];
        v[k] = keep + __shfl_xor(send, 32, 64);
    }
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const bool up = lane & 16;
        const double send = up ? v[k] : v[k + 2], keep = up ? v[k + 2] : v[k];
        v[k] = keep + __shfl_xor(send, 16, 64);
    }
    {
        const bool up = lane & 8;
        const double send = up ? v[0] : v[1], keep = up ? v[1] : v[0];
        v[0] = keep + __shfl_xor(send, 8, 64);
    }
    double r = v[0];
#pragma unroll
    for (int off = 4; off > 0; off >>= 1) r += __shfl_xor(r, off, 64);
    return r;
}

// A walk over the records, forwards or backwards: each record as full_device.h's segment, with what it shares with the
// last of its kind in the walk (lengths and whole free segments by the table's hints, to 1e-12; the offset and RF
// frequency by their bits). Uniform over the launch.
struct Walk {
    int free_bit, rf_bit;  // the walk's direction: HB_SAME_FREE, HB_SAME_RF_DT or HB_NEXT_FREE, HB_NEXT_RF_DT
    int gx = 0, gy = 0, gz = 0, b0 = 0, f = 0;
    bool free_ok = false, rf_ok = false;

    __device__ __forceinline__ explicit Walk(bool forward)
        : free_bit(forward ? HB_SAME_FREE : HB_NEXT_FREE), rf_bit(forward ? HB_SAME_RF_DT : HB_NEXT_RF_DT) {}

    __device__ __forceinline__ full::Seg next(const hb_segment& r, float frf) {
        full::Seg q;
        q.dt = r.dt64;
        q.rfx = r.rf_x, q.rfy = r.rf_y;
        q.gx = r.g_x, q.gy = r.g_y, q.gz = r.g_z, q.b0 = r.b0;
        q.frf = frf;
        q.mx = r.m_x, q.my = r.m_y, q.mz = r.m_z, q.b0a = r.b0_area;
        q.flags = r.flags;
        q.same_off = q.same_dt = q.same_free = false;
        if (r.flags & HB_RF) {
            const int x = __float_as_int(r.g_x), y = __float_as_int(r.g_y), z = __float_as_int(r.g_z);
            const int b = __float_as_int(r.b0), w = __float_as_int(frf);
            q.same_off = rf_ok && ((gx ^ x) | (gy ^ y) | (gz ^ z) | (b0 ^ b) | (f ^ w)) == 0;
            q.same_dt = rf_ok && (r.flags & rf_bit);
            gx = x, gy = y, gz = z, b0 = b, f = w, rf_ok = true;
        } else {
            q.same_free = free_ok && (r.flags & free_bit);
            free_ok = true;
        }
        return q;
    }
};

template <bool POOL, int CONC>
__device__ __forceinline__ void load_params(const hb_case& cs, const hb_mt& mt, int j, full::Params& p,
                                            full::Model& md) {
    const int np = cs.n_pad;
    const Spin sp = load_spin(cs.spins, cs.pos_lo, np, j);
    p.px = (double)sp.px + (double)sp.lx, p.py = (double)sp.py + (double)sp.ly, p.pz = (double)sp.pz + (double)sp.lz;
    p.pd = sp.pd, p.r1 = sp.r1, p.r2 = sp.r2, p.db0 = sp.db0, p.b1 = sp.b1;
    p.f = POOL ? mt.pool[j] : 0.0, p.k = POOL ? mt.pool[np + j] : 0.0;
    p.r1b = POOL ? mt.pool[2 * np + j] : 1.0, p.t2b = POOL ? mt.pool[3 * np + j] : 1.0;
    p.dw = POOL ? mt.pool[4 * np + j] : 0.0;
#pragma unroll
    for (int i = 0; i < 7; ++i) p.cc[i] = CONC != HB_CONC_NONE ? (double)mt.conc[(size_t)i * np + j] : 0.0;
    md.pool = POOL;
    md.conc = CONC;
    md.line = {mt.table, mt.lx0, mt.dlx, mt.cutoff, mt.n_table, mt.lineshape};
}

// An ADC sample's source: l += sum_c h_c conj(S_c), S of this lane's spin in registers (rows >= nc are not read).
__device__ __forceinline__ void add_source(const float* __restrict__ hrow, int nc, const float (&sr)[kMaxCoilsF],
                                           const float (&si)[kMaxCoilsF], full::St& l) {
#pragma unroll
    for (int c = 0; c < kMaxCoilsF; ++c) {
        if (c < nc) {
            const double hr = hrow[2 * c], hi = hrow[2 * c + 1];
            l.x += hr * sr[c] + hi * si[c];
            l.y += hi * sr[c] - hr * si[c];
        }
    }
}

__device__ __forceinline__ void load_sens(const float* __restrict__ sens, int nc, int np, int j,
                                          float (&sr)[kMaxCoilsF], float (&si)[kMaxCoilsF]) {
#pragma unroll
    for (int c = 0; c < kMaxCoilsF; ++c) {
        sr[c] = c < nc ? sens[(size_t)(2 * c) * np + j] : 0.0f;
        si[c] = c < nc ? sens[(size_t)(2 * c + 1) * np + j] : 0.0f;
    }
}

// Workgroups [0, n_pad / 256): the replay. With chunks, workgroups [n_pad / 256, 2 n_pad / 256): the bare adjoint from
// lam (after s1), its value after chunk c's last segment (before that segment's spoil and source) into
// lam_c[c] (4, n_pad); lam: before s0 out.
// The read-only inputs come in again as noalias parameters (the same pointers as in the structs): no store of the
// kernel can change what they point to, so the records and the h rows load through the scalar cache.
template <bool POOL, int CONC>
__global__ __launch_bounds__(kBlockF) void sweep_kernel(
    hb_case cs_in, hb_mt mt_in, hb_full_adjoint ad_in, int s0, int s1, int chunk, double* __restrict__ lam_c,
    const hb_segment* __restrict__ segs, const float* __restrict__ spins, const float* __restrict__ pos_lo,
    const float* __restrict__ pool_p, const float* __restrict__ rf_freq, const float* __restrict__ table,
    const float* __restrict__ conc, const float* __restrict__ ckpt, const float* __restrict__ ckpt_mb,
    const float* __restrict__ h, const float* __restrict__ sens) {
    hb_case cs = cs_in;
    cs.spins = spins, cs.pos_lo = pos_lo;
    hb_mt mt = mt_in;
    mt.pool = pool_p, mt.table = table, mt.conc = conc;
    const int tid = threadIdx.x, lane = tid & 63, np = cs.n_pad;
    const int n_blocks = np / kBlockF;
    const bool back = (int)blockIdx.x >= n_blocks;  // uniform
    const int j = ((int)blockIdx.x - (back ? n_blocks : 0)) * kBlockF + tid;
    full::Params p;
    full::Model md;
    load_params<POOL, CONC>(cs, mt, j, p, md);
    full::Cache ck = full::no_cache();
    Walk walk(!back);
    float warm = 0.0f;
    if (!back) {
        full::St m;
        m.x = (double)ckpt[j] + (double)ckpt[3 * np + j];
        m.y = (double)ckpt[np + j] + (double)ckpt[4 * np + j];
        m.z = (double)ckpt[2 * np + j] + (double)ckpt[5 * np + j];
        m.b = POOL ? (double)ckpt_mb[j] + (double)ckpt_mb[np + j] : 0.0;
        hb_segment nr = segs[s0];
        float nf = POOL ? rf_freq[s0] : 0.0f;
        for (int s = s0; s < s1; ++s) {
            if (((s - s0) & 63) == 0) {  // the next 64 records into the L2
                asm volatile("" ::"v"(warm));
                warm = segs[min(s + lane, s1 - 1)].dt;
            }
            float* tr = ad_in.traj + (size_t)(s - s0) * 4 * np;
            tr[j] = (float)m.x, tr[np + j] = (float)m.y, tr[2 * np + j] = (float)m.z, tr[3 * np + j] = (float)m.b;
            const hb_segment r = nr;
            const float frf = nf;
            nr = segs[min(s + 1, s1 - 1)];  // in flight while this one is stepped
            if (POOL) nf = rf_freq[min(s + 1, s1 - 1)];
            m = full::step(md, p, walk.next(r, frf), m, ck).after;
            if (r.flags & HB_SPOIL) m.x = m.y = 0.0;
        }
        return;
    }
    const int nc = ad_in.nc;
    float sr[kMaxCoilsF], si[kMaxCoilsF];
    load_sens(sens, nc, np, j, sr, si);
    full::St l = {ad_in.lam[j], ad_in.lam[np + j], ad_in.lam[2 * np + j], ad_in.lam[3 * np + j]};
    hb_segment nr = segs[s1 - 1];
    float nf = POOL ? rf_freq[s1 - 1] : 0.0f;
    for (int s = s1 - 1; s >= s0; --s) {
        const int k = s - s0;
        if (s == s1 - 1 || ((s1 - 1 - s) & 63) == 0) {
            asm volatile("" ::"v"(warm));
            warm = segs[max(s - lane, s0)].dt;
        }
        if (s == s1 - 1 || (k + 1) % chunk == 0) {
            double* o = lam_c + (size_t)(k / chunk) * 4 * np + j;
            o[0] = l.x, o[np] = l.y, o[2 * (size_t)np] = l.z, o[3 * (size_t)np] = l.b;
        }
        const hb_segment r = nr;
        const float frf = nf;
        nr = segs[max(s - 1, s0)];
        if (POOL) nf = rf_freq[max(s - 1, s0)];
        const full::Seg q = walk.next(r, frf);
        const full::Step st = full::set_up(md, p, q, ck);
        if (r.flags & HB_SPOIL) l.x = l.y = 0.0;
        if (nc > 0 && (r.flags & HB_ADC)) add_source(h + (size_t)r.pad[0] * 2 * nc, nc, sr, si, l);
        full::retreat(md, q, st, l);
    }
    ad_in.lam[j] = (float)l.x, ad_in.lam[np + j] = (float)l.y, ad_in.lam[2 * np + j] = (float)l.z;
    ad_in.lam[3 * np + j] = (float)l.b;
}

// The reverse of chunk blockIdx.y, [s0 + chunk y, ...), from the replayed states. One chunk: from lam (dL/dm after s1
// in, before s0 out), gradients added to gs and gc; several: from lam_c, the chunk's gradients into
// part[y] (N_G + 2 nc, n_pad) (the coil rows with coil gradients only).
template <bool SEG, bool POOL, int CONC>
__global__ __launch_bounds__(kBlockF) void reverse_kernel(
    hb_case cs_in, hb_mt mt_in, hb_full_adjoint ad_in, int s0, int s1, int chunk, const double* __restrict__ lam_c,
    double* __restrict__ part, const hb_segment* __restrict__ segs, const float* __restrict__ spins,
    const float* __restrict__ pos_lo, const float* __restrict__ pool_p, const float* __restrict__ rf_freq,
    const float* __restrict__ table, const float* __restrict__ conc, const float* __restrict__ traj,
    const float* __restrict__ h, const float* __restrict__ sens) {
    hb_case cs = cs_in;
    cs.spins = spins, cs.pos_lo = pos_lo;
    hb_mt mt = mt_in;
    mt.pool = pool_p, mt.table = table, mt.conc = conc;
    const hb_full_adjoint& ad = ad_in;
    extern __shared__ double gcs[];                        // coil gradients: slot a of lane tid at a * kBlockF + tid
    __shared__ double red[2][kWavesF][full::N_S];          // alternate buffers: one barrier per segment
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int j = blockIdx.x * kBlockF + tid;
    const int np = cs.n_pad;
    const int nc = ad.nc;
    const bool coil = nc > 0 && ad.coil_grads;  // uniform
    const bool parts = gridDim.y > 1;           // uniform
    const int c0 = s0 + (int)blockIdx.y * chunk, c1 = min(c0 + chunk, s1);
    float warm = segs[min(c0 + lane, c1 - 1)].dt;
    full::Params p;
    full::Model md;
    load_params<POOL, CONC>(cs, mt, j, p, md);
    float sr[kMaxCoilsF], si[kMaxCoilsF];
    load_sens(sens, nc, np, j, sr, si);
    if (coil) {
        for (int c = 0; c < 2 * nc; ++c) gcs[c * kBlockF + tid] = parts ? 0.0 : ad.gc[(size_t)c * np + j];
    }
    full::St l;
    if (parts) {
        const double* o = lam_c + (size_t)blockIdx.y * 4 * np + j;
        l = {o[0], o[np], o[2 * (size_t)np], o[3 * (size_t)np]};
    } else {
        l = {ad.lam[j], ad.lam[np + j], ad.lam[2 * np + j], ad.lam[3 * np + j]};
    }
    asm volatile("" ::"v"(warm));
    double g[full::N_G];
#pragma unroll
    for (int a = 0; a < full::N_G; ++a) g[a] = 0.0;
    int rbuf = 0;
    full::Cache ck = full::no_cache();
    Walk walk(false);
    for (int s = c1 - 1; s >= c0; --s) {
        const hb_segment r = segs[s];
        const float frf = POOL ? rf_freq[s] : 0.0f;
        const full::Seg q = walk.next(r, frf);
        const float* tr = traj + (size_t)(s - s0) * 4 * np;
        const full::St m0 = {tr[j], tr[np + j], tr[2 * np + j], tr[3 * np + j]};
        const full::Step st = full::step(md, p, q, m0, ck);
        if (r.flags & HB_SPOIL) l.x = l.y = 0.0;
        if (nc > 0 && (r.flags & HB_ADC)) {
            const float* hrow = h + (size_t)r.pad[0] * 2 * nc;
            add_source(hrow, nc, sr, si, l);
            if (coil) {
                const double ax = st.after.x, ay = st.after.y;
                for (int c = 0; c < nc; ++c) {
                    const double hr = hrow[2 * c], hi = hrow[2 * c + 1];
                    gcs[(2 * c) * kBlockF + tid] += hr * ax + hi * ay;
                    gcs[(2 * c + 1) * kBlockF + tid] += hi * ax - hr * ay;
                }
            }
        }
        double sg[full::N_S];
#pragma unroll
        for (int a = 0; a < full::N_S; ++a) sg[a] = 0.0;
        full::step_reverse(md, p, q, m0, st, l, g, sg);
        if (SEG) {  // the workgroup's sums of this segment's gradients (uniform: every lane takes it)
            const double v = seg_scatter_sums(sg, lane);
            if ((lane & 7) == 0) red[rbuf][wave][lane >> 3] = v;
            // the other buffer than the last segment's: a wave writes this one again only after every wave has
            // passed the next segment's barrier, i.e. after the reads below
            __syncthreads();
            if (tid < full::N_S) {
                double t = red[rbuf][0][tid];
#pragma unroll
                for (int w = 1; w < kWavesF; ++w) t += red[rbuf][w][tid];
                ad.gseg[((size_t)blockIdx.x * ad.k_max + (s - s0)) * 8 + tid] = (float)t;
            }
            rbuf ^= 1;
        }
    }
    if (!parts) {
        ad.lam[j] = (float)l.x, ad.lam[np + j] = (float)l.y, ad.lam[2 * np + j] = (float)l.z;
        ad.lam[3 * np + j] = (float)l.b;
#pragma unroll
        for (int a = 0; a < full::N_G; ++a) ad.gs[(size_t)a * np + j] += g[a];
        if (coil) {
            for (int c = 0; c < 2 * nc; ++c) ad.gc[(size_t)c * np + j] = gcs[c * kBlockF + tid];
        }
        return;
    }
    double* o = part + (size_t)blockIdx.y * (full::N_G + 2 * nc) * np + j;
#pragma unroll
    for (int a = 0; a < full::N_G; ++a) o[(size_t)a * np] = g[a];
    if (coil) {
        for (int c = 0; c < 2 * nc; ++c) o[(size_t)(full::N_G + c) * np] = gcs[c * kBlockF + tid];
    }
}

// Row a of the chunks' gradients added to gs (a < N_G) or gc, last chunk first; one lane per (row, spin).
__global__ __launch_bounds__(kBlockF) void chunk_sums_kernel(const double* __restrict__ part, int n_chunks, int rows,
                                                             int np, double* __restrict__ gs,
                                                             double* __restrict__ gc) {
    const int a = blockIdx.y, j = blockIdx.x * kBlockF + threadIdx.x;
    double* out = (a < full::N_G ? gs + (size_t)a * np : gc + (size_t)(a - full::N_G) * np) + j;
    double t = *out;
#pragma unroll 8
    for (int c = n_chunks - 1; c >= 0; --c) t += part[((size_t)c * rows + a) * np + j];
    *out = t;
}

// Segments per chunk of an interval of k segments of n_blocks workgroups (k: one chunk).
int chunk_for(int n_blocks, int k) {
    const int want = std::min(kFillBlocks / n_blocks, k / kMinChunk);
    return want < 2 ? k : (k + want - 1) / want;
}

template <bool POOL, int CONC>
hipError_t launch_full(const hb_case& cs, const hb_mt& mt, const hb_full_adjoint& ad, int s0, int s1, double* work,
                       hipStream_t st) {
    const int n_blocks = cs.n_pad / kBlockF, k = s1 - s0;
    const int chunk = work ? chunk_for(n_blocks, k) : k, n_chunks = (k + chunk - 1) / chunk;
    double* lam_c = work;
    double* part = work ? work + (size_t)n_chunks * 4 * cs.n_pad : nullptr;
    hipLaunchKernelGGL((sweep_kernel<POOL, CONC>), dim3(n_chunks > 1 ? 2 * n_blocks : n_blocks), dim3(kBlockF), 0, st,
                       cs, mt, ad, s0, s1, chunk, lam_c, cs.segs, cs.spins, cs.pos_lo, mt.pool, mt.rf_freq, mt.table,
                       mt.conc, ad.ckpt, ad.ckpt_mb, ad.h, ad.sens);
    const bool coil = ad.nc > 0 && ad.coil_grads;
    const size_t lds = coil ? sizeof(double) * 2 * ad.nc * kBlockF : 0;
    auto kernel = ad.seg_grads ? reverse_kernel<true, POOL, CONC> : reverse_kernel<false, POOL, CONC>;
    hipLaunchKernelGGL(kernel, dim3(n_blocks, n_chunks), dim3(kBlockF), lds, st, cs, mt, ad, s0, s1, chunk, lam_c, part,
                       cs.segs, cs.spins, cs.pos_lo, mt.pool, mt.rf_freq, mt.table, mt.conc, ad.traj, ad.h, ad.sens);
    if (n_chunks > 1)
        hipLaunchKernelGGL(chunk_sums_kernel, dim3(n_blocks, full::N_G + (coil ? 2 * ad.nc : 0)), dim3(kBlockF), 0, st,
                           part, n_chunks, full::N_G + 2 * ad.nc, cs.n_pad, ad.gs, ad.gc);
    return hipGetLastError();
}

template <bool POOL>
hipError_t launch_conc(const hb_case& cs, const hb_mt& mt, const hb_full_adjoint& ad, int s0, int s1, double* work,
                       hipStream_t st) {
    switch (mt.conc_mode) {
        case HB_CONC_LEADING: return launch_full<POOL, HB_CONC_LEADING>(cs, mt, ad, s0, s1, work, st);
        case HB_CONC_EXACT: return launch_full<POOL, HB_CONC_EXACT>(cs, mt, ad, s0, s1, work, st);
        default: return launch_full<POOL, HB_CONC_NONE>(cs, mt, ad, s0, s1, work, st);
    }
}

}  // namespace
}  // namespace hb

extern "C" int64_t hb_adjoint_full_workspace(int32_t n_pad, int32_t k_max, int32_t nc) {
    using namespace hb;
    if (n_pad < kBlockF || n_pad % kBlockF || k_max < 1 || nc < 0 || nc > kMaxCoilsF) return 0;
    // the most chunks any interval of up to k_max segments takes
    const int64_t chunks = std::max(1, std::min(kFillBlocks / (n_pad / kBlockF), k_max / kMinChunk));
    return chunks < 2 ? 0 : chunks * (4 + full::N_G + 2 * nc) * (int64_t)n_pad;
}

extern "C" int hb_adjoint_full_chunks(const hb_case* cs, const hb_mt* mt, const hb_full_adjoint* ad, int32_t s0,
                                      int32_t s1, double* work, void* stream) {
    using namespace hb;
    if (!cs || !mt || !ad || !ad->ckpt || !ad->traj || !ad->lam || !ad->gs) return hipErrorInvalidValue;
    if (cs->n_pad <= 0 || cs->n_pad % kBlockF || cs->n < 0 || cs->n > cs->n_pad) return hipErrorInvalidValue;
    if (s0 < 0 || s1 < s0 || s1 > cs->n_segments || s1 - s0 > ad->k_max) return hipErrorInvalidValue;
    if (ad->nc < 0 || ad->nc > kMaxCoilsF || (ad->nc > 0 && (!ad->h || !ad->sens))) return hipErrorInvalidValue;
    if (ad->coil_grads && ad->nc > 0 && !ad->gc) return hipErrorInvalidValue;
    if (ad->seg_grads && !ad->gseg) return hipErrorInvalidValue;
    if (mt->pool && (!mt->rf_freq || !ad->ckpt_mb)) return hipErrorInvalidValue;
    if (mt->pool && mt->lineshape == HB_LINE_SUPERLORENTZIAN && (!mt->table || mt->n_table < 2 || !(mt->dlx > 0.0f)))
        return hipErrorInvalidValue;
    if (mt->pool && mt->lineshape != HB_LINE_SUPERLORENTZIAN && mt->lineshape != HB_LINE_LORENTZIAN)
        return hipErrorInvalidValue;
    if (mt->conc_mode < HB_CONC_NONE || mt->conc_mode > HB_CONC_EXACT || (mt->conc_mode && !mt->conc))
        return hipErrorInvalidValue;
    if (s1 == s0) return hipSuccess;
    hipStream_t st = (hipStream_t)stream;
    return mt->pool ? launch_conc<true>(*cs, *mt, *ad, s0, s1, work, st)
                    : launch_conc<false>(*cs, *mt, *ad, s0, s1, work, st);
}

extern "C" int hb_adjoint_full(const hb_case* cs, const hb_mt* mt, const hb_full_adjoint* ad, int32_t s0, int32_t s1,
                               void* stream) {
    return hb_adjoint_full_chunks(cs, mt, ad, s0, s1, nullptr, stream);
}
