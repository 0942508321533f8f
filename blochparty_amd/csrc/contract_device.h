// The coil contraction of the forward kernels on the matrix cores, shared by forward.hip and mt.hip.
//
// Coil contraction, per wave: each ADC sample leaves Mxy of the wave's 64 spins; eight samples are staged in LDS as
// the columns of B (64 x 16: Re Mxy of samples 0..7, then Im), and D = A B on the matrix cores with A (16 x 64) the
// wave's sensitivities of one tile of 8 coils, rows Re S_0, Im S_0, Re S_1, Im S_1, ..., held in registers in the
// operand order. With the K index of step u at lane group g being spin 16 g + u, lane l supplies
// A[l % 16][16 (l / 16) + u] and B[16 (l / 16) + u][l % 16] and receives D[4 (l / 16) + r][l % 16], r = 0..3. The
// complex sums are then
//     P_c(t) = D[2c][t] - D[2c + 1][8 + t],   Q_c(t) = D[2c][8 + t] + D[2c + 1][t]   (signal before demodulation),
// the partner column 8 lanes away in the same row of 16 (a DPP rotation). The four waves' sums are added in LDS in a
// fixed order and written as this workgroup's partial row; hb_signal_reduce adds the workgroups in float64, in
// order. No atomics: the signal is the same bit for bit on every run.
//
// Precision of the product: for up to two tiles (16 coils) both operands are split into float16 pairs, x = hi + lo
// (x scaled into [-2^8, 2^8] by powers of two), and D = Ah Bh + Ah Bl + Al Bh on v_mfma_f32_16x16x32_f16: float16
// products are exact in the float32 accumulator, and the pairs hold each operand to 2^-24 relative (2^-33 of the bound
// at least), so D is as close to the exact sum as a float32 product would be, at six 16-cycle instructions per tile
// and flush in place of sixteen 32-cycle v_mfma_f32_16x16x4f32. More tiles use the float32 instruction, with the
// sensitivities read from memory. So does F32 (the full variant), with the sensitivities in registers as they are: it takes
// no scales, and a coil, a spin or a late echo far below the case's largest keeps its 24 bits.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace hb {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kStgStride = 68;  // floats per staged column row: 64 lanes + 4 (spreads the b128 reads over banks)
constexpr int kStgFloats = 16 * kStgStride;
constexpr int kMaxTiles = 16;   // 128 coils: LDS = 4 x 16 x 68 + 4 x 8 x 256 floats = 49 KB

// LDS: every wave's staging block, then two buffers of the waves' coil sums (flushes alternate between them).
__host__ __device__ constexpr int lds_floats(int nt) { return kWaves * kStgFloats + 2 * kWaves * 8 * 16 * nt; }

// Float16's smallest step is 2^-24, so the low part of a value scaled to 2^-6 of the bound would keep it to 2^-19 only:
// the operands are lifted by this power of two (undone exactly by out_scale), which leaves 2^8 above the bound (for an
// operand that is one such value, not a product of two).
constexpr float kLift = 256.0f;

// x of lane (jj + 8) mod 16 of this lane's row of 16 (DPP row_ror:8).
__device__ __forceinline__ float dpp_ror8(float x) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(0u, __float_as_uint(x), 0x128, 0xf, 0xf, false));
}

// x = hi + lo in float16 for eight floats: hi rounded to nearest, lo the rounded remainder (exact in float32). For
// |x| < 65504 the pair holds x to 2^-24 |x| or 2^-25, whichever is larger (lo may be subnormal: the matrix cores take
// float16 subnormals as they are).
__device__ __forceinline__ void split8(const float* x, h8& hi, h8& lo) {
#pragma unroll
    for (int e = 0; e < 8; e += 2) {  // in pairs: one v_cvt_pk_f16_f32 per pair of hi and of lo parts
        const h2 h = __builtin_convertvector((f2){x[e], x[e + 1]}, h2);
        // x - float(h) in one v_fma_mix_f32 per value, the float16 operand taken from its half of the packed pair
        // (the compiler forms a conversion and a subtraction); exact, float16 subnormals included
        const unsigned hu = __builtin_bit_cast(unsigned, h);
        float r0, r1;
        asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(hu), "v"(x[e]));
        asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r1) : "v"(hu), "v"(x[e + 1]));
        const h2 l = __builtin_convertvector((f2){r0, r1}, h2);
        hi[e] = h[0], hi[e + 1] = h[1];
        lo[e] = l[0], lo[e + 1] = l[1];
    }
}

// The wave's sensitivities as matrix-core operands. NT > 0: each tile's 16 values per lane (spins 16 g + u,
// u = 0..15, of row l % 16) scaled by the case's sens_scale and split into float16 hi and lo parts, as the A operands
// of two v_mfma_f32_16x16x32_f16 (u = 0..7 and 8..15); NT = 0: read from memory in float32 at every flush, value u of
// tile t at sa[t st + u su].
// out_scale undoes the sensitivities' and the staged values' scales (powers of two: exact).
template <int NT, bool F32 = false>
struct Sens {
    static constexpr bool kPairs = NT > 0 && !F32;
    h8 hi[kPairs ? NT : 1][2], lo[kPairs ? NT : 1][2];
    float a[NT > 0 && F32 ? NT : 1][16];
    const float *sa, *sa0;
    size_t st;
    int su, n_rows;
    float x_scale, out_scale;

    // F32: rows from n_rows on are zeros, row 0 (sa0) read in their place: every load is unconditional
    __device__ __forceinline__ float at(int t, int u, int row) const {
        if constexpr (F32) {
            const bool in = 16 * t + row < n_rows;
            const float v = (in ? sa + t * st : sa0)[(size_t)u * su];
            return in ? v : 0.0f;
        }
        return sa[t * st + (size_t)u * su];
    }

    // sa, st, su and n_rows are set; x_scale_ and sens_scale as hb_case's (0 reads as 1)
    __device__ __forceinline__ void scales(float x_scale_, float& sens_scale) {
        x_scale = x_scale_ > 0.0f ? x_scale_ : 1.0f;
        if (!(sens_scale > 0.0f)) sens_scale = 1.0f;
        if (kPairs) x_scale *= kLift, sens_scale *= kLift;
        out_scale = 1.0f / (kPairs ? x_scale * sens_scale : x_scale);
    }

    // F32: no scales
    __device__ __forceinline__ void load_f32(int lane) {
        static_assert(F32, "float32 operands");
        x_scale = out_scale = 1.0f;
        if constexpr (NT > 0) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int u = 0; u < 16; ++u) a[t][u] = at(t, u, lane & 15);
        }
    }

    __device__ __forceinline__ void load(float x_scale_, float sens_scale, int lane) {
        scales(x_scale_, sens_scale);
        if constexpr (kPairs) {
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    float x[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[e] = at(t, 8 * i + e, lane & 15) * sens_scale;
                    split8(x, hi[t][i], lo[t][i]);
                }
        }
    }
};

// The wave's complex coil sums of tile t from its product acc, into mine in the output order [sample][tile][coil][re, im].
__device__ __forceinline__ void store_pq(float* mine, int vals, int t, int lane, const f4& acc) {
    const int g = lane >> 4, jj = lane & 15;
    // rows 4 g .. 4 g + 3 of lane (g, jj) are Re S_c0, Im S_c0, Re S_c1, Im S_c1 (c0 = 2 g, c1 = 2 g + 1) at
    // column jj; the partner column jj +- 8 sits in the same row of 16 lanes: DPP row_ror:8. Lanes jj < 8 form
    // coil c0's (P, Q) at sample jj, lanes jj >= 8 coil c1's at sample jj - 8.
    const float r0 = dpp_ror8(acc[0]), r1 = dpp_ror8(acc[1]), r2 = dpp_ror8(acc[2]), r3 = dpp_ror8(acc[3]);
    const bool first = jj < 8;
    const f2 pq = first ? (f2){acc[0] - r1, r0 + acc[1]} : (f2){r2 - acc[3], acc[2] + r3};
    *reinterpret_cast<f2*>(mine + (jj & 7) * vals + 16 * t + 2 * (2 * g + (jj >> 3))) = pq;  // one 8-byte store
}

// The coil sums of the nb (<= 8) staged samples of every wave, added over the workgroup, into the partial rows
// [row, row + nb) of this workgroup. Every lane of the workgroup calls it. One barrier: a wave reads only its own
// staging block (a wave-scope fence orders its lanes' writes before the reads), and the waves' sums alternate
// between two buffers, so a flush's writes never meet the previous flush's reads (every wave has passed this
// flush's barrier, after those reads, before it can write the buffer again two flushes later).
template <int NT, bool F32>
__device__ __forceinline__ void flush_to(float* stg, float* wred2, int& par, const Sens<NT, F32>& S, int nt,
                                         int n_out_cols, float* __restrict__ out, int k_first = 8,
                                         float* __restrict__ out_rest = nullptr, int k_skip = 0) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, jj = lane & 15;
    const int vals = 16 * nt;
    float* wred = wred2 + par * (kWaves * 8 * vals);
    par ^= 1;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float b[16];
    {
        const f4* src = reinterpret_cast<const f4*>(stg + jj * kStgStride + 16 * g);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const f4 x = src[v];
            b[4 * v] = x[0], b[4 * v + 1] = x[1], b[4 * v + 2] = x[2], b[4 * v + 3] = x[3];
        }
    }
    float* mine = wred + wave * 8 * vals;
    constexpr bool kPairs = Sens<NT, F32>::kPairs;
    h8 bh[2], bl[2];
    if constexpr (kPairs) {
        split8(b, bh[0], bl[0]);
        split8(b + 8, bh[1], bl[1]);
    }
    for (int t = 0; t < nt; ++t) {
        f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (kPairs) {
            // A B = Ah Bh + Ah Bl + Al Bh (+ Al Bl, under 2^-22 of the product: dropped), small terms first; each
            // product of float16 values is exact in the float32 accumulator
#pragma unroll
            for (int i = 0; i < 2; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(S.lo[t][i], bh[i], acc, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 2; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(S.hi[t][i], bl[i], acc, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 2; ++i) acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(S.hi[t][i], bh[i], acc, 0, 0, 0);
        } else {
#pragma unroll
            for (int u = 0; u < 16; ++u)
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(NT > 0 ? S.a[NT > 0 ? t : 0][u] : S.at(t, u, jj), b[u], acc, 0,
                                                           0, 0);
        }
        store_pq(mine, vals, t, lane, acc);
    }
    __syncthreads();
    // columns [0, k_first) to out, [k_first, k_first + k_skip) dropped, the rest to out_rest (output value
    // v = sample * vals + 16 tile + 2 coil + {0: re, 1: im})
    const int n_out = n_out_cols * vals, split = k_first * vals, resume = (k_first + k_skip) * vals;
    for (int v = tid; v < n_out; v += kBlock) {
        float s = wred[v];
#pragma unroll
        for (int w = 1; w < kWaves; ++w) s += wred[w * 8 * vals + v];
        s *= S.out_scale;
        if (v < split)
            out[v] = s;
        else if (v >= resume)
            out_rest[v - resume] = s;
    }
}

// The staged samples into the partial rows [row, row + nb) of this workgroup (never past the buffer's rows).
template <int NT, bool F32>
__device__ __forceinline__ void flush(float* stg, float* wred2, int& par, const Sens<NT, F32>& S, int nt, int nb, int row,
                                      int rows, float* __restrict__ partial) {
    const int n_out = row + nb <= rows ? nb : (rows > row ? rows - row : 0);
    flush_to(stg, wred2, par, S, nt, n_out, partial + ((size_t)blockIdx.x * rows + row) * (16 * nt));
}

}  // namespace hb
