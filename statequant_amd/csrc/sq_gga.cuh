// Mixed-width GGA / STEP slot with the FP8 write window (PW-S m): one decode token per (batch row, value head).
//
// Replaces the reference's `_gga_step`, `_gga_advance`, `_gga_store`, `_gga_load`
// (/root/reference/src/statequant/kernels/_gga_triton.py:207-340) and the dual-axis fit they call
// (`_fit_parts`, /root/reference/src/statequant/kernels/_stepquant_triton.py:41-69).  Per slot (byte offsets):
//   0            int32 [4]: n (queued pairs), head (ring index of the oldest pair)
//   offs[h]      head h at its frozen width b: fp16 [d_k, d_v] (b = 16), or codes [d_k, d_v b / 8] packed
//                little-endian along d_v (u = z + qmax; b = 2: u = (z + 3) / 2), row factors fp16 [d_k] (b = 2: one
//                per 32 value columns, [d_k, d_v / 32]) and column factors fp16 [d_v]; the state is (r c) z
//   qoff + h qsz the head's window: P e4m3 [m, d_k], V e4m3 [m, d_v], PS fp32 [m], VS fp32 [m] (a ring)
// One token (Algorithm 1 of the method, as the reference implements it):
//   O_pre = a (O - beta k (k^T O));  queued left factors p_i <- R(a (p_i - beta k (k^T p_i)))  (R: FP8 per vector);
//   o = O_pre^T q + sum_i (p_i^T q) v_i + (beta k^T q) v;  window full: the oldest pair is merged, O_pre += p_0 v_0^T;
//   the state is re-fitted at its width and re-packed in place; (R(beta k), R(v)) is queued.  Pivots (b = 16) and
//   slots without a window take the new write into the state: O = Q(O_pre + beta k v^T).
//
// A workgroup of four wavefronts holds the head's [d_k, d_v] tile in registers.  Wavefront w owns a quarter of the
// columns and all rows: lane (tr, q) = (lane / 4, lane % 4) owns the columns tc CT .. tc CT + CT - 1 (tc = 4 w + q,
// CT = d_v / 16) of the rows s 16 + tr.  Sums along d_k -- the step and the fit take five of them per column -- stay
// inside a wavefront and end SPREAD over it: each of the four 16-lane rows keeps a quarter of its lanes' columns
// (gga_col_reduce), does what is to be done per column for those alone, and hands only the results that every lane
// needs back (gga_col_gather).  The one sum along d_v (the row factors of the fit) is a quad reduction plus an exchange
// of per-wavefront partials through LDS, where one thread per row then forms that row's factors for everybody.
//
// What bounds the step is the vector ALU: every head is unpacked, updated, fitted and packed at every token (some 20
// instructions per state value), while its bytes would take a tenth of the time.  So what counts is instructions, and
// enough wavefronts to hide the serial stretches between them: the fit keeps ONE copy of the tile and multiplies by the
// row factors' reciprocals again where it needs the quotients (one instruction a value; divisions only where a rounding
// could differ, see GGA_ABOVE), which leaves registers for four wavefronts per SIMD where values and quotients side by side
// left them for two.
#pragma once
#include "sq_device.cuh"
#include "sq_params.h"

namespace sq {

constexpr int GGA_THREADS = 256;
constexpr int GGA_WAVES = GGA_THREADS / WAVE;
constexpr int GGA_MMAX = 8;
constexpr int GGA_GROUP = 32;
// the slot's second counter: the ring index of the oldest pair, and above it -- while a step runs -- the heads that have
// read the counters, in 24 bits: as many as a launch has workgroups
constexpr uint32_t GGA_RING = 0xFF, GGA_TICKET = 0x100;
constexpr int GGA_GRID_Y = 65535;                       // heads along the second dimension of a launch

template <int DK_, int DV_>
struct GgaTile {
    static constexpr int DK = DK_, DV = DV_;
    static constexpr int CT = DV / 16;                  // columns per thread
    static constexpr int CO = CT / 4;                   // columns a lane keeps of a sum along d_k
    static constexpr int RPT = DK / 16;                 // rows per thread
    static constexpr int NE = DK / WAVE;                // a key vector's elements per lane (one wavefront per vector)
    static constexpr int NV = DV / WAVE;
    static constexpr int NG = DV / GGA_GROUP;           // row-factor groups of a two-bit head
    static_assert(DK % WAVE == 0 && DV % WAVE == 0 && CT % 4 == 0, "built for d_k, d_v multiples of 64");
};

struct GgaThread {
    int tid, lane, wave, tc, tr;
    int own;                                            // first of the lane's kept columns, of its CT, in quarters of CT
};
__device__ __forceinline__ GgaThread gga_thread() {
    GgaThread t;
    t.tid = threadIdx.x;
    // from a copy the compiler cannot trace back: called anew in front of a phase, what it derives does not stay in
    // registers from the kernel's top on
    asm volatile("" : "+v"(t.tid));
    t.lane = t.tid & (WAVE - 1);
    t.wave = t.tid >> 6;
    t.tc = t.wave * 4 + (t.lane & 3);
    t.tr = t.lane >> 2;
    t.own = 2 * ((t.lane >> 4) & 1) + (t.lane >> 5);
    return t;
}

__host__ __device__ constexpr int gga_qmax(int b) { return b == 2 ? 3 : (1 << (b - 1)) - 1; }
__host__ __device__ constexpr int gga_code_bytes(int b, int dk, int dv) { return dk * dv * b / 8; }

// fp16 with the fit's clamp: [2^-24, 65504], round to nearest even.
__device__ __forceinline__ float gga_half(float x) { return float(_Float16(fminf(fmaxf(x, FP16_TINY), 65504.0f))); }

// The fit's divisions go through `div_rc` / `rcp_f16` (sq_device.cuh): reciprocals once per row or column, IEEE
// quotients at a third of the instructions.
__device__ __forceinline__ float gga_div(float x, float d, float rc) { return div_rc(x, d, rc); }
__device__ __forceinline__ float gga_rcp_f16(float d) { return rcp_f16(d); }

// ---------------------------------------------------------------------------------------------------------------
// sums / maxima along d_k
// ---------------------------------------------------------------------------------------------------------------
constexpr int DPP_ROR4 = 0x124, DPP_ROR8 = 0x128;      // row_ror: lane i of a 16-lane row reads lane (i + n) % 16

template <bool MAX>
__device__ __forceinline__ float gga_combine(float a, float b) { return MAX ? fmaxf(a, b) : a + b; }

// Totals over the 16 row groups of a wavefront (lanes with the same lane % 4) of the CT columns of a lane, spread: the
// lane keeps the CO = CT / 4 columns from CO own on.  A lane swap takes two columns at once -- v_permlane16_swap(a, b)
// leaves {a's even 16-lane rows | b's even rows} and {a's odd rows | b's odd rows}, whose sum is column a's in the even
// rows and column b's in the odd ones, v_permlane32_swap the same for the halves -- so the swaps of eight columns cost 12
// instructions where handing every lane all of them costs 56.  The four lanes that keep a column hold the same bits.
// (Sums: lanes 8 and 4 apart first, then 16, then 32 -- the order decides the last bit of a sum and with it, now and
// then, which side of an fp16 rounding threshold a column factor falls on.)
template <class T, int K, bool MAX>
__device__ __forceinline__ void gga_col_reduce(float (&p)[K][T::CT], float (&own)[K][T::CO]) {
    constexpr int CT = T::CT, CO = T::CO;
    auto rows = [](float v) {
        v = gga_combine<MAX>(v, dpp<DPP_ROR8>(v));
        return gga_combine<MAX>(v, dpp<DPP_ROR4>(v));
    };
#pragma unroll
    for (int k = 0; k < K; ++k) {
        if constexpr (!MAX) {
#pragma unroll
            for (int e = 0; e < CT; ++e) p[k][e] = rows(p[k][e]);
        }
        float half[CT / 2];
#pragma unroll
        for (int e = 0; e < CT / 2; ++e) {
            const auto r = __builtin_amdgcn_permlane16_swap(as_u32(p[k][e]), as_u32(p[k][e + CT / 2]), false, false);
            half[e] = gga_combine<MAX>(as_f32(r[0]), as_f32(r[1]));
        }
#pragma unroll
        for (int e = 0; e < CO; ++e) {
            const auto r = __builtin_amdgcn_permlane32_swap(as_u32(half[e]), as_u32(half[e + CO]), false, false);
            own[k][e] = gga_combine<MAX>(as_f32(r[0]), as_f32(r[1]));
            if constexpr (MAX) own[k][e] = rows(own[k][e]);
        }
    }
}
// Every lane's CT columns from the kept ones.
template <class T>
__device__ __forceinline__ void gga_col_gather(const float (&own)[T::CO], float (&all)[T::CT]) {
    constexpr int CT = T::CT, CO = T::CO;
    float half[CT / 2];
#pragma unroll
    for (int e = 0; e < CO; ++e) {
        const auto r = __builtin_amdgcn_permlane32_swap(as_u32(own[e]), as_u32(own[e]), false, false);
        half[e] = as_f32(r[0]);
        half[e + CO] = as_f32(r[1]);
    }
#pragma unroll
    for (int e = 0; e < CT / 2; ++e) {
        const auto r = __builtin_amdgcn_permlane16_swap(as_u32(half[e]), as_u32(half[e]), false, false);
        all[e] = as_f32(r[0]);
        all[e + CT / 2] = as_f32(r[1]);
    }
}

// ---------------------------------------------------------------------------------------------------------------
// a thread's CT codes of one row: NB = CT B / 8 bytes, little-endian bit string
// ---------------------------------------------------------------------------------------------------------------
template <int NB>
__device__ __forceinline__ uint64_t gga_load_bytes(const uint8_t* p) {
    if constexpr (NB == 8) {
        const uint2 v = *reinterpret_cast<const uint2*>(p);
        return uint64_t(v.x) | (uint64_t(v.y) << 32);
    } else if constexpr (NB == 4) {
        return *reinterpret_cast<const uint32_t*>(p);
    } else if constexpr (NB == 2) {
        return *reinterpret_cast<const uint16_t*>(p);
    } else if constexpr (NB == 1) {
        return *p;
    } else if constexpr (NB == 6) {
        const uint16_t* h = reinterpret_cast<const uint16_t*>(p);
        return uint64_t(h[0]) | (uint64_t(h[1]) << 16) | (uint64_t(h[2]) << 32);
    } else {
        static_assert(NB == 3, "bytes per thread and row");
        return uint64_t(p[0]) | (uint64_t(p[1]) << 8) | (uint64_t(p[2]) << 16);
    }
}
template <int NB>
__device__ __forceinline__ void gga_store_bytes(uint8_t* p, uint64_t v) {
    if constexpr (NB == 8) {
        *reinterpret_cast<uint2*>(p) = make_uint2(uint32_t(v), uint32_t(v >> 32));
    } else if constexpr (NB == 4) {
        *reinterpret_cast<uint32_t*>(p) = uint32_t(v);
    } else if constexpr (NB == 2) {
        *reinterpret_cast<uint16_t*>(p) = uint16_t(v);
    } else if constexpr (NB == 1) {
        *p = uint8_t(v);
    } else if constexpr (NB == 6) {
        uint16_t* h = reinterpret_cast<uint16_t*>(p);
        h[0] = uint16_t(v);
        h[1] = uint16_t(v >> 16);
        h[2] = uint16_t(v >> 32);
    } else {
        static_assert(NB == 3, "bytes per thread and row");
        p[0] = uint8_t(v);
        p[1] = uint8_t(v >> 8);
        p[2] = uint8_t(v >> 16);
    }
}

// Code e of a row piece as its signed value z times 2^up(e).  The code's bits are left where they are, in the mantissa
// of 2^23: masked in, 2^23 + (bias + z) 2^up comes out as a float without a shift or a conversion, and one exact
// subtraction leaves z 2^up.  The power of two goes into the column factor (exact).  PER codes fit a mantissa at a time.
template <int B>
struct GgaCode {
    static constexpr int LOW = B == 2 ? 1 : 0;                             // two bits: z = 2 u - 3, from a word shifted by 1
    static constexpr int PER = B == 8 ? 2 : B == 6 ? 3 : B == 4 ? 4 : 8;
    __device__ static constexpr int up(int e) { return (e % PER) * B; }
    __device__ __forceinline__ static float value(uint64_t raw, int e) {
        const int at = (e / PER) * PER * B;
        const uint32_t w = LOW ? uint32_t(raw) << 1 : uint32_t(raw >> at);
        const uint32_t mask = ((1u << B) - 1) << (up(e) + LOW);
        const float bias = 8388608.0f + float((B == 2 ? 3 : gga_qmax(B)) << up(e));
        return as_f32((w & mask) | 0x4B000000u) - bias;
    }
};

// Head state of width B at S -> the thread's x[s][e] (reference: `_load_head`, _gga_triton.py:131-143).  `between` runs
// when the loads are out and before any of them is used: what else is to be requested.
template <class T, int B, class F>
__device__ __forceinline__ void gga_load_head(const uint8_t* S, const GgaThread& t, float (&x)[T::RPT][T::CT], F&& between) {
    constexpr int CT = T::CT, RPT = T::RPT, DK = T::DK, DV = T::DV;
    if constexpr (B == 16) {
        const uint16_t* H = reinterpret_cast<const uint16_t*>(S);
        uint2 v[RPT][CT / 4];
#pragma unroll
        for (int s = 0; s < RPT; ++s)
#pragma unroll
            for (int e4 = 0; e4 < CT / 4; ++e4)
                v[s][e4] = *reinterpret_cast<const uint2*>(H + (s * 16 + t.tr) * DV + t.tc * CT + 4 * e4);
        between();
#pragma unroll
        for (int s = 0; s < RPT; ++s)
#pragma unroll
            for (int e4 = 0; e4 < CT / 4; ++e4) {
                x[s][4 * e4 + 0] = f16_to_f32(uint16_t(v[s][e4].x));
                x[s][4 * e4 + 1] = f16_to_f32(uint16_t(v[s][e4].x >> 16));
                x[s][4 * e4 + 2] = f16_to_f32(uint16_t(v[s][e4].y));
                x[s][4 * e4 + 3] = f16_to_f32(uint16_t(v[s][e4].y >> 16));
            }
    } else {
        constexpr int NB = CT * B / 8;
        constexpr int RB = DV * B / 8;                                     // bytes of a row of codes
        const uint16_t* R = reinterpret_cast<const uint16_t*>(S + gga_code_bytes(B, DK, DV));
        const uint16_t* C = R + (B == 2 ? DK * T::NG : DK);
        uint64_t raw[RPT];
        uint16_t rr[RPT];
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const int i = s * 16 + t.tr;
            raw[s] = gga_load_bytes<NB>(S + i * RB + t.tc * NB);
            rr[s] = B == 2 ? R[i * T::NG + (t.tc * CT) / GGA_GROUP] : R[i];
        }
        uint32_t cw[CT / 2];
        if constexpr (CT == 8) {
            const uint4 v = *reinterpret_cast<const uint4*>(C + t.tc * CT);
            cw[0] = v.x; cw[1] = v.y; cw[2] = v.z; cw[3] = v.w;
        } else {
            const uint2 v = *reinterpret_cast<const uint2*>(C + t.tc * CT);
            cw[0] = v.x; cw[1] = v.y;
        }
        between();
        float c[CT];                                                       // column factors, over the code's scale
#pragma unroll
        for (int e = 0; e < CT; ++e)
            c[e] = f16_to_f32(uint16_t(cw[e / 2] >> (16 * (e % 2)))) * (1.0f / float(1u << GgaCode<B>::up(e)));
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const float r = f16_to_f32(rr[s]);
#pragma unroll
            for (int e = 0; e < CT; ++e) x[s][e] = (r * c[e]) * GgaCode<B>::value(raw[s], e);
            __builtin_amdgcn_sched_barrier(0);              // a row at a time: rows side by side would not fit the registers
        }
    }
}

// LDS of the fit: per-wavefront partial row sums, and every row's factors {r, 1 / r, w^2} (two-bit heads: per group
// of value columns).
template <class T>
struct GgaFitLds {
    float4 row[T::NG][T::DK];
    float sum[GGA_WAVES * T::DK];
};

constexpr float GGA_MAGIC = 12582912.0f;               // 1.5 2^23 (even: ties go to even): adding it rounds to an integer, left
                                                       // in the low mantissa bits

// The fit needs the IEEE quotients' roundings -- a code, a column's fp16 factor -- not the quotients, and products with the
// reciprocals nearly always round alike.  With u = 2^-24: RN(1 / r), RN(1 / c) and each product add at most u, IEEE x / r
// and (x / r) / c at most u each, so a product raised and lowered by 8 u (GGA_ABOVE, GGA_BELOW: a rounding or two less)
// encloses the quotient with 2 u to spare.  Where both ends round to the same number that is the quotient's; where they
// do not, the lanes' values are divided (a row step of 512 values: one in 20 at 8 bits, one in 350 at 4).  Not meant for
// overflows: from GGA_FAST_MAX on everything is divided.  6 instructions a code instead of 9 and 8, 1.5 a value instead of
// 4 for the column maxima: some 600 of a wavefront's 3400, 30.2 -> 27.4 us for 32 sequences x 32 heads of 128 x 128, the same
// bits stored.  (Leaving the clamp out where no code can need it measured 29.1: another order of the compiler's.)
constexpr float GGA_ABOVE = 1.0f + 0x1p-21f, GGA_BELOW = 1.0f - 0x1p-21f, GGA_FAST_MAX = 1e30f;

// A row's factor from its mean |x| a: {r, 1 / r, w^2}.  The division and the square root are IEEE.
__device__ __forceinline__ float4 gga_row_factor(float a, float w) {
    const float r = gga_half(sqrtf(fmaxf(a, 1e-20f) / w));
    return make_float4(r, gga_rcp_f16(r), w * w, 0.0f);
}

// STEP's dual-axis fit of the thread block's tile x at width B, packed at S (reference: `_store_head` ->
// `_fit_parts`): row factors r = half(sqrt(max(mean_j |x|, 1e-20) / w)), column factors c = half(max_i |x / r| /
// qmax), codes, one w^2-weighted least-squares refit of c with the codes fixed, codes again.  Codes and factors are
// those of IEEE divisions, as in torch (quotients are exact half-integers often enough -- one 8-bit head in eight -- that
// rounding y times a reciprocal would store other codes); the square root is IEEE.  `w` = the head's row weights.
template <class T, int B>
__device__ __forceinline__ void gga_fit_store(uint8_t* S, float (&x)[T::RPT][T::CT], const float* w,
                                              GgaFitLds<T>& L, const GgaThread& t) {
    constexpr int CT = T::CT, CO = T::CO, RPT = T::RPT, DK = T::DK, DV = T::DV;
    if constexpr (B == 16) {
        uint16_t* H = reinterpret_cast<uint16_t*>(S);
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const int i = s * 16 + t.tr;
#pragma unroll
            for (int e4 = 0; e4 < CT; e4 += 4) {
                uint2 v;
                v.x = uint32_t(f32_to_f16(x[s][e4])) | (uint32_t(f32_to_f16(x[s][e4 + 1])) << 16);
                v.y = uint32_t(f32_to_f16(x[s][e4 + 2])) | (uint32_t(f32_to_f16(x[s][e4 + 3])) << 16);
                *reinterpret_cast<uint2*>(H + i * DV + t.tc * CT + e4) = v;
            }
        }
    } else {
        constexpr int NB = CT * B / 8;
        constexpr int RB = DV * B / 8;
        constexpr float QMAX = float(gga_qmax(B));
        constexpr int COLS = B == 2 ? GGA_GROUP : DV;                       // columns sharing one row factor
        uint16_t* R = reinterpret_cast<uint16_t*>(S + gga_code_bytes(B, DK, DV));
        uint16_t* C = R + (B == 2 ? DK * T::NG : DK);
        // ---- row factors ----
        constexpr bool OWN = B == 2 && 4 * CT >= GGA_GROUP;       // a two-bit group lies inside one wavefront's columns
        const int grp = B == 2 ? (t.wave * 4 * CT) / GGA_GROUP : 0;
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            float a = 0.0f;
#pragma unroll
            for (int e = 0; e < CT; ++e) a = a + fabsf(x[s][e]);
            a = block_sum<4>(a);                            // over the wavefront's 4 CT columns
            __builtin_amdgcn_sched_barrier(0);
            if ((t.lane & 3) == 0) L.sum[OWN ? t.wave * DK + s * 16 + t.tr : (s * 16 + t.tr) * GGA_WAVES + t.wave] = a;
        }
        if constexpr (OWN) {
            wave_sync();
#pragma unroll
            for (int i = t.lane; i < DK; i += WAVE) {
                const float4 f = gga_row_factor(L.sum[t.wave * DK + i] * (1.0f / float(COLS)), w[i]);
                L.row[grp][i] = f;
                R[i * T::NG + grp] = f32_to_f16(f.x);
            }
            wave_sync();
        } else {
            constexpr int GROUPS = B == 2 ? T::NG : 1;
            static_assert(GROUPS * DK <= GGA_THREADS, "a thread per row factor");
            __syncthreads();
            if (t.tid < GROUPS * DK) {
                const int i = t.tid % DK, g = t.tid / DK;
                const float4 w4 = *reinterpret_cast<const float4*>(L.sum + i * GGA_WAVES);
                float a = (w4.x + w4.y) + (w4.z + w4.w);
                if constexpr (B == 2) a = g == 0 ? w4.x + w4.y : w4.z + w4.w;         // d_v = 64: two wavefronts
                const float4 f = gga_row_factor(a * (1.0f / float(COLS)), w[i]);
                L.row[g][i] = f;
                R[B == 2 ? i * T::NG + g : i] = f32_to_f16(f.x);
            }
            __syncthreads();
        }
        // ---- the columns' first factors, from the quotients y by the row factors ----
        // max_i (|y| / qmax) = (max_i |y|) / qmax: division is monotonic
        auto factor = [&](float m) { return gga_half(gga_div(m, QMAX, 1.0f / QMAX)); };
        float c[CO];
        bool exactly;                                       // infinities among the values: every quotient by division
        {
            float cmax[1][CT], cm[1][CO];
#pragma unroll
            for (int e = 0; e < CT; ++e) cmax[0][e] = 0.0f;
#pragma unroll
            for (int s = 0; s < RPT; s += 2) {
                const float rc0 = L.row[grp][s * 16 + t.tr].y, rc1 = L.row[grp][(s + 1) * 16 + t.tr].y;
#pragma unroll
                for (int e = 0; e < CT; ++e)
                    cmax[0][e] = fmaxf(fmaxf(cmax[0][e], fabsf(x[s][e] * rc0)), fabsf(x[s + 1][e] * rc1));
                __builtin_amdgcn_sched_barrier(0);
            }
            gga_col_reduce<T, 1, true>(cmax, cm);
            bool sure = true, tame = true;
#pragma unroll
            for (int e = 0; e < CO; ++e) {
                c[e] = factor(cm[0][e] * GGA_ABOVE);
                sure = sure && c[e] == factor(cm[0][e] * GGA_BELOW);
                tame = tame && cm[0][e] < GGA_FAST_MAX;
            }
            exactly = __builtin_amdgcn_ballot_w64(!tame) != 0;
            if (__builtin_expect(exactly || __builtin_amdgcn_ballot_w64(!sure) != 0, 0)) {
#pragma unroll
                for (int e = 0; e < CT; ++e) cmax[0][e] = 0.0f;
#pragma unroll
                for (int s = 0; s < RPT; ++s) {
                    float2 f = *reinterpret_cast<const float2*>(&L.row[grp][s * 16 + t.tr]);
                    asm volatile("" : "+v"(f.y));
#pragma unroll
                    for (int e = 0; e < CT; ++e) cmax[0][e] = fmaxf(cmax[0][e], fabsf(gga_div(x[s][e], f.x, f.y)));
                    __builtin_amdgcn_sched_barrier(0);
                }
                gga_col_reduce<T, 1, true>(cmax, cm);
#pragma unroll
                for (int e = 0; e < CO; ++e) c[e] = factor(cm[0][e]);
            }
        }
        // what a code is formed with, per column: the reciprocal of its factor, a margin up and down; two bits: twice the
        // factor
        float k[B == 2 ? CT : 1], above[B == 2 ? 1 : CT], below[B == 2 ? 1 : CT];
        auto against = [&]() {
            float f[CO];
            if constexpr (B == 2) {
#pragma unroll
                for (int e = 0; e < CO; ++e) f[e] = 2.0f * c[e];
                gga_col_gather<T>(f, k);
            } else {
                float rc[CT];
#pragma unroll
                for (int e = 0; e < CO; ++e) f[e] = gga_rcp_f16(c[e]);
                gga_col_gather<T>(f, rc);
#pragma unroll
                for (int e = 0; e < CT; ++e) {
                    above[e] = rc[e] * GGA_ABOVE;
                    below[e] = rc[e] * GGA_BELOW;
                }
            }
        };
        // rint(y / c), clamped, as GGA_MAGIC + z, of the row step's values in a row of factors {r, 1 / r}
        auto codes = [&](const float (&v)[CT], const float4& f, float (&z)[CT]) {
            float fy = f.y;
            asm volatile("" : "+v"(fy));                    // products of an earlier pass over the tile are formed again, not kept
            uint32_t differ = 0;
#pragma unroll
            for (int e = 0; e < CT; ++e) {
                const float y = v[e] * fy;
                const float up = __builtin_fmaf(y, above[e], GGA_MAGIC), down = __builtin_fmaf(y, below[e], GGA_MAGIC);
                differ |= as_u32(up) ^ as_u32(down);
                z[e] = __builtin_amdgcn_fmed3f(up, GGA_MAGIC - QMAX, GGA_MAGIC + QMAX);
            }
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(differ != 0 || exactly) != 0, 0)) {
                float g[CO], cc[CT], rc[CT];
                asm volatile("" : "+v"(fy));
#pragma unroll
                for (int e = 0; e < CO; ++e) g[e] = gga_rcp_f16(c[e]);
                gga_col_gather<T>(c, cc);
                gga_col_gather<T>(g, rc);
#pragma unroll
                for (int e = 0; e < CT; ++e)
                    z[e] = __builtin_amdgcn_fmed3f(gga_div(gga_div(v[e], f.x, fy), cc[e], rc[e]) + GGA_MAGIC,
                                                   GGA_MAGIC - QMAX, GGA_MAGIC + QMAX);
            }
        };
        // two bits: |z| is 3 where y / c >= 2, which -- rounded quotients or not -- is exactly where |x| >= r 2 c: the
        // product of two fp16 numbers is exact, and the next float below it is further off than the quotients' rounding
        auto big = [&](float v, const float4& f, int e) { return fabsf(v) >= f.x * k[e]; };
        against();
        // ---- codes, and the least-squares column factors for them ----
        float nd[2][CT], so[2][CO];
#pragma unroll
        for (int e = 0; e < CT; ++e) nd[0][e] = nd[1][e] = 0.0f;
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const float4 f = L.row[grp][s * 16 + t.tr];
            float z[CT];
            if constexpr (B != 2) codes(x[s], f, z);
            const float off = -GGA_MAGIC * f.x;             // exact, and so is r z = r (MAGIC + z) - r MAGIC
#pragma unroll
            for (int e = 0; e < CT; ++e) {
                float vv;
                if constexpr (B == 2) {
                    const float mag = big(x[s][e], f, e) ? 3.0f : 1.0f;
                    vv = f.x * (x[s][e] >= 0.0f ? mag : -mag);
                } else {
                    vv = __builtin_fmaf(f.x, z[e], off);
                }
                nd[0][e] = __builtin_fmaf(f.z * vv, x[s][e], nd[0][e]);
                nd[1][e] = __builtin_fmaf(f.z, vv * vv, nd[1][e]);
                asm volatile("" : "+v"(nd[0][e]), "+v"(nd[1][e]));      // (here, not behind the last row step's branch)
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        gga_col_reduce<T, 2, false>(nd, so);
#pragma unroll
        for (int e = 0; e < CO; ++e)
            c[e] = gga_half(so[1][e] > 0.0f ? so[0][e] / fmaxf(so[1][e], 1e-30f) : c[e]);
        against();
        // ---- codes again, packed: u = z + qmax (two bits: (z + 3) / 2) ----
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            constexpr int WB = B == 6 ? 4 : 32 / B;         // codes per word (six bits: 24 of its bits)
            constexpr int WORDS = (CT + WB - 1) / WB;
            const float4 f = L.row[grp][s * 16 + t.tr];
            float z[CT];
            if constexpr (B != 2) codes(x[s], f, z);
            uint64_t bits = 0;
#pragma unroll
            for (int d = WORDS - 1; d >= 0; --d) {
                uint32_t acc = 0, magic = 0;
#pragma unroll
                for (int j = WB - 1; j >= 0; --j) {
                    const int e = d * WB + j;
                    if (e >= CT) continue;
                    uint32_t u;
                    if constexpr (B == 2) {
                        const bool b3 = big(x[s][e], f, e);
                        u = x[s][e] >= 0.0f ? (b3 ? 3u : 2u) : (b3 ? 0u : 1u);
                    } else {                                // z on top of constant bits, which add up to a constant
                        u = as_u32(z[e]);
                        magic = (magic << B) + (0x4B400000u - uint32_t(gga_qmax(B)));
                    }
                    acc = (acc << B) + u;
                }
                bits = (bits << (B * WB % 64)) | uint64_t(acc - magic);
            }
            gga_store_bytes<NB>(S + (s * 16 + t.tr) * RB + t.tc * NB, bits);
            __builtin_amdgcn_sched_barrier(0);
        }
        if ((t.lane & 12) == 0) {                           // one of the four lanes that keep these columns
            uint16_t* at = C + t.tc * CT + t.own * CO;
            if constexpr (CO == 2) *reinterpret_cast<uint32_t*>(at) = uint32_t(f32_to_f16(c[0])) | (uint32_t(f32_to_f16(c[1])) << 16);
            else *at = f32_to_f16(c[0]);
        }
    }
}

template <class T, class F>
__device__ __forceinline__ void gga_load_any(const uint8_t* S, int bits, const GgaThread& t, float (&x)[T::RPT][T::CT],
                                             F&& between) {
    if (bits == 16) gga_load_head<T, 16>(S, t, x, between);
    else if (bits == 8) gga_load_head<T, 8>(S, t, x, between);
    else if (bits == 6) gga_load_head<T, 6>(S, t, x, between);
    else if (bits == 4) gga_load_head<T, 4>(S, t, x, between);
    else gga_load_head<T, 2>(S, t, x, between);
}
template <class T>
__device__ __forceinline__ void gga_store_any(uint8_t* S, int bits, float (&x)[T::RPT][T::CT], const float* w,
                                              GgaFitLds<T>& L) {
    const GgaThread t = gga_thread();
    if (bits == 16) gga_fit_store<T, 16>(S, x, w, L, t);
    else if (bits == 8) gga_fit_store<T, 8>(S, x, w, L, t);
    else if (bits == 6) gga_fit_store<T, 6>(S, x, w, L, t);
    else if (bits == 4) gga_fit_store<T, 4>(S, x, w, L, t);
    else gga_fit_store<T, 2>(S, x, w, L, t);
}

// ---------------------------------------------------------------------------------------------------------------
// FP8 (E4M3, finite, no infinities) vectors, one wavefront per vector, N elements per lane (reference: `_fp8_enc`,
// _gga_triton.py:182-190; torch's cast rounds to nearest even, and so does the hardware conversion)
// ---------------------------------------------------------------------------------------------------------------
__device__ __forceinline__ float fp8_to_f32(uint32_t byte) { return __builtin_amdgcn_cvt_f32_fp8(int(byte), 0); }
__device__ __forceinline__ uint32_t f32_to_fp8(float y) {
    return uint32_t(__builtin_amdgcn_cvt_pk_fp8_f32(y, 0.0f, 0, false)) & 0xFFu;
}
// codes, scale s = amax / 448 and the reconstruction of x (0 -> 0)
template <int N>
__device__ __forceinline__ float fp8_encode(const float (&x)[N], uint32_t (&code)[N], float (&rec)[N]) {
    float am = 0.0f;
#pragma unroll
    for (int t = 0; t < N; ++t) am = fmaxf(am, fabsf(x[t]));
    const float s = wave_max(am) / 448.0f;
    const float safe = s > 0.0f ? s : 1.0f;
#pragma unroll
    for (int t = 0; t < N; ++t) {
        code[t] = f32_to_fp8(fminf(fmaxf(x[t] / safe, -448.0f), 448.0f));
        rec[t] = s > 0.0f ? fp8_to_f32(code[t]) * safe : 0.0f;
    }
    return s;
}
template <int N>
__device__ __forceinline__ void fp8_store(uint8_t* p, int lane, const uint32_t (&code)[N]) {
    if constexpr (N == 2) reinterpret_cast<uint16_t*>(p)[lane] = uint16_t(code[0] | (code[1] << 8));
    else p[lane] = uint8_t(code[0]);
}
template <int N>
__device__ __forceinline__ void fp8_load(const uint8_t* p, int lane, uint32_t (&code)[N]) {
    if constexpr (N == 2) {
        const uint32_t v = reinterpret_cast<const uint16_t*>(p)[lane];
        code[0] = v & 0xFFu;
        code[1] = v >> 8;
    } else {
        code[0] = p[lane];
    }
}

// ---------------------------------------------------------------------------------------------------------------
// the decode step
// ---------------------------------------------------------------------------------------------------------------
template <class T>
struct GgaLds {
    float2 kq[T::DK];                             // k, q normalised
    float r0[T::DK];                              // left factor of the write that enters the state
    float coef[GGA_MMAX];
    GgaFitLds<T> fit;
};

// Four wavefronts per SIMD (128 registers, some spilled): the launch of 32 sequences x 32 heads of 128 x 128 then runs in
// one round of workgroups.  us per launch there, mixed widths: 44.0 with values and quotients side by side (225 registers,
// two wavefronts per SIMD) -> 34.6 at three -> 32.4 at four.  In one round every workgroup loads, computes and stores at
// the same time as all others, so what stands in front of the first value and behind the last one is paid in full: with
// the serving case's types compiled in (SPEC, as in the other families; some 200 branches on them were in the way), the
// leading arguments in registers, the state requested ahead of the counters and of the window that waits for them, the
// new pair queued ahead of the fit and the counters advanced in the same launch (a ticket, below) a layer takes 30.2 us
// where the step and a launch for the counters took 33.7 (with the fit's products, GGA_ABOVE, and today's compiler flags 27.7; one
// sequence 13.9).  SPEC 0, any token and gate type: 28.4 and 15.0 with fp32 tokens.
template <class T, int SPEC>
__global__ __launch_bounds__(GGA_THREADS, 4)
void gga_step_kernel(const int32_t* __restrict__ idx, const int32_t* __restrict__ offs, const int32_t* __restrict__ widths,
                     uint8_t* blob, uint64_t slot_stride, uint32_t rows, uint32_t head0, const GgaParams p0) {
    // (the leading arguments, copies of fields of the block, are in registers when a wavefront starts)
    GgaParams p = p0;
    assume_serving_case<SPEC>(p);
    constexpr int CT = T::CT, CO = T::CO, RPT = T::RPT, DK = T::DK, DV = T::DV, NE = T::NE, NV = T::NV;
    __shared__ __attribute__((aligned(16))) GgaLds<T> L;
    const GgaThread t = gga_thread();
    // head-major order: workgroups that run together work on the same head, hence on the same width, and share the
    // instructions of one of the five width paths (each path is ~40 KB of straight-line code)
    const uint32_t h = head0 + blockIdx.y, b = blockIdx.x;
    const uint32_t bh = b * uint32_t(p.hv) + h;
    const uint32_t hk = p.gqa_shift >= 0 ? h >> p.gqa_shift : h / uint32_t(p.gqa);
    const int32_t seq = idx[b];
    const int bits = widths[h];
    const int32_t off = offs[h];
    void* const outp = advance(p.out, p.out_dt, uint64_t(bh) * DV);
    if (seq <= 0) {
        if (t.tid < DV) store_f(outp, p.out_dt, t.tid, 0.0f);
        return;
    }
    uint8_t* const base = blob + uint64_t(seq) * slot_stride;
    uint8_t* const S = base + off;
    const bool window = p.pw && bits != 16;
    const int m = p.m;
    uint8_t* const qb = base + p.qoff + uint64_t(h) * p.qsz;
    uint8_t* const PP = qb;
    uint8_t* const VP = qb + m * DK;
    float* const PS = reinterpret_cast<float*>(qb + m * (DK + DV));
    float* const VS = PS + m;
    // the slot's counters: scalar loads (left to the compiler, vector loads: the same words are written further down)
    const auto* const ct = (const __attribute__((address_space(4))) int32_t*)(base);
    int n = ct[0], hd = ct[1];

    // ---- q, k of the key head (every wavefront on its own: lane l holds elements l NE .. l NE + NE - 1), gates ----
    const void* qp = advance(p.q, p.q_dt, uint64_t(b) * p.s_q + hk * DK);
    const void* kp = advance(p.k, p.k_dt, uint64_t(b) * p.s_k + hk * DK);
    uint32_t qr[NE], kr[NE];
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        qr[e] = load_raw(qp, p.q_dt, t.lane * NE + e);
        kr[e] = load_raw(kp, p.k_dt, t.lane * NE + e);
    }
    const uint32_t ar = load_raw_uniform(p.a, p.a_dt, uint64_t(b) * p.s_a + h);
    const uint32_t btr = load_raw_uniform(p.bt, p.bt_dt, uint64_t(b) * p.s_bt + h);
    const uint32_t alr = load_raw_uniform(p.A_log, p.A_log_dt, h);
    const uint32_t dbr = load_raw_uniform(p.dt_bias, p.dt_bias_dt, h);
    // the lane's kept columns of v and of the queued right factors (for the output), and all its columns of the write
    // that enters the state: the oldest pair of a full window, v itself without a window
    const void* vp = advance(p.v, p.v_dt, uint64_t(b) * p.s_v + h * DV);
    const int c0 = t.tc * CT, oc = c0 + t.own * CO;
    uint32_t vo[CO], v0q[CT / 4];
#pragma unroll
    for (int e = 0; e < CO; ++e) vo[e] = load_raw(vp, p.v_dt, oc + e);
    uint32_t vq[GGA_MMAX];
    float vsl = 0.0f;                                   // lane oi: the scale of the oi-th oldest right factor
    float x[RPT][CT];
    // the state goes out ahead of the window, whose addresses wait for the counters
    gga_load_any<T>(S, bits, t, x, [&] {
        asm volatile("" : "+s"(n), "+s"(hd) :: "memory");           // read here, never again: see the ticket below
        n = n < 0 ? 0 : n > m ? m : n;
        hd &= GGA_RING;                                              // (the ticket above it may be counting already)
        hd = hd >= m ? m - 1 : hd;
        if (!window) n = hd = 0;
        if (window) {
            if (t.lane < n) vsl = VS[hd + t.lane < m ? hd + t.lane : hd + t.lane - m];
#pragma unroll
            for (int oi = 0; oi < GGA_MMAX; ++oi) {      // entries beyond the queue: any of the ring, not used below
                int jj = hd + oi < m ? hd + oi : hd + oi - m;
                jj = jj < m ? jj : 0;
                if constexpr (CO == 2) vq[oi] = *reinterpret_cast<const uint16_t*>(VP + jj * DV + oc);
                else vq[oi] = VP[jj * DV + oc];
            }
            if (n == m) {
#pragma unroll
                for (int w4 = 0; w4 < CT / 4; ++w4) v0q[w4] = reinterpret_cast<const uint32_t*>(VP + hd * DV + c0)[w4];
            }
        }
    });
    const bool full = window && n == m, enters = full || !window;

    float qe[NE], ke[NE], ssq = 0.0f, ssk = 0.0f;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        qe[e] = raw_to_f(qr[e], p.q_dt);
        ke[e] = raw_to_f(kr[e], p.k_dt);
        ssq = __builtin_fmaf(qe[e], qe[e], ssq);
        ssk = __builtin_fmaf(ke[e], ke[e], ssk);
    }
    const float nq = sqrtf(wave_sum(ssq) + 1e-6f);
    const float nk = sqrtf(wave_sum(ssk) + 1e-6f);
    float a, beta;
    if (p.gate) {
        const float xg = raw_to_f(ar, p.a_dt) + raw_to_f(dbr, p.dt_bias_dt);
        const float sp = xg <= 20.0f ? logf(1.0f + expf(xg)) : xg;
        a = expf(-expf(raw_to_f(alr, p.A_log_dt)) * sp);
        beta = 1.0f / (1.0f + expf(-raw_to_f(btr, p.bt_dt)));
    } else {
        a = expf(raw_to_f(ar, p.a_dt));
        beta = raw_to_f(btr, p.bt_dt);
    }
    float bke[NE], bkq = 0.0f;
#pragma unroll
    for (int e = 0; e < NE; ++e) {
        qe[e] = qe[e] / nq * p.scale;
        ke[e] = ke[e] / nk;
        bke[e] = beta * ke[e];
        bkq = bkq + bke[e] * qe[e];
    }
    bkq = wave_sum(bkq);
    if (t.wave == 0) {
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            L.kq[t.lane * NE + e] = make_float2(ke[e], qe[e]);
            if (!window) L.r0[t.lane * NE + e] = bke[e];
        }
    }

    // ---- the queued left factors: propagate, re-encode, read out (wavefront w: entries w, w + 4) ----
    if (window) {
        for (int oi = t.wave; oi < n; oi += GGA_WAVES) {
            const int jj = hd + oi < m ? hd + oi : hd + oi - m;
            uint32_t code[NE];
            fp8_load<NE>(PP + jj * DK, t.lane, code);
            const float ps = PS[jj];
            float pv[NE], kpp = 0.0f;
#pragma unroll
            for (int e = 0; e < NE; ++e) {
                pv[e] = fp8_to_f32(code[e]) * ps;
                kpp = kpp + ke[e] * pv[e];
            }
            kpp = wave_sum(kpp);
            float ap[NE], rec[NE];
#pragma unroll
            for (int e = 0; e < NE; ++e) ap[e] = a * (pv[e] - bke[e] * kpp);
            const float sc = fp8_encode<NE>(ap, code, rec);
            if (!(full && oi == 0)) {                      // the oldest pair of a full window leaves it below
                fp8_store<NE>(PP + jj * DK, t.lane, code);
                if (t.lane == 0) PS[jj] = sc;
            }
            float cf = 0.0f;
#pragma unroll
            for (int e = 0; e < NE; ++e) cf = cf + rec[e] * qe[e];
            cf = wave_sum(cf);
            if (t.lane == 0) L.coef[oi] = cf;
            if (oi == 0) {
#pragma unroll
                for (int e = 0; e < NE; ++e) L.r0[t.lane * NE + e] = rec[e];
            }
        }
    }
    __syncthreads();
    // ---- a ticket for the slot's counters: every head of the slot reads them, the last one to have done so advances them.
    // The tickets are counted above the ring index (whose value is below 16; zero between steps), so the slot's bytes are
    // what a launch of its own behind every step left there.  This head's reads have returned (their values are in
    // registers) before its ticket goes out, so no head reads what the last one writes; the writes are seen by the next
    // launch.
    uint32_t ticket = 0;
    if (p.pw && t.tid == 0)
        ticket = __hip_atomic_fetch_add(reinterpret_cast<uint32_t*>(base) + 1, GGA_TICKET, __ATOMIC_RELAXED,
                                        __HIP_MEMORY_SCOPE_AGENT);

    // ---- k^T O and q^T O; the output: q^T O_pre = a (q^T O - (beta k . q) k^T O), the queued pairs oldest first, and
    //      this token's write -- for the lane's kept columns ----
    float kO[CT], krow[RPT];
    {
        float acc[2][CT], own[2][CO], o[CO];
#pragma unroll
        for (int e = 0; e < CT; ++e) acc[0][e] = acc[1][e] = 0.0f;
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const float2 kq = L.kq[s * 16 + t.tr];
            krow[s] = kq.x;
#pragma unroll
            for (int e = 0; e < CT; ++e) {
                acc[0][e] = __builtin_fmaf(kq.x, x[s][e], acc[0][e]);
                acc[1][e] = __builtin_fmaf(kq.y, x[s][e], acc[1][e]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        gga_col_reduce<T, 2, false>(acc, own);
        gga_col_gather<T>(own[0], kO);
#pragma unroll
        for (int e = 0; e < CO; ++e) {
            o[e] = a * __builtin_fmaf(-bkq, own[0][e], own[1][e]);
            o[e] = o[e] + bkq * raw_to_f(vo[e], p.v_dt);
        }
        if (window) {
            const float cfl = t.lane < n ? L.coef[t.lane] * vsl : 0.0f;
#pragma unroll
            for (int oi = 0; oi < GGA_MMAX; ++oi) {
                if (oi < n) {
                    const float cf = lane_bcast(cfl, oi);
#pragma unroll
                    for (int e = 0; e < CO; ++e) o[e] = __builtin_fmaf(cf, fp8_to_f32((vq[oi] >> (8 * e)) & 0xFFu), o[e]);
                }
            }
        }
        if ((t.lane & 12) == 0) {                          // one of the four lanes that keep these columns
#pragma unroll
            for (int e = 0; e < CO; ++e) store_f(outp, p.out_dt, oc + e, o[e]);
        }
    }

    // ---- O_pre = a (O - beta k (k^T O)), and the write that enters the state: the pair that leaves a full window;
    //      pivots and slots without a window take the new one ----
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
        const float bk = beta * krow[s];
#pragma unroll
        for (int e = 0; e < CT; ++e) x[s][e] = a * __builtin_fmaf(-bk, kO[e], x[s][e]);
    }
    if (enters) {
        float v0[CT];
        if (full) {
            const float s0 = lane_bcast(vsl, 0);
#pragma unroll
            for (int e = 0; e < CT; ++e) v0[e] = fp8_to_f32((v0q[e / 4] >> (8 * (e % 4))) & 0xFFu) * s0;
        } else {
#pragma unroll
            for (int e = 0; e < CT; ++e) v0[e] = raw_to_f(load_raw(vp, p.v_dt, c0 + e), p.v_dt);
        }
#pragma unroll
        for (int s = 0; s < RPT; ++s) {
            const float r0 = L.r0[s * 16 + t.tr];
#pragma unroll
            for (int e = 0; e < CT; ++e) x[s][e] = __builtin_fmaf(r0, v0[e], x[s][e]);
        }
    }

    // ---- queue (R(beta k), R(v)).  A full window's new pair replaces the oldest one, whose right factor every
    // wavefront has read for the merge: the barrier puts the store behind all of those reads (each wavefront used its
    // copy before it got here).
    if (window) {
        __syncthreads();
        const int jn = n == m ? hd : hd + n < m ? hd + n : hd + n - m;
        if (t.wave == 0) {
            uint32_t code[NE];
            float rec[NE];
            const float sc = fp8_encode<NE>(bke, code, rec);
            fp8_store<NE>(PP + jn * DK, t.lane, code);
            if (t.lane == 0) PS[jn] = sc;
        } else if (t.wave == 1) {
            float vv[NV];
#pragma unroll
            for (int e = 0; e < NV; ++e) vv[e] = raw_to_f(load_raw(vp, p.v_dt, t.lane * NV + e), p.v_dt);
            uint32_t code[NV];
            float rec[NV];
            const float sc = fp8_encode<NV>(vv, code, rec);
            fp8_store<NV>(VP + jn * DV, t.lane, code);
            if (t.lane == 0) VS[jn] = sc;
        }
    }

    // ---- re-fit and re-pack in place ----
    gga_store_any<T>(S, bits, x, p.w + h * DK, L.fit);

    // ---- the last head's: the counters of the slot, advanced (reference `_gga_advance`).  The last one is the last of all
    // rows that name the slot; who could be it counts them, in the tail of one workgroup a slot, the counter requested with
    // the indices (against no count at all, 32 sequences 27.87 -> 27.99 us, 6: 15.24 -> 15.40; the counter behind the indices
    // 28.04; the indices requested by everybody ahead of the fit 27.96 and 15.36, but 16 sequences with g and beta given
    // 18.57 -> 18.97 instead of 18.62).  A launch that names a slot twice steps its state in no order that could be relied
    // on, but the counters advance once, and no ticket is left for the next step. ----
    if (p.pw && t.tid < WAVE) {
        const uint32_t drawn = uint32_t(__builtin_amdgcn_readfirstlane(int(ticket))) / GGA_TICKET + 1;
        if (drawn >= uint32_t(p.hv)) {
            int32_t* const ct = reinterpret_cast<int32_t*>(base);
            const int n0 = ct[0];
            uint32_t named = rows == 1;
            for (uint32_t r = 0; rows > 1 && r < rows; r += WAVE)
                named += __builtin_popcountll(__builtin_amdgcn_ballot_w64(r + t.tid < rows && idx[min(r + t.tid, rows - 1)] == seq));
            if (t.tid == 0 && drawn == named * uint32_t(p.hv)) {
                const int hd0 = int(ticket & GGA_RING);
                ct[0] = n0 + 1 < m ? n0 + 1 : m;
                __hip_atomic_store(ct + 1, n0 == m ? (hd0 + 1) % m : hd0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

// Fit + pack canonical states X [rows, hv, d_k, d_v] fp32 into slots idx; zero the counters (reference `_gga_store`).
template <class T>
__global__ __launch_bounds__(GGA_THREADS, 2) void gga_store_kernel(const GgaParams p) {
    constexpr int CT = T::CT, RPT = T::RPT, DK = T::DK, DV = T::DV;
    __shared__ __attribute__((aligned(16))) GgaFitLds<T> L;
    const GgaThread t = gga_thread();
    // head-major order: workgroups that run together work on the same head, hence on the same width, and share the
    // instructions of one of the five width paths (each path is ~40 KB of straight-line code)
    const uint32_t h = blockIdx.x / uint32_t(p.rows), b = blockIdx.x - h * uint32_t(p.rows);
    const uint32_t bh = b * uint32_t(p.hv) + h;
    const int32_t seq = p.idx[b];
    if (seq <= 0) return;
    uint8_t* const base = p.blob + uint64_t(seq) * p.slot_stride;
    const float* X = p.X + uint64_t(bh) * (DK * DV);
    float x[RPT][CT];
#pragma unroll
    for (int s = 0; s < RPT; ++s) {
        const int i = s * 16 + t.tr;
#pragma unroll
        for (int e4 = 0; e4 < CT; e4 += 4) {
            const float4 v = *reinterpret_cast<const float4*>(X + i * DV + t.tc * CT + e4);
            x[s][e4] = v.x; x[s][e4 + 1] = v.y; x[s][e4 + 2] = v.z; x[s][e4 + 3] = v.w;
        }
    }
    gga_store_any<T>(base + p.offs[h], p.bits[h], x, p.w + h * DK, L);
    if (h == 0 && t.tid < 2) reinterpret_cast<int32_t*>(base)[t.tid] = 0;
}

// Unpack slots idx into canonical fp32 Y [rows, hv, d_k, d_v]: the stored state without the window (`_gga_load`).
template <class T>
__global__ __launch_bounds__(GGA_THREADS, 2) void gga_load_kernel(const GgaParams p) {
    constexpr int CT = T::CT, RPT = T::RPT, DK = T::DK, DV = T::DV;
    const GgaThread t = gga_thread();
    // head-major order: workgroups that run together work on the same head, hence on the same width, and share the
    // instructions of one of the five width paths (each path is ~40 KB of straight-line code)
    const uint32_t h = blockIdx.x / uint32_t(p.rows), b = blockIdx.x - h * uint32_t(p.rows);
    const uint32_t bh = b * uint32_t(p.hv) + h;
    const int32_t seq = p.idx[b];
    float* Y = p.Y + uint64_t(bh) * (DK * DV);
    float x[RPT][CT];
    if (seq > 0) {
        gga_load_any<T>(p.blob + uint64_t(seq) * p.slot_stride + p.offs[h], p.bits[h], t, x, [] {});
    } else {
#pragma unroll
        for (int s = 0; s < RPT; ++s)
#pragma unroll
            for (int e = 0; e < CT; ++e) x[s][e] = 0.0f;
    }
#pragma unroll
    for (int s = 0; s < RPT; ++s)
#pragma unroll
        for (int e4 = 0; e4 < CT; e4 += 4)
            *reinterpret_cast<float4*>(Y + (s * 16 + t.tr) * DV + t.tc * CT + e4) =
                make_float4(x[s][e4], x[s][e4 + 1], x[s][e4 + 2], x[s][e4 + 3]);
}

// op: 0 step, 1 store, 2 load
template <class T>
int launch_gga(const GgaParams& p, int op, hipStream_t stream) {
    const dim3 grid(p.rows * p.hv), block(GGA_THREADS);
    if (op == 0) {
        const int spec = serving_case(p);
        for (int h0 = 0; h0 < p.hv; h0 += GGA_GRID_Y) {                   // (one launch but for 65 536 heads and more)
            const dim3 tiles(p.rows, p.hv - h0 < GGA_GRID_Y ? p.hv - h0 : GGA_GRID_Y);
#define SQ_GGA_STEP(SPEC)                                                                                                \
            hipLaunchKernelGGL((gga_step_kernel<T, SPEC>), tiles, block, 0, stream, p.idx, p.offs, p.bits, p.blob,       \
                               p.slot_stride, uint32_t(p.rows), uint32_t(h0), p)
            if (spec == 2) SQ_GGA_STEP(2);
            else if (spec == 1) SQ_GGA_STEP(1);
            else SQ_GGA_STEP(0);
#undef SQ_GGA_STEP
        }
    } else if (op == 1) {
        hipLaunchKernelGGL(gga_store_kernel<T>, grid, block, 0, stream, p);
    } else {
        hipLaunchKernelGGL(gga_load_kernel<T>, grid, block, 0, stream, p);
    }
    return int(hipGetLastError());
}

}  // namespace sq
