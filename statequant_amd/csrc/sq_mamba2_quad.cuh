// Mamba2 / SSD packed decode step, one workgroup per (batch row, GH heads of one B / C group): the heads share C
// (the read-out vector, its digit planes), B (this token's key, its rounded copy for the buffer) and every product
// with the buffered keys; every wavefront owns NB 32-row blocks of one head's state (int4 / int8 codes with key-axis or
// 32-row value-axis groups, or bf16; geometry and building blocks in sq_quad.cuh).
//
// Same arithmetic per head as the one-wavefront kernel of sq_mamba2.cuh (the reference's `_m2_step`,
// /root/reference/src/statequant/kernels/_mamba2_triton.py:48-197):
//   u_n = dt x_n,  y_n = a_n [alpha S0 C + sum_{i<n} (alpha / alpha_i) (B_i . C) u_i] + (B_n . C) u_n + D x_n
//   fold (buffer full): S = alpha_m S0 + sum_i (alpha_m / alpha_i) u_i B_i^T, re-quantized out of LDS
// Division of labour inside the workgroup as in the Gated DeltaNet kernel (sq_gdn_quad.cuh): all loads first, one
// wavefront each for C and B, per head dt and the decays, then per wavefront the state pass, its share of the
// buffered keys, its rows' epilogue, append and fold.
#pragma once
#include "sq_gdn_quad.cuh"

namespace sq {

template <class T, class Q>
struct Mamba2Loads {
    uint16_t sc[Q::NB][T::NG];             // scales of rows (block bi, lane % 32)
    ColScales<T> scv[Q::NB];               // value-axis groups: the block's scales of the lane's columns
    Raw4<T::QBUF> uraw[Q::UT], kraw[Q::KT];
    uint16_t kbs[Q::KT], ubs;
    float gbl, gcur;
    int np;
    uint32_t xr[Q::NE], xr2[Q::NE], g0, g1, g2, g3, vr;
};

// SPEC > 0 compiles the serving case in (as in the Gated DeltaNet kernel): bf16 x / B / C / out, fp32 A, D and
// dt_bias (dt comes as fp32 or bf16: one scalar load); 1: head counts that are powers of two (128 heads 36.0 -> 33.9 us
// per launch against SPEC 0), 2: others.  SPEC = 0 reads all of it from the arguments.
template <class T, int NB, int GH, int WPE, int SPEC>
__global__ __launch_bounds__((Quad<T, NB, GH>::THREADS), WPE)
void mamba2_quad_kernel(const int32_t* __restrict__ idx, const int32_t* __restrict__ order, const uint8_t* codes,
                        const int32_t* counters, int per_xcd, int hv, int hv_shift, uint32_t codes_stride,
                        uint32_t counters_stride, uint32_t start_ramp, const Mamba2Params p) {
    constexpr bool FIX = SPEC > 0, POW2 = SPEC == 1;
    const int x_dt = FIX ? int(BF16) : p.x_dt, B_dt = FIX ? int(BF16) : p.B_dt, C_dt = FIX ? int(BF16) : p.C_dt;
    const int out_dt = FIX ? int(BF16) : p.out_dt, dt_dt = p.dt_dt, A_dt = FIX ? int(F32) : p.A_dt;
    const int D_dt = FIX ? int(F32) : p.D_dt, dt_bias_dt = FIX ? int(F32) : p.dt_bias_dt;
    using Q = Quad<T, NB, GH>;
    using L = QuadLds<T, NB, GH, 2, 1>;
    constexpr int DK = T::DK, DV = T::DV, NW = Q::NW, NWH = Q::NWH, MM = T::MMAX, NE = Q::NE, NG = T::NG, DKP = Q::DKP;
    constexpr int RQ = 1 % NW, RK = 3 % NW, RX = 2 % NW;          // which wavefront plays which shared role
    __shared__ __attribute__((aligned(16))) uint8_t lds[L::BYTES];
    uint8_t* lds_kbr = lds + L::KBR;
    float* lds_xn = reinterpret_cast<float*>(lds + L::XN);         // [0]: C, [1]: B
    uint8_t* lds_pl = lds + L::PL;
    float* lds_xs = reinterpret_cast<float*>(lds + L::XS);
    float* lds_dots = reinterpret_cast<float*>(lds + L::DOTS);
    float* lds_kbsf = reinterpret_cast<float*>(lds + L::KBSF);
    float* lds_red = reinterpret_cast<float*>(lds + L::RED);

    const int lane0 = threadIdx.x & (WAVE - 1);
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int hl = w / NWH, wh = w % NWH;                         // head of the group, wavefront of the head
    const int m = p.m;
    uint8_t* lds_ubr = lds + L::UBR + hl * (MM * DV * T::BE);     // this head's buffered values
    float* lds_ubsf = reinterpret_cast<float*>(lds + L::UBSF) + hl * MM;
    float* lds_scal = reinterpret_cast<float*>(lds + L::SCAL) + hl * 8;
    float* lds_gsc = reinterpret_cast<float*>(lds + L::SCAL) + GH * 8;   // the group's scalars (B . C)
    float* lds_gbf = reinterpret_cast<float*>(lds + L::GBF) + hl * MM;
    uint16_t* lds_sc = reinterpret_cast<uint16_t*>(lds + L::SC) + hl * (DV * NG);
    uint8_t* my_codes = lds + L::CODES + hl * Q::HEAD + wh * NB * Q::BLK;

    // ---- this workgroup's item: (batch row, head group), dealt so that every XCD walks a contiguous range ----
    const int ngrp = hv / GH;
    int b, grp, slot;
    {
        const int wg = blockIdx.x;
        const int item = per_xcd ? (wg & 7) * per_xcd + (wg >> 3) : wg;
        b = (POW2 || hv_shift >= 0) ? item >> (hv_shift - ilog2(GH)) : item / ngrp;
        grp = item - b * ngrp;
        if (order) b = order[b];                    // the caller's dispatch order: position -> batch row
        slot = idx ? idx[b] : b;
    }
    const uint32_t h = grp * GH + hl;
    const uint32_t hk = (POW2 || p.gqa_shift >= 0) ? h >> p.gqa_shift : h / uint32_t(p.gqa);

    const int lane = lane0;
    const int n32 = lane & 31, kb = lane >> 5;
    // the row of the head this lane finishes after the pass (NB = 2: the wavefront's halves take a block each)
    const int row_ = (wh * NB + (NB == 2 ? kb : 0)) * T::MR + n32;
    // d_v may end inside the last row block (80): its lanes beyond repeat the last row and keep the result to themselves
    const bool rlive = !T::RAGV || row_ < DV;
    const int row = rlive ? row_ : DV - 1;
    const int rows_left = DV - wh * NB * T::MR;                   // of this wavefront's blocks

    Mamba2Loads<T, Q> F;
    const int vl = Q::vec_lane(lane);                             // whose elements of a d_k vector this lane loads
    // ---- issue every load: first the token's own operands (their addresses need the batch row only; being older
    //      than the row blocks they are back before them) ...
    if constexpr (RQ == RK) {                                     // a single wavefront carries both vectors
        if (w == RQ) {
            load_vec<NE>(advance(p.C, C_dt, uint64_t(uint32_t(b)) * p.s_C + hk * DK), C_dt, vl, F.xr);
            load_vec<NE>(advance(p.B, B_dt, uint64_t(uint32_t(b)) * p.s_B + hk * DK), B_dt, vl, F.xr2);
        }
    } else if (w == RQ || w == RK) {
        const bool isq = w == RQ;
        const void* base = isq ? advance(p.C, C_dt, uint64_t(uint32_t(b)) * p.s_C + hk * DK)
                               : advance(p.B, B_dt, uint64_t(uint32_t(b)) * p.s_B + hk * DK);
        load_vec<NE>(base, isq ? C_dt : B_dt, vl, F.xr);
    }
    if (wh == 0) {
        F.g0 = load_raw_uniform(p.dt, dt_dt, uint64_t(uint32_t(b)) * p.s_dt + h);
        F.g1 = load_raw_uniform(p.A, A_dt, h);
        F.g2 = load_raw_uniform(p.dt_bias, dt_bias_dt, h);      // absent: the C ABI points them at A, so the loads
        F.g3 = load_raw_uniform(p.D, D_dt, h);                  // need no branch
    }
    F.vr = load_raw(advance(p.x, x_dt, uint64_t(uint32_t(b)) * p.s_x + h * DV), x_dt, uint32_t(row));
    void* const outp = advance(p.out, out_dt, uint64_t(uint32_t(b)) * p.s_out + h * DV);
    if (idx && slot <= 0) {                              // padding row: zero output, touch nothing else
        for (int r = wh * WAVE + lane; r < DV; r += NWH * WAVE) store_f(outp, out_dt, r, 0.0f);
        return;
    }
    // ... then the slot's big side, from the preloaded leading arguments alone: the row blocks, straight into their
    // LDS image, and the fill counter (a scalar load; sq_quad.cuh) behind them ...
    quad_start_wait<Q, WPE>(start_ramp);                  // the launch's first workgroups: spread over a ramp
    quad_dma_blocks<Q, NB, T::RAGV>(field(codes, uint32_t(slot), codes_stride, h * (DV * T::ROW_BYTES)) + wh * NB * Q::GBLK, my_codes, lane, rows_left);
    F.np = quad_dma_counter(field(counters, uint32_t(slot), counters_stride, h));
    __builtin_amdgcn_sched_barrier(0);
    // ... and the rest of the slot
    const uint32_t seq = slot, um = m;
    uint8_t* const Sh = field(p.st.S, seq, p.st.sS, h * (DV * T::ROW_BYTES));
    float* const gcp = field(p.st.GCUR, seq, p.st.sGC, h);
    int32_t* const np = field(p.st.NPTR, seq, p.st.sN, h);
    F.gcur = *gcp;
    uint16_t* const SCh = field(p.st.SC, seq, p.st.sSC, h * T::SC_ELEMS);
    uint8_t* const KBp = p.st.KB + (uint64_t(seq) * p.st.sKB + hk * um * DK) * T::BE;
    uint8_t* const UBp = p.st.UB + (uint64_t(seq) * p.st.sUB + h * um * DV) * T::BE;
    uint16_t* const KBSp = field(p.st.KBS, seq, p.st.sKBS, hk * um);
    uint16_t* const UBSp = field(p.st.UBS, seq, p.st.sUBS, h * um);
    float* const GBh = field(p.st.GB, seq, p.st.sGB, h * um);
#pragma unroll
    for (int bi = 0; bi < NB; ++bi) {
        if constexpr (T::AXV) {
            F.scv[bi].load(SCh + (wh * NB + bi) * DK, lane);
        } else if constexpr (!T::FLT) {
#pragma unroll
            for (int g = 0; g < NG; ++g) F.sc[bi][g] = stream_load(SCh + uint32_t((T::RAGV ? row : (wh * NB + bi) * T::MR + n32) * NG + g));
        }
    }
    // the buffer, live slots only (the others repeat the last live one: no new memory traffic); the fill count,
    // requested ahead of the row blocks, is here by now
    quad_dma_counter_wait(F.np);
    const uint32_t nfill = uint32_t(F.np & (m - 1));
    const uint32_t nl = nfill > 0 ? nfill : 1u;
    const int ucol = T::RAGV ? min(4 * (lane % Q::LU), rows_left - 4) : 4 * (lane % Q::LU);
    // buffered values of this wavefront's rows: lane (slot = lane / LU + SU t, rows 4 (lane % LU) ..)
#pragma unroll
    for (int t = 0; t < Q::UT; ++t) {
        const uint32_t i = lane / Q::LU + Q::SU * t;
        const uint32_t ic = i < nl ? i : nl - 1;
        F.uraw[t] = stream_raw4<T::QBUF>(UBp + (ic * DV + wh * Q::RW + ucol) * T::BE);
    }
    // buffered keys, dealt over the workgroup: lane (slot = SPP (NW t + w) + lane / LPS, columns 4 (lane % LPS) ..)
#pragma unroll
    for (int t = 0; t < Q::KT; ++t) {
        const uint32_t i = Q::SPP * (NW * t + w) + lane / Q::LPS;
        const uint32_t ic = i < nl ? i : nl - 1;
        F.kraw[t] = stream_raw4<T::QBUF>(KBp + (ic * DK + Q::key_col(lane)) * T::BE);
        F.kbs[t] = T::QBUF ? KBSp[ic] : uint16_t(0);
    }
    {   // per slot of this head, lane i: cumulative decay and value scale
        const uint32_t li = uint32_t(lane) < nl ? lane : 0;
        F.gbl = GBh[li];
        F.ubs = T::QBUF ? UBSp[li] : uint16_t(0);
    }
    // every load is in flight from here on: keep the compiler from sinking any of them to its use, and from
    // scheduling a use (a conversion, with its wait) up among them
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);

    // ---- shared roles: C (planes + fp32 copy), B (fp32 copy) ----
    auto role_vector = [&](uint32_t (&raw)[NE], int dt, int v) {
        float xe[NE];
        // (opened here: what both roles begin with the compiler has all wavefronts do, and wait for, first)
#pragma unroll
        for (int t = 0; t < NE; ++t) asm volatile("" : "+v"(raw[t]));
#pragma unroll
        for (int t = 0; t < NE; ++t) xe[t] = Q::vec_live(lane) ? vec_elem<NE>(raw, dt, t) : 0.0f;
        if constexpr (NE == 1) lds_xn[v * DKP + lane] = xe[0];
        else if constexpr (NE == 2) *reinterpret_cast<float2*>(lds_xn + v * DKP + 2 * lane) = make_float2(xe[0], xe[1]);
        else *reinterpret_cast<float4*>(lds_xn + v * DKP + 4 * lane) = make_float4(xe[0], xe[1], xe[2], xe[3]);
        if constexpr (!T::AXV && !T::FLT) {
            if (v == 0) quad_stage_planes<Q, T, NE>(xe, 0, lane, lds_pl, lds_xs);
        }
    };
    if constexpr (RQ == RK) {
        if (w == RQ) {
            role_vector(F.xr, C_dt, 0);
            role_vector(F.xr2, B_dt, 1);
        }
    } else {
        if (w == RQ) role_vector(F.xr, C_dt, 0);
        if (w == RK) role_vector(F.xr, B_dt, 1);
    }
    if (wh == 0) {                                       // this head's step size and decays
        float dt = raw_to_f(F.g0, dt_dt);
        if (p.has_dt_bias) dt = dt + raw_to_f(F.g2, dt_bias_dt);
        if (p.dt_softplus) dt = dt <= 20.0f ? logf(1.0f + expf(dt)) : dt;
        if (p.dt_clamp) dt = fminf(fmaxf(dt, p.dt_min), p.dt_max);
        const float g = raw_to_f(F.g1, A_dt) * dt;     // rounded on its own (no contraction into gcur + g)
        if (lane == 0) {
            lds_scal[0] = dt;
            lds_scal[1] = expf(F.gcur);
            lds_scal[2] = expf(g);
            lds_scal[3] = F.gcur + g;
            lds_scal[4] = p.has_D ? raw_to_f(F.g3, D_dt) : 0.0f;
        }
    }
    // ---- the loads land: LDS images of the row blocks, scales, raw buffer pieces ----
    const int n = F.np & (m - 1);
    const float gcur = F.gcur;
    const uint32_t vr = F.vr;
    uint16_t scw[NB][NG];
#pragma unroll
    for (int bi = 0; bi < NB; ++bi) {
        if constexpr (!T::AXV && !T::FLT) {
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                scw[bi][g] = F.sc[bi][g];
                if (kb == 0) lds_sc[(T::RAGV ? row : (wh * NB + bi) * T::MR + n32) * NG + g] = F.sc[bi][g];
            }
        }
    }
#pragma unroll
    for (int t = 0; t < Q::UT; ++t) {
        const int i = lane / Q::LU + Q::SU * t;
        if (Q::SU * Q::UT == MM || i < MM) store_raw4<T::QBUF>(lds_ubr + (i * DV + wh * Q::RW + ucol) * T::BE, F.uraw[t]);
    }
#pragma unroll
    for (int t = 0; t < Q::KT; ++t) {
        const int i = Q::SPP * (NW * t + w) + lane / Q::LPS;
        if (Q::SPP * NW * Q::KT == MM || i < MM) {
            store_raw4<T::QBUF>(lds_kbr + (i * DKP + 4 * (lane % Q::LPS)) * T::BE, F.kraw[t]);
            if (T::QBUF && lane % Q::LPS == 0) lds_kbsf[i] = f16_to_f32(F.kbs[t]);
        }
    }
    if (wh == 0 && lane < m) {
        lds_gbf[lane] = F.gbl;
        if constexpr (T::QBUF) lds_ubsf[lane] = f16_to_f32(F.ubs);
    }
    quad_dma_landed();                                             // the row blocks are in LDS
    const bool full = n == m - 1;
    lds_barrier();

    // ---- every wavefront: state pass over its row blocks (one read-out vector: the lanes of the upper half idle) ----
    float sq;                                            // (S0 C)[row], scales applied
    {
        float own[NB];
        if constexpr (T::AXV) {
#pragma unroll
            for (int bi = 0; bi < NB; ++bi)
                own[bi] = quad_block_pass_v<Q, T, 1>(my_codes + bi * Q::BLK, lds_xn, F.scv[bi], lds_pl + w * L::PL_BYTES,
                                                     lds_xs + w * (L::XS_BYTES / 4), lane);
        } else if constexpr (T::FLT) {
#pragma unroll
            for (int bi = 0; bi < NB; ++bi) own[bi] = quad_block_pass_f<Q, T, 1>(my_codes + bi * Q::BLK, lds_xn, lane);
        } else {
            v4i aop[Q::NKS];
            quad_fetch_planes<Q, T, 1>(lds_pl, lane, aop);
            float xs[NG];
#pragma unroll
            for (int g = 0; g < NG; ++g) xs[g] = lds_xs[g];
#pragma unroll
            for (int bi = 0; bi < NB; ++bi) {
                float sc[NG];
#pragma unroll
                for (int g = 0; g < NG; ++g) sc[g] = f16_to_f32(scw[bi][g]);
                own[bi] = quad_block_pass<Q, T>(my_codes + bi * Q::BLK, aop, xs, sc, lane);
            }
        }
        if constexpr (NB == 2) {                         // lane (n, kb) takes over row n of block kb
            const auto r = __builtin_amdgcn_permlane32_swap(as_u32(own[0]), as_u32(own[1]), false, false);
            sq = as_f32(r[0]);
        } else {
            sq = pair32(own[0]).lo;
        }
    }
    // ---- B_i . C of this wavefront's share of the slots ----
    {
        float x[4];
        {
            const float4 f = *reinterpret_cast<const float4*>(lds_xn + 4 * (lane % Q::LPS));
            x[0] = f.x; x[1] = f.y; x[2] = f.z; x[3] = f.w;
        }
#pragma unroll
        for (int t = 0; t < Q::KT; ++t) {
            const int i = Q::SPP * (NW * t + w) + lane / Q::LPS;
            const int ic = Q::SPP * NW * Q::KT == MM ? i : i < m ? i : m - 1;      // (a slot that does not exist: discarded)
            float kf[4];
            decode_raw4<T::QBUF>(load_raw4<T::QBUF>(lds_kbr + (ic * DKP + 4 * (lane % Q::LPS)) * T::BE), kf);
            if constexpr (T::QBUF) {
                const float s = lds_kbsf[ic];
#pragma unroll
                for (int c = 0; c < 4; ++c) kf[c] = kf[c] * s;
            }
            float pr = kf[0] * x[0];
#pragma unroll
            for (int c = 1; c < 4; ++c) pr = __builtin_fmaf(kf[c], x[c], pr);
            pr = lanes_sum<Q::LPS>(pr);
            if (lane % Q::LPS == 0 && i < MM) lds_dots[i] = pr;
        }
    }
    // ---- B . C ----
    if (w == RK) {
        float bcp = 0.0f;
#pragma unroll
        for (int t = 0; t < NE; ++t) bcp = __builtin_fmaf(lds_xn[DKP + NE * lane + t], lds_xn[NE * lane + t], bcp);
        bcp = lanes_sum<WAVE>(bcp);
        if (lane == 0) lds_gsc[0] = bcp;
    }
    // ---- the buffered key of this token: the rounded B, for this workgroup's folds and (first head group of the
    //      B / C group only) for the slot; whoever still reads slot n discards what it reads ----
    if (w == RX) {
        float kxe[NE], kmax = 0.0f;
#pragma unroll
        for (int t = 0; t < NE; ++t) {
            kxe[t] = lds_xn[DKP + NE * lane + t];
            kmax = fmaxf(kmax, fabsf(kxe[t]));
        }
        float ks = 1.0f;
        if constexpr (T::QBUF) ks = fp16_scale(lanes_max<WAVE>(kmax), 127.0f);
        const bool live = Q::vec_live(lane), write = live && h - hl == hk * uint32_t(p.gqa);
        if (T::QBUF && lane == 0) {
            lds_kbsf[n] = ks;
            if (write) KBSp[n] = f32_to_f16(ks);
        }
        if constexpr (T::QBUF) {
            uint32_t pk = 0;
#pragma unroll
            for (int t = 0; t < NE; ++t) pk |= (uint32_t(int(round_buf(kxe[t], ks))) & 0xFFu) << (8 * t);
            uint8_t* dl = lds_kbr + n * DKP + NE * lane;
            uint8_t* dg = KBp + n * DK + NE * lane;
            if constexpr (NE == 1) { *dl = uint8_t(pk); if (write) *dg = uint8_t(pk); }
            else if constexpr (NE == 2) {
                *reinterpret_cast<uint16_t*>(dl) = uint16_t(pk);
                if (write) *reinterpret_cast<uint16_t*>(dg) = uint16_t(pk);
            } else {
                *reinterpret_cast<uint32_t*>(dl) = pk;
                if (write) *reinterpret_cast<uint32_t*>(dg) = pk;
            }
        } else {
#pragma unroll
            for (int t = 0; t < NE; ++t) {
                const uint16_t hb = f32_to_bf16(kxe[t]);
                reinterpret_cast<uint16_t*>(lds_kbr)[n * DKP + NE * lane + t] = hb;
                if (write) reinterpret_cast<uint16_t*>(KBp)[n * DK + NE * lane + t] = hb;
            }
        }
    }

    // a slot's decay and value scale, lane i of every 16: what its coefficients need besides the dot products
    const int ls = lane & 15, li = ls < m ? ls : 0;
    const float dec_i = expf(gcur - lds_gbf[li]), us_i = T::QBUF ? lds_ubsf[li] : 1.0f;
    // this token's write, u = dt x, and its largest magnitude in the head: known ahead of the state's sums
    const float xt = raw_to_f(vr, x_dt);
    const float u = rlive ? lds_scal[0] * xt : 0.0f;
    float amax = 0.0f;
    if constexpr (T::QBUF) {
        amax = lanes_max<WAVE>(fabsf(u));
        if (NWH > 1 && lane == 0) lds_red[w] = amax;
    }
    lds_barrier();

    // ---- this wavefront's rows: buffer term, u, y ----
    const float alpha = lds_scal[1], a = lds_scal[2], gnew = lds_scal[3], dd = lds_scal[4];
    const float bc = lds_gsc[0];
    // coefficients of the head's slots, lane i of every 16: c[i] = exp(gcur - G_i) (B_i . C), times the slot's value scale; dead
    // slots (i >= n) may hold anything: select, never multiply
    float cq = lds_dots[li];
    float uv[MM];
#pragma unroll
    for (int i = 0; i < MM; ++i) uv[i] = lds_raw<T::QBUF>(lds_ubr, i * DV + row);
    asm volatile("" : "+v"(cq));                         // (read with the others, not behind a branch)
    cq = ls < n ? (T::QBUF ? (dec_i * cq) * us_i : dec_i * cq) : 0.0f;
    float accq = alpha * sq;
    static_for<MM>([&](auto i) {
        const float u_i = T::QBUF ? uv[i] : (i < n ? uv[i] : 0.0f);
        accq = fma_row_bcast<decltype(i)::value>(cq, u_i, accq);
    });
    float y = __builtin_fmaf(bc, u, a * accq);
    if (p.has_D) y = __builtin_fmaf(dd, xt, y);
    if (rlive && (NB == 2 || kb == 0)) store_f(outp, out_dt, row, y);

    // ---- append ----
    float us = 1.0f;
    if constexpr (T::QBUF) {
        if constexpr (NWH > 1) {
#pragma unroll
            for (int ww = 0; ww < NWH; ++ww) amax = as_f32(umax(as_u32(amax), as_u32(lds_red[hl * NWH + ww])));
        }
        us = fp16_scale(amax, 127.0f);
        if (wh == 0 && lane == 0) { UBSp[n] = f32_to_f16(us); lds_ubsf[n] = us; }
    }
    if (rlive && (NB == 2 || kb == 0)) {
        if constexpr (T::QBUF) {
            const int8_t c = int8_t(int(round_buf(u, us)));
            reinterpret_cast<int8_t*>(UBp)[n * DV + row] = c;
            reinterpret_cast<int8_t*>(lds_ubr)[n * DV + row] = c;
        } else {
            const uint16_t hb = f32_to_bf16(u);
            reinterpret_cast<uint16_t*>(UBp)[n * DV + row] = hb;
            reinterpret_cast<uint16_t*>(lds_ubr)[n * DV + row] = hb;
        }
    }
    if (wh == 0 && lane == 0) {
        GBh[n] = gnew;
        *gcp = full ? 0.0f : gnew;                       // advance
        *np = full ? 0 : n + 1;
    }

    // ---- fold ----
    if (full) {
        lds_barrier();                                   // `full` is the same in every head of a slot
        // lane offsets derived anew (from a copy of the lane id the compiler cannot trace back), so that the ones
        // formed at the top of the kernel are not kept in registers all the way to here
        int lf = lane;
        asm volatile("" : "+v"(lf));
        const float cmul = expf(gnew);
        if constexpr (T::AXV) {
            constexpr int MT = (MM + 1) / 2;
            const int fj = lf & 31, fkb = lf >> 5;
            float decf[MT];                              // decay ratios a_m / a_i of the lane's slots 2 t + kb
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const int sl = 2 * t + fkb;
                decf[t] = sl < m - 1 ? expf(gnew - lds_gbf[sl < m - 1 ? sl : 0]) : 1.0f;
            }
            float ksf[MT];                           // ... their key scales; 0 for slots that do not exist
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const int sl = 2 * t + fkb;
                ksf[t] = T::QBUF && sl < m ? lds_kbsf[sl] : 0.0f;
            }
            auto key = [&](int t, int col) {
                const int sl = 2 * t + fkb;
                const float kv = lds_raw<T::QBUF>(lds_kbr, (T::QBUF || sl < m ? sl : 0) * DKP + col);
                return T::QBUF ? kv * ksf[t] : sl < m ? kv : 0.0f;
            };
#pragma unroll
            for (int bi = 0; bi < NB; ++bi) {
                uint8_t* blk = my_codes + bi * Q::BLK;
                const int grp = wh * NB + bi;
                uint16_t* old = reinterpret_cast<uint16_t*>(lds_pl + w * L::PL_BYTES);      // the planes are done with
                F.scv[bi].store(old, lf);
                wave_sync();
                float dop[MT];
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int sl = 2 * t + fkb;
                    const int sc_ = sl < m ? sl : 0;
                    float fv = lds_raw<T::QBUF>(lds_ubr, sc_ * DV + grp * T::MR + fj);
                    if constexpr (T::QBUF) fv = fv * lds_ubsf[sc_];
                    fv = decf[t] * fv;
                    dop[t] = sl < m ? fv : 0.0f;
                }
                quad_fold_block_v<Q, T>(blk, key, dop, [&](int) { return cmul; }, cmul == 1.0f, old,
                                        SCh + grp * DK, lf);
                quad_store_block<Q>(Sh + grp * Q::GBLK, blk, lf);
            }
        } else {
            constexpr int MT4 = (MM + 3) / 4, CL = DKP / 4;
            const int fn = lf & 15, fq = lf >> 4;
            float decf[MT4];                                 // decay ratios a_m / a_i of the lane's slots 4 t + q
#pragma unroll
            for (int t = 0; t < MT4; ++t) {
                const int sl = 4 * t + fq;
                decf[t] = sl < m - 1 ? expf(gnew - lds_gbf[sl < m - 1 ? sl : 0]) : 1.0f;
            }
            const int fg = min((fq * CL) / T::KGROUP, NG - 1);
            FoldKeys<T> kop;
            quad_fold_keys<T>(lds_kbr, lds_kbsf, m, lf, kop);
#pragma unroll
            for (int bi = 0; bi < NB; ++bi) {
                uint8_t* blk = my_codes + bi * Q::BLK;
#pragma unroll
                for (int hf = 0; hf < 2; ++hf) {
                    if (T::RAGV && 16 * hf >= rows_left) continue;
                    const int frow = (wh * NB + bi) * T::MR + 16 * hf + fn;
                    float bop[MT4];
#pragma unroll
                    for (int t = 0; t < MT4; ++t) {
                        const int sl = 4 * t + fq;
                        const int sc_ = sl < m ? sl : 0;
                        float fv = lds_raw<T::QBUF>(lds_ubr, sc_ * DV + frow);
                        if constexpr (T::QBUF) fv = fv * lds_ubsf[sc_];
                        fv = decf[t] * fv;
                        bop[t] = sl < m ? fv : 0.0f;
                    }
                    if constexpr (T::FLT)
                        quad_fold_half_f<Q, T>(blk, hf, kop, bop, cmul, lf);
                    else
                        quad_fold_half<Q, T>(blk, hf, kop, bop, cmul, f16_to_f32(lds_sc[frow * NG + fg]),
                                                SCh + frow * NG + fg, lf);
                }
                wave_sync();
                quad_store_block<Q, T::RAGV>(Sh + (wh * NB + bi) * Q::GBLK, blk, lf, rows_left);
            }
        }
    }
}

template <class T, int NB, int GH, int WPE, int SPEC>
int launch_mamba2_quad(const Mamba2Params& p0, hipStream_t stream) {
    Mamba2Params p = p0;
    p.per_xcd = (p.per_xcd % GH == 0) ? p.per_xcd / GH : 0;          // dealing over head groups
    const uint32_t grid = uint32_t(p.rows) * uint32_t(p.hv / GH);
    hipLaunchKernelGGL((mamba2_quad_kernel<T, NB, GH, WPE, SPEC>), dim3(grid), dim3(Quad<T, NB, GH>::THREADS),
                       quad_lds_pad(), stream, p.idx, p.order, p.st.S, p.st.NPTR, p.per_xcd, p.hv, p.hv_shift, p.st.sS, p.st.sN,
                       quad_start_ramp<Quad<T, NB, GH>, WPE>(grid, 24), p);
    return int(hipGetLastError());
}

}  // namespace sq
