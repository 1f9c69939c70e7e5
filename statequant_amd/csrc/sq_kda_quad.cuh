// KDA packed decode step, one workgroup per (batch row, head): every wavefront owns one 32-row block of the head's state
// (int4 / int8 codes, key-axis groups or value-axis groups of one row block, or bf16; geometry and building blocks in
// sq_quad.cuh).
//
// Same arithmetic as the one-wavefront kernel of sq_kda.cuh (the reference's `_kda_step`,
// /root/reference/src/statequant/kernels/_kda_triton.py:38-149), with A = exp(G_n), G_n = G_{n-1} + g_n per channel:
//   c_x[i] = sum_j k_i[j] exp(G_n[j] - G_i[j]) x[j];   u = beta (v - S0^T (A k) - sum_i c_k[i] u_i);
//   o = S0^T (A q) + sum_i c_q[i] u_i + (k.q) u;   fold: S = S0 diag(A) + sum_i u_i (exp(G_n - G_i) k_i)^T
// KDA has no grouped keys, so a head is a workgroup.  What its one-wavefront kernel does in sequence is dealt out:
//   issue            every wavefront: its row block, scales, its rows of v and of the buffered values, its share of the
//                    buffered keys with their decays; one wavefront each q and k, both with g and the running decay
//   roles            q / k normalised, A q / A k as digit planes; G_n and A for all                       [barrier]
//   per wavefront    its row block's read-outs; c_q, c_k of its share of the slots                        [barrier]
//                    buffer term, u, o of its rows; max |u|; one wavefront each: the key, the decays      [barrier]
//                    append;  with a full buffer: fold of its row block out of LDS (one read of the codes)
// One row block per wavefront (four wavefronts for d_v 128): two per wavefront measured the same at 128
// sequences and 3 % faster at 256 (int4), but a third slower at 16 and slower everywhere on int8.
// us per launch, one wavefront per head -> this (32 heads of 128 x 128, sequences out of step): int4 g32 1 sequence
// 7.6 -> 4.2, 16: 17.7 -> 7.4, 128: 30.0 -> 21.8 (in order 18.8), 256: 47.8 -> 36.6 (in order 33.2; in lockstep 35.0 -> 33.7);
// when it was built, int8 g32 1: 7.8 -> 4.6, 256: 59.0 -> 43.4, value-axis int4 128: 33.6 -> 22.1, int8 256: 60.0 -> 45.0.  Bound at
// small batches by the chain of a head's life, at large ones by the vector ALU (int4, 256 sequences: 337 instructions per
// wavefront, 903 with a fold; 11.0 M and 29.6 M a launch, where the one-wavefront kernel has 9.1 M and 29.4 M).
#pragma once
#include "sq_gdn_quad.cuh"
#include "sq_kda.cuh"

namespace sq {

template <class T, class Q>
struct KdaLoads {
    uint16_t sc[T::NG];                    // scales of row lane % 32 of the block
    ColScales<T> scv;                      // value-axis groups: the block's scales of the lane's columns
    Raw4<T::QBUF> uraw[Q::UT], kraw[Q::KT];
    float4 gb[Q::KT];                      // cumulative decays beside kraw
    uint16_t kbs[Q::KT], ubs;
    int np;
    uint32_t xr[Q::NE], xr2[Q::NE], gr[Q::NE], beta, vr;
    float gc[Q::NE];
};

template <class T>
struct KdaLds {
    using Q = Quad<T, 1, 1>;
    using B = QuadLds<T, 1, 1, 2, 2>;                                // read-out vectors: q, k (normalised)
    static constexpr int GN = B::BYTES;                              // [DKP] G_n
    static constexpr int CM = GN + Q::DKP * 4;                       // [DKP] A = exp(G_n)
    static constexpr int XA = CM + Q::DKP * 4;                       // [2][DKP] A q, A k (value-axis groups: planes per block)
    static constexpr int KD = XA + (T::AXV || T::FLT ? 2 * Q::DKP * 4 : 0);  // [m][DKP] buffered keys x decay ratio, fp32
    static constexpr int BYTES = KD + T::MMAX * Q::DKP * 4;
};

// SPEC = 1: the serving case compiled in -- bf16 q / k / v / out, fp32 g and beta, a power-of-two
// head count where d_k is one too.
template <class T, int WPE, int SPEC>
__global__ __launch_bounds__((Quad<T, 1, 1>::THREADS), WPE)
void kda_quad_kernel(const int32_t* __restrict__ idx, const int32_t* __restrict__ order, const uint8_t* codes,
                     const int32_t* counters, int per_xcd, int hv, int hv_shift, uint32_t codes_stride,
                     uint32_t counters_stride, SQ_TL_PARAM const KdaParams p) {
    // (the leading arguments without gaps between them: 13 of the 14 words that are in registers when a wavefront starts)
    SQ_MARK(0);                                                   // entry
    constexpr bool FIX = SPEC > 0;
    const int q_dt = FIX ? int(BF16) : p.q_dt, k_dt = FIX ? int(BF16) : p.k_dt, v_dt = FIX ? int(BF16) : p.v_dt;
    const int out_dt = FIX ? int(BF16) : p.out_dt, g_dt = FIX ? int(F32) : p.g_dt, beta_dt = FIX ? int(F32) : p.beta_dt;
    using Q = Quad<T, 1, 1>;
    using L = QuadLds<T, 1, 1, 2, 2>;
    using K = KdaLds<T>;
    constexpr int DK = T::DK, DV = T::DV, NW = Q::NW, MM = T::MMAX, NE = Q::NE, NG = T::NG, DKP = Q::DKP;
    constexpr int RQ = 1 % NW, RK = 3 % NW, RX = 2 % NW, RG = 0;  // which wavefront plays which shared role
    __shared__ __attribute__((aligned(16))) uint8_t lds[K::BYTES];
    float* lds_xn = reinterpret_cast<float*>(lds + L::XN);
    uint8_t* lds_pl = lds + L::PL;
    float* lds_xs = reinterpret_cast<float*>(lds + L::XS);
    float* lds_dots = reinterpret_cast<float*>(lds + L::DOTS);
    float* lds_red = reinterpret_cast<float*>(lds + L::RED);
    float* lds_scal = reinterpret_cast<float*>(lds + L::SCAL);
    uint8_t* lds_ubr = lds + L::UBR;
    float* lds_ubsf = reinterpret_cast<float*>(lds + L::UBSF);
    uint16_t* lds_sc = reinterpret_cast<uint16_t*>(lds + L::SC);
    float* lds_gn = reinterpret_cast<float*>(lds + K::GN);
    float* lds_cm = reinterpret_cast<float*>(lds + K::CM);
    float* lds_xa = reinterpret_cast<float*>(lds + K::XA);
    float* lds_kd = reinterpret_cast<float*>(lds + K::KD);

    const int lane = threadIdx.x & (WAVE - 1);
    const int w = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    const int m = p.m;
    const uint32_t um = m;
    uint8_t* blk = lds + L::CODES + w * Q::BLK;                   // this wavefront's row block

    const TileId tid = tile_id_lead<(FIX && heads_pow2(T::DK))>(order, per_xcd, hv, hv_shift);
    const uint32_t b = tid.b, h = tid.h;
    const int32_t slot = idx ? idx[b] : int32_t(b);
    const int n32 = lane & 31, kb = lane >> 5;
    const int row = w * T::MR + n32;                              // the row of the head this lane finishes after the pass

    KdaLoads<T, Q> F;
    const int vl = Q::vec_lane(lane);                             // whose elements of a d_k vector this lane loads
    // ---- issue every load: first the token's own operands (their addresses need the batch row only) ...
    if (w == RQ)
        load_vec<NE>(advance(p.q, q_dt, uint64_t(b) * p.s_q + h * DK), q_dt, vl, F.xr);
    if (w == RK)
        load_vec<NE>(advance(p.k, k_dt, uint64_t(b) * p.s_k + h * DK), k_dt, vl, RQ == RK ? F.xr2 : F.xr);
    if (w == RQ || w == RK) load_vec<NE>(advance(p.g, g_dt, uint64_t(b) * p.s_g + h * DK), g_dt, vl, F.gr);
    F.beta = load_raw_uniform(p.beta, beta_dt, uint64_t(b) * p.s_beta + h);
    F.vr = load_raw(advance(p.v, v_dt, uint64_t(b) * p.s_v + h * DV), v_dt, uint32_t(row));
    void* const outp = advance(p.out, out_dt, uint64_t(b) * p.s_out + h * DV);
    if (idx && slot <= 0) {                              // padding row: zero output, touch nothing of a slot
        for (int r = w * WAVE + lane; r < DV; r += NW * WAVE) store_f(outp, out_dt, r, 0.0f);
        return;
    }
    SQ_MARK(1);                                                   // slot known, the token's loads issued
    const uint32_t seq = slot;
    float* const gch = field(p.st.GCUR, seq, p.st.sGC, h * DK);
    if (w == RQ || w == RK) {                            // the running decay, ahead of the row blocks: the roles wait for it
#pragma unroll
        for (int t = 0; t < NE; ++t) F.gc[t] = gch[NE * vl + t];
    }
    // ... then the row blocks, straight into their LDS image, and the fill counter (a scalar load; sq_quad.cuh) ...
    quad_dma_blocks<Q, 1>(field(codes, seq, codes_stride, h * (DV * T::ROW_BYTES)) + w * Q::GBLK, blk, lane);
    F.np = quad_dma_counter(field(counters, seq, counters_stride, h));
    __builtin_amdgcn_sched_barrier(0);
    // ... and the rest of the slot: scales and -- once the fill counter is here -- the live part of the decode buffer
    uint8_t* const Sh = field(p.st.S, seq, p.st.sS, h * (DV * T::ROW_BYTES));
    uint16_t* const SCh = field(p.st.SC, seq, p.st.sSC, h * T::SC_ELEMS);
    BufAddr<T> buf;
    buf.KB = p.st.KB + (uint64_t(seq) * p.st.sKB + h * um * DK) * T::BE;
    buf.UB = p.st.UB + (uint64_t(seq) * p.st.sUB + h * um * DV) * T::BE;
    buf.KBS = field(p.st.KBS, seq, p.st.sKBS, h * um);
    buf.UBS = field(p.st.UBS, seq, p.st.sUBS, h * um);
    float* const GBh = field(p.st.GB, seq, p.st.sGB, h * um * DK);
    if constexpr (T::AXV) {
        F.scv.load(SCh + w * DK, lane);
    } else if constexpr (!T::FLT) {
#pragma unroll
        for (int g = 0; g < NG; ++g) F.sc[g] = stream_load(SCh + uint32_t(row * NG + g));
    }
    quad_dma_counter_wait(F.np);
    const uint32_t nfill = uint32_t(F.np & (m - 1));
    const uint32_t nl = nfill > 0 ? nfill : 1u;
#pragma unroll
    for (int t = 0; t < Q::UT; ++t) {                    // lane (slot = lane / LU + SU t, rows 4 (lane % LU) ..)
        const uint32_t i = lane / Q::LU + Q::SU * t;
        const uint32_t ic = i < nl ? i : nl - 1;
        F.uraw[t] = stream_raw4<T::QBUF>(buf.UB + (ic * DV + w * Q::RW + 4 * (lane % Q::LU)) * T::BE);
    }
#pragma unroll
    for (int t = 0; t < Q::KT; ++t) {                    // lane (slot = SPP (NW t + w) + lane / LPS, columns 4 (lane % LPS) ..)
        const uint32_t i = Q::SPP * (NW * t + w) + lane / Q::LPS;
        const uint32_t ic = i < nl ? i : nl - 1;
        F.kraw[t] = stream_raw4<T::QBUF>(buf.KB + (ic * DK + Q::key_col(lane)) * T::BE);
        typedef float v4fl __attribute__((ext_vector_type(4)));
        const v4fl g4 = stream_load(reinterpret_cast<const v4fl*>(GBh + ic * DK + Q::key_col(lane)));
        F.gb[t] = make_float4(g4.x, g4.y, g4.z, g4.w);
        F.kbs[t] = T::QBUF ? buf.KBS[ic] : uint16_t(0);
    }
    F.ubs = T::QBUF ? buf.UBS[uint32_t(lane) < nl ? lane : 0] : uint16_t(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    SQ_MARK(2);                                                   // fill count here, every load issued

    // ---- roles: q and k normalised, times A the read-out vectors of the stored state; G_n, A ----
    auto role_vector = [&](const uint32_t (&raw)[NE], int dt, float post, int v) {
        float xe[NE], xa[NE], ss = 0.0f;
        // (opened here: both roles add the decays, and the compiler would have all wavefronts do it, and wait for them, first)
#pragma unroll
        for (int t = 0; t < NE; ++t) asm volatile("" : "+v"(F.gr[t]), "+v"(F.gc[t]));
#pragma unroll
        for (int t = 0; t < NE; ++t) {
            xe[t] = Q::vec_live(lane) ? vec_elem<NE>(raw, dt, t) : 0.0f;
            ss = __builtin_fmaf(xe[t], xe[t], ss);
        }
        const Quotient nrm(sqrtf(lanes_sum<WAVE>(ss) + 1e-6f));
#pragma unroll
        for (int t = 0; t < NE; ++t) {
            xe[t] = nrm.of(xe[t]) * post;
            const float gn = F.gc[t] + vec_elem<NE>(F.gr, g_dt, t);
            const float A = kda_exp(gn);
            xa[t] = A * xe[t];
            lds_xn[v * DKP + NE * lane + t] = xe[t];
            if (v == 0) {
                lds_gn[NE * lane + t] = gn;
                lds_cm[NE * lane + t] = A;
            }
            if constexpr (T::AXV || T::FLT) lds_xa[v * DKP + NE * lane + t] = xa[t];
        }
        if constexpr (!T::AXV && !T::FLT) quad_stage_planes<Q, T, NE>(xa, v, lane, lds_pl, lds_xs);
    };
    if (w == RQ) role_vector(F.xr, q_dt, p.scale, 0);
    if (w == RK) role_vector(RQ == RK ? F.xr2 : F.xr, k_dt, 1.0f, 1);
    // ---- the loads land ----
    const int n = F.np & (m - 1);
    const bool full = n == m - 1;
    uint16_t scw[NG];
    if constexpr (!T::AXV && !T::FLT) {
#pragma unroll
        for (int g = 0; g < NG; ++g) {
            scw[g] = F.sc[g];
            if (kb == 0) lds_sc[row * NG + g] = F.sc[g];
        }
    }
#pragma unroll
    for (int t = 0; t < Q::UT; ++t) {
        const int i = lane / Q::LU + Q::SU * t;
        if (Q::SU * Q::UT == MM || i < MM) store_raw4<T::QBUF>(lds_ubr + (i * DV + w * Q::RW + 4 * (lane % Q::LU)) * T::BE, F.uraw[t]);
    }
    if (w == RG && T::QBUF && lane < m) lds_ubsf[lane] = f16_to_f32(F.ubs);
    quad_dma_landed();                                             // the row blocks are in LDS
    SQ_MARK(3);                                                   // vectors, scales, buffered values here and staged
    lds_barrier();

    // ---- c_q, c_k of this wavefront's share of the slots: the decay ratio rides on the key ----
    {
        float x[2][4], gn[4];
        const int c4 = 4 * (lane % Q::LPS);
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const float4 f = *reinterpret_cast<const float4*>(lds_xn + v * DKP + c4);
            x[v][0] = f.x; x[v][1] = f.y; x[v][2] = f.z; x[v][3] = f.w;
        }
        {
            const float4 f = *reinterpret_cast<const float4*>(lds_gn + c4);
            gn[0] = f.x; gn[1] = f.y; gn[2] = f.z; gn[3] = f.w;
        }
#pragma unroll
        for (int t = 0; t < Q::KT; ++t) {
            const int i = Q::SPP * (NW * t + w) + lane / Q::LPS;
            // dead slots may hold anything, and the columns beyond d_k pair one channel's G_n with another's G_i, a ratio
            // that can overflow: discard both (an infinity times the vectors' zeros there would be a NaN in the sums)
            const bool alive = i < n && (!Q::PADK || c4 < DK);
            float kf[4];
            decode_raw4<T::QBUF>(F.kraw[t], kf);
            const float ks = f16_to_f32(F.kbs[t]);
            const float gi[4] = {F.gb[t].x, F.gb[t].y, F.gb[t].z, F.gb[t].w};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if constexpr (T::QBUF) kf[c] = kf[c] * ks;
                kf[c] = alive ? kf[c] * kda_exp(gn[c] - gi[c]) : 0.0f;
            }
            if (full && i < n) *reinterpret_cast<float4*>(lds_kd + i * DKP + c4) = make_float4(kf[0], kf[1], kf[2], kf[3]);
            float pr[2];                             // both sums side by side, then both stores
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                pr[v] = kf[0] * x[v][0];
#pragma unroll
                for (int c = 1; c < 4; ++c) pr[v] = __builtin_fmaf(kf[c], x[v][c], pr[v]);
            }
            lanes_sum2<Q::LPS>(pr);
            if (lane % Q::LPS == 0 && i < MM) {
                lds_dots[i] = pr[0];
                lds_dots[MM + i] = pr[1];
            }
        }
    }
    if (w == RK) {                                                // k . q
        float kqp = 0.0f;
#pragma unroll
        for (int t = 0; t < NE; ++t) kqp = __builtin_fmaf(lds_xn[DKP + NE * lane + t], lds_xn[NE * lane + t], kqp);
        kqp = lanes_sum<WAVE>(kqp);
        if (lane == 0) lds_scal[0] = kqp;
    }
    SQ_MARK(4);                                                   // buffered keys and decays here, coefficients done
    // ---- state pass against A q, A k ----
    float sq, sk;
    {
        float own;
        if constexpr (T::AXV) {
            own = quad_block_pass_v<Q, T, 2>(blk, lds_xa, F.scv, lds_pl + w * L::PL_BYTES, lds_xs + w * (L::XS_BYTES / 4), lane);
        } else if constexpr (T::FLT) {
            own = quad_block_pass_f<Q, T, 2>(blk, lds_xa, lane);
        } else {
            v4i aop[Q::NKS];
            quad_fetch_planes<Q, T, 2>(lds_pl, lane, aop);
            float xs[NG], sc[NG];
#pragma unroll
            for (int g = 0; g < NG; ++g) xs[g] = lds_xs[kb * NG + g];
#pragma unroll
            for (int g = 0; g < NG; ++g) sc[g] = f16_to_f32(scw[g]);
            own = quad_block_pass<Q, T>(blk, aop, xs, sc, lane);
        }
        const Pair qk = pair32(own);
        sq = qk.lo;
        sk = qk.hi;
    }
    SQ_MARK(5);                                                   // state pass done
    lds_barrier();

    // ---- append the key (its decay ratio within this buffer is 1) and the decays ----
    if (w == RX) {
        float kxe[NE], kmax = 0.0f;
#pragma unroll
        for (int t = 0; t < NE; ++t) {
            kxe[t] = lds_xn[DKP + NE * lane + t];
            kmax = fmaxf(kmax, fabsf(kxe[t]));
        }
        float ks = 1.0f;
        if constexpr (T::QBUF) ks = fp16_scale(lanes_max<WAVE>(kmax), 127.0f);
        if (T::QBUF && lane == 0) buf.KBS[n] = f32_to_f16(ks);
        uint32_t pk = 0;
#pragma unroll
        for (int t = 0; t < NE; ++t) {
            float kr;
            if constexpr (T::QBUF) {
                const float c = round_buf(kxe[t], ks);
                kr = c * ks;
                pk |= (uint32_t(int(c)) & 0xFFu) << (8 * t);
            } else {
                const uint16_t hb = f32_to_bf16(kxe[t]);
                kr = bf16_to_f32(hb);
                if (Q::vec_live(lane)) reinterpret_cast<uint16_t*>(buf.KB)[n * DK + NE * lane + t] = hb;
            }
            if (full) lds_kd[n * DKP + NE * lane + t] = kr;
        }
        if (T::QBUF && Q::vec_live(lane)) {
            uint8_t* dg = buf.KB + n * DK + NE * lane;
            if constexpr (NE == 1) *dg = uint8_t(pk);
            else if constexpr (NE == 2) *reinterpret_cast<uint16_t*>(dg) = uint16_t(pk);
            else *reinterpret_cast<uint32_t*>(dg) = pk;
        }
    }
    if (w == RG && Q::vec_live(lane)) {
#pragma unroll
        for (int t = 0; t < NE; ++t) {
            const float gn = lds_gn[NE * lane + t];
            GBh[n * DK + NE * lane + t] = gn;
            gch[NE * lane + t] = full ? 0.0f : gn;
        }
    }
    // ---- this wavefront's rows: buffer term, u, o ----
    const float kq = lds_scal[0], beta = raw_to_f(F.beta, beta_dt);
    const int ls = lane & 15, li = ls < m ? ls : 0;      // lane i of every 16: the coefficients of slot i
    const float us_i = T::QBUF ? lds_ubsf[li] : 1.0f;
    const bool alive = ls < n;
    float cq = lds_dots[li], ck = lds_dots[MM + li];
    float uv[MM];
#pragma unroll
    for (int i = 0; i < MM; ++i) uv[i] = lds_raw<T::QBUF>(lds_ubr, i * DV + row);
    asm volatile("" : "+v"(cq), "+v"(ck));               // (read with the others, not each behind a branch on `alive`)
    cq = alive ? (T::QBUF ? cq * us_i : cq) : 0.0f;
    ck = alive ? (T::QBUF ? ck * us_i : ck) : 0.0f;
    float accq = sq, acck = sk;
    static_for<MM>([&](auto i) {
        const float u_i = T::QBUF ? uv[i] : (i < n ? uv[i] : 0.0f);
        accq = fma_row_bcast<decltype(i)::value>(cq, u_i, accq);
        acck = fma_row_bcast<decltype(i)::value>(ck, u_i, acck);
    });
    const float u = beta * (raw_to_f(F.vr, v_dt) - acck);
    const float o = __builtin_fmaf(kq, u, accq);
    if (kb == 0) store_f(outp, out_dt, row, o);
    SQ_MARK(6);                                                   // outputs stored
    float us = 1.0f;
    if constexpr (T::QBUF) {
        float amax = lanes_max<WAVE>(fabsf(u));
        if constexpr (NW > 1) {
            if (lane == 0) lds_red[w] = amax;
            lds_barrier();
#pragma unroll
            for (int ww = 0; ww < NW; ++ww) amax = as_f32(umax(as_u32(amax), as_u32(lds_red[ww])));
        }
        us = fp16_scale(amax, 127.0f);
        if (w == RG && lane == 0) { buf.UBS[n] = f32_to_f16(us); lds_ubsf[n] = us; }
    }
    if (kb == 0) {
        if constexpr (T::QBUF) {
            const int8_t c = int8_t(int(round_buf(u, us)));
            reinterpret_cast<int8_t*>(buf.UB)[n * DV + row] = c;
            reinterpret_cast<int8_t*>(lds_ubr)[n * DV + row] = c;
        } else {
            const uint16_t hb = f32_to_bf16(u);
            reinterpret_cast<uint16_t*>(buf.UB)[n * DV + row] = hb;
            reinterpret_cast<uint16_t*>(lds_ubr)[n * DV + row] = hb;
        }
    }
    if (w == RG && lane == 0) *field(p.st.NPTR, seq, p.st.sN, h) = full ? 0 : n + 1;
    SQ_MARK(7);                                                   // appended, counter advanced
    // ---- fold ----
    if (full) {
        lds_barrier();
        int lf = lane;                                   // (offsets derived anew: see the GDN kernel)
        asm volatile("" : "+v"(lf));
        if constexpr (T::AXV) {
            constexpr int MT = (MM + 1) / 2;
            const int fj = lf & 31, fkb = lf >> 5;
            auto key = [&](int t, int col) {
                const int sl = 2 * t + fkb;
                const float kv = lds_kd[(sl < m ? sl : 0) * DKP + col];
                return sl < m ? kv : 0.0f;
            };
            auto cm = [&](int col) { return lds_cm[col]; };
            uint16_t* old = reinterpret_cast<uint16_t*>(lds_pl + w * L::PL_BYTES);      // the planes are done with
            F.scv.store(old, lf);
            wave_sync();
            float dop[MT];
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                const int sl = 2 * t + fkb;
                const int sc_ = sl < m ? sl : 0;
                float uv_ = lds_raw<T::QBUF>(lds_ubr, sc_ * DV + w * T::MR + fj);
                if constexpr (T::QBUF) uv_ = uv_ * lds_ubsf[sc_];
                dop[t] = sl < m ? uv_ : 0.0f;
            }
            quad_fold_block_v<Q, T>(blk, key, dop, cm, false, old, SCh + w * DK, lf);
        } else {
            constexpr int MT4 = (MM + 3) / 4, CL = DKP / 4;
            const int fn = lf & 15, fq = lf >> 4;
            const int fg = min((fq * CL) / T::KGROUP, NG - 1);
            FoldKeys<T, true> kop;
            quad_fold_keys_f32<T>(lds_kd, m, lf, kop);
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) {
                const int frow = w * T::MR + 16 * hf + fn;
                float bop[MT4];
#pragma unroll
                for (int t = 0; t < MT4; ++t) {
                    const int sl = 4 * t + fq;
                    const int sc_ = sl < m ? sl : 0;
                    float uv_ = lds_raw<T::QBUF>(lds_ubr, sc_ * DV + frow);
                    if constexpr (T::QBUF) uv_ = uv_ * lds_ubsf[sc_];
                    bop[t] = sl < m ? uv_ : 0.0f;
                }
                if constexpr (T::FLT)
                    quad_fold_half_f<Q, T, true>(blk, hf, kop, bop, 1.0f, lf, lds_cm);
                else
                    quad_fold_half<Q, T, true>(blk, hf, kop, bop, 1.0f, f16_to_f32(lds_sc[frow * NG + fg]),
                                               SCh + frow * NG + fg, lf, lds_cm);
            }
            wave_sync();
        }
        quad_store_block<Q>(Sh + w * Q::GBLK, blk, lf);
    }
    SQ_MARK(8);                                                   // folded (a full buffer)
}

template <class T, int NB, int GH, int WPE, int SPEC>
int launch_kda_quad(const KdaParams& p, hipStream_t stream) {
    static_assert(NB == 1 && GH == 1, "a row block per wavefront; no grouped keys");
    const uint32_t grid = uint32_t(p.rows) * uint32_t(p.hv);
    using Q = Quad<T, 1, 1>;
#ifdef SQ_TIMELINE
    const SqTimelineBuf tl = sq_timeline_buffer();
    hipLaunchKernelGGL((kda_quad_kernel<T, WPE, SPEC>), dim3(grid), dim3(Q::THREADS), quad_lds_pad(), stream, p.idx, p.order,
                       p.st.S, p.st.NPTR, p.per_xcd, p.hv, p.hv_shift, p.st.sS, p.st.sN, tl.p, tl.cap, p);
#else
    hipLaunchKernelGGL((kda_quad_kernel<T, WPE, SPEC>), dim3(grid), dim3(Q::THREADS), quad_lds_pad(), stream, p.idx, p.order,
                       p.st.S, p.st.NPTR, p.per_xcd, p.hv, p.hv_shift, p.st.sS, p.st.sN, p);
#endif
    return int(hipGetLastError());
}

}  // namespace sq
