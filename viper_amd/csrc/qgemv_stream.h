// M = 1 quantized GEMV for rows that no exact tiling of qgemv_m1.h covers (any
// K that is a multiple of the group) and for the long rows it serves better:
// persistent workgroups that stage the activation once and stream their weight
// rows wave by wave.
#pragma once

#include "qgemv_m1.h"

namespace vq {

// Work split.  A unit is UR = 64 / TS * R consecutive output rows, read by one
// wave: teams of TS lanes, R rows per team, CPL 16-byte chunk slots per lane
// and row (lanes of the last slot past the row read nothing).  Workgroup b (in
// XCD order) owns `upw` consecutive units and its waves take them in turn.
// The row's weight scales come with one 16-byte load per lane (the rows of a
// unit are contiguous) and reach the lanes through a wave-private LDS block,
// so no wave waits for another after the activation's barrier.  Each wave has
// a second unit's loads in flight while it sums one; loads past its last unit
// are not issued (an out-of-range load still takes the address unit's 16
// clocks: issued anyway, they cost 0.5 us of a short launch).
// K of more than TS * CPL chunks (shapes of ST_MAX slots) is read in segments.
//
// What bounds it: the weight stream, once a launch is long (Q4, K = 11008,
// N = 28672, 168 MB: 27.4-28.3 us, 6.0 TB/s); short ones the dispatch, the
// activation's quantize and a unit's dots after its data (the barrier passes
// 1.0 us after the start at K = 4096, and a 16-row workgroup ends 1.9 us
// later).  The general path of qgemv_m1_kernel that this replaced loaded every
// chunk's scale with a 2-byte load of its own, ran one unit per wave and
// quantized the activation in every workgroup: Q4, K = 4096, N = 4096 / 11008
// 4.15 / 7.4 -> 3.7 / 5.9 us, K = 8896, N = 11008 17.4 -> 10.9 us, Q6, K = 8896,
// N = 4096 10.2 -> 7.4 us, W8, K = 4096, N = 11008 13.5 -> 9.5 us.
//
// The activation is staged exactly as in qgemv_m1_kernel (same LDS row, same
// prologues); the swiglu pair reads a unit's gate rows and up rows as two
// tiles of one wave, so its epilogue needs no exchange between waves.

// 256 and 1024 threads were within 5 % of 512 or slower over K = 512..16384
// and N = 1024..28672 once two workgroups share a CU where they can.
constexpr int ST_NTT = 512;  // threads per workgroup
// Weight-issue delay, s_sleep units, as in qgemv_m1_kernel.  Without one the
// bf16 row's calls are 1-2 % faster (K = 5120, N = 1024 2.44 against 2.51 us) and
// those with a second input 3-5 % slower, whose loads then queue behind the
// weights (swiglu, Q4, K = 10240, N = 1024 4.13 against 4.05; K = 12288, N = 2560
// 5.84 / 5.65); 5 is slower than 2 by 1 %.
constexpr int ST_DELAY = 2;
// Most chunk slots per lane (two units of more of Q5 / Q6 pass 256 registers).
template <int F>
constexpr int ST_MAX = F == 5 || F == 6 ? 8 : 10;
constexpr int ST_SCALE_LDS = 1024;  // wave-private scale block: 64 lanes x 16 bytes

template <int F>
__host__ __device__ constexpr size_t st_lds_bytes(int K, int segw) {
    const int slots = (K / Fmt<F>::CK + segw - 1) / segw * segw;
    return (size_t)slots * (Fmt<F>::CK + 8) + 128 + (size_t)(ST_NTT / 64) * ST_SCALE_LDS;
}

// team_sum of values that both lanes of a chunk pair hold
template <int TS>
__device__ __forceinline__ float pair_team_sum(float v) {
    v += dpp_f<DPP_SWAP2>(v);
    if constexpr (TS >= 8) v += dpp_f<DPP_HALF_MIRROR>(v);
    if constexpr (TS >= 16) v += dpp_f<DPP_MIRROR>(v);
    return team_sum_rows<TS>(v);
}

template <int F, int CPL, int R>
struct StTile {
    u32x4 wv[R][CPL];
    uint32_t h0[R][CPL], h1[R][CPL];
    u32x4 sc;
    uint32_t res;
};

// Activation octets per thread loaded ahead of the weights: the whole row of a
// single-segment shape; rows of several segments (shapes of ST_MAX slots) up
// to K = 20480, the longest the folded prologues take.
template <int F>
__host__ __device__ constexpr int st_rounds(int ts, int cpl) {
    return cpl == ST_MAX<F> ? 20480 / 8 / ST_NTT : (ts * cpl * Fmt<F>::CK / 8 + ST_NTT - 1) / ST_NTT;
}

// kw: K / 32 in bits 0..11, units per workgroup in bits 12..21, workgroups
// per XCD in bits 22..31 (0: blocks in dispatch order).
template <int F, int TS, int CPL, int R, int SENC, int MODE, int PRO>
__global__ void __launch_bounds__(ST_NTT)
qgemv_stream_kernel(const void* x, const uint8_t* w0, const uint16_t* s0, uint16_t* y0, int kw, int n0, int e0, int e1,
                    const uint16_t* res, const void* xa, float eps, uint16_t* __restrict__ xout,
                    int32_t* __restrict__ part, const uint8_t* w1, const uint16_t* s1, uint16_t* y1, int n1,
                    const uint8_t* w2, const uint16_t* s2, uint16_t* y2, int n2) {
    using FT = Fmt<F>;
    constexpr bool TLM = MODE == M1_TL;
    uint64_t tstamp[M1_TL_STAMPS];
    auto stamp = [&](int i) {
        if constexpr (TLM) tstamp[i] = __builtin_amdgcn_s_memrealtime();
    };
    stamp(0);
    constexpr bool PART = MODE == M1_PART;
    constexpr bool SWI = MODE == M1_SWIGLU;
    constexpr bool PRE = PRO == PRO_INT8;
    constexpr bool TWO = PRO == PRO_RMSNORM || PRO == PRO_SWIGLU;
    constexpr int NTT = ST_NTT, XS = st_rounds<F>(TS, CPL);
    constexpr int UR = 64 / TS * R, W = NTT / 64, SEGW = TS * CPL;
    // slots that lie inside the row on every lane: all but the last one, as the
    // team has no more lanes than st_shape's rule needs (none certain in the
    // last segment of a longer row, shapes of ST_MAX slots)
    constexpr int FULL = CPL == ST_MAX<F> ? 0 : CPL - 1;
    constexpr int HB = FT::HIW * 4;
    constexpr int OPC = FT::CK / 8, OPG = FT::G / 8;
    const int K = (kw & 0xfff) * 32, upw = (kw >> 12) & 0x3ff, gx = (int)((unsigned)kw >> 22);
    const int CPR = K / FT::CK, NGR = K / FT::G, noct = K / 8;
    const int nseg = (CPR + SEGW - 1) / SEGW;
    extern __shared__ __align__(16) uint8_t smem[];
    // (rounded up to whole segments: slots past the row read what lies there,
    // and their scale is 0)
    const int slots = nseg * SEGW;
    int8_t* lxq = (int8_t*)smem;                                // [slots][CK]
    u32x2* lcs = (u32x2*)(smem + slots * FT::CK);               // [slots]
    float* lred = (float*)(smem + slots * (FT::CK + 8));        // 32 floats
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint8_t* wsc = smem + slots * (FT::CK + 8) + 128 + wave * ST_SCALE_LDS;
    const int l = lane % TS, rr = lane / TS;
    const bool lead = (l & 1) == 0;
    // matrix of this workgroup: matrix 0's arguments are preloaded, the others
    // are the rare path (as in qgemv_m1_kernel)
    int bid = gx ? ((int)blockIdx.x & 7) * gx + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
    const uint8_t* w = w0;
    const uint16_t* ws = s0;
    uint16_t* y = y0;
    int N = n0 & M1_N_MASK;
    const bool extra_out = (n0 & M1_N_EXTRA) != 0;
    if (!SWI && __builtin_expect(bid >= e0, 0)) {
        res = nullptr;
        if (bid >= e1) {
            bid -= e1;
            w = w2;
            ws = s2;
            y = y2;
            N = n2;
        } else {
            bid -= e0;
            w = w1;
            ws = s1;
            y = y1;
            N = n1;
        }
    }
    const uint32_t rbytes = (uint32_t)CPR * 16;
    const int uend = min((bid + 1) * upw, (N + UR - 1) / UR);
    if (bid * upw >= uend) return;  // a grid rounded up to whole XCD turns

    // a wave's tiles in order: its units, per unit the segments of K (the
    // pair: gate's, then up's)
    struct Cur {
        int u, seg;
    };
    const int ntile = SWI ? 2 * nseg : nseg;
    auto advance = [&](Cur& c) {
        if (++c.seg == ntile) {
            c.seg = 0;
            c.u += W;
        }
    };
    using Tile = StTile<F, CPL, R>;
    auto load = [&](Tile& T, const Cur& c) {
        const bool up = SWI && c.seg >= nseg;
        const uint8_t* wm = up ? (const uint8_t*)res : w;
        const uint16_t* sm = up ? (const uint16_t*)(((uint64_t)(uint32_t)e1 << 32) | (uint32_t)e0) : ws;
        const int seg = up ? c.seg - nseg : c.seg, row0 = c.u * UR;
        const int n = c.u < uend ? min(UR, N - row0) : 0;
        // the unit's scales (of this segment): from the 16-byte word that
        // holds the first one
        const size_t sb = ((size_t)row0 * NGR + (size_t)seg * (SEGW / 2)) * 2;
        const size_t stot = (size_t)N * NGR * 2;
        const int wsd = (int)(sb & 15);
        const size_t left = stot - (sb - wsd);
        const uint32_t sn = n ? (uint32_t)(left < ST_SCALE_LDS ? (left & ~(size_t)3) : ST_SCALE_LDS) : 0u;
        const int need = wsd + (nseg == 1 ? n * NGR * 2 : min(SEGW / 2, NGR - seg * (SEGW / 2)) * 2);
        T.sc = bload16(buf((const uint8_t*)sm + (sb - wsd), sn), lane * 16 < need ? lane * 16 : OOB);
        if constexpr (!SWI)
            T.res = bload2(buf(res + row0, res != nullptr ? (uint32_t)n * 2 : 0u), l < R ? (rr * R + l) * 2 : OOB);
        const auto wr = buf(wm + (size_t)row0 * rbytes, (uint32_t)n * rbytes);
        const auto hr = buf(wm + (size_t)N * (K / 2) + (size_t)row0 * CPR * HB, (uint32_t)n * CPR * HB);
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int j = 0; j < CPL; ++j) {
                const int ch = seg * SEGW + j * TS + l;
                // (one row per unit: the resource ends with the row)
                const bool in = UR == 1 || j < FULL || ch < CPR;
                T.wv[r][j] = bload16<AUX_NT>(wr, in ? (rr * R + r) * (int)rbytes + ch * 16 : OOB);
                T.h0[r][j] = 0u;
                T.h1[r][j] = 0u;
                if constexpr (FT::HIW == 1) {
                    T.h0[r][j] = bload4<AUX_NT>(hr, in ? ((rr * R + r) * CPR + ch) * HB : OOB);
                } else if constexpr (FT::HIW == 2) {
                    const u32x2 hh = bload8<AUX_NT>(hr, in ? ((rr * R + r) * CPR + ch) * HB : OOB);
                    T.h0[r][j] = hh.x;
                    T.h1[r][j] = hh.y;
                }
            }
    };

    // 1. activation octets, then the first two tiles' weights
    const auto xr = buf(x, (uint32_t)K * (PRE ? 1 : 2));
    const auto xsr = buf(xa, PRE ? (uint32_t)NGR * 4 : TWO ? (uint32_t)K * 2 : 0u);
    auto load_x = [&](int o) -> u32x4 {
        if constexpr (PRE) {
            const u32x2 q = bload8(xr, o * 8);
            const uint32_t sb = bload4(xsr, (o % OPC == 0) ? (o / OPG) * 4 : OOB);
            return u32x4{q.x, q.y, sb, 0u};
        } else {
            return bload16(xr, o * 16);
        }
    };
    // (rounds past the row are not issued where the shape does not fix their number)
    constexpr bool SKIP = CPL == ST_MAX<F>;
    u32x4 xv[XS], av[XS];
#pragma unroll
    for (int i = 0; i < XS; ++i) {
        if (SKIP && NTT * i >= noct) break;
        if constexpr (PRE) {
            const u32x2 q = bload8(xr, (tid + NTT * i) * 8);
            xv[i] = u32x4{q.x, q.y, 0u, 0u};
        } else {
            xv[i] = bload16(xr, (tid + NTT * i) * 16);
        }
    }
    issue_fence();
    if constexpr (PRE || TWO) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < XS; ++i) {
            if (SKIP && NTT * i >= noct) break;
            const int o = tid + NTT * i;
            if constexpr (PRE) xv[i].z = bload4(xsr, (o % OPC == 0) ? (o / OPG) * 4 : OOB);
            else av[i] = bload16(xsr, o * 16);
        }
        issue_fence();
    }
    float epsv = eps;
    if constexpr (PRO == PRO_RMSNORM) {
        epsv = __uint_as_float(bload4(m1_kernargs(), (int)offsetof(M1KernArgs, eps)));
        issue_fence();
    }
    stamp(1);
    if constexpr (ST_DELAY > 0) __builtin_amdgcn_s_sleep(ST_DELAY);
    // quantize the activation into LDS (the tiles in flight meanwhile)
    auto stage = [&] {
        stamp(2);
        float inv = 0.0f;
        if constexpr (PRO == PRO_RMSNORM) {
            float ss = 0.0f;
#pragma unroll
            for (int i = 0; i < XS; ++i) {
                if (SKIP && NTT * i >= noct) break;
                const u32x4 v = xv[i];  // octets past the row are zero
                const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float f = bf16f((wd[j >> 1] >> (16 * (j & 1))) & 0xffffu);
                    ss = __builtin_fmaf(f, f, ss);
                }
            }
            ss = team_sum<64>(ss);
            if (lane == 0) lred[wave] = ss;
            lds_barrier();
            float t = 0.0f;
#pragma unroll
            for (int i = 0; i < W; ++i) t += lred[i];
            inv = __builtin_amdgcn_rsqf(t / (float)K + epsv);
        }
        auto quant_store = [&](int o, const u32x4& v) { m1_quant_store<F, PRE>(o, v, noct, lxq, lcs); };
        const int wave0 = tid & ~63;
#pragma unroll
        for (int i = 0; i < XS; ++i) {
            if (wave0 + NTT * i < noct) {
                const int o = tid + NTT * i;
                if constexpr (TWO) {
                    const u32x4 v = m1_produce<PRO>(xv[i], av[i], inv);
                    if (PRO == PRO_RMSNORM && __builtin_expect(extra_out, 0) && blockIdx.x == 0) {
                        uint16_t* xo = m1_xout();
                        if (xo != nullptr && o < noct) *(u32x4*)(xo + (size_t)o * 8) = v;
                    }
                    quant_store(o, v);
                } else {
                    quant_store(o, xv[i]);
                }
            }
        }
        if constexpr (!TWO)
            if (__builtin_expect(noct > XS * NTT, 0))
                for (int o = tid + XS * NTT; (o & ~63) < noct; o += NTT) quant_store(o, load_x(o));
        stamp(3);
        lds_barrier();
        stamp(4);
    };

    // 2. a tile's products
    float acc[R] = {};
    uint16_t gate = 0;
    auto compute = [&](Tile& T, const Cur& c) {
        const bool up = SWI && c.seg >= nseg;
        const int seg = up ? c.seg - nseg : c.seg, row0 = c.u * UR;
        const int n = min(UR, N - row0);
        const size_t sb = ((size_t)row0 * NGR + (size_t)seg * (SEGW / 2)) * 2;
        const int wsd = (int)(sb & 15);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        *(u32x4*)(wsc + lane * 16) = T.sc;
        // a scale array of an odd number of entries ends within a dword: its
        // last entry is read on its own
        const size_t stot = (size_t)N * NGR * 2;
        if (__builtin_expect((stot & 2) != 0 && stot - (sb - wsd) < ST_SCALE_LDS, 0)) {
            const uint32_t last = bload2(buf((const uint8_t*)(up ? (const uint16_t*)(((uint64_t)(uint32_t)e1 << 32) | (uint32_t)e0) : ws) + stot - 2, 2u), lane == 0 ? 0 : OOB);
            if (lane == 0) *(uint16_t*)(wsc + (stot - 2 - (sb - wsd))) = (uint16_t)last;
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        // operands of every slot first: the LDS reads overlap each other and
        // the wait for the weights
        u32x4 A0[CPL], A1[CPL];
        u32x2 CS[CPL];
        uint32_t SR[R][CPL];
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            const int ch = seg * SEGW + j * TS + l;
            CS[j] = lcs[ch];
            const u32x4* a = (const u32x4*)(lxq + (size_t)ch * FT::CK);
            A0[j] = a[0];
            A1[j] = FT::OFF ? a[1] : a[0];
#pragma unroll
            for (int r = 0; r < R; ++r)
                SR[r][j] = *(const uint16_t*)(wsc + wsd + ((rr * R + r) * NGR + j * (TS / 2) + (l >> 1)) * 2);
        }
#pragma unroll
        for (int j = 0; j < CPL; ++j) {
            const int ch = seg * SEGW + j * TS + l;
            const bool in = j < FULL || ch < CPR;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                int dot;
                if constexpr (F == 4) dot = chunk_dot_q4(T.wv[r][j], A0[j], A1[j], (int)CS[j].x);
                else dot = chunk_dot<F>(T.wv[r][j], T.h0[r][j], T.h1[r][j], A0[j], A1[j], (int)CS[j].x);
                dot += dpp_i<DPP_SWAP1>(dot);
                if constexpr (PART)
                    if (lead && in && rr * R + r < n) part[(size_t)(row0 + rr * R + r) * NGR + (ch >> 1)] = dot;
                const float sc = (SENC ? bf16f(SR[r][j]) : f16f(SR[r][j])) * __uint_as_float(CS[j].y);
                acc[r] = __builtin_fmaf(in ? sc : 0.0f, (float)dot, acc[r]);
            }
            if (TLM && j == 0 && c.u == bid * upw + wave && c.seg == 0) stamp(5);
        }
        if (seg + 1 < nseg) return;  // more segments of these rows
        stamp(6);
        // the team's R rows, one per lane 0..R-1
        float v = pair_team_sum<TS>(acc[0]);
        acc[0] = 0.0f;
#pragma unroll
        for (int r = 1; r < R; ++r) {
            const float t = pair_team_sum<TS>(acc[r]);
            acc[r] = 0.0f;
            v = l == r ? t : v;
        }
        const int rl = rr * R + l;  // the lane's row of the unit
        const bool st = l < R && rl < n;
        if constexpr (SWI) {
            const uint16_t vb = f2bf(v);
            if (!up) {
                gate = vb;
                if (__builtin_expect(extra_out, 0) && st && y1 != nullptr) y1[row0 + rl] = vb;
            } else {
                if (__builtin_expect(extra_out, 0) && st && y2 != nullptr) y2[row0 + rl] = vb;
                if (st) y0[row0 + rl] = f2bf(silu_mul(bf16f(gate), bf16f(vb)));
            }
        } else {
            if (st) y[row0 + rl] = f2bf(res != nullptr ? v + bf16f(T.res) : v);
        }
    };
    // 3. tiles in order, one in flight while the other is summed.  Separate code
    // for waves with no tile, and for the last: a load that may or may not
    // have been issued would make every wait behind it one for both, and one
    // out of range still takes the address unit's time (waves past the units
    // issuing theirs: Q6, K = 10752, N = 1024 4.6 -> 3.7 us without; N = 1536
    // 5.25 -> 4.9).  (A second tile ahead of the quantize: 5 % faster where no
    // wave has a third and the tiles are small, 2-11 % slower else, as the
    // activation then queues behind it.)  Every wave runs stage(), hence its
    // barriers, exactly once.
    Cur lc{bid * upw + wave, 0}, cc = lc;
    Tile T0, T1;
    if (lc.u >= uend) {
        stage();
    } else {
        load(T0, lc);
        issue_fence();
        stage();
        for (;;) {
            advance(lc);
            if (lc.u >= uend) {
                compute(T0, cc);
                break;
            }
            load(T1, lc);
            issue_fence();
            compute(T0, cc);
            advance(cc);
            advance(lc);
            if (lc.u >= uend) {
                compute(T1, cc);
                break;
            }
            load(T0, lc);
            issue_fence();
            compute(T1, cc);
            advance(cc);
        }
    }
    if constexpr (TLM) {
        if (bid * upw + wave >= uend) {  // a wave with no unit
            stamp(5);
            stamp(6);
        }
        stamp(7);
        if (lane == 0) {
            uint64_t* o = (uint64_t*)part + ((size_t)bid * W + wave) * M1_TL_STAMPS;
#pragma unroll
            for (int i = 0; i < M1_TL_STAMPS; ++i) o[i] = tstamp[i];
        }
    }
}

// Launch shapes: (team size, chunk slots per lane, rows per team of a unit).
// The team is the narrowest that covers the row in two slots up to 64 chunks
// (K = 2048; W8 1024; one slot up to 8 chunks), then 64 lanes with as many slots as the row needs.  The
// timeline only for the rows its entry point takes that no tiling always
// covers: 160 to 640 chunks.
template <int F, int SENC, int MODE, int PRO>
m1_fn st_kernel_v(int ts, int cpl, int r) {
#define VQ_ST(TS_, CPL_, R_) \
    if constexpr (CPL_ <= ST_MAX<F> && (MODE != M1_TL || (CPL_ == 3 && F != 8) || CPL_ == 5 || CPL_ == 6 || CPL_ == ST_MAX<F>)) \
        if (ts == TS_ && cpl == CPL_ && r == R_) return qgemv_stream_kernel<F, TS_, CPL_, R_, SENC, MODE, PRO>;
    VQ_ST(8, 1, 1) VQ_ST(8, 2, 1) VQ_ST(16, 2, 1) VQ_ST(32, 2, 1) VQ_ST(64, 2, 1) VQ_ST(64, 2, 2) VQ_ST(64, 3, 1) VQ_ST(64, 4, 1)
    VQ_ST(64, 5, 1) VQ_ST(64, 6, 1) VQ_ST(64, 7, 1) VQ_ST(64, 8, 1) VQ_ST(64, 9, 1) VQ_ST(64, 10, 1)
#undef VQ_ST
    return nullptr;
}
// The partials and the timeline are built for the bf16 prologue, the swiglu
// pair for the bf16 and rmsnorm ones (as for the exact tilings).
template <int F, int PRO>
m1_fn st_pick_pro(int ts, int cpl, int r, int senc, int mode) {
    if constexpr (PRO == PRO_BF16) {
        if (mode == M1_PART) return senc ? st_kernel_v<F, 1, M1_PART, PRO>(ts, cpl, r) : st_kernel_v<F, 0, M1_PART, PRO>(ts, cpl, r);
        if (mode == M1_TL) return senc ? st_kernel_v<F, 1, M1_TL, PRO>(ts, cpl, r) : st_kernel_v<F, 0, M1_TL, PRO>(ts, cpl, r);
    }
    if constexpr (PRO == PRO_BF16 || PRO == PRO_RMSNORM)
        if (mode == M1_SWIGLU)
            return senc ? st_kernel_v<F, 1, M1_SWIGLU, PRO>(ts, cpl, r) : st_kernel_v<F, 0, M1_SWIGLU, PRO>(ts, cpl, r);
    if (mode == M1_PLAIN) return senc ? st_kernel_v<F, 1, M1_PLAIN, PRO>(ts, cpl, r) : st_kernel_v<F, 0, M1_PLAIN, PRO>(ts, cpl, r);
    return nullptr;
}

// Kernels of format F (each defined in its own translation unit).
template <int F>
m1_fn st_pick(int ts, int cpl, int r, int senc, int mode, int pro);

#define VQ_ST_PICK(F)                                                            \
    template <>                                                                  \
    m1_fn st_pick<F>(int ts, int cpl, int r, int senc, int mode, int pro) {      \
        switch (pro) {                                                           \
            case PRO_INT8: return st_pick_pro<F, PRO_INT8>(ts, cpl, r, senc, mode);       \
            case PRO_RMSNORM: return st_pick_pro<F, PRO_RMSNORM>(ts, cpl, r, senc, mode); \
            case PRO_SWIGLU: return st_pick_pro<F, PRO_SWIGLU>(ts, cpl, r, senc, mode);   \
            default: return st_pick_pro<F, PRO_BF16>(ts, cpl, r, senc, mode);             \
        }                                                                        \
    }

}  // namespace vq
