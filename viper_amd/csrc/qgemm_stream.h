// Skinny GEMM on the i8 matrix cores of gfx950 for every K that is a multiple
// of the group: one template, instantiated per format in
// qgemm_stream_{q4,q5,q6,w8}.hip; dispatch in qgemm_stream.hip.
//
// Semantics are those of the reference's multi-row path
// (kernels/ops/linear_multim.cu:64-130): per group, the int32 dot of the
// weight codes with the int8 activations, scaled by ws * xs in fp32 and
// summed over groups.
//
// What bounds it: HBM reads of the weights and, with only two or three tiles
// of rows per workgroup, the latency from the launch to the first products
// (K = 4096, N = 10240, Q4: the activations' loads 0.8 us, the first tile in
// LDS after 2.6 us, then 0.85 us per 16 rows).  So:
//  * a workgroup of 8 waves owns N / CUs consecutive rows (persistent: one
//    workgroup per CU), so the activations are read and unpacked once per CU;
//  * the waves split K by whole groups, contiguous per wave, and keep their
//    groups' activation operands in registers; a group never spans lanes of
//    two waves, so any number of groups works (an odd number too);
//  * weights arrive as 16-byte chunks, contiguous along the wave's part of
//    each row, one tile of 16 rows ahead of the products, and reach the
//    matrix-core layout through wave-private LDS (no workgroup barrier);
//  * the cross-wave sum is double-buffered: one barrier per tile, and one
//    wave adds and stores while the others go on;
//  * for at most 8 rows, two groups share an accumulator (the activations of
//    group h in columns 0..7 for even h, 8..15 for odd h, zeros elsewhere):
//    half the scaling work.
// K too long for the registers runs in phases; the row sums of earlier phases
// wait in LDS.
//
// Measured (us per launch in a graph, distinct weights per launch; before:
// the v_dot4 and chunk-gathering matrix-core kernels this one replaced for K
// not a multiple of four groups, the row-contiguous kernel (qgemm_rc.h) else):
//   bf16 x, Q4, K = 3520, N = 2560 / 10240, M = 8: 19.3 -> 6.1 / 24.0 -> 9.8
//   bf16 x, Q6, K = 3520, N = 8192, M = 8: 23.8 -> 9.9 (2.4 TB/s of weights)
//   fragments, Q4, K = 4096, N = 10240, M = 16: 12.2 -> 9.0
//   fragments, Q4, K = 6144, N = 10240, M = 16: 19.3 -> 11.7 (2.9 TB/s)
//   fragments, W8, K = 3072, N = 10240, M = 16: 16.3 -> 11.0
// (16 waves per workgroup, 128 registers, spill; tiles of 32 and 48 rows took
// 15% longer at K = 2560, N = 2560 and the same, within 2%, at N = 10240.)
#pragma once

#include "qgemm_rc.h"

namespace vq {

constexpr int SG_W = 8;   // waves per workgroup
constexpr int SG_XR = 8;  // RC_BF16: octet pairs per thread

// Per format: high-plane bytes per row and group; the weight bytes of a
// product are SC * w (the code shifted to the top of the byte, its offset
// removed by flipping the top bit), so a group dot is SC * D and the
// activation scales carry 1 / SC (both exact).
template <int F> struct SgFmt;
template <> struct SgFmt<4> { static constexpr int HB = 0, SC = 16, SH = 4; };
template <> struct SgFmt<5> { static constexpr int HB = 8, SC = 8, SH = 3; };
template <> struct SgFmt<6> { static constexpr int HB = 16, SC = 4, SH = 2; };
template <> struct SgFmt<8> { static constexpr int HB = 0, SC = 1, SH = 0; };

// Four codes of a packed byte quadruple as SC * w in int8: word I of a
// quarter's two (see decode_word); H the quarter's high-plane word.
template <int F, int I>
__device__ __forceinline__ void sg_decode(uint32_t p, uint32_t H, uint32_t& even, uint32_t& odd) {
    if constexpr (F == 4) {
        even = ((p << 4) & 0xf0f0f0f0u) ^ 0x80808080u;
        odd = (p & 0xf0f0f0f0u) ^ 0x80808080u;
    } else if constexpr (F == 5) {  // bit 4 of the even (odd) codes: H bit 2I (2I + 1) of each byte
        even = ((p << 3) & 0x78787878u) | (~(H << (7 - 2 * I)) & 0x80808080u);
        odd = ((p >> 1) & 0x78787878u) | (~(H << (6 - 2 * I)) & 0x80808080u);
    } else {  // bits 4..5: H bits 4I (4I + 2) of each byte
        even = (((p << 2) & 0x3c3c3c3cu) | (shl<6 - 4 * I>(H) & 0xc0c0c0c0u)) ^ 0x80808080u;
        odd = (((p >> 2) & 0x3c3c3c3cu) | (shl<4 - 4 * I>(H) & 0xc0c0c0c0u)) ^ 0x80808080u;
    }
}

// LDS of one wave: the 16 weight rows of a tile (GWX groups) in row order, the
// high planes, the scales as [group][row].
template <int F, int NI>
struct SgShape {
    static constexpr int HB = SgFmt<F>::HB;
    static constexpr int GWX = 2 * NI;                  // most groups per wave and phase
    static constexpr int NH = HB ? (NI + 1) / 2 : 1;    // high-plane loads per lane
    static constexpr int NS = (GWX / 2 + 1 + 3) / 4;    // scale dwords per lane
    static constexpr int STR = GWX * 32 + 16;           // row strides
    static constexpr int HSTR = HB ? GWX * HB + HB : 0;
    static constexpr int SSTR = 32;                     // group stride of the scales (bytes)
    static constexpr int SCB = (GWX + 1) / 2 * 2 * SSTR;  // whole packs of groups
    static constexpr int WAVE = 16 * (STR + HSTR) + SCB;
    static constexpr int LDS = SG_W * WAVE + 2 * SG_W * 1024;  // and two buffers of cross-wave sums
    struct Tile {
        u32x4 v[NI];
        u32x4 h[NH];
        uint32_t sc[NS];
    };
};

// RC_BF16: LDS of the quantized rows, fragments [group][4][rows][QB] and scales
// [group][rows]
__host__ __device__ constexpr size_t sg_act_lds(int g, int rows, int ng) { return (size_t)ng * g * rows + (size_t)ng * rows * 4; }

// Arguments (the preloaded dwords hold all the common path reads): kk = K / 32
// in bits 0..19, groups per phase - 1 in bits 20..28; ms = M - 1 in bits 0..3,
// the scale encoding in bit 4; rg = rows per workgroup in bits 0..11,
// workgroups per XCD in bits 12..31.  AM, as in qgemm_rc.h: RC_FRAG, RC_NAT or
// RC_BF16 (xq = x; one phase).  PK: groups per accumulator, 2 for M <= 8, else
// 1.  SE: scale encoding, 2 = from ms.  PART: also store every int32 group dot
// (test and debug entry point).  TLM (measurement): `part` receives per-wave
// timestamps instead, as in qgemm_rc.h.
template <int F, int NI, int PK, int AM, int SE, bool PART, bool TLM = false>
__global__ void __launch_bounds__(64 * SG_W)
qgemm_stream_kernel(const int8_t* xq, const float* xs, const uint8_t* w, const uint16_t* ws, uint16_t* y, unsigned kk,
                    int N, unsigned rg, unsigned ms, const uint16_t* res, int32_t* __restrict__ part, const uint8_t* w1,
                    const uint16_t* ws1, uint16_t* y1) {
    using SH = SgShape<F, NI>;
    using Tile = typename SH::Tile;
    static_assert(!TLM || (!PART && AM == RC_FRAG), "timeline: fragment input");
    uint64_t tstamp[RC_TL_STAMPS];
    auto stamp = [&](int i) {
        if constexpr (TLM) tstamp[i] = __builtin_amdgcn_s_memrealtime();
    };
    stamp(0);
    constexpr int G = F == 8 ? 32 : 64, QB = F == 8 ? 8 : 16, HB = SH::HB, W = SG_W, NTT = 64 * SG_W, GWX = SH::GWX, NH = SH::NH, NS = SH::NS;
    constexpr int R2 = 16 / PK;               // columns per group: the rows of x, rounded up
    constexpr int NPK = (GWX + PK - 1) / PK;  // accumulator groups per wave and phase
    constexpr float XSC = 1.0f / SgFmt<F>::SC;
    const int K = (int)(kk & 0xfffffu) * 32, PG = (int)((kk >> 20) & 0x1ffu) + 1;
    const int M = (int)(ms & 15u) + 1;
    const bool senc = SE == 2 ? (ms & 16u) != 0 : SE == 1;
    const int rpw = (int)(rg & 0xfffu), gx = (int)(rg >> 12);
    const int NG = K / G, GW = (PG + W - 1) / W, NP = (NG + PG - 1) / PG;
    extern __shared__ __align__(16) uint8_t smem[];
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n16 = lane & 15, kb = lane >> 4, qi = ((kb & 1) << 1) | (kb >> 1);
    const int m = n16 & (R2 - 1), pj = n16 / R2;  // this lane's activation row and group of the pack

    int bid = ((int)blockIdx.x & 7) * gx + ((int)blockIdx.x >> 3);
    const int nb0 = (int)(((unsigned)N + (unsigned)rpw - 1) / (unsigned)rpw);
    if (__builtin_expect(bid >= nb0, 0)) {  // second matrix of a pair, or past a grid of whole XCD turns
        bid -= nb0;
        if (w1 == nullptr || bid >= nb0) return;
        w = w1;
        ws = ws1;
        y = y1;
        res = nullptr;
    }
    const int rbeg = bid * rpw, rend = rbeg + min(N - rbeg, rpw);
    const int ntile = (rend - rbeg + 15) / 16;
    uint8_t* tb = smem + wave * SH::WAVE;
    uint8_t* hb = tb + 16 * SH::STR;
    uint8_t* sb = hb + 16 * SH::HSTR;
    float* red = (float*)(smem + W * SH::WAVE);             // [2][W][64 lanes][4]
    uint8_t* ext = smem + SH::LDS;
    float* lac = (float*)ext;                               // NP > 1: [rpw][16] sums of earlier phases

    const int rbytes = NG * 32, hrb = NG * HB;
    // groups of phase p this wave owns: g0 .. g0 + gn - 1
    int g0 = wave * GW, gn = max(0, min(GW, min(NG, PG) - g0));
    // 16-byte chunk i * 64 + lane of the wave's rows is chunk c of row r
    int lo[NI], wo[NI], hl[NH], ho[NH];
    auto set_offsets = [&] {
        const float ic = 1.0f / (float)max(1, 2 * gn), ih = 1.0f / (float)max(1, gn);
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int idx = i * 64 + lane, r = (int)(((float)idx + 0.5f) * ic), c = idx - r * 2 * gn;
            const bool in = gn > 0 && r < 16;
            lo[i] = in ? r * rbytes + c * 16 : OOB;
            wo[i] = in ? r * SH::STR + c * 16 : -1;
        }
        if constexpr (HB != 0) {
#pragma unroll
            for (int i = 0; i < NH; ++i) {
                const int idx = i * 64 + lane, r = (int)(((float)idx + 0.5f) * ih), c = idx - r * gn;
                const bool in = gn > 0 && r < 16;
                hl[i] = in ? r * hrb + c * HB : OOB;
                ho[i] = in ? r * SH::HSTR + c * HB : -1;
            }
        }
    };
    auto load = [&](Tile& T, int t) {
        const int row0 = rbeg + t * 16, n = gn > 0 ? min(16, rend - row0) : 0;
        // scales: the wave's gn entries of each row, as dwords from the one
        // that holds the first (the array starts 16-byte aligned)
        const size_t sbyte = (size_t)row0 * NG * 2;
        const int rel = (int)(sbyte & 2);
        const size_t left = ((size_t)N * NG * 2 - (sbyte - rel)) & ~(size_t)3;
        const uint32_t want = (uint32_t)((rel + n * NG * 2 + 3) & ~3);
        const auto sr = buf((const uint8_t*)ws + (sbyte - rel), n ? (left < want ? (uint32_t)left : want) : 0u);
        const int b0 = (rel + (n16 * NG + g0) * 2) & ~3;
#pragma unroll
        for (int i = 0; i < NS; ++i) T.sc[i] = bload4(sr, kb + 4 * i <= gn / 2 ? b0 + (kb + 4 * i) * 4 : OOB);
        const auto wr = buf(w + (size_t)row0 * rbytes + (size_t)g0 * 32, n ? (uint32_t)(n * rbytes - g0 * 32) : 0u);
#pragma unroll
        for (int i = 0; i < NI; ++i) T.v[i] = bload16<AUX_NT>(wr, lo[i]);
        if constexpr (HB != 0) {
            const auto hr = buf(w + (size_t)N * rbytes + (size_t)row0 * hrb + (size_t)g0 * HB,
                                n ? (uint32_t)(n * hrb - g0 * HB) : 0u);
#pragma unroll
            for (int i = 0; i < NH; ++i) {
                if constexpr (HB == 8) {
                    const u32x2 t = bload8<AUX_NT>(hr, hl[i]);
                    T.h[i] = u32x4{t.x, t.y, 0u, 0u};
                } else {
                    T.h[i] = bload16<AUX_NT>(hr, hl[i]);
                }
            }
        }
    };

    // Activation operands of the wave's groups: for group h the lane's k-slot
    // of row m where h is the lane's group of its pack, else zero, so that the
    // products of a pack's groups add up in one accumulator, each in its own
    // columns; and the lane's scale of each pack (0 past the wave's groups).
    i32x4 B[GWX];
    float X[NPK];
    const auto xr = buf(xq, AM == RC_BF16 ? (uint32_t)(M * K) * 2 : AM == RC_NAT ? (uint32_t)(M * K) : (uint32_t)NG * 64 * QB);
    const auto xsr = buf(xs, AM == RC_BF16 ? 0u : AM == RC_NAT ? (uint32_t)(M * NG) * 4 : (uint32_t)NG * 64);
    auto act_load = [&] {
#pragma unroll
        for (int h = 0; h < GWX; ++h) {
            const int g = g0 + h;
            const bool in = h < gn && h % PK == pj && (AM != RC_NAT || m < M);
            const int o = !in ? OOB : AM == RC_NAT ? m * K + g * G + qi * QB : (g * 64 + 16 * kb + m) * QB;
            if constexpr (QB == 16) {
                const u32x4 v = bload16(xr, o);
                B[h] = i32x4{(int)v.x, (int)v.y, (int)v.z, (int)v.w};
            } else {
                const u32x2 v = bload8(xr, o);
                B[h] = i32x4{(int)v.x, (int)v.y, 0, 0};
            }
        }
#pragma unroll
        for (int p = 0; p < NPK; ++p) {
            const int h = p * PK + pj, g = g0 + h;
            const bool in = h < gn && (AM != RC_NAT || m < M);
            X[p] = __uint_as_float(bload4(xsr, !in ? OOB : AM == RC_NAT ? (m * NG + g) * 4 : (g * 16 + m) * 4));
        }
    };
    auto act_ready = [&] {
        if constexpr (AM == RC_NAT && F != 8) {  // k order -> [even | odd] per octet
#pragma unroll
            for (int h = 0; h < GWX; ++h) {
                const u32x4 v = {(uint32_t)B[h].x, (uint32_t)B[h].y, (uint32_t)B[h].z, (uint32_t)B[h].w};
                B[h] = i32x4{(int)__builtin_amdgcn_perm(v.y, v.x, 0x06040200u), (int)__builtin_amdgcn_perm(v.y, v.x, 0x07050301u),
                             (int)__builtin_amdgcn_perm(v.w, v.z, 0x06040200u), (int)__builtin_amdgcn_perm(v.w, v.z, 0x07050301u)};
            }
        }
#pragma unroll
        for (int p = 0; p < NPK; ++p) X[p] *= XSC;
    };

    set_offsets();
    Tile T0, T1;
    if constexpr (AM == RC_BF16) {
        // every workgroup quantizes the rows into LDS while its first tile's
        // weights are in flight (one phase)
        int8_t* lxa = (int8_t*)ext;
        float* lxs = (float*)(ext + (size_t)NG * G * R2);
        const int np = M * K / 16;  // octet pairs
        u32x4 xv[SG_XR], xw[SG_XR];
#pragma unroll
        for (int i = 0; i < SG_XR; ++i) {
            if (NTT * i >= np) break;  // uniform: an out-of-range load is not free
            xv[i] = bload16(xr, (tid + NTT * i) * 32);
            xw[i] = bload16(xr, (tid + NTT * i) * 32 + 16);
        }
        issue_fence();
        load(T0, 0);
        issue_fence();
#pragma unroll
        for (int i = 0; i < SG_XR; ++i) {
            const int j = tid + NTT * i;
            if (j - lane >= np) break;  // whole waves, so that every group reduction sees whole groups
            uint32_t d0, d1, d2, d3;
            float sc;
            quantize_octet_pair<G, (F != 8)>(xv[i], xw[i], d0, d1, d2, d3, sc);
            if (j < np) {
                const int kp = K / 16, mm = j / kp, k2 = j - mm * kp;  // pair k2 of row mm
                if constexpr (G == 64) {
                    const int g = k2 >> 2, q = k2 & 3, ks = ((q & 1) << 1) | (q >> 1);
                    *(u32x4*)(lxa + ((size_t)(g * 4 + ks) * R2 + mm) * 16) = u32x4{d0, d1, d2, d3};
                    if (q == 0) lxs[g * R2 + mm] = sc;
                } else {
                    const int g = k2 >> 1, q0 = (k2 & 1) * 2, q1 = q0 + 1;
                    const int s0 = ((q0 & 1) << 1) | (q0 >> 1), s1 = ((q1 & 1) << 1) | (q1 >> 1);
                    *(u32x2*)(lxa + ((size_t)(g * 4 + s0) * R2 + mm) * 8) = u32x2{d0, d1};
                    *(u32x2*)(lxa + ((size_t)(g * 4 + s1) * R2 + mm) * 8) = u32x2{d2, d3};
                    if (q0 == 0) lxs[g * R2 + mm] = sc;
                }
            }
        }
        lds_barrier();
#pragma unroll
        for (int h = 0; h < GWX; ++h) {
            const int hc = min(h, max(gn, 1) - 1), g = min(g0 + hc, NG - 1);
            const bool in = h < gn && h % PK == pj;
            if constexpr (QB == 16) {
                const u32x4 v = *(const u32x4*)(lxa + ((size_t)(g * 4 + kb) * R2 + m) * 16);
                B[h] = i32x4{in ? (int)v.x : 0, in ? (int)v.y : 0, in ? (int)v.z : 0, in ? (int)v.w : 0};
            } else {
                const u32x2 v = *(const u32x2*)(lxa + ((size_t)(g * 4 + kb) * R2 + m) * 8);
                B[h] = i32x4{in ? (int)v.x : 0, in ? (int)v.y : 0, 0, 0};
            }
        }
#pragma unroll
        for (int p = 0; p < NPK; ++p) {
            const int h = p * PK + pj, g = min(g0 + h, NG - 1);
            const float v = lxs[g * R2 + m];
            X[p] = h < gn ? v : 0.0f;
        }
    } else {
        act_load();
        issue_fence();
        stamp(1);
        load(T0, 0);
        issue_fence();
        stamp(2);
    }
    // scales past the wave's groups stay zero (their products must be finite)
    for (int i = lane; i < SH::SCB / 4; i += 64) ((uint32_t*)sb)[i] = 0u;
    act_ready();

    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    };
    // The residual's values are requested by the wave that will sum the tile, once
    // the tile is in LDS: a wait for them at the store held every wave at the
    // next barrier (Q4, M = 10, K = 3200, N = 23260 16.9 us without a residual,
    // 20.4 with).  The shapes with no register left wait there.
    constexpr bool AHEAD = !PART && !(F == 4 && NI == 6) && !(F == 8 && NI == 8);
    int rb = 0;
    auto compute = [&](Tile& T, int t, int p) {
        const int row0 = rbeg + t * 16, n = min(16, rend - row0);
        wave_sync();
        const int rel = (int)(((size_t)row0 * NG * 2) & 2);
        const int odd = ((rel >> 1) + n16 * NG + g0) & 1;
#pragma unroll
        for (int i = 0; i < NS; ++i) {
            const int ga = 2 * (kb + 4 * i) - odd;  // groups ga, ga + 1
            uint16_t* o = (uint16_t*)(sb + ga * SH::SSTR) + n16;
            if (ga >= 0 && ga < gn) o[0] = (uint16_t)T.sc[i];
            if (ga + 1 < gn) o[16] = (uint16_t)(T.sc[i] >> 16);
        }
        // a scale array of an odd number of entries ends within a dword: its
        // last entry is read on its own
        if (__builtin_expect((N & NG & 1) && row0 + n == N && gn > 0 && g0 + gn == NG, 0)) {
            const uint32_t last = bload2(buf(ws + (size_t)N * NG - 1, 2u), lane == 0 ? 0 : OOB);
            if (lane == 0) *((uint16_t*)(sb + (gn - 1) * SH::SSTR) + n - 1) = (uint16_t)last;
        }
#pragma unroll
        for (int i = 0; i < NI; ++i)
            if (wo[i] >= 0) *(u32x4*)(tb + wo[i]) = T.v[i];
        if constexpr (HB != 0) {
#pragma unroll
            for (int i = 0; i < NH; ++i)
                if (ho[i] >= 0) {
                    if constexpr (HB == 8) *(u32x2*)(hb + ho[i]) = u32x2{T.h[i].x, T.h[i].y};
                    else *(u32x4*)(hb + ho[i]) = T.h[i];
                }
        }
        wave_sync();
        if (TLM && t == 0 && p == 0) stamp(3);
        const bool sums = (t & (W - 1)) == wave, add = res != nullptr && p + 1 == NP;
        const size_t o0 = (size_t)n16 * N + row0 + 4 * kb;
        uint16_t rv[4] = {0, 0, 0, 0};
        if (AHEAD && __builtin_expect(add, 0) && sums && n16 < M) {
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (4 * kb + r < n) rv[r] = res[o0 + r];
        }
        float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        const uint8_t* tp = tb + n16 * SH::STR + qi * 8;
        const uint8_t* hp = hb + n16 * SH::HSTR + (HB == 8 ? (qi >> 1) * 4 : qi * 4);
        const uint8_t* sp = sb + pj * SH::SSTR + kb * 8;
        // four groups at a time: their LDS reads, then the products, then the
        // scaling, so that the LDS and matrix-core latencies overlap
        constexpr int U = 4, UP = U / PK;
        static_assert(GWX % U == 0 || GWX % U == 2, "whole packs");
#pragma unroll
        for (int h0 = 0; h0 < GWX; h0 += U) {
            if (h0 < gn) {
                u32x2 P[U], Z[UP];
                uint32_t H[U];
                i32x4 C[UP];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (h0 + u >= GWX) continue;
                    P[u] = *(const u32x2*)(tp + (h0 + u) * 32);
                    H[u] = 0u;
                    if constexpr (HB == 8) H[u] = *(const uint32_t*)(hp + (h0 + u) * 8) >> (4 * (qi & 1));
                    else if constexpr (HB == 16) H[u] = *(const uint32_t*)(hp + (h0 + u) * 16);
                    if (u % PK == 0) Z[u / PK] = *(const u32x2*)(sp + (h0 + u) * SH::SSTR);
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    if (h0 + u >= GWX) continue;
                    const i32x4 C0 = u % PK == 0 ? i32x4{0, 0, 0, 0} : C[u / PK];
                    const u32x2 q = P[u];
                    const i32x4 b = B[h0 + u < GWX ? h0 + u : 0];
                    if constexpr (F == 8) {
                        C[u / PK] = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                            (long)(((uint64_t)q.y << 32) | q.x), (long)(((uint64_t)(uint32_t)b.y << 32) | (uint32_t)b.x), C0, 0,
                            0, 0);
                    } else {
                        uint32_t e0, d0, e1, d1;
                        sg_decode<F, 0>(q.x, H[u], e0, d0);
                        sg_decode<F, 1>(q.y, H[u], e1, d1);
                        C[u / PK] =
                            __builtin_amdgcn_mfma_i32_16x16x64_i8(i32x4{(int)e0, (int)d0, (int)e1, (int)d1}, b, C0, 0, 0, 0);
                    }
                }
#pragma unroll
                for (int v = 0; v < UP; ++v) {
                    if (h0 + v * PK >= GWX) continue;
                    const u32x2 z = Z[v];
                    const uint32_t zr[4] = {z.x & 0xffffu, z.x >> 16, z.y & 0xffffu, z.y >> 16};
                    const float x = X[h0 / PK + v < NPK ? h0 / PK + v : 0];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float wsf = senc ? bf16f(zr[r]) : f16f(zr[r]);
                        acc[r] = __builtin_fmaf(wsf * x, (float)C[v][r], acc[r]);
                    }
                    if constexpr (PART) {
                        const int h = h0 + v * PK + pj;
                        if (h < gn && m < M)
#pragma unroll
                            for (int r = 0; r < 4; ++r)
                                if (4 * kb + r < n)
                                    part[((size_t)m * N + row0 + 4 * kb + r) * NG + g0 + h] = C[v][r] >> SgFmt<F>::SH;
                    }
                }
            }
            if (TLM && h0 == 0 && t == 0 && p == 0) stamp(4);
        }
        stamp(5);
        // the pack's groups, then the waves in order (two buffers in turn: one
        // barrier per tile), by one wave, in turn
        float* rd = red + rb * (W * 256);
        rb ^= 1;
        if constexpr (PK == 2) {
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] += dpp_f<0x128>(acc[r]);  // row_ror:8
        }
        *(float4*)(rd + (wave * 64 + lane) * 4) = make_float4(acc[0], acc[1], acc[2], acc[3]);
        lds_barrier();
        stamp(6);
        stamp(7);
        if (!sums) return;
        float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < W; ++u) {
            const float4 a = *(const float4*)(rd + (u * 64 + lane) * 4);
            v[0] += a.x;
            v[1] += a.y;
            v[2] += a.z;
            v[3] += a.w;
        }
        if (n16 < M) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int nl = 4 * kb + r;
                if (nl >= n) continue;
                float* ac = lac + (t * 16 + nl) * 16 + n16;  // written and read by this lane only
                float z = v[r];
                if (p > 0) z += *ac;
                if (p + 1 < NP) {
                    *ac = z;
                } else {
                    if (__builtin_expect(add, 0)) z += bf16f(AHEAD ? rv[r] : res[o0 + r]);
                    y[o0 + r] = f2bf(z);
                }
            }
        }
        stamp(7);
    };
    for (int p = 0;;) {
        // (separate code for the last tile, so that no wait counts loads that
        // may not have been issued)
        for (int t = 0;;) {
            if (t + 1 == ntile) {
                compute(T0, t, p);
                break;
            }
            load(T1, t + 1);
            issue_fence();
            compute(T0, t, p);
            if (t + 2 == ntile) {
                compute(T1, t + 1, p);
                break;
            }
            load(T0, t + 2);
            issue_fence();
            compute(T1, t + 1, p);
            t += 2;
        }
        if (AM == RC_BF16 || ++p == NP) break;
        // the next phase's groups
        g0 = p * PG + wave * GW;
        gn = max(0, min(GW, min(NG, (p + 1) * PG) - g0));
        set_offsets();
        act_load();
        issue_fence();
        load(T0, 0);
        issue_fence();
        wave_sync();
        for (int i = lane; i < SH::SCB / 4; i += 64) ((uint32_t*)sb)[i] = 0u;
        act_ready();
    }
    if constexpr (TLM) {
        // (no second matrix: bid counts the workgroups that have rows; the
        // points of the K split repeat the last one)
        if (lane == 0) {
            uint64_t* o = (uint64_t*)part + ((size_t)bid * W + wave) * RC_TL_STAMPS;
#pragma unroll
            for (int i = 0; i < RC_TL_STAMPS; ++i) o[i] = tstamp[i < 7 ? i : 7];
        }
    }
}

// ------------------------------------------------------------------ host side

typedef void (*sg_fn)(const int8_t*, const float*, const uint8_t*, const uint16_t*, uint16_t*, unsigned, int, unsigned, unsigned,
                      const uint16_t*, int32_t*, const uint8_t*, const uint16_t*, uint16_t*);

// Most chunk loads per lane (groups per wave / 2) that keep two tiles in
// flight without spilling.
__host__ __device__ constexpr int sg_ni_max(int F, int am, bool part) {
    return F == 8 ? (am == RC_NAT || part ? 6 : 8) : F == 4 ? 6 : 4;
}

template <int F, int NI>
sg_fn sg_pick_ni(int am, bool pack, bool part, int senc) {
    if constexpr (NI <= sg_ni_max(F, RC_NAT, true)) {
        if (part) return qgemm_stream_kernel<F, NI, 1, RC_FRAG, 2, true>;
        if (am == RC_NAT) {
            if (pack) return senc ? qgemm_stream_kernel<F, NI, 2, RC_NAT, 1, false> : qgemm_stream_kernel<F, NI, 2, RC_NAT, 0, false>;
            return senc ? qgemm_stream_kernel<F, NI, 1, RC_NAT, 1, false> : qgemm_stream_kernel<F, NI, 1, RC_NAT, 0, false>;
        }
    }
    if (part || am == RC_NAT) return nullptr;
    if (am == RC_BF16)
        return senc ? qgemm_stream_kernel<F, NI, 2, RC_BF16, 1, false> : qgemm_stream_kernel<F, NI, 2, RC_BF16, 0, false>;
    if (pack) return senc ? qgemm_stream_kernel<F, NI, 2, RC_FRAG, 1, false> : qgemm_stream_kernel<F, NI, 2, RC_FRAG, 0, false>;
    return senc ? qgemm_stream_kernel<F, NI, 1, RC_FRAG, 1, false> : qgemm_stream_kernel<F, NI, 1, RC_FRAG, 0, false>;
}

// The kernel for gw groups per wave and its LDS without the mode's own (nullptr:
// gw needs phases).
template <int F>
sg_fn sg_pick(int gw, int am, bool pack, bool part, int senc, size_t* lds) {
#define VQ_SG(NI_)                                              \
    if constexpr (NI_ <= sg_ni_max(F, RC_FRAG, false))          \
        if (gw <= 2 * NI_) {                                    \
            *lds = SgShape<F, NI_>::LDS;                        \
            return sg_pick_ni<F, NI_>(am, pack, part, senc);    \
        }
    VQ_SG(1) VQ_SG(2) VQ_SG(3) VQ_SG(4) VQ_SG(6) VQ_SG(8)
#undef VQ_SG
    return nullptr;
}

// Timeline kernels (fragments; the groups per wave of K past one quad of the
// row-contiguous kernel, whose measurement entry point launches them).
template <int F>
sg_fn sg_pick_tl(int gw, bool pack) {
#define VQ_SG_TL(NI_)                                           \
    if constexpr (NI_ <= sg_ni_max(F, RC_FRAG, false))          \
        if (gw <= 2 * NI_)                                      \
            return pack ? qgemm_stream_kernel<F, NI_, 2, RC_FRAG, 2, false, true> : qgemm_stream_kernel<F, NI_, 1, RC_FRAG, 2, false, true>;
    if (gw <= 4) return nullptr;
    VQ_SG_TL(3) VQ_SG_TL(4) VQ_SG_TL(6) VQ_SG_TL(8)
#undef VQ_SG_TL
    return nullptr;
}
sg_fn sg_pick_tl4(int gw, bool pack);
sg_fn sg_pick_tl8(int gw, bool pack);

sg_fn sg_pick_q4(int gw, int am, bool pack, bool part, int senc, size_t* lds);
sg_fn sg_pick_q5(int gw, int am, bool pack, bool part, int senc, size_t* lds);
sg_fn sg_pick_q6(int gw, int am, bool pack, bool part, int senc, size_t* lds);
sg_fn sg_pick_w8(int gw, int am, bool pack, bool part, int senc, size_t* lds);

}  // namespace vq
