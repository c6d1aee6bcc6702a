// Host side of the streaming skinny GEMM (qgemm_stream.h): launch shape, and
// the choice between it and the row-contiguous kernel (qgemm_rc.h).
#include "qgemm_stream.h"

namespace vq {

// Groups per wave and phase, phases, and rows per workgroup: one workgroup per
// CU, every CU the same rows (both matrices of a pair together), at most 1024
// a workgroup so that the phases' row sums (64 bytes a row) fit LDS.
struct SgLaunch {
    int np, pg, rpw;
    sg_fn fn;
    size_t lds;
};
constexpr int SG_RPW_MAX = 1024;

static long sg_rows(int N, bool pair) { return pair ? 2L * N : N; }

static bool sg_launch(int qtype, long rows_total, int K, int M, int am, bool part, int senc, SgLaunch& l) {
    const int F = qtype == VIPER_QTYPE_W8_G32 ? 8 : qtype, G = group_of(qtype), NG = K / G;
    const int most = SG_W * 2 * sg_ni_max(F, am, part);
    const long rpw = (rows_total + device_cus() - 1) / device_cus();
    l.np = (NG + most - 1) / most;
    l.pg = (NG + l.np - 1) / l.np;
    l.rpw = (int)(rpw < SG_RPW_MAX ? rpw : SG_RPW_MAX);
    const int gw = (l.pg + SG_W - 1) / SG_W;
    const bool pack = M <= 8;
    switch (qtype) {
        case VIPER_QTYPE_Q4_G64: l.fn = sg_pick_q4(gw, am, pack, part, senc, &l.lds); break;
        case VIPER_QTYPE_Q5_G64: l.fn = sg_pick_q5(gw, am, pack, part, senc, &l.lds); break;
        case VIPER_QTYPE_Q6_G64: l.fn = sg_pick_q6(gw, am, pack, part, senc, &l.lds); break;
        default: l.fn = sg_pick_w8(gw, am, pack, part, senc, &l.lds); break;
    }
    if (l.fn == nullptr) return false;
    if (am == RC_BF16) l.lds += sg_act_lds(G, 8, NG);
    else if (l.np > 1) l.lds += (size_t)l.rpw * 64;
    return l.lds <= (size_t)device_lds_max();
}

// Phases over K: the groups one workgroup's waves hold in registers.
int sg_phases(int qtype, int K, int am) {
    const int F = qtype == VIPER_QTYPE_W8_G32 ? 8 : qtype, most = SG_W * 2 * sg_ni_max(F, am, false);
    return (K / group_of(qtype) + most - 1) / most;
}

// RC_BF16: at most 8 rows (the slots of the LDS copy), one phase, every row's
// octet pairs in SG_XR rounds.
bool sg_bf16_ok(int qtype, int N, int K, int M, bool pair) {
    if (M > 8 || (long)M * K > (long)SG_XR * 64 * SG_W * 16) return false;
    SgLaunch l;
    return sg_launch(qtype, sg_rows(N, pair), K, M, RC_BF16, false, 0, l) && l.np == 1;
}

// Which calls of whole group quads the streaming kernel takes from the
// row-contiguous kernel: those whose rows exceed one round of its workgroups
// (its two-quad and segment-loop kernels, see rc_capped), where that ran the
// chip in several rounds (fragments, M = 16, us, row-contiguous / streaming: Q4
// N = 10240 K = 4096 12.2 / 9.0, K = 5120 13.7 / 10.9, K = 6144 19.3 / 11.7; Q5
// N = 10240 K = 4096 13.7 / 10.3; Q6 13.2 / 11.4; W8 N = 10240 K = 3072 16.3 /
// 11.0; and where it holds them: Q4 N = 5120 K = 4096 6.4 / 6.8, K = 5120
// 7.0 / 8.3, N = 10240 K = 3072 6.4 / 7.7).
// Of those only K of one phase, or two of Q4 (K = 11776, N = 13696, M = 16
// 40.8 / 30.6): serial phases cost more than rounds of workgroups (Q5, four
// phases, K = 12800, N = 6400, M = 6 26.1 / 29.2; K = 12544, N = 7815, M = 3
// 26.6 / 29.4).
// Where both kernels' rounds cover the same padded rows (16-row tiles here, its
// workgroups' rows there) and the waves' groups leave part of a step of four
// idle, up to 4 bf16 rows of Q4 and more than 8 int8 rows of all but Q6 stay
// there (Q4, N = 13312..16384, row-contiguous / streaming: 4 bf16 rows of K =
// 3328 9.7 / 10.5, 16 int8 rows of K = 4608 14.4 / 16.3; of K = 4096, whole steps,
// 13.9 / 11.9; fragments of K = 3328 10.4 / 10.0, 7 int8 rows of a pair of K =
// 3584 20.8 / 18.6; Q6, N = 10000, 4 bf16 rows of K = 3328 12.1 / 10.7).
// Two bf16 rows, up to 64 per CU, also leave the other kernels of that family
// for one that pads fewer rows (Q5, K = 2048, N = 14000 11.3 / 8.3).
bool sg_takes(int qtype, int N, int K, int M, bool pair, int am) {
    if (!rc_ok(qtype, K)) return true;
    const long total = sg_rows(N, pair);
    const int phases = sg_phases(qtype, K, RC_FRAG);
    if (phases > (qtype == VIPER_QTYPE_Q4_G64 ? 2 : 1)) return false;
    int rows;
    const int rounds = rc_rounds(qtype, total, K, &rows);
    const long per_cu = (total + device_cus() - 1) / device_cus();
    if (!rc_capped(qtype, total, K))
        return am == RC_BF16 && M == 2 && !pair && rounds > 1 && per_cu <= 64 && (per_cu + 15) / 16 * 16 < (long)rounds * rows;
    const int gw = (K / group_of(qtype) + SG_W - 1) / SG_W;
    const bool even = rows > 16 && (per_cu + 15) / 16 * 16 == (long)rounds * rows && gw % 4 != 0;
    return !(even && !pair && ((am == RC_NAT && M > 8 && qtype != VIPER_QTYPE_Q6_G64) ||
                               (am == RC_BF16 && M <= 4 && qtype == VIPER_QTYPE_Q4_G64)));
}

// K of an even number of groups, not a multiple of four: this kernel, or the
// one that gathers group pairs (qgemm_mfma.hip)?  That one has the shorter
// chain after a workgroup's weights arrive (no LDS transpose, four waves up to
// 40 groups, one load segment up to 80) and as many workgroups as there are
// row blocks; this one streams.  So it takes, us, pairs / streaming:
//  * short rows: up to 24 groups (Q4, M = 16, K = 384, N = 2048 / 24576, two
//    launches 3.9 / 4.5 and 7.2 / 10.3; int8 rows 2.1 / 2.3, 5.7 / 7.5, but N =
//    256 the other way by 6 %), up to 40 after a quantize launch, for W8, or for
//    at most 16 rows per CU;
//  * few rows per CU (16) where one load segment of it holds what this kernel
//    needs more steps for (Q4, M = 16, N = 2048, K = 4224 6.0 / 6.8; Q6, M = 8
//    8.3 / 9.5, and there, in two phases, up to 40: N = 6144 12.0 / 13.3);
//  * 9 and more rows of Q4 / W8 over many short rows, more tiles than its waves
//    can hide (M = 16, N = 24000, K = 3712 18.5 / 20.2 with a residual, W8, K =
//    2112 18.1 / 23.0; N = 10240 the other way);
//  * few rows per CU and a K of several phases (Q4, M = 16, N = 2048, K = 8320
//    11.0 / 13.3), where those are not nearly full (Q5, K = 6784 10.0 / 9.6).  Of
//    int8 rows, which that kernel gathers, only 9 and more of 128 groups (Q4,
//    M = 16, K = 8320 1.06 times, M = 8 0.98; K = 7552 8.4 against 9.9 here).
// Never for more groups than its staged scales hold (W8, M = 12, K = 13248, N =
// 256 25.7 / 20.5).  A call of one launch here (up to 8 bf16 rows of one phase) is compared with
// its two: there only many short rows (Q4, K = 384, N = 24576, M = 8 9.0 / 10.4;
// N = 16384 equal) and many values a workgroup quantizes (Q4, M = 8, K = 4224,
// N = 2048 6.6 / 7.3).
bool sg_over_mf(int qtype, int N, int K, int M, bool pair, int am) {
    if (M < 2 || !mf_ok(qtype, K)) return true;
    const int NG = K / group_of(qtype), F = qtype == VIPER_QTYPE_W8_G32 ? 8 : qtype;
    const long per_cu = (sg_rows(N, pair) + device_cus() - 1) / device_cus();
    const bool wide = F == 5 || F == 6, nat = am == RC_NAT;
    if (nat ? NG > 384 || per_cu <= 1 : !mf_frag_ok(qtype, N, K)) return true;
    if (am == RC_BF16) return !((NG <= (wide ? 12 : F == 8 ? 24 : 40) && per_cu > 80) || ((long)M * K >= 32768 && per_cu <= 16));
    if (NG <= 40 && (per_cu <= 16 || NG <= (wide && nat ? 8 : 24) || !nat || F == 8)) return false;
    if (NG > 64 && NG <= 80 && per_cu <= (wide && !nat ? 40 : 16)) return false;
    if (!nat && M > 8 && !wide && NG <= 80 && per_cu > (F == 8 ? 48 : 80)) return false;
    const int phases = sg_phases(qtype, K, am), cap = phases * SG_W * 2 * sg_ni_max(F, am, false);
    if (phases == 1 || per_cu > 16) return true;
    return nat ? M <= 8 || wide || NG < 128 : wide && NG * 20 >= cap * (phases == 2 ? 15 : 16);
}

int launch_sg(int qtype, const void* w, const void* s, int senc, int N, int K, const void* xq, const void* xs, int am,
              int M, void* y, const void* res, int32_t* part, const void* w1, const void* s1, void* y1, hipStream_t st) {
    const bool pair = w1 != nullptr;
    if (M < 1 || M > 16 || (part != nullptr && am != RC_FRAG)) return VIPER_INTERNAL;
    if (am == RC_BF16 && !sg_bf16_ok(qtype, N, K, M, pair)) return VIPER_INTERNAL;
    // (the limit of the row-contiguous kernel's argument word, for every K of whole group pairs)
    if (M >= 2 && (K / group_of(qtype)) % 2 == 0 && N >= (1 << 27)) return VIPER_INVALID_ARGUMENT;
    SgLaunch l;
    if (!sg_launch(qtype, sg_rows(N, pair), K, M, am, part != nullptr, senc, l)) return VIPER_INTERNAL;
    const unsigned nb = ((unsigned)N + (unsigned)l.rpw - 1) / (unsigned)l.rpw * (pair ? 2u : 1u), gx = (nb + 7) / 8;
    if (gx >= 1u << 20) return VIPER_INVALID_ARGUMENT;
    const int8_t* a0 = (const int8_t*)xq;
    const float* a1 = (const float*)xs;
    const uint8_t* a2 = (const uint8_t*)w;
    const uint16_t* a3 = (const uint16_t*)s;
    uint16_t* a4 = (uint16_t*)y;
    const uint16_t* a5 = (const uint16_t*)res;
    const uint8_t* b0 = (const uint8_t*)w1;
    const uint16_t* b1 = (const uint16_t*)s1;
    uint16_t* b2 = (uint16_t*)y1;
    unsigned kk = (unsigned)(K / 32) | (unsigned)(l.pg - 1) << 20;
    unsigned rg = (unsigned)l.rpw | gx << 12, ms = (unsigned)(M - 1) | (senc ? 16u : 0u);
    void* args[] = {&a0, &a1, &a2, &a3, &a4, &kk, &N, &rg, &ms, &a5, &part, &b0, &b1, &b2};
    launch((const void*)l.fn, 8 * gx, 64 * SG_W, l.lds, st, args);
    return status_of(hipGetLastError());
}

int launch_sg_timeline(int qtype, const void* w, const void* s, int senc, int N, int K, const void* xq, const void* xs, int M,
                       void* y, uint64_t* stamps, size_t stamp_bytes, int* workgroups, int* waves, hipStream_t st) {
    SgLaunch l;
    if (M < 2 || M > 16 || N >= (1 << 27) || !sg_launch(qtype, N, K, M, RC_FRAG, false, senc, l)) return VIPER_INVALID_ARGUMENT;
    const int gw = (l.pg + SG_W - 1) / SG_W;
    l.fn = qtype == VIPER_QTYPE_W8_G32 ? sg_pick_tl8(gw, M <= 8) : qtype == VIPER_QTYPE_Q4_G64 ? sg_pick_tl4(gw, M <= 8) : nullptr;
    if (l.fn == nullptr) return VIPER_INVALID_ARGUMENT;
    const unsigned nb = ((unsigned)N + (unsigned)l.rpw - 1) / (unsigned)l.rpw, gx = (nb + 7) / 8;
    if (gx >= 1u << 20 || stamps == nullptr || stamp_bytes < (size_t)nb * SG_W * RC_TL_STAMPS * sizeof(uint64_t))
        return VIPER_INVALID_ARGUMENT;
    if (workgroups != nullptr) *workgroups = (int)nb;
    if (waves != nullptr) *waves = SG_W;
    const void* none = nullptr;
    unsigned kk = (unsigned)(K / 32) | (unsigned)(l.pg - 1) << 20;
    unsigned rg = (unsigned)l.rpw | gx << 12, ms = (unsigned)(M - 1) | (senc ? 16u : 0u);
    void* args[] = {&xq, &xs, &w, &s, &y, &kk, &N, &rg, &ms, &none, &stamps, &none, &none, &none};
    launch((const void*)l.fn, 8 * gx, 64 * SG_W, l.lds, st, args);
    return status_of(hipGetLastError());
}

}  // namespace vq
