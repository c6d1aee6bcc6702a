// Host side of the M = 1 GEMV: launch shape and dispatch.
#include "qgemv_stream.h"

namespace vq {

struct M1Shape {
    int ts, ntt, cpl;
};

static m1_fn m1_kernel(int qtype, const M1Shape& sh, int senc, int mode, bool exact, int pro, int mr = 1) {
    const bool folded = pro == PRO_RMSNORM || pro == PRO_SWIGLU;
    const int ts = sh.ts, ntt = sh.ntt, cpl = sh.cpl;
    switch (qtype) {
        case VIPER_QTYPE_Q4_G64:
            return folded ? m1_pick_folded<4>(ts, ntt, cpl, senc, mode, exact, pro, mr)
                          : m1_pick_plain<4>(ts, ntt, cpl, senc, mode, exact, pro, mr);
        case VIPER_QTYPE_Q5_G64:
            return folded ? m1_pick_folded<5>(ts, ntt, cpl, senc, mode, exact, pro, mr)
                          : m1_pick_plain<5>(ts, ntt, cpl, senc, mode, exact, pro, mr);
        case VIPER_QTYPE_Q6_G64:
            return folded ? m1_pick_folded<6>(ts, ntt, cpl, senc, mode, exact, pro, mr)
                          : m1_pick_plain<6>(ts, ntt, cpl, senc, mode, exact, pro, mr);
        default:
            return folded ? m1_pick_folded<8>(ts, ntt, cpl, senc, mode, exact, pro, mr)
                          : m1_pick_plain<8>(ts, ntt, cpl, senc, mode, exact, pro, mr);
    }
}

// A launch shape takes the exact-tiling kernels: TS * CPL chunks per row and
// a row's scales in whole 16-byte words.
static bool m1_exact(const M1Shape& sh, int cpr, int ngr) { return cpr == sh.ts * sh.cpl && ngr % 8 == 0; }

// Per-CU row load of a shape: ceil(ceil(N / rows) / CUs) * rows (rows per
// workgroup are halved for the swiglu pair, whose workgroups also read the
// same rows of the second matrix).
static long m1_load(const M1Shape& sh, int N, int cus, bool pair = false) {
    const long rows = pair ? sh.ntt / sh.ts / 2 : sh.ntt / sh.ts;
    const long groups = (N + rows - 1) / rows;
    return ((groups + cus - 1) / cus) * rows;
}

// Launch shape.  Exact tilings (TS * CPL == chunks per row) come first: their
// lanes need no masking and their scales arrive in one block.  Among them the
// smallest per-CU row load wins, then a workgroup that stages the activation
// row in one round (noct <= NTT: one octet per thread, a single quantize
// pass), then fewer chunk slots per lane (more lanes per row, so each lane's
// dot chain after the weights arrive is shorter), then the smaller workgroup
// (two 320-thread workgroups per CU beat one of 640 on the north-star shape:
// each quantizes and passes its barrier on its own).  One row of any other K
// takes the streaming kernel (st_shape).  MR > 1 rows with no exact tiling:
// the smallest team covering a row in 10 slots per lane (longer rows loop over
// segments of 64 lanes), workgroup size by row load, ties to more rows per
// workgroup (fewer redundant activation quantizations).
// MR > 1 rows: only the shapes m1_mr_shape_ok instantiates, with every row
// staged in M1_XS_MR rounds; there a workgroup that stages the rows in at
// most two rounds is taken first (the rows' quantize is repeated by every
// workgroup, so fewer, larger workgroups do less of it: 4 rows at K = 2560,
// 6.7 us with 640 threads against 7.4 us with 320), and the one-round
// preference does not apply (2 rows: 5.04 us with 320 threads, 5.03 us with
// 640).
static M1Shape m1_shape(int cpr, int N, int cus, int min_ntt, int noct, bool pair = false, int mr = 1) {
    M1Shape best{0, 0, 0};
    long best_load = -1;
    auto extra = [&](const M1Shape& c) { const int r = (noct + c.ntt - 1) / c.ntt; return r > 2 ? r - 2 : 0; };
    auto consider = [&](const M1Shape& c) {
        const long load = m1_load(c, N, cus, pair);
        const bool one = mr == 1 && c.ntt >= noct, best_one = mr == 1 && best.ntt >= noct;
        const int xr = extra(c), bxr = best.ntt ? extra(best) : 0;
        const bool take = best_load < 0 || load < best_load ||
                          (load == best_load &&
                           (xr < bxr ||
                            (xr == bxr &&
                             (one > best_one ||
                              (one == best_one && (c.cpl < best.cpl || (c.cpl == best.cpl && c.ntt < best.ntt)))))));
        if (take) {
            best = c;
            best_load = load;
        }
    };
    for (const auto& s : M1_SHAPES) {
        const M1Shape c{s[0], s[1], s[2]};
        if (c.ntt < min_ntt || c.ts * c.cpl != cpr || (pair && !m1_pair_ok(c.ts, c.ntt))) continue;
        if (mr > 1 && !m1_mr_shape_ok(c.ts, c.ntt, c.cpl)) continue;
        consider(c);
    }
    if (best.ntt != 0) return best;
    if (mr == 1) return best;
    int ts = 8;
    while (ts < 64 && ts * 10 < cpr) ts *= 2;
    for (const auto& s : M1_SHAPES) {
        const M1Shape c{s[0], s[1], s[2]};
        if (c.ts != ts || c.cpl != 10 || c.ntt < min_ntt || !m1_mr_shape_ok(c.ts, c.ntt, c.cpl)) continue;
        const long load = m1_load(c, N, cus);
        if (best_load < 0 || load < best_load || (load == best_load && c.ntt > best.ntt)) {
            best = c;
            best_load = load;
        }
    }
    return best;
}

// The reference engine's gate / up matrices (K = 3072, N = 10752) on the
// 384-thread tiling (24 rows, 448 workgroups) load some CUs with 48 rows
// against a 42-row mean.  One Q4 / Q5 matrix there takes the 44-row
// workgroup (M1_WIDE96, 245 workgroups) when its grid still covers 95 % of
// the CUs and it lowers the per-CU rows: N = 10752 Q4 5.06-5.16 -> 4.63-4.68
// us (int8 row 4.90-4.93 -> 4.72-4.73), Q5 6.04-6.09 -> 5.87-5.90 us,
// N = 11000 Q4 5.10-5.17 -> 4.69-4.70 us.  Not for Q6 (6.41-6.49 -> 7.03-7.14
// us) nor a grid that leaves CUs idle (Q4 N = 9000, 205 workgroups:
// 4.19-4.21 -> 4.25-4.38 us).
static M1Shape m1_wide96(int qtype, int cpr, int N, int cus, const M1Shape& sh) {
    if ((qtype != VIPER_QTYPE_Q4_G64 && qtype != VIPER_QTYPE_Q5_G64) || cpr != 96 || sh.ntt == 0) return sh;
    const M1Shape c{M1_WIDE96[0], M1_WIDE96[1], M1_WIDE96[2]};
    const long rows = c.ntt / c.ts, groups = (N + rows - 1) / rows;
    if (groups * 20 < (long)cus * 19) return sh;
    return m1_load(c, N, cus) < m1_load(sh, N, cus) ? c : sh;
}

// Q5 from a bf16 row on the 16-lane tiling of K = 2560: where one 40-row
// workgroup per CU carries as many rows as two of 20, it is faster (the
// north-star shape, config 4: 4.92-4.99 -> 4.79-4.80 us); Q4 keeps two
// workgroups of 20 (their quantize and barrier run independently: 3.8
// against 3.97 us), and so do Q5 from an int8 row (4.86-4.88 against
// 5.04-5.09 us) and Q6 (equal).
static M1Shape m1_q5_bf16(int qtype, int pro, int N, int cus, const M1Shape& sh) {
    if (qtype != VIPER_QTYPE_Q5_G64 || pro != PRO_BF16 || sh.ts != 16 || sh.ntt != 320 || sh.cpl != 5) return sh;
    const M1Shape c{16, 640, 5};
    return m1_load(c, N, cus) == m1_load(sh, N, cus) ? c : sh;
}

// Upper bound over the launch shapes (an exact tiling's scale block holds at
// most NTT * CPL bytes).
size_t lds_m1(int qtype, int K) {
    constexpr int kBlockMax = 640 * 10;
    switch (qtype) {
        case VIPER_QTYPE_Q4_G64: return m1_lds_bytes<4>(K, 0) + kBlockMax;
        case VIPER_QTYPE_Q5_G64: return m1_lds_bytes<5>(K, 0) + kBlockMax;
        case VIPER_QTYPE_Q6_G64: return m1_lds_bytes<6>(K, 0) + kBlockMax;
        default: return m1_lds_bytes<8>(K, 0) + kBlockMax;
    }
}

static size_t lds_m1_launch(int qtype, int K, int rows, bool exact, int mr = 1) {
    const int r = exact ? rows : 0;
    switch (qtype) {
        case VIPER_QTYPE_Q4_G64: return m1_lds_bytes<4>(K, r, mr);
        case VIPER_QTYPE_Q5_G64: return m1_lds_bytes<5>(K, r, mr);
        case VIPER_QTYPE_Q6_G64: return m1_lds_bytes<6>(K, r, mr);
        default: return m1_lds_bytes<8>(K, r, mr);
    }
}

static int m1_mr(int M) { return M <= 1 ? 1 : (M == 2 ? 2 : 4); }

bool m1_rows_ok(int qtype, int K, int M) {
    // every row is staged in the first M1_XS_MR rounds of the workgroup, and
    // some multi-row shape tiles the row (the shape does not depend on N)
    if (M < 2 || M > 4 || (long)M * (K / 8) > (long)M1_XS_MR * 640) return false;
    const int ck = qtype == VIPER_QTYPE_W8_G32 ? 16 : 32, noct = M * (K / 8);
    const M1Shape sh = m1_shape(K / ck, 1 << 14, device_cus(), (noct + M1_XS_MR - 1) / M1_XS_MR, noct, false, m1_mr(M));
    constexpr int kBlockMax = 640 * 10;
    return sh.ntt != 0 && lds_m1_launch(qtype, K, 0, false, m1_mr(M)) + kBlockMax <= (size_t)LDS_MAX;
}

bool m1_rows_exact(int qtype, int K, int M) {
    if (!m1_rows_ok(qtype, K, M)) return false;
    const int ck = qtype == VIPER_QTYPE_W8_G32 ? 16 : 32, noct = M * (K / 8);
    const M1Shape sh = m1_shape(K / ck, 1 << 14, device_cus(), (noct + M1_XS_MR - 1) / M1_XS_MR, noct, false, m1_mr(M));
    return m1_exact(sh, K / ck, K / group_of(qtype));
}

bool m1_rows_pair(int qtype, int K, int M) {
    // the multi-row shape stages its rows two octets per thread (m1_pairs)
    if (qtype != VIPER_QTYPE_Q4_G64 || !m1_rows_ok(qtype, K, M)) return false;
    const int noct = M * (K / 8);
    const M1Shape sh = m1_shape(K / 32, 1 << 14, device_cus(), (noct + M1_XS_MR - 1) / M1_XS_MR, noct, false, m1_mr(M));
    return m1_pairs<4>(m1_exact(sh, K / 32, K / 64), sh.ntt, m1_mr(M), PRO_BF16);
}

// The folded prologues hold the whole row after one load round.
bool m1_folded_ok(int qtype, int K) { return K <= 20480 && lds_m1(qtype, K) <= (size_t)LDS_MAX; }

// ------------------------------------------------------- streaming launches

// Launch shape of the streaming kernel: teams, slots and rows per unit, units
// per workgroup, workgroups per XCD (0: dispatch order) and workgroups per
// matrix.
struct StShape {
    int ts, cpl, r, upw, gx, grid, nb[3];
};

static StShape st_shape(int qtype, int K, const int* n, int nouts, int cus) {
    const int cpr = K / (qtype == VIPER_QTYPE_W8_G32 ? 16 : 32);
    StShape s{};
    s.ts = cpr <= 16 ? 8 : cpr <= 32 ? 16 : cpr <= 64 ? 32 : 64;
    const bool wide = qtype == VIPER_QTYPE_Q5_G64 || qtype == VIPER_QTYPE_Q6_G64;  // high-plane registers
    const int slots = (cpr + s.ts - 1) / s.ts, most = wide ? ST_MAX<5> : ST_MAX<4>;
    s.cpl = slots > most ? most : slots;  // (every slot but the last full, see the kernel)
    s.r = 1;
    auto units = [&](int rows) { const int ur = 64 / s.ts * s.r; return (rows + ur - 1) / ur; };
    auto total = [&] {
        long u = 0;
        for (int i = 0; i < nouts; ++i) u += units(n[i]);
        return u;
    };
    // Two rows per unit where a row fills two slots of 64 lanes (the
    // activation is then read from LDS once for both) and every wave still
    // has a unit (Q4, K = 3520, N = 4096 / 11008: 3.70 / 6.85 -> 3.42 / 5.52 us;
    // N = 1024: 2.51 -> 2.65 us, so not there).
    if (s.ts == 64 && s.cpl == 2 && total() >= 10L * cus) s.r = 2;
    const long u = total();
    // One workgroup per CU, or two where there are enough units for both and
    // the kernel's registers let two sit on a CU (at most 128 per lane): small
    // tiles from 10 units per CU on (Q4, K = 2048, N = 8192 / 20000: 3.72 / 6.5
    // -> 3.49 / 5.55 us; N = 4096, 8 units: 2.88 -> 3.01 us; Q5, K = 4096, N =
    // 4608, 9 units: 4.35 -> 4.67), larger ones from
    // 24 on (K = 7168, N = 8192 / 3000: 7.55 / 4.15 -> 7.22 / 4.61 us).
    const bool two = s.cpl <= 2 ? u >= 10L * cus : s.cpl <= (wide ? 4 : 5) && u >= 24L * cus;
    const long wgs = (two ? 2L : 1L) * cus;
    long upw = (u + wgs - 1) / wgs;
    s.upw = (int)(upw < 1 ? 1 : upw > 1023 ? 1023 : upw);
    long g = 0;
    for (int i = 0; i < nouts; ++i) {
        s.nb[i] = (units(n[i]) + s.upw - 1) / s.upw;
        g += s.nb[i];
    }
    s.gx = (int)((g + 7) / 8);
    s.grid = 8 * s.gx;
    if (s.gx > 1023) {
        s.gx = 0;
        s.grid = (int)g;
    }
    return s;
}

static m1_fn st_kernel(int qtype, const StShape& s, int senc, int mode, int pro) {
    switch (qtype) {
        case VIPER_QTYPE_Q4_G64: return st_pick<4>(s.ts, s.cpl, s.r, senc, mode, pro);
        case VIPER_QTYPE_Q5_G64: return st_pick<5>(s.ts, s.cpl, s.r, senc, mode, pro);
        case VIPER_QTYPE_Q6_G64: return st_pick<6>(s.ts, s.cpl, s.r, senc, mode, pro);
        default: return st_pick<8>(s.ts, s.cpl, s.r, senc, mode, pro);
    }
}

static size_t st_lds(int qtype, int K, const StShape& s) {
    switch (qtype) {
        case VIPER_QTYPE_Q4_G64: return st_lds_bytes<4>(K, s.ts * s.cpl);
        case VIPER_QTYPE_Q5_G64: return st_lds_bytes<5>(K, s.ts * s.cpl);
        case VIPER_QTYPE_Q6_G64: return st_lds_bytes<6>(K, s.ts * s.cpl);
        default: return st_lds_bytes<8>(K, s.ts * s.cpl);
    }
}

static int st_kw(int K, const StShape& s) { return (int)((unsigned)(K / 32) | (unsigned)s.upw << 12 | (unsigned)s.gx << 22); }

static bool folded_pro(int pro) { return pro == PRO_RMSNORM || pro == PRO_SWIGLU; }

// The exact tiling one row of this K would run on (ntt 0: none).
static M1Shape m1_one(int qtype, int K, int N, int cus, int pro, bool pair) {
    const bool w8 = qtype == VIPER_QTYPE_W8_G32;
    const int cpr = K / (w8 ? 16 : 32), noct = K / 8;
    M1Shape sh{0, 0, 0};
    if (!m1_tiles(w8 ? 8 : qtype, cpr)) return sh;
    // The folded prologues run fastest with one octet per thread (rmsnorm's
    // row sum and swiglu's element work are then a single pass): take such a
    // workgroup where a tiling allows it, even at a higher row load.
    if (folded_pro(pro)) sh = m1_shape(cpr, N, cus, noct < 640 ? noct : 640, noct, pair);
    if (sh.ntt == 0) sh = m1_shape(cpr, N, cus, 0, noct, pair);
    return sh;
}

// One row takes the exact tiling `sh`, or the streaming kernel?  80 and 96
// chunks (W8 also 160 and 192) always the tiling (K = 2560, N = 2560 / 10240
// 2.70 / 4.5 us against 2.83 / 4.5).  Longer rows where the streaming kernel's
// eight waves take a second and third turn and the tiling gives every CU one
// workgroup with rows within 20 / 17 of the mean: Q4, 160 chunks, up to 20
// rows per CU (K = 5120, N = 4608 / 5120 3.90 / 4.05 us against 4.23 / 4.36;
// N = 6144, 40 rows on the fullest CU, 5.2 / 4.8), with the swiglu prologue,
// one octet per thread there, uneven too (N = 3072 3.6 / 3.9); 192 chunks up
// to 12 (K = 6144, N = 2560 3.3 / 3.5); 320 up to 10 (int8 row, K = 10240, N =
// 2560 4.19 / 4.37; W8, K = 5120 3.90 / 4.03).  640 chunks, two segments or ten
// slots there, for 5..10 rows (Q5, K = 20480, N = 1536 / 2560 7.4 / 9.1 against
// 8.2 / 10.5; N = 3072 15.6 / 12.2; W8, K = 10240, N = 1536 4.77 / 4.9).
// Only where no other launch's outputs have to have the same bits (alone): the
// gate/up pair's equal those of viper_hip_qlinear_m1 from the same row, for
// any N, and the streaming kernel sums a row in one order whatever N.
static bool m1_tiled(int qtype, int K, const M1Shape& sh, int N, int cus, int pro, bool alone) {
    if (sh.ntt == 0) return false;
    const bool w8 = qtype == VIPER_QTYPE_W8_G32;
    const int cpr = K / (w8 ? 16 : 32);
    if (cpr <= 96 || (w8 && cpr <= 192)) return true;
    if (!alone) return false;
    const long rows = (N + cus - 1) / cus, load = m1_load(sh, N, cus);
    if (cpr == 640) return rows > 4 && rows <= 10;
    if (cpr == 192 && pro == PRO_SWIGLU) return false;  // (Q4, N = 3072 4.4 / 4.1)
    if (rows <= 8 || rows > (cpr == 160 ? 20 : cpr == 192 ? 12 : 10)) return false;
    return load * 17 <= rows * 20 || (cpr == 160 && pro == PRO_SWIGLU);
}

int launch_m1(int qtype, int senc, int K, int pro, const void* x, const void* xa, float eps, void* xout,
              const M1Out* outs, int nouts, const void* res, int32_t* part, hipStream_t st, int M, bool plain) {
    if (nouts < 1 || nouts > 3) return VIPER_INVALID_ARGUMENT;
    const int mr = m1_mr(M);
    if (mr > 1 && (nouts != 1 || (pro != PRO_BF16 && pro != PRO_INT8) || !m1_rows_ok(qtype, K, M)))
        return VIPER_INVALID_ARGUMENT;
    const int ck = qtype == VIPER_QTYPE_W8_G32 ? 16 : 32;
    const bool folded = pro == PRO_RMSNORM || pro == PRO_SWIGLU;
    int ntot = 0;
    for (int i = 0; i < nouts; ++i) {
        // n0's high bits carry flags
        if (outs[i].n >= M1_N_EXTRA || ntot > INT32_MAX - outs[i].n) return VIPER_INVALID_ARGUMENT;
        ntot += outs[i].n;
    }
    const int noct = M * (K / 8);
    const int cus = device_cus();
    m1_fn fn;
    unsigned grid, threads;
    size_t lds;
    int nb[3] = {0, 0, 0};
    int kg;  // the K slot: streaming launches pack more into it, exact tilings carry the grid size
    M1Shape sh = mr == 1 ? m1_one(qtype, K, ntot, cus, pro, false) : M1Shape{0, 0, 0};
    const bool alone = nouts == 1 && (plain || pro == PRO_INT8 || pro == PRO_SWIGLU);
    if (mr == 1 && !m1_tiled(qtype, K, sh, ntot, cus, pro, alone)) {
        const int n[3] = {outs[0].n, nouts > 1 ? outs[1].n : 0, nouts > 2 ? outs[2].n : 0};
        const StShape ss = st_shape(qtype, K, n, nouts, cus);
        fn = st_kernel(qtype, ss, senc, part != nullptr ? M1_PART : M1_PLAIN, pro);
        for (int i = 0; i < nouts; ++i) nb[i] = ss.nb[i];
        grid = (unsigned)ss.grid;
        threads = ST_NTT;
        lds = st_lds(qtype, K, ss);
        kg = st_kw(K, ss);
    } else {
        if (mr > 1) sh = m1_shape(K / ck, ntot, cus, (noct + M1_XS_MR - 1) / M1_XS_MR, noct, false, mr);
        if (sh.ntt == 0) return VIPER_INVALID_ARGUMENT;
        if (!folded && nouts == 1 && mr == 1) sh = m1_q5_bf16(qtype, pro, ntot, cus, m1_wide96(qtype, K / ck, ntot, cus, sh));
        const int group = qtype == VIPER_QTYPE_W8_G32 ? 32 : 64;
        const bool exact = m1_exact(sh, K / ck, K / group);
        fn = m1_kernel(qtype, sh, senc, part != nullptr ? M1_PART : M1_PLAIN, exact, pro, mr);
        const int rows = sh.ntt / sh.ts;
        lds = lds_m1_launch(qtype, K, rows, exact, mr);
        if (lds > (size_t)LDS_MAX) return VIPER_INVALID_ARGUMENT;
        for (int i = 0; i < nouts; ++i) nb[i] = (outs[i].n + rows - 1) / rows;
        grid = (unsigned)(nb[0] + nb[1] + nb[2]);
        threads = (unsigned)sh.ntt;
        kg = exact ? (int)grid : K;
    }
    if (fn == nullptr) return VIPER_INTERNAL;
    const M1Out o0 = outs[0], o1 = nouts > 1 ? outs[1] : outs[0], o2 = nouts > 2 ? outs[2] : outs[0];
    const uint8_t *w0 = (const uint8_t*)o0.w, *w1 = (const uint8_t*)o1.w, *w2 = (const uint8_t*)o2.w;
    const uint16_t *s0 = (const uint16_t*)o0.s, *s1 = (const uint16_t*)o1.s, *s2 = (const uint16_t*)o2.s;
    uint16_t *y0 = (uint16_t*)o0.y, *y1 = (uint16_t*)o1.y, *y2 = (uint16_t*)o2.y;
    int n0 = o0.n | (pro == PRO_RMSNORM && xout != nullptr ? M1_N_EXTRA : 0);
    int n1 = nouts > 1 ? o1.n : 0, n2 = nouts > 2 ? o2.n : 0;
    int e0 = nb[0], e1 = nb[0] + nb[1];
    if (mr > 1) e1 = M;  // one matrix: e1 carries the activation rows
    const uint16_t* r = (const uint16_t*)res;
    void* args[] = {&x, &w0, &s0, &y0, &kg, &n0, &e0, &e1, &r, &xa, &eps, &xout, &part,
                    &w1, &s1, &y1, &n1, &w2, &s2, &y2, &n2};
    launch((const void*)fn, grid, threads, lds, st, args);
    return status_of(hipGetLastError());
}

int launch_m1_timeline(int qtype, int senc, int K, const void* x, const void* w, const void* s, void* y, int N,
                       uint64_t* stamps, size_t stamp_bytes, int* workgroups, int* waves, hipStream_t st) {
    // rows of 5 or 10 (6) slots of 16, 32 or 64 lanes, or of 336 chunks, whose
    // scales fill whole 16-byte words, on the kernel that the call runs
    const int ck = qtype == VIPER_QTYPE_W8_G32 ? 16 : 32, group = qtype == VIPER_QTYPE_W8_G32 ? 32 : 64;
    const int cpr = K / ck;
    if ((cpr != 80 && cpr != 160 && cpr != 320 && cpr != 640 && cpr != 96 && cpr != 192 && cpr != 384 && cpr != 336) ||
        (K / group) % 8 != 0)
        return VIPER_INVALID_ARGUMENT;
    const int cus = device_cus();
    m1_fn fn;
    int nwg, threads, kg;  // as launch_m1
    unsigned grid;
    size_t lds;
    M1Shape sh = m1_one(qtype, K, N, cus, PRO_BF16, false);
    if (m1_tiled(qtype, K, sh, N, cus, PRO_BF16, true)) {
        sh = m1_q5_bf16(qtype, PRO_BF16, N, cus, m1_wide96(qtype, cpr, N, cus, sh));
        fn = m1_kernel(qtype, sh, senc, M1_TL, true, PRO_BF16);
        const int rows = sh.ntt / sh.ts;
        nwg = (N + rows - 1) / rows;
        grid = (unsigned)nwg;
        threads = sh.ntt;
        lds = lds_m1_launch(qtype, K, rows, true);
        kg = nwg;
    } else {
        const StShape ss = st_shape(qtype, K, &N, 1, cus);
        fn = st_kernel(qtype, ss, senc, M1_TL, PRO_BF16);
        nwg = ss.nb[0];
        grid = (unsigned)ss.grid;
        threads = ST_NTT;
        lds = st_lds(qtype, K, ss);
        kg = st_kw(K, ss);
    }
    if (fn == nullptr) return VIPER_INTERNAL;
    const size_t need = (size_t)nwg * (threads / 64) * M1_TL_STAMPS * sizeof(uint64_t);
    if (stamps == nullptr || stamp_bytes < need) return VIPER_INVALID_ARGUMENT;
    if (workgroups != nullptr) *workgroups = nwg;
    if (waves != nullptr) *waves = threads / 64;
    const uint8_t* w0 = (const uint8_t*)w;
    const uint16_t* s0 = (const uint16_t*)s;
    uint16_t* y0 = (uint16_t*)y;
    int n0 = N, e0 = nwg, e1 = nwg, nz = 0;
    const uint16_t* r = nullptr;
    const void* xa = nullptr;
    float eps = 0.0f;
    uint16_t* xout = nullptr;
    int32_t* part = (int32_t*)stamps;
    const void* nul = nullptr;
    void* args[] = {&x, &w0, &s0, &y0, &kg, &n0, &e0, &e1, &r, &xa, &eps, &xout, &part,
                    &nul, &nul, &nul, &nz, &nul, &nul, &nul, &nz};
    launch((const void*)fn, grid, (unsigned)threads, lds, st, args);
    return status_of(hipGetLastError());
}

int launch_m1_swiglu(int qtype, int senc, int K, int pro, const void* x, const void* xa, float eps, void* xout,
                     const void* wg, const void* sg, const void* wu, const void* su, int N, void* h, void* g_out,
                     void* u_out, hipStream_t st) {
    if (pro != PRO_BF16 && pro != PRO_RMSNORM) return VIPER_INVALID_ARGUMENT;
    if (N >= M1_N_EXTRA) return VIPER_INVALID_ARGUMENT;  // n0's high bits carry flags
    const int cus = device_cus();
    m1_fn fn;
    unsigned grid, threads;
    size_t lds;
    int kg;  // as in launch_m1
    const M1Shape sh = m1_one(qtype, K, N, cus, pro, true);
    if (!m1_tiled(qtype, K, sh, N, cus, pro, false)) {
        const StShape ss = st_shape(qtype, K, &N, 1, cus);
        fn = st_kernel(qtype, ss, senc, M1_SWIGLU, pro);
        grid = (unsigned)ss.grid;
        threads = ST_NTT;
        lds = st_lds(qtype, K, ss);
        kg = st_kw(K, ss);
    } else {
        fn = m1_kernel(qtype, sh, senc, M1_SWIGLU, true, pro);
        const int rows = sh.ntt / sh.ts;
        grid = (unsigned)((N + rows / 2 - 1) / (rows / 2));
        threads = (unsigned)sh.ntt;
        lds = lds_m1_launch(qtype, K, rows, true);
        kg = (int)grid;
    }
    if (fn == nullptr) return VIPER_INTERNAL;
    // every workgroup is a pair of gate and up rows; the up matrix goes in the
    // residual's slot (weights) and e0 / e1 (scales), the product to y0, the
    // optional gate / up outputs to y1 / y2 (flagged in n0)
    const bool extra = g_out != nullptr || u_out != nullptr || (pro == PRO_RMSNORM && xout != nullptr);
    int n0 = N | (extra ? M1_N_EXTRA : 0), n1 = N, n2 = N;
    const uint64_t su_bits = (uint64_t)(uintptr_t)su;
    int e0 = (int)(uint32_t)su_bits, e1 = (int)(uint32_t)(su_bits >> 32);
    const uint8_t *w0 = (const uint8_t*)wg, *w1 = nullptr, *w2 = nullptr;
    const uint16_t *s0 = (const uint16_t*)sg, *s1 = nullptr, *s2 = nullptr;
    uint16_t *y0 = (uint16_t*)h, *y1 = (uint16_t*)g_out, *y2 = (uint16_t*)u_out;
    const uint16_t* r = (const uint16_t*)wu;
    int32_t* part = nullptr;
    void* args[] = {&x, &w0, &s0, &y0, &kg, &n0, &e0, &e1, &r, &xa, &eps, &xout, &part,
                    &w1, &s1, &y1, &n1, &w2, &s2, &y2, &n2};
    launch((const void*)fn, grid, threads, lds, st, args);
    return status_of(hipGetLastError());
}

}  // namespace vq
