// Quantized linear for MI355X (gfx950): y = bf16( sum_g ws*xs*D_g [+ res] ).
//
// Semantics follow the reference's int8 decode path (itzrnvr/viper):
// activation quantize as kernels/ops/rmsnorm_quantize.cu:71-104 and
// linear_multim.cu:21-61 (per-row, per-group amax/127 floored at 1e-8,
// round-to-nearest-even of x/scale), group dot + fp32 combine as
// kernels/ops/dp4a_smem_kernel.cu:25-74 and linear_multim.cu:64-130, weight
// layout as tools/convert/convert.cpp:91-127.  The design is gfx950's own.
//
// M = 1 (the decode GEMV; qgemv_m1_kernel in qgemv_m1.h where its tilings fit
// the row exactly, else qgemv_stream_kernel in qgemv_stream.h): teams of 8-64
// lanes stream output rows with 16-byte non-temporal loads; each workgroup
// quantizes the bf16 activation into LDS while its weights are in flight,
// the int32 group dots are exact (v_dot8 on split activation nibbles for Q4,
// v_dot4 on offset codes for Q5/Q6/W8) and the fp32 combine is reduced with
// DPP in a fixed order (deterministic).
//
// M = 2..16 (qgemm_rc.h, qgemm_stream.h, qgemm_mfma.hip; which one is the Route
// of a call below): few rows are quantized by every workgroup, more are quantized once into a caller workspace in the
// matrix-core fragment order or supplied by the caller, and every weight byte
// is read once for all M rows.
//
// The activation quantizer never divides per element: with s the group scale
// (an IEEE divide amax/127, once per group) and r = rcp(s) (the hardware
// reciprocal, within 1 ulp), q0 = x*r and q1 = fma(fma(-q0, s, x), r, q0);
// adding 1.5*2^23 rounds q1 to the nearest even integer and leaves it, two's
// complement, in the low byte.  For every finite bf16 pair (amax, x) the byte
// equals RNE(x/s): check_quantizer_kernel verifies that exhaustively on the
// device (and the CPU oracle the same steps with an IEEE 1/s).

#include "qlinear_host.h"

#include <mutex>

namespace vq {

// ------------------------------------------------ allocation-free entry point

// The workspace of viper_hip_qlinear_static: a file-scope device array, one
// copy on every device the library runs on, held until the process ends.  In
// host code `scratch` names a host-side stand-in, never device memory: the
// device address comes from hipGetSymbolAddress, taken once per device with
// that device current and kept in scratch_dev.
constexpr size_t STATIC_SCRATCH_BYTES = VIPER_QLINEAR_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) uint8_t scratch[STATIC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
static std::mutex scratch_mu;
static void* scratch_dev[MAX_DEVICES];

// Device address of the current device's scratch (looked up on its first use).
static int scratch_address(void** out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return VIPER_DEVICE_ERROR;
    if (dev < 0 || dev >= MAX_DEVICES) return VIPER_INTERNAL;
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (scratch_dev[dev] == nullptr) {
        void* p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || p == nullptr) return VIPER_DEVICE_ERROR;
        scratch_dev[dev] = p;
    }
    *out = scratch_dev[dev];
    return VIPER_OK;
}

// ------------------------------------------------ standalone activation quantize

// MF: the fragment order the matrix-core kernels read (xs transposed to
// [K/G][16]; 64-groups use quantize_frag64_kernel); else xq [M][K] in k order
// and xs [M][K/G].
template <int G, bool MF>
__global__ void __launch_bounds__(NT)
quantize_act_kernel(const uint16_t* x, int8_t* __restrict__ xq,
                    float* __restrict__ xs, int oct_total, int K) {
    const int o = (int)blockIdx.x * NT + (int)threadIdx.x;
    const bool ok = o < oct_total;
    u32x4 v = {0u, 0u, 0u, 0u};
    if (ok) v = *(const u32x4*)(x + (size_t)o * 8);
    uint32_t d0, d1;
    float s;
    quantize_octet<G, MF && G == 64>(v, d0, d1, s);
    if (ok) {
        if constexpr (MF) {
            // group g, k-slot kb of the octet's quarter, row m (matrix-core
            // fragment order: quarter qi of a group sits in k-slot
            // kb = bit-swap(qi), Q bytes per fragment); written through like
            // quantize_frag64_kernel's stores
            constexpr int Q = G == 64 ? 16 : 8;
            const int opr = K / 8;
            const int m = o / opr, og = o % opr;
            const int g = og / (G / 8), k0 = (og % (G / 8)) * 8;
            const int qi = k0 / Q;
            const int kb = ((qi & 1) << 1) | (qi >> 1);
            const auto xw = buf(xq, (uint32_t)(K / G) * 64u * (uint32_t)Q);
            const auto sw = buf(xs, (uint32_t)(K / G) * 64u);
            bstore8<AUX_SC1>(xw, ((g * 4 + kb) * 16 + m) * Q + k0 % Q, u32x2{d0, d1});
            if ((o & (G / 8 - 1)) == 0) bstore4<AUX_SC1>(sw, (g * 16 + m) * 4, __float_as_uint(s));
        } else {
            *(u32x2*)(xq + (size_t)o * 8) = u32x2{d0, d1};
            if ((o & (G / 8 - 1)) == 0) xs[(size_t)o * 8 / G] = s;
        }
    }
}

// Fragment order of 64-groups, one wave per group: lane l = 16 * kb + m
// quantizes row m's quarter bit-swap(kb) of the group (16 values) and stores
// its 16-byte fragment, so a wave writes the group's 1 KB contiguously.  The
// group amax is the max over the 4 lanes of row m (lanes m, m + 16, m + 32,
// m + 48).  Rows m >= M are neither read nor written.
__global__ void __launch_bounds__(64)
quantize_frag64_kernel(const uint16_t* x, int M, int K, int8_t* __restrict__ xq, float* __restrict__ xs) {
    const int L = (int)threadIdx.x, g = (int)blockIdx.x;
    const int m = L & 15, kb = L >> 4, qi = ((kb & 1) << 1) | (kb >> 1);
    const bool ok = m < M;
    const auto xr = buf(x, (uint32_t)M * (uint32_t)K * 2u);
    const int off = ok ? (m * K + g * 64 + 16 * qi) * 2 : OOB;
    const u32x4 v0 = bload16(xr, off), v1 = bload16(xr, off + 16);
    const uint32_t wd[8] = {v0.x, v0.y, v0.z, v0.w, v1.x, v1.y, v1.z, v1.w};
    float f[16];
    float a = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        f[i] = bf16f((wd[i >> 1] >> (16 * (i & 1))) & 0xffffu);
        a = fmaxf(a, fabsf(f[i]));
    }
    a = fmaxf(a, __shfl_xor(a, 16, 64));
    a = fmaxf(a, __shfl_xor(a, 32, 64));
    float s, r;
    group_scale(a, s, r);
    uint32_t t[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) t[i] = qbits(f[i], s, r);
    const u32x4 o = {bytes4(t[0], t[2], t[4], t[6]), bytes4(t[1], t[3], t[5], t[7]), bytes4(t[8], t[10], t[12], t[14]),
                     bytes4(t[9], t[11], t[13], t[15])};
    // written through (the matrix-core kernel reads them right after this
    // launch; 0.2 us of the M = 16 verify)
    const auto xw = buf(xq, (uint32_t)(K / 64) * 1024u);
    const auto sw = buf(xs, (uint32_t)(K / 64) * 64u);
    bstore16<AUX_SC1>(xw, ok ? (g * 64 + L) * 16 : OOB, o);
    bstore4<AUX_SC1>(sw, (ok && kb == 0) ? (g * 16 + m) * 4 : OOB, __float_as_uint(s));
}

// ----------------------------------------------- bf16 rounding self-check

// Every fp32 bit pattern through the kernels' conversion (f2bf2, the
// hardware v_cvt_pk_bf16_f32) and its arithmetic statement f2bf_sw; *count
// receives the number of disagreements (each thread covers a contiguous
// range of patterns, two per conversion).
constexpr int BFC_GRID = 4096, BFC_NT = 256;
__global__ void __launch_bounds__(BFC_NT) check_bf16_kernel(unsigned long long* __restrict__ count) {
    constexpr unsigned long long per = (1ull << 32) / ((unsigned long long)BFC_GRID * BFC_NT);
    const unsigned long long base = ((unsigned long long)blockIdx.x * BFC_NT + threadIdx.x) * per;
    unsigned bad = 0;
    for (unsigned long long k = 0; k < per; k += 2) {
        const float a = __uint_as_float((uint32_t)(base + k)), b = __uint_as_float((uint32_t)(base + k + 1));
        const uint32_t hw = f2bf2(a, b);
        bad += (hw & 0xffffu) != f2bf_sw(a);
        bad += (hw >> 16) != f2bf_sw(b);
    }
    if (bad) atomicAdd(count, (unsigned long long)bad);
}

// --------------------------------------------------- quantizer self-check

__global__ void __launch_bounds__(NT) check_quantizer_kernel(int ab0, int32_t* __restrict__ counts) {
    __shared__ int red[NT];
    const int ab = ab0 + (int)blockIdx.x;
    const float amax = bf16f((uint32_t)ab);
    float s, r;
    group_scale(amax, s, r);
    const float s_ieee = fmaxf(amax / 127.0f, 1e-8f);
    int bad = s != s_ieee;
    for (int xb = (int)threadIdx.x; xb <= ab; xb += NT) {
        const float xv = bf16f((uint32_t)xb);
        const int fast = (int8_t)(qbits(xv, s, r) & 0xffu);
        const int fastn = (int8_t)(qbits(-xv, s, r) & 0xffu);
        const float ex = fminf(fmaxf(__builtin_rintf(xv / s_ieee), -127.0f), 127.0f);
        bad += fast != (int)ex;
        bad += fastn != -(int)ex;
    }
    red[threadIdx.x] = bad;
    __syncthreads();
    for (int step = NT / 2; step > 0; step >>= 1) {
        if ((int)threadIdx.x < step) red[threadIdx.x] += red[threadIdx.x + step];
        __syncthreads();
    }
    if (threadIdx.x == 0) counts[blockIdx.x] = red[0];
}

static int launch_quantize(int group, const void* x, int M, int K, void* xq, void* xs, bool mf, hipStream_t st) {
    const int oct_total = M * K / 8;
    const unsigned grid = (unsigned)((oct_total + NT - 1) / NT);
    const uint16_t* a0 = (const uint16_t*)x;
    int8_t* a1 = (int8_t*)xq;
    float* a2 = (float*)xs;
    if (mf && group == 64) {
        void* fargs[] = {&a0, &M, &K, &a1, &a2};
        launch((const void*)quantize_frag64_kernel, (unsigned)(K / 64), 64, 0, st, fargs);
        return status_of(hipGetLastError());
    }
    void* args[] = {&a0, &a1, &a2, (void*)&oct_total, &K};
    const void* fn;
    if (group == 64) fn = (const void*)quantize_act_kernel<64, false>;
    else fn = mf ? (const void*)quantize_act_kernel<32, true> : (const void*)quantize_act_kernel<32, false>;
    launch(fn, grid, NT, 0, st, args);
    return status_of(hipGetLastError());
}

// M = 1 is fused when the quantized activation and its per-chunk records fit
// the LDS budget.
static bool fused_ok(int qtype, int M, int K) {
    return M == 1 && lds_m1(qtype, K) <= (size_t)LDS_MAX;
}

// Workspace of a call with M > 1 (zero-filled before its first use): the
// K split's control words and block counters at offset 0 for every shape
// (RC_CTL_BYTES: the missed-sum count, then RC_CNT_MAX counters from byte
// 256), then (long K on the matrix cores) the K split's records of part sums,
// one per row block at the same offset for every shape, then xq ([M][K], or
// fragment order with room for 16 rows) and xs ([M][K/G], or [K/G][16])
// fp32.  Offsets in bytes.
struct WsLayout {
    size_t cnt, sp, xq, xs, total;
    int blocks;  // row blocks of the K split (0: no split)
};
static size_t workspace_xq(int K) { return align16((size_t)16 * K); }
static size_t workspace_xs(int qtype, int K) { return align16((size_t)(K / group_of(qtype)) * 16 * 4); }
static size_t split_record_bytes(int blocks) { return (size_t)blocks * RC_REC_SLOTS * 8; }

static WsLayout workspace_layout(int qtype, int N, int K, int M) {
    WsLayout l{0, 0, 0, 0, 0, 0};
    const int G = group_of(qtype);
    if (G == 0 || M <= 0 || K <= 0 || N <= 0 || K % G != 0) return l;
    if (fused_ok(qtype, M, K)) return l;
    l.blocks = M >= 2 && M <= 16 ? rc_split_blocks(qtype, N, K) : 0;
    l.cnt = (size_t)RC_CTL_CNT * 4;
    l.sp = RC_CTL_BYTES;
    l.xq = l.sp + split_record_bytes(l.blocks);
    l.xs = l.xq + workspace_xq(K);
    l.total = l.xs + workspace_xs(qtype, K);
    return l;
}

// Workspace of the fragment-input entry points: the control words and, for
// long K, the K split's records (0: the launch needs none).
static size_t frag_workspace_need(int qtype, int N, int K, int M) {
    const int G = group_of(qtype);
    if (G == 0 || M < 2 || M > 16 || N <= 0 || K <= 0 || K % G != 0) return 0;
    const int blocks = rc_split_blocks(qtype, N, K);
    return blocks > 0 ? RC_CTL_BYTES + split_record_bytes(blocks) : 0;
}

static size_t workspace_need(int qtype, int N, int K, int M) { return workspace_layout(qtype, N, K, M).total; }

// Optional second matrix of the same shape applied to the same activation in
// the same launch (the reference's fused2: k and v, gate and up).
struct Second {
    const void* w = nullptr;
    const void* s = nullptr;
    void* y = nullptr;
};

static int validate_second(const Second& b, int qtype, int senc, int group, int N, int K, int M,
                           const void* res, const int32_t* part) {
    if (b.w == nullptr && b.s == nullptr && b.y == nullptr) return VIPER_OK;
    if (b.y == nullptr || res != nullptr || part != nullptr) return VIPER_INVALID_ARGUMENT;
    if (misaligned(b.y, 2)) return VIPER_INVALID_ARGUMENT;
    return validate_weights(qtype, b.w, b.s, senc, group, N, K, M);
}

// Two to four rows of one matrix: on the M = 1 kernel's dot path, or on the
// matrix cores?  The dot path's exact multi-row tilings (K = 2560, 5120, 10240:
// Q4, 2 rows, K = 5120, N = 4096 / 10240 4.4 / 7.4 us against 4.7 / 10.2), and K
// beyond one phase of the streaming kernel, where its serial phases or a
// second launch cost more (one: K has one phase; Q4, 2 rows, N = 2560, dot /
// matrix cores: K = 9600 8.9 / 11.7; K = 6144 7.3 / 5.0, K = 4096 6.9 / 4.1,
// K = 3072 6.4 / 3.7, K = 512 4.3 / 2.7; 4 rows K = 4096, N = 10240 11.2 / 9.0).
// Two rows also where the streaming kernel (takes) would fill its last tile
// least while one round of 40-row workgroups holds them here, 33..40 rows per
// CU (N = 10240: Q4 K = 2112 5.6 / 6.5, K = 4608 8.1 / 9.7; Q6 K = 2112 6.9 / 7.7;
// W8 K = 1760 5.4 / 6.2; N = 8192 the other way; Q4, K = 4096, N = 11005, two
// rounds, 12.3 / 8.2; up to 36 groups of Q4 also those two rounds, 49..80 rows:
// N = 14080, K = 1280 6.8 / 7.05, K = 2304 7.8 / 8.6), short rows of W8, which decodes cheapest, from there on
// (N = 16384, K = 704 4.8 / 5.8, K = 1056 5.9 / 6.7), and few long ones of it,
// whose tiles take the most steps (K = 3520, N = 2560 6.3 / 6.5; K = 4096, N =
// 4256 6.7 / 8.9, N = 6144 equal).
static bool dot_rows(int qtype, int N, int K, int M, bool one, bool takes) {
    if (!m1_rows_ok(qtype, K, M)) return false;
    if (m1_rows_exact(qtype, K, M) || !one) return true;
    if (M > 2 || !takes) return false;
    const bool w8 = qtype == VIPER_QTYPE_W8_G32, q4 = qtype == VIPER_QTYPE_Q4_G64;
    const long per_cu = (N + (long)device_cus() - 1) / device_cus();
    if (q4 && K <= 2304 && per_cu > 48 && per_cu <= 80) return true;
    return (per_cu > 32 && (per_cu <= 40 || (w8 && K <= 1152))) || (w8 && K > 96 * 32 && per_cu <= 20);
}

// The kernel a call runs, from its sizes alone (the routes of include/viper_qlinear.h).
enum Route {
    R_M1 = VIPER_ROUTE_M1,
    R_ROWS = VIPER_ROUTE_ROWS,
    R_RC_BF16 = VIPER_ROUTE_RC_BF16,
    R_SG_BF16 = VIPER_ROUTE_STREAM_BF16,
    R_SPLIT = VIPER_ROUTE_RC_SPLIT,
    R_RC = VIPER_ROUTE_RC,
    R_SG = VIPER_ROUTE_STREAM,
    R_MF = VIPER_ROUTE_PAIRS,
};

// bf16 rows.  Few rows: every workgroup quantizes the rows itself, one launch
// (the workspace stays required for M > 1 whichever kernel runs).  Two to four
// rows of one matrix on the M = 1 kernel's dot path; 5..8 rows (and fused
// pairs of 3..8) on the matrix cores with the quantize into LDS
// (north-star shape: M = 5 6.63 us, 8 7.49 us against 8.21 / 8.25 us for
// the next-best path; at M >= 10 the rows' quantize in every workgroup
// costs more than the quantize launch).
static Route linear_route(int qtype, int N, int K, int M, bool pair, bool part) {
    if (fused_ok(qtype, M, K)) return R_M1;
    const bool rc_k = M >= 2 && rc_ok(qtype, K);
    // K or rows beyond the row-contiguous kernel: the streaming one, which also
    // quantizes up to 8 rows itself (Q4, M = 8, us, one launch / two: K = 3520,
    // N = 2560 6.1 / 7.0, N = 10240 9.8 / 10.6; K = 4096, N = 10240 9.9 / 10.6).
    const bool one = sg_bf16_ok(qtype, N, K, M, pair);
    const bool takes = sg_takes(qtype, N, K, M, pair, one ? RC_BF16 : RC_FRAG);
    const bool dot = !pair && dot_rows(qtype, N, K, M, one, takes);
    int wg_rows;
    const int rounds = rc_k ? rc_rounds(qtype, pair ? 2L * N : N, K, &wg_rows) : 0;
    // (two rows past 64 per CU, several rounds of the row-contiguous kernel of up
    // to 48 rows: the dots where rounds of their 40 pad fewer; Q4, K = 1536, N =
    // 17366 7.4 us against 9.9 on the streaming kernel, K = 2048, N = 20480 8.4 /
    // 9.7; Q6, K = 1536, N = 25600 12.7 against 15.3 on the row-contiguous one; Q4,
    // K = 2048, N = 24320 10.1 / 9.6)
    const long per_cu = (N + (long)device_cus() - 1) / device_cus();
    const bool dots_pad = !pair && !takes && rounds > 1 && per_cu > 64 && (per_cu + 39) / 40 * 40 < (long)rounds * wg_rows &&
                          m1_rows_ok(qtype, K, M);
    if (M == 2 && (dot || dots_pad)) return R_ROWS;
    // With the rows staged two octets per thread (64-groups), the row-contiguous
    // kernel's one-launch path also wins for Q4 at 3-4 rows (5.45 / 5.74 against
    // 5.6 / 5.9 us on the dot kernel) and 9-10 rows (6.76 / 7.00 against 7.27 us
    // in two launches; 12 and 16 rows stay two launches: 7.5 / 8.2 against 7.3
    // us), and for Q5 / Q6 at 8 rows (7.90 / 8.22 against 8.37 / 8.58 us).  W8
    // keeps 3-4 rows on the dot kernel and 5-8 here.  Every round of its
    // workgroups quantizes the rows again: where the streaming kernel would
    // take two launches, up to 12 rows times rounds (Q4, K = 7168: 3 rows, N =
    // 10240 15.6 against 16.5 us, 5 rows, N = 8192 / 10240 13.4 / 18.7 against
    // 13.5 / 16.5); a pair's two rows of Q5 and Q6 and a K of one phase up to two
    // rounds (Q5, K = 2048, N = 20000 22.1 against 20.7 us in two launches; Q4 16.2 /
    // 17.5; Q5, K = 5504 45.7 / 61.4).
    const bool q4 = qtype == VIPER_QTYPE_Q4_G64;
    const int bf_max = q4 && !pair ? 10 : 8;
    const bool rc_bf16 = rc_k && M <= bf_max && rc_bf16_ok(qtype, N, K, M, pair) && (!takes || (!one && M * rounds <= 12)) &&
                         !(pair && M == 2 && rounds > 2 && !q4 && qtype != VIPER_QTYPE_W8_G32 && sg_phases(qtype, K, RC_FRAG) == 1);
    // Long K splits over workgroups in the two-launch path (down shape
    // K = 10240, 4 rows 9.5 us against 10.3 us without the split), unless one
    // launch serves a K of one phase (Q4, 6 rows, K = 6144, N = 3072 6.8 us
    // against 8.5; 7 and 8 rows have none there: 8.5 against 9.2 on the segment
    // loop).  (Every workgroup quantizing the bf16 rows of its own part of K,
    // in one launch, measured slower at every row count: down shape 3 / 8 / 16
    // rows 10.4 / 12.6 / 15.9 us against 8.4 / 9.4 / 9.8 us.)
    const bool split = rc_k && !pair && rc_split_blocks(qtype, N, K) > 0 && !(takes && rc_split_capped(qtype, N, K)) &&
                       !(one && (takes || rc_bf16));
    // Q5/Q6/W8 (K = 2560, N = 10240, 5% outlier channels): 3 or 4 rows of one
    // matrix run faster on the multi-row dot kernel below (Q5 4 rows 7.86
    // against 8.10 us; W8 3 / 4 rows 7.47 / 7.77 against 8.9 / 9.17 us); 5-8
    // rows of every format stay on the one-launch path.
    // (Q4 rows staged two octets per thread also past that size: down shape
    // K = 10240, 4 rows 8.4 us against 9.0-9.1 us for two launches with the K
    // split)
    // (but not where the streaming kernel takes a K of whole quads, the rows
    // have no exact tiling and there are more than 40 per CU: Q4, 4 rows, K =
    // 7168, N = 16384 35.6 us against 20.5 in its two launches; 3 rows, K = 9216,
    // N = 4352 11.4 / 15.3)
    const bool rows_ok = dot && ((long)M * K <= 32768 || m1_rows_pair(qtype, K, M)) &&
                         !(takes && (one || (rc_k && !m1_rows_exact(qtype, K, M) && N > 40L * device_cus())));
    if (rc_bf16 && !split && (M > 4 || !rows_ok || q4)) return R_RC_BF16;
    // (3 or 4 rows here also where the LDS copy does not fit: while every
    // workgroup's share of the rows' quantize stays small; down shape
    // K = 10240: 3 rows 8.8 us against about 9.5 us for two launches with the K
    // split)
    if (rows_ok) return R_ROWS;
    if (split) return R_SPLIT;
    if (takes && one && !part && sg_over_mf(qtype, N, K, M, pair, RC_BF16)) return R_SG_BF16;
    if (rc_k) return takes ? R_SG : R_RC;
    return sg_over_mf(qtype, N, K, M, pair, RC_FRAG) ? R_SG : R_MF;
}

// int8 rows in the layout of viper_hip_quantize_act.
static Route prequant_route(int qtype, int N, int K, int M, bool pair) {
    if (fused_ok(qtype, M, K)) return R_M1;
    const bool one = sg_phases(qtype, K, RC_NAT) == 1, takes = sg_takes(qtype, N, K, M, pair, RC_NAT);
    const bool rc_k = M >= 2 && rc_ok(qtype, K);
    // (3 and 4 rows of a nibble format and K of one phase: the matrix cores, also
    // against an exact tiling, Q4, 4 rows, K = 5120, N = 512 / 4096 4.6 / 5.4 us
    // against 5.2 / 5.9; not in several rounds, 3 rows, K = 2560, N = 28160 13.8
    // against 11.4)
    int wg_rows;
    const bool rows34 = M > 2 && one && rc_k && qtype != VIPER_QTYPE_W8_G32 && (takes || rc_rounds(qtype, N, K, &wg_rows) == 1);
    if (!pair && !rows34 && dot_rows(qtype, N, K, M, one, takes)) return R_ROWS;
    if (rc_k) return takes ? R_SG : R_RC;
    return sg_over_mf(qtype, N, K, M, pair, RC_NAT) ? R_SG : R_MF;
}

// int8 fragments; ws: with a workspace the K split may use.
static Route frag_route(int qtype, int N, int K, int M, bool pair, bool ws) {
    const bool takes = sg_takes(qtype, N, K, M, pair, RC_FRAG);
    if (ws && !pair && frag_workspace_need(qtype, N, K, M) > 0 && !(takes && rc_split_capped(qtype, N, K))) return R_SPLIT;
    return takes ? R_SG : R_RC;
}

// The rows' limit of a call that neither the M = 1 kernels nor the
// row-contiguous kernel take: one row, or K of an odd number of groups.  (The
// entry points' limit: their callers' refusals stay, whichever kernel runs.)
static bool rows_refused(int qtype, int M, int K) {
    return (M < 2 || (K / group_of(qtype)) % 2 != 0) && lds_pre(qtype, M, K) > (size_t)LDS_MAX;
}

static int qlinear_common(int qtype, const void* w, const void* s, int senc, int group, int N,
                          int K, const void* x, int M, void* y, const void* res, void* wsp,
                          size_t wsp_bytes, int32_t* part, void* stream, Second b = Second()) {
    int rc = validate_weights(qtype, w, s, senc, group, N, K, M);
    if (rc != VIPER_OK) return rc;
    if (x == nullptr || y == nullptr) return VIPER_INVALID_ARGUMENT;
    if (misaligned(x, 16) || misaligned(y, 2) || misaligned(res, 2) || misaligned(part, 4))
        return VIPER_INVALID_ARGUMENT;
    rc = validate_second(b, qtype, senc, group, N, K, M, res, part);
    if (rc != VIPER_OK) return rc;
    hipStream_t st = (hipStream_t)stream;
    const bool pair = b.w != nullptr;
    if (fused_ok(qtype, M, K)) {
        const M1Out outs[2] = {{w, s, y, N}, {b.w, b.s, b.y, N}};
        return launch_m1(qtype, senc, K, PRO_BF16, x, nullptr, 0.0f, nullptr, outs, pair ? 2 : 1, res, part, st);
    }
    const size_t need = workspace_need(qtype, N, K, M);
    if (wsp == nullptr || wsp_bytes < need || misaligned(wsp, 16)) return VIPER_INVALID_ARGUMENT;
    const Route route = linear_route(qtype, N, K, M, pair, part != nullptr);
    if (route == R_RC_BF16)
        return launch_rc(qtype, w, s, senc, N, K, x, nullptr, RC_BF16, M, y, res, part, b.w, b.s, b.y, st);
    if (route == R_ROWS) {
        const M1Out outs[1] = {{w, s, y, N}};
        return launch_m1(qtype, senc, K, PRO_BF16, x, nullptr, 0.0f, nullptr, outs, 1, res, part, st, M);
    }
    if (rows_refused(qtype, M, K)) return VIPER_INVALID_ARGUMENT;
    if (route == R_SG_BF16)
        return launch_sg(qtype, w, s, senc, N, K, x, nullptr, RC_BF16, M, y, res, nullptr, b.w, b.s, b.y, st);
    const WsLayout lay = workspace_layout(qtype, N, K, M);
    if (route == R_SPLIT && lay.blocks == 0) return VIPER_INTERNAL;
    uint8_t* xq = (uint8_t*)wsp + lay.xq;
    float* xs = (float*)((uint8_t*)wsp + lay.xs);
    // long K on the matrix cores: the K split (control words and counters at
    // the workspace's start, then the records of part sums)
    uint64_t* sp = route == R_SPLIT ? (uint64_t*)((uint8_t*)wsp + lay.sp) : nullptr;
    unsigned* sc = route == R_SPLIT ? (unsigned*)wsp : nullptr;
    rc = launch_quantize(group, x, M, K, xq, xs, true, st);
    if (rc != VIPER_OK) return rc;
    if (route == R_SG)
        return launch_sg(qtype, w, s, senc, N, K, xq, xs, RC_FRAG, M, y, res, part, b.w, b.s, b.y, st);
    if (route == R_MF)
        return launch_mf(qtype, w, s, senc, N, K, xq, xs, false, M, y, res, part, b.w, b.s, b.y, st);
    return launch_rc(qtype, w, s, senc, N, K, xq, xs, RC_FRAG, M, y, res, part, b.w, b.s, b.y, st, sp, sc);
}

static int prequant_common(int qtype, const void* w, const void* s, int senc, int group, int N,
                           int K, const void* xq, const void* xs, int M, void* y, const void* res,
                           void* stream, Second b = Second()) {
    int rc = validate_weights(qtype, w, s, senc, group, N, K, M);
    if (rc != VIPER_OK) return rc;
    if (xq == nullptr || xs == nullptr || y == nullptr) return VIPER_INVALID_ARGUMENT;
    if (misaligned(xq, 8) || misaligned(xs, 4) || misaligned(y, 2) || misaligned(res, 2))
        return VIPER_INVALID_ARGUMENT;
    rc = validate_second(b, qtype, senc, group, N, K, M, res, nullptr);
    if (rc != VIPER_OK) return rc;
    hipStream_t st = (hipStream_t)stream;
    const Route route = prequant_route(qtype, N, K, M, b.w != nullptr);
    if (route == R_M1 || route == R_ROWS) {
        const M1Out outs[2] = {{w, s, y, N}, {b.w, b.s, b.y, N}};
        return launch_m1(qtype, senc, K, PRO_INT8, xq, xs, 0.0f, nullptr, outs, b.w ? 2 : 1, res, nullptr, st, M);
    }
    if (rows_refused(qtype, M, K)) return VIPER_INVALID_ARGUMENT;
    if (route == R_SG)
        return launch_sg(qtype, w, s, senc, N, K, xq, xs, RC_NAT, M, y, res, nullptr, b.w, b.s, b.y, st);
    if (route == R_MF)
        return launch_mf(qtype, w, s, senc, N, K, xq, xs, true, M, y, res, nullptr, b.w, b.s, b.y, st);
    return launch_rc(qtype, w, s, senc, N, K, xq, xs, RC_NAT, M, y, res, nullptr, b.w, b.s, b.y, st);
}

// 2..16 int8 rows already in the matrix-core fragment order (a producer's
// fragment output): one launch of the row-contiguous matrix-core kernel, or of
// the streaming one where the rows exceed one round of it.  Long K splits over
// workgroups when a workspace of frag_workspace_need bytes is given (no launch
// before it: the split keeps its own counters), else runs the segment loop.
static int prequant_frag(int qtype, const void* w, const void* s, int senc, int group, int N, int K,
                         const void* xf, const void* xsf, int M, void* y, const void* res, void* wsp,
                         size_t wsp_bytes, void* stream, Second b = Second()) {
    int rc = validate_weights(qtype, w, s, senc, group, N, K, M);
    if (rc != VIPER_OK) return rc;
    if (xf == nullptr || xsf == nullptr || y == nullptr || M < 2 || !rc_ok(qtype, K)) return VIPER_INVALID_ARGUMENT;
    if (misaligned(xf, 16) || misaligned(xsf, 16) || misaligned(y, 2) || misaligned(res, 2))
        return VIPER_INVALID_ARGUMENT;
    rc = validate_second(b, qtype, senc, group, N, K, M, res, nullptr);
    if (rc != VIPER_OK) return rc;
    if (wsp != nullptr && misaligned(wsp, 16)) return VIPER_INVALID_ARGUMENT;
    const size_t need = b.w == nullptr ? frag_workspace_need(qtype, N, K, M) : 0;
    if (wsp != nullptr && need > 0 && wsp_bytes < need) return VIPER_INVALID_ARGUMENT;
    const Route route = frag_route(qtype, N, K, M, b.w != nullptr, wsp != nullptr);
    if (route == R_SG)
        return launch_sg(qtype, w, s, senc, N, K, xf, xsf, RC_FRAG, M, y, res, nullptr, b.w, b.s, b.y, (hipStream_t)stream);
    uint64_t* sp = route == R_SPLIT ? (uint64_t*)((uint8_t*)wsp + RC_CTL_BYTES) : nullptr;
    unsigned* sc = route == R_SPLIT ? (unsigned*)wsp : nullptr;
    return launch_rc(qtype, w, s, senc, N, K, xf, xsf, RC_FRAG, M, y, res, nullptr, b.w, b.s, b.y,
                     (hipStream_t)stream, sp, sc);
}

}  // namespace vq

// ------------------------------------------------------------------- C ABI

extern "C" int viper_hip_abi_version(void) { return VIPER_QLINEAR_ABI_VERSION; }

extern "C" int viper_hip_group_size(int qtype) { return vq::group_of(qtype); }

extern "C" size_t viper_hip_qlinear_workspace_bytes(int qtype, int N, int K, int M) {
    return vq::workspace_need(qtype, N, K, M);
}

extern "C" size_t viper_hip_qlinear_workspace_layout(int qtype, int N, int K, int M, size_t* offsets) {
    const vq::WsLayout l = vq::workspace_layout(qtype, N, K, M);
    if (offsets != nullptr) {
        offsets[0] = l.total ? (size_t)vq::RC_CTL_MISS * 4 : SIZE_MAX;
        offsets[1] = l.total ? l.cnt : SIZE_MAX;
        offsets[2] = l.blocks ? l.sp : SIZE_MAX;
        offsets[3] = l.total ? l.xq : SIZE_MAX;
        offsets[4] = l.total ? l.xs : SIZE_MAX;
        offsets[5] = (size_t)l.blocks;
    }
    return l.total;
}

extern "C" size_t viper_hip_qlinear_frag_workspace_bytes(int qtype, int N, int K, int M) {
    return vq::frag_workspace_need(qtype, N, K, M);
}

extern "C" int viper_hip_qlinear(int qtype, const void* w_packed, const void* w_scales,
                                 int scale_enc, int group, int N, int K, const void* x_bf16, int M,
                                 void* y_bf16, const void* residual_bf16, void* workspace,
                                 size_t workspace_bytes, void* stream) {
    return vq::qlinear_common(qtype, w_packed, w_scales, scale_enc, group, N, K, x_bf16, M, y_bf16,
                              residual_bf16, workspace, workspace_bytes, nullptr, stream);
}

extern "C" int viper_hip_qlinear_static(int qtype, const void* w_packed, const void* w_scales, int scale_enc,
                                        int group, int N, int K, const void* x_bf16, int M, void* y_bf16,
                                        const void* residual_bf16, void* stream) {
    const size_t need = vq::workspace_need(qtype, N, K, M);
    if (need > vq::STATIC_SCRATCH_BYTES) return VIPER_INVALID_ARGUMENT;
    void* wsp = nullptr;
    if (need > 0) {
        const int rc = vq::scratch_address(&wsp);
        if (rc != VIPER_OK) return rc;
    }
    return vq::qlinear_common(qtype, w_packed, w_scales, scale_enc, group, N, K, x_bf16, M, y_bf16, residual_bf16,
                              wsp, need > 0 ? vq::STATIC_SCRATCH_BYTES : 0, nullptr, stream);
}

extern "C" int viper_hip_qlinear_partials(int qtype, const void* w_packed, const void* w_scales,
                                          int scale_enc, int group, int N, int K,
                                          const void* x_bf16, int M, void* y_bf16,
                                          const void* residual_bf16, void* workspace,
                                          size_t workspace_bytes, int32_t* partials,
                                          void* stream) {
    if (partials == nullptr) return VIPER_INVALID_ARGUMENT;
    return vq::qlinear_common(qtype, w_packed, w_scales, scale_enc, group, N, K, x_bf16, M, y_bf16,
                              residual_bf16, workspace, workspace_bytes, partials, stream);
}

extern "C" int viper_hip_qlinear_route(int qtype, int input, int N, int K, int M, int matrices) {
    const int G = vq::group_of(qtype);
    if (G == 0 || N <= 0 || K <= 0 || M <= 0 || M > VIPER_QLINEAR_MAX_M || K > VIPER_QLINEAR_MAX_K || K % G != 0 ||
        matrices < 1 || matrices > 2)
        return -1;
    const bool pair = matrices == 2;
    switch (input) {
        case VIPER_INPUT_BF16: return vq::linear_route(qtype, N, K, M, pair, false);
        case VIPER_INPUT_INT8: return vq::prequant_route(qtype, N, K, M, pair);
        case VIPER_INPUT_FRAG: return M < 2 || !vq::rc_ok(qtype, K) ? -1 : (int)vq::frag_route(qtype, N, K, M, pair, true);
        default: return -1;
    }
}

extern "C" int viper_hip_quantize_act(int group, const void* x_bf16, int M, int K, void* xq,
                                      void* xs, void* stream) {
    if (group != 64 && group != 32) return VIPER_INVALID_ARGUMENT;
    if (x_bf16 == nullptr || xq == nullptr || xs == nullptr) return VIPER_INVALID_ARGUMENT;
    if (M <= 0 || K <= 0 || K % group != 0) return VIPER_INVALID_ARGUMENT;
    if ((int64_t)M * K > INT32_MAX / 2) return VIPER_INVALID_ARGUMENT;
    if (vq::misaligned(x_bf16, 16) || vq::misaligned(xq, 8) || vq::misaligned(xs, 4))
        return VIPER_INVALID_ARGUMENT;
    return vq::launch_quantize(group, x_bf16, M, K, xq, xs, false, (hipStream_t)stream);
}

extern "C" int viper_hip_qlinear_prequantized(int qtype, const void* w_packed,
                                              const void* w_scales, int scale_enc, int group,
                                              int N, int K, const void* xq, const void* xs, int M,
                                              void* y_bf16, const void* residual_bf16,
                                              void* stream) {
    return vq::prequant_common(qtype, w_packed, w_scales, scale_enc, group, N, K, xq, xs, M, y_bf16,
                               residual_bf16, stream);
}

extern "C" int viper_hip_qlinear_fused2(int qtype, const void* w0_packed, const void* w0_scales,
                                        const void* w1_packed, const void* w1_scales, int scale_enc,
                                        int group, int N, int K, const void* x_bf16, int M,
                                        void* y0_bf16, void* y1_bf16, void* workspace,
                                        size_t workspace_bytes, void* stream) {
    if (w1_packed == nullptr || w1_scales == nullptr || y1_bf16 == nullptr) return VIPER_INVALID_ARGUMENT;
    return vq::qlinear_common(qtype, w0_packed, w0_scales, scale_enc, group, N, K, x_bf16, M, y0_bf16,
                              nullptr, workspace, workspace_bytes, nullptr, stream,
                              vq::Second{w1_packed, w1_scales, y1_bf16});
}

extern "C" int viper_hip_qlinear_fused2_prequantized(int qtype, const void* w0_packed,
                                                     const void* w0_scales, const void* w1_packed,
                                                     const void* w1_scales, int scale_enc, int group,
                                                     int N, int K, const void* xq, const void* xs,
                                                     int M, void* y0_bf16, void* y1_bf16,
                                                     void* stream) {
    if (w1_packed == nullptr || w1_scales == nullptr || y1_bf16 == nullptr) return VIPER_INVALID_ARGUMENT;
    return vq::prequant_common(qtype, w0_packed, w0_scales, scale_enc, group, N, K, xq, xs, M, y0_bf16,
                               nullptr, stream, vq::Second{w1_packed, w1_scales, y1_bf16});
}

extern "C" int viper_hip_qlinear_prequantized_frag(int qtype, const void* w_packed, const void* w_scales,
                                                   int scale_enc, int group, int N, int K, const void* xfrag,
                                                   const void* xsfrag, int M, void* y_bf16,
                                                   const void* residual_bf16, void* workspace, size_t workspace_bytes,
                                                   void* stream) {
    return vq::prequant_frag(qtype, w_packed, w_scales, scale_enc, group, N, K, xfrag, xsfrag, M, y_bf16,
                             residual_bf16, workspace, workspace_bytes, stream);
}

extern "C" int viper_hip_qlinear_fused2_prequantized_frag(int qtype, const void* w0_packed,
                                                          const void* w0_scales, const void* w1_packed,
                                                          const void* w1_scales, int scale_enc, int group,
                                                          int N, int K, const void* xfrag, const void* xsfrag,
                                                          int M, void* y0_bf16, void* y1_bf16, void* stream) {
    if (w1_packed == nullptr || w1_scales == nullptr || y1_bf16 == nullptr) return VIPER_INVALID_ARGUMENT;
    return vq::prequant_frag(qtype, w0_packed, w0_scales, scale_enc, group, N, K, xfrag, xsfrag, M, y0_bf16,
                             nullptr, nullptr, 0, stream, vq::Second{w1_packed, w1_scales, y1_bf16});
}

extern "C" int viper_hip_qlinear_frag_timeline(int qtype, const void* w_packed, const void* w_scales, int scale_enc,
                                               int group, int N, int K, const void* xfrag, const void* xsfrag, int M,
                                               void* y_bf16, uint64_t* stamps, size_t stamp_bytes, int* workgroups,
                                               int* waves_per_workgroup, void* workspace, size_t workspace_bytes,
                                               void* stream) {
    int rc = vq::validate_weights(qtype, w_packed, w_scales, scale_enc, group, N, K, M);
    if (rc != VIPER_OK) return rc;
    if (xfrag == nullptr || xsfrag == nullptr || y_bf16 == nullptr || vq::misaligned(xfrag, 16) ||
        vq::misaligned(xsfrag, 16) || vq::misaligned(y_bf16, 2) || vq::misaligned(stamps, 8) ||
        vq::misaligned(workspace, 16))
        return VIPER_INVALID_ARGUMENT;
    const size_t need = vq::frag_workspace_need(qtype, N, K, M);
    if (workspace != nullptr && (need == 0 || workspace_bytes < need)) return VIPER_INVALID_ARGUMENT;
    // the kernel the production call runs, and only the calls its first kernel took
    if (vq::frag_route(qtype, N, K, M, false, workspace != nullptr) == vq::R_SG) {
        if (!vq::rc_timeline_ok(qtype, N, K, M, workspace != nullptr)) return VIPER_INVALID_ARGUMENT;
        return vq::launch_sg_timeline(qtype, w_packed, w_scales, scale_enc, N, K, xfrag, xsfrag, M, y_bf16, stamps, stamp_bytes,
                                      workgroups, waves_per_workgroup, (hipStream_t)stream);
    }
    return vq::launch_rc_timeline(qtype, w_packed, w_scales, scale_enc, N, K, xfrag, xsfrag, M, y_bf16, stamps,
                                  stamp_bytes, workgroups, waves_per_workgroup, (unsigned*)workspace,
                                  (hipStream_t)stream);
}

extern "C" int viper_hip_qlinear_m1(int qtype, int scale_enc, int group, int K, int prologue, const void* a,
                                    const void* b, float eps, void* norm_out, int n_out,
                                    const void* const* w_packed, const void* const* w_scales, const int* N,
                                    void* const* y_bf16, const void* residual_bf16, void* stream) {
    if (n_out < 1 || n_out > 3 || w_packed == nullptr || w_scales == nullptr || N == nullptr || y_bf16 == nullptr)
        return VIPER_INVALID_ARGUMENT;
    if (prologue < VIPER_PROLOGUE_BF16 || prologue > VIPER_PROLOGUE_SWIGLU) return VIPER_INVALID_ARGUMENT;
    vq::M1Out outs[3];
    for (int i = 0; i < n_out; ++i) {
        const int rc = vq::validate_weights(qtype, w_packed[i], w_scales[i], scale_enc, group, N[i], K, 1);
        if (rc != VIPER_OK) return rc;
        if (y_bf16[i] == nullptr || vq::misaligned(y_bf16[i], 2)) return VIPER_INVALID_ARGUMENT;
        outs[i] = vq::M1Out{w_packed[i], w_scales[i], y_bf16[i], N[i]};
    }
    if (a == nullptr || (prologue != VIPER_PROLOGUE_BF16 && b == nullptr)) return VIPER_INVALID_ARGUMENT;
    const size_t align_a = prologue == VIPER_PROLOGUE_INT8 ? 8 : 16;
    const size_t align_b = prologue == VIPER_PROLOGUE_INT8 ? 4 : 16;
    if (vq::misaligned(a, align_a) || vq::misaligned(b, align_b) || vq::misaligned(norm_out, 16) ||
        vq::misaligned(residual_bf16, 2))
        return VIPER_INVALID_ARGUMENT;
    if (norm_out != nullptr && prologue != VIPER_PROLOGUE_RMSNORM) return VIPER_INVALID_ARGUMENT;
    if (vq::lds_m1(qtype, K) > (size_t)vq::LDS_MAX) return VIPER_INVALID_ARGUMENT;
    if ((prologue == VIPER_PROLOGUE_RMSNORM || prologue == VIPER_PROLOGUE_SWIGLU) && !vq::m1_folded_ok(qtype, K))
        return VIPER_INVALID_ARGUMENT;
    return vq::launch_m1(qtype, scale_enc, K, prologue, a, b, eps, norm_out, outs, n_out, residual_bf16, nullptr,
                         (hipStream_t)stream, 1, false);
}

extern "C" int viper_hip_qlinear_m1_swiglu(int qtype, int scale_enc, int group, int K, int prologue, const void* a,
                                           const void* b, float eps, void* norm_out, const void* w_gate,
                                           const void* s_gate, const void* w_up, const void* s_up, int N,
                                           void* h_bf16, void* gate_bf16, void* up_bf16, void* stream) {
    if (prologue != VIPER_PROLOGUE_BF16 && prologue != VIPER_PROLOGUE_RMSNORM) return VIPER_INVALID_ARGUMENT;
    int rc = vq::validate_weights(qtype, w_gate, s_gate, scale_enc, group, N, K, 1);
    if (rc != VIPER_OK) return rc;
    rc = vq::validate_weights(qtype, w_up, s_up, scale_enc, group, N, K, 1);
    if (rc != VIPER_OK) return rc;
    if (h_bf16 == nullptr || vq::misaligned(h_bf16, 2) || vq::misaligned(gate_bf16, 2) || vq::misaligned(up_bf16, 2))
        return VIPER_INVALID_ARGUMENT;
    if (a == nullptr || (prologue == VIPER_PROLOGUE_RMSNORM && b == nullptr)) return VIPER_INVALID_ARGUMENT;
    if (vq::misaligned(a, 16) || vq::misaligned(b, 16) || vq::misaligned(norm_out, 16)) return VIPER_INVALID_ARGUMENT;
    if (norm_out != nullptr && prologue != VIPER_PROLOGUE_RMSNORM) return VIPER_INVALID_ARGUMENT;
    if (vq::lds_m1(qtype, K) > (size_t)vq::LDS_MAX) return VIPER_INVALID_ARGUMENT;
    if (prologue == VIPER_PROLOGUE_RMSNORM && !vq::m1_folded_ok(qtype, K)) return VIPER_INVALID_ARGUMENT;
    return vq::launch_m1_swiglu(qtype, scale_enc, K, prologue, a, b, eps, norm_out, w_gate, s_gate, w_up, s_up, N,
                                h_bf16, gate_bf16, up_bf16, (hipStream_t)stream);
}

extern "C" int viper_hip_qlinear_timeline(int qtype, const void* w_packed, const void* w_scales, int scale_enc,
                                          int group, int N, int K, const void* x_bf16, void* y_bf16, uint64_t* stamps,
                                          size_t stamp_bytes, int* workgroups, int* waves_per_workgroup,
                                          void* stream) {
    const int rc = vq::validate_weights(qtype, w_packed, w_scales, scale_enc, group, N, K, 1);
    if (rc != VIPER_OK) return rc;
    if (x_bf16 == nullptr || y_bf16 == nullptr || vq::misaligned(x_bf16, 16) || vq::misaligned(y_bf16, 2) ||
        vq::misaligned(stamps, 8))
        return VIPER_INVALID_ARGUMENT;
    return vq::launch_m1_timeline(qtype, scale_enc, K, x_bf16, w_packed, w_scales, y_bf16, N, stamps, stamp_bytes,
                                  workgroups, waves_per_workgroup, (hipStream_t)stream);
}

extern "C" int viper_hip_check_bf16_rounding(unsigned long long* count, void* stream) {
    if (count == nullptr || vq::misaligned(count, 8)) return VIPER_INVALID_ARGUMENT;
    void* args[] = {&count};
    vq::launch((const void*)vq::check_bf16_kernel, vq::BFC_GRID, vq::BFC_NT, 0, (hipStream_t)stream, args);
    return vq::status_of(hipGetLastError());
}

extern "C" int viper_hip_check_quantizer(int exp_lo, int exp_hi, int32_t* counts, void* stream) {
    if (counts == nullptr || exp_lo < 0 || exp_hi > 254 || exp_lo > exp_hi)
        return VIPER_INVALID_ARGUMENT;
    if (vq::misaligned(counts, 4)) return VIPER_INVALID_ARGUMENT;
    int ab0 = exp_lo << 7;
    int32_t* c = counts;
    void* args[] = {&ab0, &c};
    const unsigned grid = (unsigned)((exp_hi - exp_lo + 1) << 7);
    vq::launch((const void*)vq::check_quantizer_kernel, grid, vq::NT, 0, (hipStream_t)stream, args);
    return vq::status_of(hipGetLastError());
}
