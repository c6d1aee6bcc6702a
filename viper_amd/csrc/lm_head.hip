// LM head: bf16 GEMV (the reference's linear_bf16,
// kernels/ops/linear_bf16_kernel.cu:15-70) and greedy argmax
// (sampling_greedy_bf16, kernels/ops/sampling_kernel.cu:11-80).
//
// GEMV: y[m][n] = bf16_RNE(sum_k w[n][k] * x[m][k]) with fp32 accumulation.
// The matrix (vocab x hidden, e.g. 166144 x 2560 = 850 MB) is streamed once
// from HBM: a team of TS lanes owns a row and each lane issues its 16-byte
// chunks of the row at once (non-temporal loads), after the activation loads
// (loads retire in issue order, so x is staged into LDS while the weights
// are in flight).  Each 16-byte chunk is 8 bf16 and costs 4 v_dot2_f32_bf16
// per activation row; teams are reduced with DPP in a fixed order.  More rows
// take the matrix-core kernel below (head_mfma_kernel).
//
// Argmax: one workgroup per logits row; every lane requests all of its
// 16-byte octets at once, keeps the first octet holding its largest value
// (octet maxima by v_max, compared with strict >, so NaN never wins and ties
// keep the smaller index), then finds the first element of that octet equal
// to it; lanes and waves combine by (value, then smaller index).

#include "qlinear_host.h"

namespace vq {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c,
                                           false);
}

constexpr int LH_CPL = 10;  // 16-byte chunk slots per lane per row segment
constexpr int LH_XS = 4;    // activation octets per thread loaded before the weights

template <int TS, int NTT, int MT, bool EXACT>
__global__ void __launch_bounds__(NTT)
gemv_bf16_kernel(const uint16_t* __restrict__ w, const uint16_t* x, uint16_t* __restrict__ y,
                 int M, int N, int K) {
    constexpr int ROWS = NTT / TS;
    extern __shared__ __align__(16) u32x4 lx[];  // [M][K/8]
    const int tid = (int)threadIdx.x;
    const int l = tid % TS;
    const int rr = tid / TS;
    // row blocks in XCD order (each XCD streams one contiguous range of rows):
    // 121.5 -> 117.3 us for the 166144 x 2560 head
    const int row0 = xcd_block((int)blockIdx.x, (int)gridDim.x) * ROWS;
    const int row = row0 + rr;
    const int nrows = min(ROWS, N - row0);
    const bool row_ok = rr < nrows;
    const int CPR = K / 8;
    const int nx = M * CPR;

    // 1. activation octets, then the weight chunks of the first segment
    const auto xr = buf(x, (uint32_t)nx * 16);
    u32x4 xv[LH_XS];
#pragma unroll
    for (int i = 0; i < LH_XS; ++i) xv[i] = bload16(xr, (tid + NTT * i) * 16);
    issue_fence();
    const uint32_t rbytes = (uint32_t)K * 2;
    const auto wr = buf(w + (size_t)row0 * K, (uint32_t)nrows * rbytes);
    const int segw = TS * LH_CPL;
    const int nseg = EXACT ? 1 : (CPR + segw - 1) / segw;
    u32x4 wv[LH_CPL];
    auto load_seg = [&](int seg) {
#pragma unroll
        for (int j = 0; j < LH_CPL; ++j) {
            const int c = seg * segw + j * TS + l;
            const bool in = EXACT || c < CPR;
            wv[j] = bload16<AUX_NT>(wr, in ? rr * (int)rbytes + c * 16 : OOB);
        }
    };
    load_seg(0);

    // 2. stage x into LDS
#pragma unroll
    for (int i = 0; i < LH_XS; ++i)
        if (tid + NTT * i < nx) lx[tid + NTT * i] = xv[i];
    for (int i = tid + NTT * LH_XS; i < nx; i += NTT) lx[i] = bload16(xr, i * 16);
    lds_barrier();

    // 3. dots
    float acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = 0.0f;
    for (int seg = 0; seg < nseg; ++seg) {
        if (seg) load_seg(seg);
#pragma unroll
        for (int j = 0; j < LH_CPL; ++j) {
            const int c = seg * segw + j * TS + l;
            const bool ok = EXACT || c < CPR;
            const int cc = EXACT ? c : min(c, CPR - 1);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (m < M) {
                    const u32x4 a = lx[m * CPR + cc];
                    float t = acc[m];
                    t = dot2_bf16(wv[j].x, a.x, t);
                    t = dot2_bf16(wv[j].y, a.y, t);
                    t = dot2_bf16(wv[j].z, a.z, t);
                    t = dot2_bf16(wv[j].w, a.w, t);
                    acc[m] = ok ? t : acc[m];  // a lane past the row adds nothing (not even 0 * inf)
                }
            }
        }
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        if (m < M) {
            const float v = team_sum<TS>(acc[m]);
            if (l == 0 && row_ok) y[(size_t)m * N + row] = f2bf(v);
        }
    }
}

// More rows on the matrix cores.  The dot kernel reads every activation row
// from LDS for each weight chunk, so at 8 rows it is bound by LDS (166144 x
// 2560: 117 us for 2 rows, 240 for 8, 455 for 12).  Here a weight tile of 16
// rows is the A operand of v_mfma_f32_16x16x32_bf16 and the activation rows
// the 16 columns of B, read once per tile.  A fragment load straight from
// memory (16 rows x 64 bytes per instruction) streams at 4.9 TB/s, so each
// wave loads 2 rows x 512 contiguous bytes per instruction and turns its 16
// rows x 512 bytes through an LDS buffer of its own (row stride 528 bytes:
// conflict-free 16-byte reads).  Persistent workgroups stage the activation
// once; each wave keeps the next 8 KB segment (of the next tile, too) in
// flight while it multiplies one.  Bound by the weight stream: 127 us for 2..6
// rows, 129 for 8, 132 for 12 (850 MB, 6.5-6.7 TB/s; the dot kernel's one row
// 117 us).  tpw tiles per workgroup; SHARE: a workgroup's few tiles go to 1 << lk
// waves each, one tile a wave (hm_split).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int HM_NTT = 512;
constexpr int HM_SC = 32;              // 16-byte chunks of a row per segment
constexpr int HM_STR = HM_SC * 16 + 16;  // LDS row stride of the wave's buffer
constexpr int HM_XS = LDS_MAX / 16 / HM_NTT;  // activation chunks per thread (at most 64 KiB of rows)

__host__ __device__ constexpr size_t hm_lds_bytes(int M, int K) {
    return (size_t)((K / 8 + HM_SC - 1) / HM_SC * HM_SC) * M * 16 + (size_t)(HM_NTT / 64) * 16 * HM_STR;
}

template <bool SHARE>
__global__ void __launch_bounds__(HM_NTT)
head_mfma_kernel(const uint16_t* w, const uint16_t* x, uint16_t* y, int M, int N, int K, int tpw, int gx, int lk) {
    constexpr int W = HM_NTT / 64, RI = 64 / HM_SC;
    extern __shared__ __align__(16) u32x4 lx[];  // x as [chunk][M], zeros past the row; then the waves' buffers
    const int tid = (int)threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q = lane >> 4;
    const int CPR = K / 8, NS = (CPR + HM_SC - 1) / HM_SC, KP = NS * HM_SC;
    uint8_t* tb = (uint8_t*)(lx + (size_t)KP * M) + wave * (16 * HM_STR);
    // workgroup blocks in XCD order; a grid rounded up to whole XCD turns
    const int bid = ((int)blockIdx.x & 7) * gx + ((int)blockIdx.x >> 3);
    const int tend = min((bid + 1) * tpw, (N + 15) / 16);
    if (bid * tpw >= tend) return;
    const int ks = SHARE ? 1 << lk : 1, s0 = SHARE ? wave & (ks - 1) : 0;  // segments s0, s0 + ks, ... of its tiles
    const int t0 = bid * tpw + (SHARE ? wave >> lk : wave);
    const int nx = M * CPR;
    const auto xr = buf(x, (uint32_t)nx * 16);
    u32x4 xv[HM_XS];
#pragma unroll
    for (int i = 0; i < HM_XS; ++i) xv[i] = bload16(xr, (tid + HM_NTT * i) * 16);
    issue_fence();

    struct Seg {
        u32x4 v[16 / RI];
    };
    struct Cur {
        int t, s;  // tile, segment of the row
    };
    const uint32_t rbytes = (uint32_t)K * 2;
    auto advance = [&](Cur& c) {
        if ((c.s += ks) >= NS) {
            c.s = s0;
            c.t += SHARE ? W >> lk : W;
        }
    };
    auto load = [&](Seg& S, const Cur& c) {
        const int row0 = c.t * 16, n = min(16, N - row0);
        const auto wr = buf(w + (size_t)row0 * K, (uint32_t)n * rbytes);
        const int ch = c.s * HM_SC + lane % HM_SC;
#pragma unroll
        for (int i = 0; i < 16 / RI; ++i)
            S.v[i] = bload16<AUX_NT>(wr, ch < CPR ? (i * RI + lane / HM_SC) * (int)rbytes + ch * 16 : OOB);
    };
    Cur lc{!SHARE || s0 < NS ? t0 : tend, s0}, cc = lc;
    Seg S0, S1;
    if (lc.t < tend) load(S0, lc);
    issue_fence();
#pragma unroll
    for (int i = 0; i < HM_XS; ++i) {
        const int t = tid + HM_NTT * i;
        if (t < nx) {
            const int m = t / CPR, c = t - m * CPR;
            lx[c * M + m] = xv[i];
        }
    }
    for (int t = nx + tid; t < KP * M; t += HM_NTT) lx[t] = u32x4{0u, 0u, 0u, 0u};
    lds_barrier();

    const int mr = min(l16, M - 1);  // columns past M repeat the last row and are not stored
    f32x4 a0 = {0.0f, 0.0f, 0.0f, 0.0f}, a1 = a0;
    // the lane holds rows 4q .. 4q + 3 of a tile for activation row l16
    auto store = [&](int t, const f32x4& v) {
        const int n0 = t * 16 + 4 * q;
        const uint32_t p0 = f2bf2(v[0], v[1]), p1 = f2bf2(v[2], v[3]);
        if (l16 < M) {
            uint16_t* o = y + (size_t)l16 * N + n0;
            if (n0 < N) o[0] = (uint16_t)p0;
            if (n0 + 1 < N) o[1] = (uint16_t)(p0 >> 16);
            if (n0 + 2 < N) o[2] = (uint16_t)p1;
            if (n0 + 3 < N) o[3] = (uint16_t)(p1 >> 16);
        }
    };
    auto compute = [&](const Seg& S, const Cur& c) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int i = 0; i < 16 / RI; ++i)
            *(u32x4*)(tb + (i * RI + lane / HM_SC) * HM_STR + (lane % HM_SC) * 16) = S.v[i];
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
        // k-slot q of each product: chunk q of its four (the same for both operands)
#pragma unroll
        for (int kb = 0; kb < HM_SC / 8; ++kb) {
            const u32x4 w0 = *(const u32x4*)(tb + l16 * HM_STR + (kb * 8 + q) * 16);
            const u32x4 w1 = *(const u32x4*)(tb + l16 * HM_STR + (kb * 8 + 4 + q) * 16);
            const u32x4 x0 = lx[(c.s * HM_SC + kb * 8 + q) * M + mr], x1 = lx[(c.s * HM_SC + kb * 8 + 4 + q) * M + mr];
            a0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w0), __builtin_bit_cast(bf16x8, x0),
                                                         a0, 0, 0, 0);
            a1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w1), __builtin_bit_cast(bf16x8, x1),
                                                         a1, 0, 0, 0);
        }
        if (SHARE || c.s + 1 < NS) return;
        store(c.t, a0 + a1);
        a0 = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        a1 = a0;
    };
    // (separate code for the last segment, so that no wait counts loads that
    // may not have been issued)
    if (cc.t < tend) {
        for (;;) {
            advance(lc);
            if (lc.t >= tend) {
                compute(S0, cc);
                break;
            }
            load(S1, lc);
            issue_fence();
            compute(S0, cc);
            advance(cc);
            advance(lc);
            if (lc.t >= tend) {
                compute(S1, cc);
                break;
            }
            load(S0, lc);
            issue_fence();
            compute(S1, cc);
            advance(cc);
        }
    }
    if constexpr (SHARE) {
        // the waves of a tile meet in LDS, added in wave order
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
        __builtin_amdgcn_wave_barrier();
        *(f32x4*)(tb + lane * 16) = a0 + a1;
        lds_barrier();
        if (s0 != 0 || t0 >= tend) return;
        f32x4 v = *(const f32x4*)(tb + lane * 16);
        for (int u = 1; u < ks; ++u) v += *(const f32x4*)(tb + u * (16 * HM_STR) + lane * 16);
        store(t0, v);
    }
}

// (value, index) order of the greedy pick: larger value, then smaller index
__device__ __forceinline__ void better(float& v, int& i, float ov, int oi) {
    if (ov > v || (ov == v && oi < i)) {
        v = ov;
        i = oi;
    }
}

constexpr int AM_NT = 1024;
constexpr int AM_PT = 24;  // octets per lane in flight at once (the whole 166144-logit row in one pass)

// Largest of the 8 bf16 values of an octet (v_max_f32 / v_max3_f32 return
// the non-NaN operand, so NaN never wins, as with the strict > scan).
__device__ __forceinline__ float octet_max(const u32x4& q) {
    const float f0 = __uint_as_float(q.x << 16), f1 = __uint_as_float(q.x & 0xffff0000u);
    const float f2 = __uint_as_float(q.y << 16), f3 = __uint_as_float(q.y & 0xffff0000u);
    const float f4 = __uint_as_float(q.z << 16), f5 = __uint_as_float(q.z & 0xffff0000u);
    const float f6 = __uint_as_float(q.w << 16), f7 = __uint_as_float(q.w & 0xffff0000u);
    return fmaxf(fmaxf(fmaxf(f0, f1), fmaxf(f2, f3)), fmaxf(fmaxf(f4, f5), fmaxf(f6, f7)));
}

__global__ void __launch_bounds__(AM_NT)
argmax_bf16_kernel(const uint16_t* logits, int32_t* __restrict__ out, int V) {
    __shared__ float sv[AM_NT / 64];
    __shared__ int si[AM_NT / 64];
    const int b = (int)blockIdx.x;
    const int tid = (int)threadIdx.x;
    const uint16_t* row = logits + (size_t)b * V;
    // octets (16-byte loads when the row is 16-byte aligned): per lane the
    // first octet holding its largest value (octets are visited in increasing
    // order per lane, strict >), all of a pass's loads in flight at once
    // (buffer loads: past the row they read zero and are skipped by the
    // index bound)
    const bool vec = ((((uintptr_t)row) & 15) == 0);
    const int noct = vec ? V / 8 : 0;
    const auto rr = buf(row, (uint32_t)noct * 16);
    float best = -__builtin_inff();
    int boct = -1;
    for (int o0 = tid; o0 < noct; o0 += AM_NT * AM_PT) {
        u32x4 q[AM_PT];
#pragma unroll
        for (int i = 0; i < AM_PT; ++i) q[i] = bload16(rr, (o0 + i * AM_NT) * 16);
#pragma unroll
        for (int i = 0; i < AM_PT; ++i) {
            const int o = o0 + i * AM_NT;
            const float m = octet_max(q[i]);
            if (o < noct && m > best) {
                best = m;
                boct = o;
            }
        }
    }
    // the first element of that octet equal to its maximum
    int idx = 0;
    if (boct >= 0) {
        const u32x4 q = bload16(rr, boct * 16);
        const uint32_t wd[4] = {q.x, q.y, q.z, q.w};
        idx = boct * 8 + 7;
#pragma unroll
        for (int j = 7; j >= 0; --j)
            if (bf16f((wd[j >> 1] >> (16 * (j & 1))) & 0xffffu) == best) idx = boct * 8 + j;
    }
    // elements past the last octet (or an unaligned row), one per lane
    for (int v = noct * 8 + tid; v < V; v += AM_NT) {
        const float f = bf16f(row[v]);
        if (f > best) {
            best = f;
            idx = v;
        }
    }
    // Indices increase per lane but interleave across lanes, so equal maxima
    // resolve in the combine below (larger value, then smaller index).
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(best, off, 64);
        const int oi = __shfl_xor(idx, off, 64);
        better(best, idx, ov, oi);
    }
    if ((tid & 63) == 0) {
        sv[tid >> 6] = best;
        si[tid >> 6] = idx;
    }
    __syncthreads();
    if (tid == 0) {
        for (int i = 1; i < AM_NT / 64; ++i) better(best, idx, sv[i], si[i]);
        out[b] = idx;
    }
}

// Split argmax: P workgroups per row, each over GR_NT * PT consecutive octets
// (GR_NT threads, PT octets each, all requested at once; greedy_octets), meet
// through a 64-bit key per row in the caller's workspace:
//   key = (order(value) << 32) | (0xFFFFFFFF - index),
// where order maps floats to unsigned integers in the same order (+0 for
// both zeros, which compare equal), so the largest key is the largest value
// at its smallest index, the reference's (value, then smaller index) pick.
// Each workgroup takes the max into the row's key, then (after the max has
// returned, so it is performed first) counts itself on the row's counter;
// the workgroup that counts last swaps the key for 0, resets the counter and
// writes the index.  All four accesses are agent-scope atomics, performed in
// the order each workgroup issues them, so the last count sees every max.
// A workgroup with nothing above -inf offers (-inf, 0): a row with nothing
// above -inf gives 0, as the single-workgroup kernel does.
constexpr int GR_NT = 256;

__device__ __forceinline__ uint64_t greedy_key(float v, int i) {
    const uint32_t u = v == 0.0f ? 0u : __float_as_uint(v);
    const uint32_t o = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ((uint64_t)o << 32) | (uint64_t)(0xFFFFFFFFu - (uint32_t)i);
}

template <int PT>
__global__ void __launch_bounds__(GR_NT)
argmax_split_kernel(const uint16_t* logits, int32_t* __restrict__ out, int V, int P, uint64_t* keys,
                    unsigned* cnt) {
    __shared__ float sv[GR_NT / 64];
    __shared__ int si[GR_NT / 64];
    constexpr int OCT = GR_NT * PT;
    const int b = (int)blockIdx.x / P, p = (int)blockIdx.x % P;
    const int tid = (int)threadIdx.x;
    const int noct = V / 8;  // whole octets (the host takes this kernel for V % 8 == 0 only)
    const int o0 = p * OCT;
    const int n = min(OCT, noct - o0);
    const auto rr = buf(logits + (size_t)b * V + (size_t)o0 * 8, (uint32_t)n * 16);
    u32x4 q[PT];
#pragma unroll
    for (int i = 0; i < PT; ++i) q[i] = bload16(rr, (tid + i * GR_NT) * 16);
    float best = -__builtin_inff();
    int boct = -1;
#pragma unroll
    for (int i = 0; i < PT; ++i) {
        const int o = tid + i * GR_NT;
        const float m = octet_max(q[i]);
        if (o < n && m > best) {
            best = m;
            boct = o;
        }
    }
    int idx = 0;
    if (boct >= 0) {
        const u32x4 v = bload16(rr, boct * 16);
        const uint32_t wd[4] = {v.x, v.y, v.z, v.w};
        idx = (o0 + boct) * 8 + 7;
#pragma unroll
        for (int j = 7; j >= 0; --j)
            if (bf16f((wd[j >> 1] >> (16 * (j & 1))) & 0xffffu) == best) idx = (o0 + boct) * 8 + j;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(best, off, 64);
        const int oi = __shfl_xor(idx, off, 64);
        better(best, idx, ov, oi);
    }
    if ((tid & 63) == 0) {
        sv[tid >> 6] = best;
        si[tid >> 6] = idx;
    }
    __syncthreads();
    if (tid == 0) {
        for (int i = 1; i < GR_NT / 64; ++i) better(best, idx, sv[i], si[i]);
        const uint64_t prev =
            __hip_atomic_fetch_max(keys + b, greedy_key(best, idx), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // the count depends on the returned max (no key is all ones), so it
        // is issued only after the max is performed
        const unsigned inc = 1u + (unsigned)(prev == ~0ull);
        const unsigned t = __hip_atomic_fetch_add(cnt + b, inc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (t == (unsigned)(P - 1)) {
            const uint64_t k = __hip_atomic_exchange(keys + b, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(cnt + b, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            out[b] = (int32_t)(0xFFFFFFFFu - (uint32_t)k);
        }
    }
}

// ---- host

typedef void (*lh_fn)(const uint16_t*, const uint16_t*, uint16_t*, int, int, int);

template <int TS, bool EXACT>
static lh_fn lh_pick_mt(int mt) {
    switch (mt) {
        case 1: return gemv_bf16_kernel<TS, 256, 1, EXACT>;
        default: return gemv_bf16_kernel<TS, 256, 4, EXACT>;
    }
}
template <int TS>
static lh_fn lh_pick(int mt, bool exact) {
    return exact ? lh_pick_mt<TS, true>(mt) : lh_pick_mt<TS, false>(mt);
}

// The matrix-core kernel's tiles per workgroup and (log2) waves per tile.  Up to
// 16 tiles per CU: one round of workgroups, and where a workgroup has half as
// many tiles as waves or fewer the waves split the rows of each, so that no
// wave reads a row alone while others idle (8 rows of 2560, N = 1024 / 4096 /
// 16384 18.6 / 19.1 / 22.3 us with nine tiles to eight waves -> 5.7 / 6.8 / 16.2;
// 2 waves per tile at N = 4096 8.2, none 8.8; a second round of workgroups, 0.1
// to 0.8 of the chip, is as long as the first: N = 40000 50 -> 36.5, N = 50257 52
// -> 45).  Beyond, about three workgroups per CU in turn, each of an odd number
// of tiles (131072 x 4096: 157 us; 256 workgroups, whose first rows then lie
// 4 MB apart and meet in the same memory channels, 178 us; N = 65536, 4 rows of
// 8192, 16 tiles each 205 us, 9 each 185).
static void hm_split(int tiles, int segs, int& tpw, int& lk) {
    const int cus = device_cus(), waves = HM_NTT / 64;
    lk = 0;
    if (tiles < 16 * cus) {
        tpw = (tiles + cus - 1) / cus;
        while (lk < 3 && tpw <= waves >> (lk + 1) && (1 << lk) < segs) ++lk;
    } else {
        tpw = (tiles + 3 * cus - 1) / (3 * cus);
        tpw = (tpw < waves ? waves : tpw) | 1;
    }
}

// Several rows on the matrix cores, or on the dot kernel?  The dot kernel for
// the few rows whose LDS reads hide behind the weights (M x K up to 4 x 2560:
// 121 us against 127; 3 rows of 4096: N = 65536 88 against 94, N = 131072 175
// against 180; 4 rows of 3072 99 against 87 the other way, 5 rows of 1024: 43.7
// against 40.2), for up to 4 rows also where N is small (3 rows of 4096, N = 300
// / 1024 / 2560 5.3 / 5.9 / 8.4 us against 6.2 / 6.4 / 7.2), and for two rows of
// a large head (8192, N = 16384 / 32000 / 65536 53.6 / 91 / 171 against 47 / 97 / 185).
static bool hm_takes(int M, int N, int K) {
    if (M > 4) return true;
    if (M < 2 || N < 2048) return false;
    if (M == 4) return K >= 3072;
    return M * K > 12288 && (M == 3 || (N + 15) / 16 <= 4 * device_cus());
}

// Octets per thread of the split argmax.  Every workgroup's two atomics go to
// the one or two cache lines that hold all rows' keys and counters and are
// performed one after another there, ~15 ns a workgroup: with two octets per thread
// 166144 logits took 4.0 / 5.0 / 6.8 / 9.3 / 14.0 us for 1 / 2 / 4 / 8 / 16 rows,
// with eight (a quarter of the workgroups) 4.1 / 4.1 / 4.5 / 5.0 / 6.0; 32000
// logits 3.7 / 3.9 / 4.3 / 5.0 for 1 / 4 / 8 / 16 rows against 3.9 / 4.1 / 4.2 /
// 4.2.  So eight from 49 workgroups of two octets on.  (512 threads of four or
// eight octets 5.2 us for 8 rows, 1024 threads 5.8-6.3.)
constexpr int GR_WGS = 48;
static long greedy_wgs(int B, int V, int pt) { return (long)B * ((V / 8 + GR_NT * pt - 1) / (GR_NT * pt)); }
static int greedy_octets(int B, int V) { return greedy_wgs(B, V, 2) > GR_WGS ? 8 : 2; }

}  // namespace vq

extern "C" int viper_hip_linear_bf16(const void* w_bf16, const void* x_bf16, void* y_bf16, int M, int N,
                                     int K, void* stream) {
    if (w_bf16 == nullptr || x_bf16 == nullptr || y_bf16 == nullptr) return VIPER_INVALID_ARGUMENT;
    if (M <= 0 || N <= 0 || K <= 0 || M > VIPER_QLINEAR_MAX_M || K % 8 != 0) return VIPER_INVALID_ARGUMENT;
    if (vq::misaligned(w_bf16, 16) || vq::misaligned(x_bf16, 16) || vq::misaligned(y_bf16, 2))
        return VIPER_INVALID_ARGUMENT;
    const size_t lds = (size_t)M * K * 2;
    if (lds > (size_t)vq::LDS_MAX || (size_t)K * 2 * 256 > (size_t)INT32_MAX) return VIPER_INVALID_ARGUMENT;
    if (vq::hm_takes(M, N, K)) {
        const int tiles = (N + 15) / 16;
        int tpw = 0, lk = 0;
        vq::hm_split(tiles, (K / 8 + vq::HM_SC - 1) / vq::HM_SC, tpw, lk);
        int gx = ((tiles + tpw - 1) / tpw + 7) / 8;
        const void* fn = lk ? (const void*)vq::head_mfma_kernel<true> : (const void*)vq::head_mfma_kernel<false>;
        void* args[] = {&w_bf16, &x_bf16, &y_bf16, &M, &N, &K, &tpw, &gx, &lk};
        (void)hipLaunchKernel(fn, dim3((unsigned)(8 * gx)), dim3(vq::HM_NTT), args, vq::hm_lds_bytes(M, K), (hipStream_t)stream);
        return vq::status_of(hipGetLastError());
    }
    const int cpr = K / 8;
    int ts = 8;
    while (ts < 64 && ts * vq::LH_CPL < cpr) ts *= 2;
    const bool exact = cpr == ts * vq::LH_CPL;
    const int mt = M == 1 ? 1 : 4;
    vq::lh_fn fn;
    switch (ts) {
        case 8: fn = vq::lh_pick<8>(mt, exact); break;
        case 16: fn = vq::lh_pick<16>(mt, exact); break;
        case 32: fn = vq::lh_pick<32>(mt, exact); break;
        default: fn = vq::lh_pick<64>(mt, exact); break;
    }
    const int rows = 256 / ts;
    const unsigned grid = (unsigned)((N + rows - 1) / rows);
    const uint16_t* a0 = (const uint16_t*)w_bf16;
    const uint16_t* a1 = (const uint16_t*)x_bf16;
    uint16_t* a2 = (uint16_t*)y_bf16;
    void* args[] = {&a0, &a1, &a2, &M, &N, &K};
    (void)hipLaunchKernel((const void*)fn, dim3(grid), dim3(256), args, lds, (hipStream_t)stream);
    return vq::status_of(hipGetLastError());
}

extern "C" int viper_hip_sampling_greedy(const void* logits_bf16, int32_t* out_token, int B, int V,
                                         void* stream) {
    if (logits_bf16 == nullptr || out_token == nullptr || B <= 0 || V <= 0) return VIPER_INVALID_ARGUMENT;
    if (vq::misaligned(logits_bf16, 2) || vq::misaligned(out_token, 4)) return VIPER_INVALID_ARGUMENT;
    const uint16_t* a0 = (const uint16_t*)logits_bf16;
    void* args[] = {&a0, &out_token, &V};
    (void)hipLaunchKernel((const void*)vq::argmax_bf16_kernel, dim3((unsigned)B), dim3(vq::AM_NT), args, 0,
                          (hipStream_t)stream);
    return vq::status_of(hipGetLastError());
}

extern "C" size_t viper_hip_sampling_greedy_workspace_bytes(int B) {
    return B > 0 ? (size_t)B * 16 : 0;
}

extern "C" int viper_hip_sampling_greedy_split(const void* logits_bf16, int32_t* out_token, int B, int V,
                                               void* workspace, size_t workspace_bytes, void* stream) {
    if (logits_bf16 == nullptr || out_token == nullptr || workspace == nullptr || B <= 0 || V <= 0)
        return VIPER_INVALID_ARGUMENT;
    if (vq::misaligned(logits_bf16, 2) || vq::misaligned(out_token, 4) || vq::misaligned(workspace, 8) ||
        workspace_bytes < viper_hip_sampling_greedy_workspace_bytes(B))
        return VIPER_INVALID_ARGUMENT;
    // rows that are not whole 16-byte octets take the one-workgroup kernel
    if (vq::misaligned(logits_bf16, 16) || V % 8 != 0)
        return viper_hip_sampling_greedy(logits_bf16, out_token, B, V, stream);
    if (vq::greedy_wgs(B, V, 2) > (long)INT32_MAX) return VIPER_INVALID_ARGUMENT;
    const int pt = vq::greedy_octets(B, V);
    int P = (int)vq::greedy_wgs(1, V, pt);
    const void* fn = pt == 8 ? (const void*)vq::argmax_split_kernel<8> : (const void*)vq::argmax_split_kernel<2>;
    const uint16_t* a0 = (const uint16_t*)logits_bf16;
    uint64_t* keys = (uint64_t*)workspace;
    unsigned* cnt = (unsigned*)(keys + B);
    void* args[] = {&a0, &out_token, &V, &P, &keys, &cnt};
    (void)hipLaunchKernel(fn, dim3((unsigned)(P * B)), dim3(vq::GR_NT), args, 0, (hipStream_t)stream);
    return vq::status_of(hipGetLastError());
}
