// IQ4_NL conversion of routed-expert weights on the GPU.
//
// The reference converts on the CPU (engine/qconv.cpp:202-227, convert_experts):
// each source row is widened to fp32 (dequant_rows, :17-43) and quantized by
// ggml's IQ4_NL quantizer (quant_row, :91-98: ggml_quantize_chunk with no
// importance matrix), and the fp16 scale and 16 code bytes of every 32-element
// block go to the row's scale and code areas.  ggml's algorithm per block
// (quantize_row_iq4_nl_impl, one 32-block per super-block, ntry = 7):
//   m = the first element of largest |x|; |m| < 1e-15 -> scale 0;
//   a candidate inverse scale s assigns q_j = nearest codebook entry of s*x_j
//   and is scored by S_xq = sum (x_j^2 q_j) x_j, S_qq = sum (x_j^2 q_j) q_j in
//   element order; s0 = 1/(m/127) gives d = S_xq/S_qq, best = d*S_xq; then
//   s = (t-127)/m, t = -7..7, replaces them when S_qq > 0 and
//   S_xq^2 > best*S_qq; the scale is stored as fp16 and the codes are the
//   nearest entries of (1/d)*x_j with the fp32 d.
//
// Here one thread quantizes one block, and the bytes are identical to the CPU
// checker's (the library builds with -ffp-contract=off and correctly rounded
// division).  Scoring all sixteen candidates with that sequence is 16 x 32 table reads
// and about 5,000 VALU instructions per block; instead:
//   * Over the fifteen scales s = -n/m, n = 120..134, an element's nearest entry changes
//     at most once: neighbouring midpoints are more than a factor 134/120 apart (the
//     closest, 115.5 and 93.5, a factor 1.235).  So two reads, at n = 120 and n = 134,
//     give both entries; their sum, twice the midpoint between them, gives the n where
//     the change happens, and one exact evaluation at the nearest integer decides
//     between it and the next (every other n is further from the midpoint than rounding
//     reaches).  Each change is added to the bin of its n; prefix sums over the bins give
//     S_xq and S_qq of every candidate.  All their terms have one sign (bar an opposite
//     entry 1, below 1e-4 of the sum), so the relative errors are at most the roundings
//     on a term's way, of 2^-24 each: 3 + 31 in the sequence, 2 + 8 + 2 + 14 here, and up
//     to 31 more on what met in one bin (at most 0.21 of S_xq and 0.36 of S_qq).
//   * A candidate whose approximate score S_xq^2 / S_qq is below the largest by more than
//     3e-5 (2 x 102 roundings of the sequence's score, 2 x 102 of this one: 2.4e-5, and the
//     last operations) cannot be the last to win; what is left -- mostly one candidate --
//     is evaluated with the fp32 operations of the sequence, in its order, starting from
//     s0's exact score.  The first is evaluated by the block's own lane, the others -- about
//     one block in three has any -- by the wave's lanes in turn.  Candidates with no change between them assign alike and
//     score alike, and only the first is evaluated.  (No change is lost in S_xq's sum: the
//     smallest adds 11 (4.5/134)^3 |m|^3 = 4.2e-4 |m|^3, and half an ulp of the largest sum,
//     32 x 127 |m|^3, is at most 2.5e-4 |m|^3.  A test of the bin alone spills registers.)
//   * Blocks whose largest element lies outside [1e-6, 1e4], where the products could
//     underflow or overflow, or that hold a NaN, take the sequence over all sixteen.  Where
//     three lanes of a wave in four have such a block, each evaluates its own.
//
// nearest(a): ggml bisects the codebook and keeps the lower of the two
// bracketing entries when a - lo < hi - a.  Both differences are exact
// wherever the comparison is close (every midpoint lies at |a| >= 4.5 and the
// entries are integers), so that test is a < (lo + hi)/2.  The brackets have
// integer ends and the midpoints are multiples of 1/2, so nearest(a) is
// constant on every half-unit slot [k/2, (k+1)/2): one LDS table of the slot
// values answers it.  The slot comes from 8a, whose floor rounded down to a
// multiple of 4 is the byte offset 4 floor(2a) of a 4-byte entry; 8a is exact
// (a power-of-two scaling), so it is 8 times the a that ggml rounds.
//
// In the candidate loop |a| <= |s m| <= 134.02 (|x_j| <= |m|, |s| <= 134/|m|)
// or a is NaN (a NaN or infinite input; v_cvt_flr_i32_f32 gives 0), so the
// table spans a in [-135.5, 135.5) and needs no clamp there.  The final pass
// uses s = 1/d, which has no such bound, and clamps.
#include "../../include/qe_moe.h"
#include "qe_kernels.h"

namespace {

constexpr int NL4_HALF = 271;          // slots k = -271 .. 270
constexpr int NL4_SLOTS = 2 * NL4_HALF; // 542 entries

__device__ inline int kv_at(int i) {
    const uint32_t w = i < 4 ? QE_NL4_W0 : i < 8 ? QE_NL4_W1 : i < 12 ? QE_NL4_W2 : QE_NL4_W3;
    return (int)(int8_t)(w >> (8 * (i & 3)));
}

// slot k holds a in [k/2, (k+1)/2): value and index of the nearest entry
__device__ inline void build_table(float *tab_q, int *tab_c) {
    for (int t = threadIdx.x; t < NL4_SLOTS; t += blockDim.x) {
        const int k = t - NL4_HALF;
        const int fl = k >> 1; // floor(a)
        int lo = 0;
        for (int i = 1; i < 16; ++i)
            if (kv_at(i) <= fl) lo = i;
        // a < (v_lo + v_hi)/2  <=>  k + 1/2 < v_lo + v_hi  <=>  k < v_lo + v_hi
        const int c = lo < 15 && k >= kv_at(lo) + kv_at(lo + 1) ? lo + 1 : lo;
        tab_q[t] = (float)kv_at(c);
        tab_c[t] = c;
    }
}

// byte offset of the slot of a, from a8 = 8a: 4 floor(2a) = floor(a8) & ~3
__device__ inline int slot_bytes(float a8) {
    int k;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(k) : "v"(a8));
    return k & ~3;
}

template <typename T> __device__ inline T tab_at(const T *tab0, int bytes) {
    return *(const T *)((const char *)tab0 + bytes);
}

// S_xq and S_qq of inverse scale s (given as s8 = 8 s), in element order
__device__ inline void nl4_fit(const float (&x)[32], float s8, const float *tab0, float &sxq, float &sqq) {
    float a = 0.f, b = 0.f;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        const float q = tab_at(tab0, slot_bytes(s8 * x[j]));
        const float wq = (x[j] * x[j]) * q;
        a = a + wq * x[j];
        b = b + wq * q;
    }
    sxq = a;
    sqq = b;
}

template <int TYPE>
__device__ inline void load_block(const uint8_t *src, uint32_t g, float (&x)[32]) {
    if constexpr (TYPE == QE_SRC_F32) {
        const float4 *p = (const float4 *)(src + (size_t)g * 128);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float4 v = p[i];
            x[4 * i] = v.x; x[4 * i + 1] = v.y; x[4 * i + 2] = v.z; x[4 * i + 3] = v.w;
        }
    } else if constexpr (TYPE == QE_SRC_F16 || TYPE == QE_SRC_BF16) {
        const uint4 *p = (const uint4 *)(src + (size_t)g * 64);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint4 v = p[i];
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if constexpr (TYPE == QE_SRC_F16) {
                    x[8 * i + 2 * k] = qe_f16_to_f32((uint16_t)w[k]);
                    x[8 * i + 2 * k + 1] = qe_f16_to_f32((uint16_t)(w[k] >> 16));
                } else {
                    x[8 * i + 2 * k] = __uint_as_float(w[k] << 16);
                    x[8 * i + 2 * k + 1] = __uint_as_float(w[k] & 0xffff0000u);
                }
            }
        }
    } else { // Q8_0: fp16 d, then 32 int8; blocks are 34 bytes, so 2-byte aligned
        const uint16_t *p = (const uint16_t *)(src + (size_t)g * 34);
        const float d = qe_f16_to_f32(p[0]);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const uint16_t v = p[1 + i];
            x[2 * i] = d * (float)(int8_t)(v & 0xff);
            x[2 * i + 1] = d * (float)(int8_t)(v >> 8);
        }
    }
}

// 8 n / -m for n = 120..134, correctly rounded, from mn = -m / 8 and rn = 1 / mn: the
// quotient estimate and one remainder step (equal to the division for all 2^23
// mantissas of m and every n, checked exhaustively; no exponent in use here over- or
// underflows).
__device__ inline float scale8(float n, float mn, float rn) {
    const float q = n * rn;
    return fmaf(fmaf(-q, mn, n), rn, q);
}

// WPS: waves per SIMD the registers are cut for (qe_launch_nl4_quant).  At four, F16
// spills 6 VGPRs and BF16 one (16 and 8 bytes of scratch a lane); F32 and Q8_0 none.
// What bounds it: VALU issue (3,090 instructions a wave of 64 blocks, of half rate where
// they convert, clamp or mask) and the slot reads' bank conflicts (36 % of the cycles).
// One Q8_0 layer (25 M blocks): 2,455 us scoring all candidates, 1,590 now; 32,768 bf16
// blocks 14.8 -> 11.7 us.  Measured on the way: the bins by LDS float atomics 9,020 us;
// every lane evaluating its own remaining candidates 1,750 (four rounds a wave instead of
// about 1.4).
template <int TYPE, int WPS>
__global__ __launch_bounds__(256, WPS) void k_nl4_quant(QeNl4Args a) {
    constexpr int N0 = 120, NC = 15; // candidates s = -n/m, n = N0 .. N0 + NC - 1 (t = 127 - n)
    __shared__ float s_q[NL4_SLOTS];
    __shared__ int s_c[NL4_SLOTS];
    __shared__ float2 s_bin[NC - 1][256]; // [n - N0 - 1][thread]: what S_xq, S_qq change by from n - 1 to n
    build_table(s_q, s_c);
    __syncthreads();
    const uint32_t g = blockIdx.x * 256u + threadIdx.x;
    const bool live = g < a.nblk; // lanes past the end stay for the wave's exchange
    float x[32];
    if (live) {
        load_block<TYPE>(a.src, g, x);
    } else {
#pragma unroll
        for (int j = 0; j < 32; ++j) x[j] = 0.f;
    }
    const float *q0 = s_q + NL4_HALF;

    float amax = 0.f, m = 0.f;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        if (fabsf(x[j]) > amax) { amax = fabsf(x[j]); m = x[j]; }
    }
    float d = 0.f, best_rest = 0.f;
    uint32_t rest = 0u; // candidates left
    if (amax >= 1e-15f) {
        float sxq, sqq;
        nl4_fit(x, 8.f * (1.f / (m / 127.f)), q0, sxq, sqq);
        d = sxq / sqq;
        float best = d * sxq;
        uint32_t cand = (1u << NC) - 1u; // candidates to evaluate, bit n - N0
        const float mn = -0.125f * m, rn = 1.f / mn;
        if (amax >= 1e-6f && amax <= 1e4f) {
            float2 *bin = &s_bin[0][threadIdx.x]; // this thread's column
#pragma unroll
            for (int i = 0; i < NC - 1; ++i) bin[256 * i] = make_float2(0.f, 0.f);
            const float slo = scale8((float)N0, mn, rn), shi = scale8((float)(N0 + NC - 1), mn, rn), hm = 4.f * mn;
            float A4[4] = {0.f, 0.f, 0.f, 0.f}, B4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                const float ql = tab_at(q0, slot_bytes(slo * x[j])), qh = tab_at(q0, slot_bytes(shi * x[j]));
                const float sum = ql + qh, dq = qh - ql;
                const float w = x[j] * x[j], p = w * x[j];
                A4[j & 3] = fmaf(p, ql, A4[j & 3]);
                B4[j & 3] = fmaf(w * ql, ql, B4[j & 3]);
                // the change lies at n = (ql + qh) / 2 * -m / x; without one (or x = 0) the
                // result is any bin and nothing is added
                const float n0 = rintf(fminf(fmaxf(sum * hm * __builtin_amdgcn_rcpf(x[j]), (float)N0), (float)(N0 + NC - 1)));
                const bool outer = (scale8(n0, mn, rn) * x[j] >= 4.f * sum) == (dq > 0.f); // at n0 already qh
                const int i = min((int)n0 - N0 - 1 + (outer ? 0 : 1), NC - 2);
                float2 *bj = bin + 256 * max(i, 0);
                const float2 v = *bj;
                *bj = make_float2(fmaf(p, dq, v.x), fmaf(w * dq, sum, v.y));
            }
            float A = (A4[0] + A4[1]) + (A4[2] + A4[3]), B = (B4[0] + B4[1]) + (B4[2] + B4[3]);
            float sc[NC], top = sxq * sxq * __builtin_amdgcn_rcpf(sqq);
            uint32_t same = 0u; // bit n - N0: n assigns as n + 1 does
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                if (i > 0) {
                    const float2 v = bin[256 * (i - 1)];
                    if (A + v.x == A) same |= 1u << (i - 1);
                    A += v.x;
                    B += v.y;
                }
                sc[i] = A * A * __builtin_amdgcn_rcpf(B);
                top = fmaxf(top, sc[i]);
            }
            if (A == A) { // no NaN in the block
                const float thr = top * (1.f - 3e-5f);
                cand = 0u;
#pragma unroll
                for (int i = 0; i < NC; ++i)
                    if (sc[i] >= thr) cand |= 1u << i;
                cand &= ~same;
            }
        }
        rest = cand;
        best_rest = best;
    }
    // In the sequence's order, n from 134 down (the general division: this also serves
    // blocks outside scale8's range).  Each lane evaluates its block's first; while three
    // lanes in four have more -- blocks that keep all fifteen, mostly -- also the next: a
    // round of the list below costs about 4/3 of one here (blocks of 1e-7: 15.4 us for
    // 4,096 scoring all candidates in turn, 20.1 with the list alone, 16.1 so; 4 M blocks 431,
    // 507, 430).
    unsigned long long more; // lanes with candidates left
    do {
        if (rest) {
            const int i = 31 - __builtin_clz(rest);
            rest &= ~(1u << i);
            float sxq, sqq;
            nl4_fit(x, 8.f * ((float)(-N0 - i) / m), q0, sxq, sqq);
            if (sqq > 0.f && sxq * sxq > best_rest * sqq) {
                d = sxq / sqq;
                best_rest = d * sxq;
            }
        }
        more = __ballot(rest != 0);
    } while (__popcll(more) >= 48);
    if (more) {
        // The wave's list of (lane, candidate), in its lanes' bins (64 columns of 14
        // slots, read out by now): an entry is evaluated by lane k % 64, from the block in
        // memory, and replaced by its sums, which the owner takes in order.
        const int lane = threadIdx.x & 63, cnt = __popc(rest);
        int off = cnt;
#pragma unroll
        for (int s = 1; s < 64; s <<= 1) {
            const int v = __shfl_up(off, s);
            if (lane >= s) off += v;
        }
        const int total = __builtin_amdgcn_readlane(off, 63);
        off -= cnt;
        float2 *wbin = &s_bin[0][threadIdx.x & ~63]; // slot k: row k / 64, column k % 64 of the wave
        auto slot = [&](int k) -> float2 & { return wbin[256 * (k >> 6) + (k & 63)]; };
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        uint32_t left = rest;
        for (int k = off; left; ++k) {
            const int i = 31 - __builtin_clz(left);
            left &= ~(1u << i);
            slot(k) = make_float2(__int_as_float(lane), __int_as_float(i));
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int k0 = 0; k0 < total; k0 += 64) {
            const int k = k0 + lane;
            const float2 e = k < total ? slot(k) : make_float2(__int_as_float(lane), 0.f);
            const int o = __float_as_int(e.x) & 63;
            const float mo = __shfl(m, o);
            if (k < total) {
                float y[32], sxq, sqq;
                load_block<TYPE>(a.src, g - lane + o, y);
                nl4_fit(y, 8.f * ((float)(-N0 - __float_as_int(e.y)) / mo), q0, sxq, sqq);
                slot(k) = make_float2(sxq, sqq);
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        for (int k = off; k < off + cnt; ++k) {
            const float2 v = slot(k);
            if (v.y > 0.f && v.x * v.x > best_rest * v.y) {
                d = v.x / v.y;
                best_rest = d * v.x;
            }
        }
    }
    if (!live) return;
    const float s8 = 8.f * (d != 0.f ? 1.f / d : 0.f);
    const int *c0 = s_c + NL4_HALF;
    uint32_t c[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        const float a8 = fminf(fmaxf(s8 * x[j], -1080.f), 1079.f); // NaN -> -1080
        const uint32_t code = (uint32_t)tab_at(c0, slot_bytes(a8));
        c[(j & 15) >> 2] |= code << (8 * (j & 3) + (j >> 4) * 4);
    }
    const uint32_t row = g / a.nb, b = g - row * a.nb;
    const uint32_t grp = row / a.rows_per_group, r = row - grp * a.rows_per_group;
    uint8_t *dst = a.dst + (size_t)grp * a.group_stride + (size_t)r * a.row_stride;
    *(uint4 *)(dst + 16 * b) = make_uint4(c[0], c[1], c[2], c[3]);
    *(uint16_t *)(dst + 16 * a.nb + 2 * b) = qe_f32_to_f16(d);
}

} // namespace

hipError_t qe_launch_nl4_quant(const QeNl4Args &a, int src_type, hipStream_t st) {
    if (a.nblk == 0) return hipSuccess;
    const dim3 grid((a.nblk + 255) / 256), block(256);
    // up to three workgroups per CU: all run at once, and what counts is one wave's own
    // pace, which more registers help (32,768 blocks 13.0 -> 11.5 us); beyond, the fourth
    // wave per SIMD does (25 M blocks 1,727 -> 1,590)
    const auto go = [&](auto small, auto large) {
        if (grid.x <= 3 * 256) small<<<grid, block, 0, st>>>(a);
        else large<<<grid, block, 0, st>>>(a);
    };
    switch (src_type) {
    case QE_SRC_F32: go(k_nl4_quant<QE_SRC_F32, 3>, k_nl4_quant<QE_SRC_F32, 4>); break;
    case QE_SRC_F16: go(k_nl4_quant<QE_SRC_F16, 3>, k_nl4_quant<QE_SRC_F16, 4>); break;
    case QE_SRC_BF16: go(k_nl4_quant<QE_SRC_BF16, 3>, k_nl4_quant<QE_SRC_BF16, 4>); break;
    case QE_SRC_Q8_0: go(k_nl4_quant<QE_SRC_Q8_0, 3>, k_nl4_quant<QE_SRC_Q8_0, 4>); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}
