// Kernel argument blocks and host launchers of the MoE block (internal).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "qe_device.h"

#define QE_SMALL_T 8   /* calls of up to this many tokens take the persistent decode kernel */
// The router's K splits at T tokens (subtrees of 64 / nz chunks, whose partials
// k_topk merges): enough workgroups of 64 tokens x 128 experts to fill the GPU, and
// no more, since every split writes T x 256 partials (8192 tokens: 4 splits 96 + 13 us
// with k_topk, 8 splits 102 + 18; 1999: 8 splits 32 + 7, 16 splits 39 + 9; 512 in the
// fused launch: 16 splits 21.3, 32 splits 25).
// From QE_RS_SPLIT_T tokens the router and the shared gate/up tiles run as two
// launches of larger tiles (1024 tokens: 43 us fused, 47 apart; 1999: 88 against 67).
#define QE_RS_SPLIT_T 1280
static inline int qe_router_splits(int T) { return T < 256 ? 32 : T < QE_RS_SPLIT_T ? 16 : T < 4096 ? 8 : 4; }
static inline size_t qe_rpart_rows(size_t t_max) { // token rows of partials that calls of up to t_max tokens write
    size_t n = 0;
    for (size_t end : {(size_t)255, (size_t)QE_RS_SPLIT_T - 1, (size_t)4095, t_max}) {
        const size_t t = end < t_max ? end : t_max, rows = t * qe_router_splits((int)t);
        n = n > rows ? n : rows;
    }
    return n;
}
#define QE_MFMA_MC 64 /* pairs per work item of the prefill MFMA grouped GEMMs (up to four 16-row tiles) */

// Pairs per work item: QE_MFMA_MC, or 32 in a call of fewer than QE_ITEM32_T tokens
// whose pairs fall on at most QE_ITEM32_E experts (k_disp_scatter counts them).  Few
// experts leave the GPU partly empty, and then an expert's 33..64 pairs in one item make
// the longest workgroups; items of 32 halve them.  With more experts the GPU is full and
// the second decode of the weights costs more.  us per layer with items of 64 / 32:
// 100 tokens over 66 experts 95 / 83; 200 tokens over 50 experts 100 / 89, over 98 97 / 93,
// over 140 105 / 113; 223 tokens over 146 110 / 120.  In longer calls the line would have
// to fall with T: 300 tokens over 105 experts 4 % slower, 400 over 80 11 %.
#define QE_ITEM32_T 224
#define QE_ITEM32_E 112
static inline int qe_item32_experts(int T) { return T < QE_ITEM32_T ? QE_ITEM32_E : 0; }
// Gate/up of items of up to 32 pairs: activations straight to registers (gu_small) where
// more than qe_direct_experts(T) experts have pairs, staged through LDS elsewhere.  In
// small calls, and over nearly all experts, items hold a few pairs each and their weights'
// latency decides; with more pairs the four waves' separate reads of the activations cost
// more than the staging.  us per layer direct / staged: 100 tokens over 248 experts 141 /
// 147; 144 over 253 153 / 158, over 70 87 / 89; 180 over 132 106 / 95, over 94 96 / 89;
// 223 over 103 107 / 98; 1000 over 256 260 / 241.
#define QE_DIRECT_T 152  /* always direct below */
#define QE_DIRECT_T2 256 /* never from here on */
#define QE_DIRECT_E 224
static inline int qe_direct_experts(int T) { return T < QE_DIRECT_T ? 0 : T < QE_DIRECT_T2 ? QE_DIRECT_E : QE_N_EXPERT; }
// upper bound of the items of T tokens: those of more than half the pairs, and one
// smaller per expert
static inline int qe_max_items(int T) {
    return T * QE_K_USED / ((qe_item32_experts(T) ? 32 : QE_MFMA_MC) / 2 + 1) + 1 + QE_N_EXPERT;
}

// One layer's weights inside the context.
struct QeLayerPtrs {
    const uint8_t *arena;     // 256 expert blobs
    const float *router;      // [257][2048]
    const float *bias;        // [256] or nullptr
    const uint8_t *sh_gu;     // Q8 [1024][2048]
    const uint8_t *sh_dn;     // Q8 [2048][512]
    const float *post_norm;   // [2048]
};

// Optional per-kernel event timing (host side): when `on`, every launch of
// qe_launch_layer is bracketed by two events on its stream.
enum { QP_DECODE, QP_NORMQ, QP_ROUTER, QP_SHGU, QP_TOPK, QP_DISPATCH, QP_GU, QP_HQUANT, QP_DOWN_LARGE, QP_SHDN,
       QP_COMBINE, QP_N };
struct QeProf {
    bool on = false;
    int used = 0, cap = 0, dropped = 0;
    hipEvent_t *ev = nullptr; // 2*cap events
    int *kid = nullptr;       // kernel id per pair
};

// Event bracket of one launch when per-kernel timing is on.
struct ProfScope {
    QeProf *p;
    hipStream_t st;
    int slot = -1;
    ProfScope(QeProf *p_, int kid, hipStream_t s) : p(p_), st(s) {
        if (!p || !p->on) return;
        if (p->used >= p->cap) { p->dropped++; return; }
        slot = p->used++;
        p->kid[slot] = kid;
        (void)hipEventRecord(p->ev[2 * slot], st);
    }
    ~ProfScope() {
        if (slot >= 0) (void)hipEventRecord(p->ev[2 * slot + 1], st);
    }
};

// Scratch of a context, sized for t_max tokens.
struct QeScratch {
    float *xn; int8_t *xqp; float *xs;      // [T][2048] normed x, its int8 quantisation (operand layout), [T][64] scales
    _Float16 *xhl;                          // [T][2048] normed x as fp16 hi|lo halves (store_hilo16 layout)
    float *logits;                          // [T][257]
    float *shgu;                            // prefill: shared silu(g)*u as [T][512] fp16 hi|lo halves
    float *rpart;                           // [nz][T][256] router subtree partials (qe_router_splits)
    int32_t *ids; float *wts; float *shg;   // [T][8], [T][8], [T]
    int32_t *off; int32_t *pairs;           // [257], [T*8]
    int4 *items; int32_t *n_items;          // work items (expert, first pair, count); n_items[0] items, the first n_items[1] of more than 32 pairs; n_items[2]: small ones direct
    int8_t *hqp; float *hs;                 // [T*8][512] quantised h (operand layout), [T*8][16] scales
    float *sd;                              // [T][2048] shared-expert output
    float *yp;                              // [T*8][2048] weighted expert outputs
    int32_t *chunk_hist;                    // [T*8/1024][256]
    int32_t *item_done;                     // [max items] finished gate/up workgroups per item (fused launch)
    unsigned *err; unsigned err_val;        // a fused launch's wait that gave up stores err_val to *err
    int spin_cap;                           // reads such a wait may take
    int wait_extra;                         // test hook: gate/up workgroups a fused down wait expects beyond its item's
    int t_max;
    QeProf *prof;                           // host-side timing, may be nullptr
};

struct QeCombineArgs {
    int T;
    const float *yp; const float *sd; const float *shg; const float *x2;
    float *out;
    const float *nw; float *xn; // optional exit norm: xn = RMSNorm(out) * nw (nw == nullptr: none)
};

// Persistent decode kernel (qe_decode.hip): T <= QE_SMALL_T tokens through
// layers first_layer .. first_layer + n_layers - 1 in one cooperative launch.
struct QeDecodeArgs {
    const uint8_t *arena; const float *router; const float *bias; const uint8_t *bias_on;
    const uint8_t *sh_gu; const uint8_t *sh_dn; const float *post_norm;
    int first_layer, n_layers, T, norm, residual;
    const float *x_in; float *x_out;
    uint64_t *ex;        // exchange words {value, tag}, QE_DECODE_EX_WORDS of them (qe_decode.hip)
    // routing sink of the last layer (plain stores by workgroup 0)
    float *logits; int32_t *ids; float *wts; float *shg; int32_t *off; int32_t *pairs; float *sd_out; float *xn_out;
    unsigned *sync;      // QE_DECODE_SYNC_WORDS: [0] launch epoch, [32] exit counter
    unsigned *err;       // host-mapped: set to 1 + epoch when a poll of the launch timed out
    int spin_cap;        // reads an exchange poll makes before it gives up (QE_DECODE_SPIN_CAP)
    const float *exit_norm; float *exit_xn; // optional: exit_xn = RMSNorm(x_out) * exit_norm
};
hipError_t qe_launch_decode(const QeDecodeArgs &a, hipStream_t st);
#ifndef QE_DEC_REP
#define QE_DEC_REP 4 /* copies of every decode exchange buffer */
#endif
#define QE_DECODE_EX_WORDS \
    (QE_DEC_REP * (2 * QE_SMALL_T * QE_D + QE_SMALL_T * QE_ROUTER_ROWS + QE_SMALL_T * QE_FF_SH + QE_SMALL_T * 8 * 16 * 9 + \
                   8 * QE_FF_EXP + 2 * QE_SMALL_T * 256))
#define QE_DECODE_SYNC_WORDS 64 /* launch epoch, exit counter */
#define QE_DECODE_SPIN_CAP (1 << 22) /* poll reads (s_sleep 1 between) before an exchange wait gives up */
#define QE_DECODE_SPIN_CAP_LATE 16  /* the cap of a wave's polls after one of them gave up */

// Launchers (qe_kernels.hip).  xin: layer input; post_norm: nullptr = input is
// already normalised; x2: residual added to the output or nullptr.
// tokens of the largest call (the API's limit): the down epilogue's 32-bit store
// offsets rely on its pair count staying below 2^19
#define QE_LAYER_T_MAX 65536
hipError_t qe_launch_layer(const QeLayerPtrs &L, const QeScratch &S, const float *xin, bool norm, const float *x2,
                           float *out, int T, hipStream_t st, const float *exit_norm = nullptr,
                           float *exit_xn = nullptr);
hipError_t qe_launch_dispatch(const QeScratch &S, int T, hipStream_t st);
// The same dispatch with its scratch in a static device array (no allocation);
// off and pairs are the caller's device buffers.
#define QE_DISPATCH_NOALLOC_T_MAX 16384
hipError_t qe_launch_dispatch_noalloc(const int32_t *ids, int T, int32_t *off, int32_t *pairs, hipStream_t st);
// the current device's address of that array, looked up once per device
hipError_t qe_noalloc_prepare(uint8_t **base);
hipError_t qe_launch_expert_mfma(const QeLayerPtrs &L, const QeScratch &S, int T, hipStream_t st);
hipError_t qe_launch_router_shgu(const QeLayerPtrs &L, const QeScratch &S, int T, hipStream_t st);

// IQ4_NL conversion (qe_convert.hip): block g (of nblk, nb per row) of the
// source goes to row g / nb of the destination, rows grouped rows_per_group
// at a time (one expert's matrix) at group_stride, row_stride within a group.
struct QeNl4Args {
    const uint8_t *src; uint8_t *dst;
    uint32_t nblk, nb, rows_per_group;
    size_t group_stride, row_stride;
};
hipError_t qe_launch_nl4_quant(const QeNl4Args &a, int src_type, hipStream_t st);

hipError_t qe_launch_synth_layer(uint8_t *arena_l, float *router_l, uint8_t *sh_gu_l, uint8_t *sh_dn_l,
                                 float *post_norm_l, uint64_t seed, int layer, hipStream_t st);
hipError_t qe_launch_synth_x(float *out, uint64_t seed, int inst, int64_t n, hipStream_t st);
