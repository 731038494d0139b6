// How a prefill call of T tokens is cut up, and the workspace that takes.  Plain C++ without
// HIP: the host code, the kernels' launchers and the CPU tests read the same rules.
#pragma once
#include <stddef.h>

#include <initializer_list>

#include "qe_format.h"

// The router's K splits at T tokens (subtrees of 64 / nz chunks, whose partials
// k_topk merges): enough workgroups of 64 tokens x 128 experts to fill the GPU, and
// no more, since every split writes T x 256 partials (8192 tokens: 4 splits 96 + 13 us
// with k_topk, 8 splits 102 + 18; 1999: 8 splits 32 + 7, 16 splits 39 + 9; 512 in the
// fused launch: 16 splits 21.3, 32 splits 25).
// From QE_RS_SPLIT_T tokens the router and the shared gate/up tiles run as two
// launches of larger tiles (1024 tokens: 43 us fused, 47 apart; 1999: 88 against 67).
#define QE_RS_SPLIT_T 1280
static inline int qe_router_splits(int T) { return T < 256 ? 32 : T < QE_RS_SPLIT_T ? 16 : T < 4096 ? 8 : 4; }
// token rows of partials that calls of up to t_max tokens write: the largest call, or the
// last before a line at which the splits fall
static inline size_t qe_rpart_rows(size_t t_max) {
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
// to fall with T: 300 tokens over about 110 experts 10 % slower, 400 over about 85 11 %.
// (Up to 16 tokens no expert has more than 16 pairs and the items are the same either way.)
#define QE_ITEM32_T 224
#define QE_ITEM32_E 112
static inline int qe_item32_experts(int T) { return T > 16 && T < QE_ITEM32_T ? QE_ITEM32_E : 0; }

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
// the same over all calls of up to t_max tokens, whose largest need not be the last
static inline int qe_max_items_upto(int t_max) {
    const int n = qe_max_items(t_max), m = t_max >= QE_ITEM32_T ? qe_max_items(QE_ITEM32_T - 1) : 0;
    return n > m ? n : m;
}
