// The launches of one decode step, enqueued in one call (kx_internal.h).  Host code only.
#include <algorithm>

#include "kx_attn_merge.h"
#include "kx_gemv_fused.h"
#include "kx_hip.h"
#include "kx_internal.h"
#include "kx_tile_order.h"

namespace {

constexpr int kHeadDim = 128;

// Enqueues the launches and stops at the first that is refused.
struct Enqueue {
    int rc = KX_OK;
    template <class F>
    void operator()(F&& launch) {
        if (rc == KX_OK) rc = launch();
    }
};

}  // namespace

static_assert(sizeof(kx_step_layer) == 19 * 8, "nineteen eight-byte words");

extern "C" size_t kx_step_desc_bytes(void) {
    return sizeof(kx_step_desc);
}

extern "C" size_t kx_step_layer_bytes(void) {
    return sizeof(kx_step_layer);
}

// Every workgroup of the o projection repeats the merge of its two heads, so merging there, a launch less, pays while the
// projection has one round of workgroups (hidden 4096 and 32 heads: 256 of them, 1.1 to 2.3 us per layer faster; 5120 and 64: 640, 0.7 to
// 2.7 us slower than the separate merge kernel) and, up to two, while the heads have few chunks.  us per layer, in the projection /
// separate, at 1000, 3000 and 5000 positions: 320 workgroups of 40 heads 34.1 / 35.0, 36.8 / 36.7, 39.5 / 38.4, 400 38.6 / 38.8, 40.4 /
// 40.7, 43.2 / 42.4, 384 of 64 34.3 / 34.8, 37.4 / 36.2, 40.7 / 38.2.
extern "C" int kx_step_merges_in_o(int32_t hidden, int32_t n_q, int32_t max_positions) {
    if (max_positions < 1 || kx::attn_chunks_of(max_positions) > kx::kMergeParts * kx::kMergeHold) return -1;
    const int64_t columns = (hidden + kx::kTileCols - 1) / kx::kTileCols;
    const int64_t workgroups = columns * std::max(1, n_q * kHeadDim / 256);  // 256 rows of K each
    const int64_t chunks = static_cast<int64_t>(n_q) * kx::attn_chunks_of(max_positions);
    return workgroups <= 256 || (workgroups <= 512 && chunks <= 1920) ? 1 : 0;
}

extern "C" int kx_decode_step_bf16(const kx_step_desc* d, const kx_step_layer* layers, void* stream) {
    if (!d || (!layers && d->layers > 0)) return KX_ERR_NULL_POINTER;
    Enqueue run;
    const auto chain = [&](const kx_chain_desc& link, const kx_step_matrix& w, int K, int N) {
        run([&] {
            return kx_gemv_awq_chain_bf16(&link, w.qweight, w.scales, w.qzeros, K, N, d->group, d->gemv_workspace,
                                          d->gemv_workspace_bytes, stream);
        });
    };
    const auto normed_row = [&](const uint16_t* gain) {
        kx_chain_desc link{};
        link.in_kind = KX_IN_NORM;
        link.norm_row = d->x;
        link.norm_sumsq = d->sumsq;
        link.norm_parts = d->norm_parts;
        link.norm_gain = gain;
        link.norm_eps = d->eps;
        return link;
    };
    const auto into_residual = [&] {
        kx_chain_desc link{};
        link.out_kind = KX_OUT_RESIDUAL;
        link.residual_in = d->x;
        link.residual_out = d->x;
        link.sumsq_out = d->sumsq;
        return link;
    };
    const int H = d->hidden, I = d->intermediate;
    const int qkv_out = (d->n_q + 2 * d->n_kv) * kHeadDim;
    run([&] { return kx_embedding_bf16(d->embed, d->token, d->x, d->embed_rows, H, stream); });
    for (int li = 0; li < d->layers && run.rc == KX_OK; li++) {
        const kx_step_layer& L = layers[li];
        if (li == 0) {  // the embedding row comes without its sums of squares
            run([&] {
                return kx_gemv_awq_qkv_rope_bf16(d->x, nullptr, L.in_norm, d->eps, nullptr, L.qkv.qweight, L.qkv.scales,
                                                 L.qkv.qzeros, L.q_norm, L.k_norm, d->q, L.k_cache, L.v_cache, d->n_q,
                                                 d->n_kv, kHeadDim, d->pos, static_cast<int32_t>(L.cache_positions),
                                                 d->rope_theta, d->eps, H, d->group, d->gemv_workspace,
                                                 d->gemv_workspace_bytes, stream);
            });
        } else {
            kx_chain_desc link = normed_row(L.in_norm);
            link.out_kind = KX_OUT_QKV_ROPE;
            link.q_out = d->q;
            link.pos = d->pos;
            link.rope_n_q_heads = d->n_q;
            link.rope_n_kv_heads = d->n_kv;
            link.rope_theta = d->rope_theta;
            link.qk_eps = d->eps;
            link.q_gain = L.q_norm;
            link.k_gain = L.k_norm;
            link.k_cache = L.k_cache;
            link.v_cache = L.v_cache;
            link.cache_positions = static_cast<int32_t>(L.cache_positions);
            chain(link, L.qkv, H, qkv_out);
        }
        kx_chain_desc o = into_residual();
        if (d->merge_in_o) {
            run([&] {
                return kx_attn_decode_partial_bf16(d->q, L.k_cache, L.v_cache, d->n_q, d->n_kv, kHeadDim, d->pos,
                                                   d->max_positions, d->attn_workspace, d->attn_workspace_bytes, stream);
            });
            o.in_kind = KX_IN_ATTN;
            o.attn_workspace = d->attn_workspace;
            o.attn_workspace_bytes = d->attn_workspace_bytes;
            o.n_q_heads = d->n_q;
            o.n_kv_heads = d->n_kv;
            o.max_positions = d->max_positions;
        } else {
            run([&] {
                return kx_attn_decode_bf16(d->q, L.k_cache, L.v_cache, d->attn, d->n_q, d->n_kv, kHeadDim, d->pos,
                                           d->max_positions, d->attn_workspace, d->attn_workspace_bytes, stream);
            });
            o.in_kind = KX_IN_ROW;
            o.x = d->attn;
        }
        chain(o, L.o, d->n_q * kHeadDim, H);
        kx_chain_desc mlp = normed_row(L.post_norm);
        mlp.out_kind = KX_OUT_ROW;
        mlp.y = d->gate_up;
        chain(mlp, L.gate_up, H, 2 * I);
        kx_chain_desc down = into_residual();
        down.in_kind = KX_IN_SWIGLU;
        down.gate = d->gate_up;
        down.up = d->gate_up + I;
        chain(down, L.down, I, H);
    }
    run([&] { return kx_rmsnorm_bf16(d->x, d->final_norm, d->h, 1, H, d->eps, stream); });
    if (d->lm_head) {
        run([&] { return kx_gemv_bf16(d->h, d->lm_head, d->logits, 1, H, d->head_rows, nullptr, 0, stream); });
        run([&] { return kx_argmax_bf16(d->logits, d->logits_n, d->next_token, stream); });
    }
    return run.rc;
}
