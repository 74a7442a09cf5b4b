/*
 * Entry points of libkx_hip.so that are not part of the drop-in boundary (include/kx_hip.h): what the
 * tests and the benchmark need to put one particular kernel under a shape, and the decode step of the Python
 * driver in one call.  No state is kept: everything travels with the call.
 */
#ifndef KX_INTERNAL_H
#define KX_INTERNAL_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define KX_POLICY_BY_SHAPE 0   /* what kx_gemv_awq_bf16 does: one row on the vector kernel with the fixed-point exchange
                                  wherever that applies, several rows on the MFMA kernel */
#define KX_POLICY_VECTOR 1     /* the vector-ALU kernel with the ordered fp32 exchange (any accepted shape): the sums of
                                  the launches with a prologue or an epilogue, bit for bit */
#define KX_POLICY_MFMA 2       /* the one-shot MFMA kernel where N allows, else the vector kernel */
#define KX_POLICY_MFMA_NO_WAIT 3  /* the same, and workgroups that finish a column tile together give up waiting at once:
                                  the path a workgroup takes whose neighbours cannot start while it waits */

/* kx_gemv_awq_bf16 with the kernel chosen by the caller. */
int kx_gemv_awq_bf16_policy(const uint16_t* x, const int32_t* qweight, const uint16_t* scales,
                            const int32_t* qzeros, uint16_t* y, int32_t M, int32_t K, int32_t N,
                            int32_t group_size, void* workspace, size_t workspace_bytes, void* stream,
                            int32_t policy);

/* One decode step of one sequence (mykuiperllama_amd.decode, the chained form): the same calls of include/kx_hip.h in the
 * same order as the Python driver would make, from native code.  Through ctypes a call costs the host 9 us, more than
 * most of the launches take on the GPU: a step of 28 layers of 1024 hidden that is not captured in a graph took 1380 us,
 * and takes 800 this way.  Stops at the first call that is refused and returns its code; the pointers are read during
 * the call only.  A layer is nineteen eight-byte words. */
typedef struct kx_step_matrix {
    const int32_t* qweight;
    const uint16_t* scales;
    const int32_t* qzeros;
} kx_step_matrix;

typedef struct kx_step_layer {
    kx_step_matrix qkv, o, gate_up, down;
    const uint16_t *in_norm, *post_norm, *q_norm, *k_norm;
    uint16_t *k_cache, *v_cache;
    int64_t cache_positions;
} kx_step_layer;

typedef struct kx_step_desc {
    const uint16_t* embed;
    const int32_t* token;
    const int32_t* pos;
    const uint16_t* final_norm;
    const uint16_t* lm_head; /* null: the step ends with the normalised row */
    uint16_t *x, *h, *q, *attn, *gate_up, *logits;
    float* sumsq;
    int32_t* next_token;
    void* gemv_workspace;
    size_t gemv_workspace_bytes;
    void* attn_workspace;
    size_t attn_workspace_bytes;
    int32_t layers, hidden, intermediate, n_q, n_kv, group, max_positions, norm_parts, merge_in_o;
    int32_t embed_rows, head_rows, logits_n;
    float rope_theta, eps;
} kx_step_desc;

int kx_decode_step_bf16(const kx_step_desc* desc, const kx_step_layer* layers, void* stream);

/* Where a step of one sequence merges the chunks of the attention: 1 on the way into the o projection, 0 in a launch of its own,
 * which is then the faster, -1 in a launch of its own because the cache has more chunks than the projection merges. */
int kx_step_merges_in_o(int32_t hidden, int32_t n_q_heads, int32_t max_positions);

/* Column tile and K tile of workgroup `id` of a grid whose neighbouring column tiles share memory lines (csrc/kx_tile_order.h):
 * 1, or 0 where such a grid is too small or too large for it and a workgroup takes the tile of its own number. */
int kx_shared_line_tile(int32_t coltiles, int32_t ktiles, int32_t id, int32_t* ct, int32_t* kt);

/* Whether a matrix-core launch whose column tiles share memory lines has its workgroups take the tiles of their own numbers all the
 * same: rows, 32-row steps per wave, output columns, the grid, and whether its workgroups finish a column tile together. */
int kx_tiles_by_number(int32_t M, int32_t steps, int32_t N, int32_t coltiles, int32_t ktiles, int32_t together);

/* The form of csrc/kx_bf16_gemv.hip's kernel for two to sixteen rows and K <= 8192 that a launch takes, by whether every row of W
 * starts on a memory line: waves, elements of K per unit, units of a wave, waves that split K, runs of four blocks (0 or 1).
 * Returns 1, or 0 for sizes that the kernel does not take (among them two rows where the kernel for one and two is faster). */
int kx_bf16_held_form(int32_t whole_lines, int32_t M, int32_t K, int32_t N, int32_t* form);

/* Bytes of a kx_step_desc and of a kx_step_layer as the library was compiled: a binding that mirrors them compares. */
size_t kx_step_desc_bytes(void);
size_t kx_step_layer_bytes(void);

#ifdef __cplusplus
}
#endif
#endif /* KX_INTERNAL_H */
