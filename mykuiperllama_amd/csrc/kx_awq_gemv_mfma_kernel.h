// Fused INT4 AWQ dequantise + GEMV on the matrix cores (gfx950, v_mfma_f32_16x16x32_bf16), M <= 16.
//
//   y[m,n] = sum_k x[m,k] * (q[k,n] - z[k/G,n]) * s[k/G,n]
//
// One MFMA multiplies A = activations (16 rows m x 32 k) by B = weights (32 k x 16 columns n) into a
// 16 x 16 fp32 tile.  Lane l of the wave supplies, for both operands, the eight k values
// 8*(l/16) .. 8*(l/16)+7 of row / column l%16, and receives D[4*(l/16)+v][l%16], v = 0..3.
//
// A lane (c = l%16, b = l/16) loads the two packed words (c-th pair of the tile's 32 word columns)
// of the eight rows 8b .. 8b+7 of a 32-row step: sixteen columns x eight rows of codes.  Nibble p of
// word h of those eight rows is exactly the B operand of column 8*(2c+h) + ORDER[p], so sixteen
// MFMAs per step - one per (h, p) - cover the lane's sixteen columns, all with the same A operand,
// which is a plain 16-byte load of x.  A code becomes a bf16 by OR-ing it into the mantissa of
// 128.0 (0x4300 | q = 128 + q, exact), two rows per register; the +128 joins the zero point:
//
//   sum_k x*(q - z) = sum_k x*(128 + q)  -  (128 + z) * sum_k x
//
// and sum_k x comes out of one more MFMA against a B operand of ones, in the same register layout.
// Raw sums of the waves of a workgroup meet in LDS; the thread that owns a column applies zero point and scale once per
// wave, whose steps lie in one quantisation group (groups are multiples of 32, and the host picks KS so that KS*32 divides
// the group), and takes part in the split-K exchange.  With FINE the steps of a wave lie in groups of their own: zero point
// and scale are applied per step in registers, and what meets in LDS are scaled sums.
// The offset that cancels is 128 where the vector kernel has 16, which shows in the last bits of the fp32 sum: its error against
// float64 is 1.3 to 4 times as large, and up to 1 in 1000 bf16 outputs is not the correctly rounded sum where on the vector
// kernel next to none are (groups of 32, K 9216 and 12288).  The rounding itself is the larger part by far: the bf16 outputs
// of both are 1.63e-3 to 1.70e-3 off, equal to six digits (K 512 to 25600, x of mean 0 and 1).
//
// Cost per weight: one VALU operation to build the operand (two byte permutes, three shifts and
// eight and/or pairs per sixteen weights) and 1/512 of an MFMA, whatever M is.
//
// The activations may be produced on the way in (PRO: SwiGLU of two tensors, or an RMSNorm whose sum of
// squares arrives per 256 columns) and the result may be added to a residual stream on the way out (EPI),
// with the arithmetic and rounding points of the stand-alone kernels.  A produced activation is staged
// in LDS as bf16, the workgroup's K range of every row, and the A operand is read from there.
#ifndef KX_AWQ_GEMV_MFMA_KERNEL_H
#define KX_AWQ_GEMV_MFMA_KERNEL_H

#include "kx_common.h"
#include "kx_gemv_fused.h"
#include "kx_rope.h"
#include "kx_splitk_exchange.h"

namespace kx {

constexpr int kStepRows = 32;  // rows of K per MFMA step

// Column (0..7) inside a word -> nibble that holds it (inverse of order_of).
__host__ __device__ constexpr int nibble_of(int col) {
    return (col & 1) ? 4 + (col >> 1) : (col >> 1);
}

// Two bf16 128.0 in a register whose value the compiler cannot see.  (v & 0x000F000F) | magic then
// selects as one v_and_or_b32 (a literal and a register); with two literals it would be split into
// v_and + v_or.  The conversion itself stays ordinary C so that the compiler keeps track of the
// registers the matrix instructions are still reading.
__device__ __forceinline__ uint32_t opaque_bf16_128_pair() {
    uint32_t out;
    asm volatile("v_mov_b32 %0, 0x43004300" : "=v"(out));
    return out;
}

__device__ __forceinline__ uint32_t code_pair_to_bf16(uint32_t v, uint32_t magic) {
    return (v & 0x000F000Fu) | magic;
}

// Two neighbouring bf16 as floats.
__device__ __forceinline__ float low_bf16(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float high_bf16(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }

// Sums of the waves in LDS, [wave][word half h][row][128 columns 16 c + 8 h + j], c < 16, j < 8: lane (c, b) writes two 16-byte
// pieces per row.  The two change places in every other group of four lanes, so that eight lanes side by side write to all
// banks.  What bounds this phase is the number of LDS writes: a ds_write_b128 takes the compute unit 13.5 cycles however many
// of its lanes are active (22 to 33 where they meet in a quarter of the banks), a ds_read_b128 4.5.  So from four rows on the
// lanes without a row of their own take over a part of the others' (v_permlane32_swap, v_permlane16_swap), which leaves
// 16 / 8 / 4 writes per wave at 16 / 8 / 4 rows instead of 32 / 16 / 16, and a thread reads and stores four columns at a time.
// us per launch, before -> now, M = 4 / 8 / 16: 4096 -> 1024 6.6 / 7.1 / 8.3 -> 6.4 / 6.9 / 7.5, 4096 -> 4096 into the residual
// stream 7.8 / 8.2 / 9.5 -> 7.6 / 7.8 / 8.8, 12288 -> 4096 behind SwiGLU 13.5 / 15.1 / 17.8 -> 13.5 / 14.4 / 16.5,
// 4096 -> 24576 behind a norm 16.9 / 21.1 / 24.3 -> 16.8 / 20.2 / 23.0; one and two rows alike.
constexpr int kHalfCols = 128;
__device__ __forceinline__ int red_piece(int piece) {  // 16-byte piece 0 .. 31 of a row of 128 columns -> where it lies
    return piece ^ ((piece >> 3) & 1);
}

// 128 + zero point, indexed by nibble.
__device__ __forceinline__ void zero_offsets(uint32_t zeros, float (&out)[8]) {
    const uint32_t even = (zeros & 0x0F0F0F0Fu) | 0x80808080u, odd = ((zeros >> 4) & 0x0F0F0F0Fu) | 0x80808080u;
#pragma unroll
    for (int i = 0; i < 8; i++) out[i] = static_cast<float>(((i % 2 ? odd : even) >> (8 * (i / 2))) & 0xFFu);
}

// Half `which` of the lanes of `a`, then of `b`; lanes 0 .. 15 of `a`, then of `b` (and the same of lanes 32 .. 63).
__device__ __forceinline__ float half_wave_pack(float a, float b, int which) {
    return __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false)[which]);
}
__device__ __forceinline__ float quarter_wave_pack(float a, float b) {
    return __uint_as_float(__builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false)[0]);
}

// A thread's columns: their sums, and the scales as loaded.
template <int COLS>
struct alignas(4 * COLS) FloatsOf {
    float v[COLS];
    __device__ __forceinline__ float& operator[](int i) { return v[i]; }
    __device__ __forceinline__ float operator[](int i) const { return v[i]; }
};
template <int COLS>
struct ScaleBits {
    struct alignas(2 * COLS) type {
        uint16_t v[COLS];
        __device__ __forceinline__ uint16_t operator[](int i) const { return v[i]; }
    };
};

template <bool LONE>
struct WordPair {
    typedef u32x2 type;
};
template <>
struct WordPair<true> {
    typedef u32x2 __attribute__((aligned(4))) type;
};

// How a launch divides the matrix between workgroups.
struct MfmaGrid {
    int coltiles;
    int ktiles;
    int side;              // column tiles side by side in the grid (gridDim.x, whose own load is a trip to memory)
    int run;               // blocks of K whose sums are added up first: by a workgroup that walks over them (WALK), or by
                           // the one that reads the partial sums back, so that every launch of a shape adds alike
    int sliced;            // all K tiles of a column tile finish it together (splitk_exchange_sliced)
    uint32_t group_magic;  // ceil(2^32 / (G / 32)), 0 for groups of 32
    uint32_t wait_ticks;   // how long a workgroup waits for the others of its tile
    TileOrder order;       // which tile a workgroup takes where not that of its own number
};

// Quantisation group of a 32-row step: step / (G / 32) for any number of steps a matrix can have.
__device__ __forceinline__ int group_of_step(const MfmaGrid& g, int step) {
    return g.group_magic ? static_cast<int>(__umulhi(static_cast<uint32_t>(step), g.group_magic)) : step;
}

// KS: consecutive 32-row steps per wave (they share a quantisation group, or FINE);
// MC: activation rows a workgroup reduces per LDS round (1, 2, 4 or 8); ROUNDS: 2 for M > 8, else 1;
// WALK: a workgroup works through grid.run blocks of KB rows of K, one behind the other, and adds their sums up in
// registers (make_mfma_plan says when; carrying the loop costs the other launches up to a microsecond);
// FINE: a wave's steps lie in groups of their own, and scale and zero point are applied per step, to the sums in registers:
// groups that are no multiple of 128 with four steps per wave (make_mfma_plan says what that is worth).  The scales go through
// LDS, each loaded once per workgroup (a lane's own take as many loads as the weights); the waves' sums then only add up;
// LONE: N is an odd multiple of eight (a template parameter: the moves cost 20 registers, an occupancy step).
// With a prologue, `x` is not read: fi.a / fi.b (/ fi.gain) are 16-byte aligned, fi.ld a multiple of eight.
// Three workgroups per compute unit (168 registers) at sixteen rows with one or two steps per wave.  One step is held to it: us
// per launch, two -> three, groups of 32, M = 9 / 16: 1024 -> 34816 15.9 / 16.7 -> 15.4 / 16.5, behind a norm 16.8 / 17.7 -> 16.0 /
// 17.1, 1024 -> 24576 11.4 / 11.8 -> 11.2 / 11.7.  Two steps take 167 by themselves; held to it, the plain launch spilled 19: spilled
// -> left alone, groups of 64, 2048 -> 24576 14.7 / 15.9 -> 13.7 / 14.9, 2048 -> 16896 15.2 / 16.9 -> 13.4 / 15.1, 2048 -> 51200 24.3 /
// 28.2 -> 23.0 / 26.6; grids of up to 512 workgroups alike.
//
// Four steps per wave at five and more rows, stored: 185 registers leave two to a compute unit, so that a grid of 513 to 768
// comes in two rounds and cannot finish its tiles together.  With four nibbles' operands at a time and a step's activations read
// when it comes they fit 168 (what still goes to memory at sixteen rows behind a norm, 80 bytes a lane, belongs to the single
// reader's read-back; the plain form, which has none, keeps all but two words).
// Behind a norm every such launch takes this form: us per launch, M = 9 / 16, two -> three and finishing together, 4096 -> 24576 20.0 /
// 20.8 -> 18.0 / 18.7, 5120 -> 15360 20.9 / 21.6 -> 16.9 / 17.4, 8192 -> 10240 at M = 6 / 9 / 16 17.9 / 21.9 / 22.3 -> 17.2 / 18.1 / 20.2;
// two -> three alone, larger grids, M = 6 / 16, 4096 -> 32768 22.8 / 25.7 -> 22.8 / 24.3, 5120 -> 51200 43.8 /
// 48.2 -> 43.8 / 46.2, and smaller ones, 4096 -> 12288 12.3 / 13.9 -> 12.2 / 13.9.  A plain launch takes it where make_mfma_plan
// says so (TRIO): larger grids at sixteen rows lose by it, 4096 -> 32768 23.5 -> 26.1.
template <int KS, int ROWS, int PRO, int EPI, bool WALK, bool FINE, bool TRIO>
constexpr bool kThreePerUnit = KS == 4 && ROWS >= 8 && EPI == kEpiStore && !WALK && !FINE && (PRO == kProPreNorm || TRIO);
template <int WAVES, int KS, int MC, int ROUNDS, int PRO = kProNone, int EPI = kEpiStore, bool LONE = false, bool WALK = false, bool FINE = false,
          bool TRIO = false>
__global__ __launch_bounds__(WAVES * kWave, ((KS == 1 && ROUNDS == 2 && EPI == kEpiStore) || kThreePerUnit<KS, MC * ROUNDS, PRO, EPI, WALK, FINE, TRIO> ? 3 : 2)) void awq_gemv_mfma_kernel(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ qweight,
    const uint16_t* __restrict__ scales, const uint32_t* __restrict__ qzeros,
    uint16_t* __restrict__ y, float* __restrict__ partials, uint32_t* __restrict__ counters,
    int M, int K, int N, MfmaGrid grid, FusedInput fi, ResidualTarget res, RopeTarget rope,
    size_t cache_stride) {
    constexpr int WROWS = KS * kStepRows;  // rows of K per wave
    constexpr int KB = WAVES * WROWS;      // rows of K per workgroup
    constexpr int ROWS = MC * ROUNDS;      // activation rows this kernel carries (>= M)
    static_assert(!WALK || (KS == 4 && ROWS >= 8), "the launches that walk");
    static_assert(!FINE || (KS == 4 && !WALK), "the launches whose waves cross groups");
    constexpr int THREADS = WAVES * kWave;
    static_assert(THREADS >= kTileCols, "one thread per tile column");
    static_assert(PRO == kProNone || PRO == kProSwiGLU || PRO == kProPreNorm, "prologues of the matrix-core kernel");
    static_assert(EPI == kEpiStore || EPI == kEpiResidual || EPI == kEpiQkRope, "epilogues of the matrix-core kernel");
    constexpr bool STAGED = PRO != kProNone;
    constexpr bool THREE = kThreePerUnit<KS, ROWS, PRO, EPI, WALK, FINE, TRIO>;
    static_assert(!TRIO || (THREE && PRO == kProNone), "plain launches, three to a compute unit");
    // The loads of the next block go out while the waves of this one meet, except at sixteen rows behind a prologue, whose
    // operands do not fit the registers beside the weights and the sums: there the other workgroup of the compute unit
    // has to cover the gap.
    constexpr bool AHEAD = PRO == kProNone || ROUNDS == 1;
    // Those launches are short of registers.  What is cheap to work out is worked out per block (the addresses of the rows) or per
    // round (the scales as floats) instead of kept: spilled addresses came back behind the weights, so that a block waited for
    // them before it produced its activations.  us per launch behind SwiGLU, kept -> worked out, M = 9 / 16: 18432 -> 5120
    // 29.9 / 30.7 -> 24.1 / 24.5, 25600 -> 5120 34.5 / 35.8 -> 26.7 / 27.2.
    constexpr bool SHORT_OF_REGISTERS = WALK && !AHEAD;
    // Launches of a shape that walks elsewhere (make_mfma_plan): behind a prologue at sixteen rows or with an odd number
    // of words, and the rotary epilogue.
    constexpr bool RUNS = !WALK && !FINE && KS == 4 &&
                          ((ROWS == 16 && PRO != kProNone) || (ROWS >= 8 && (EPI == kEpiQkRope || (LONE && PRO != kProNone))));
    // A staged row is the workgroup's K range plus 16 bytes, so that the rows a wave reads together
    // start in different banks.
    constexpr int XPITCH = KB + 8;
    constexpr int KPIECES = KB / 8;             // 16-byte pieces per staged row
    constexpr int PIECES = ROWS * KPIECES;
    constexpr int PPT = (PIECES + THREADS - 1) / THREADS;  // pieces a thread produces, of the same k in every THREADS / KPIECES-th row
    static_assert(THREADS % KPIECES == 0, "a thread's pieces share their k");

    // From eight rows on a thread owns pieces of four columns, so that the sums are read, multiplied and stored sixteen bytes at
    // a time: word half tid / 128, piece tid % 32 of its 128 columns, rows tid / 32 % 4 + 4 i.  Up to four rows a thread owns
    // one column of each (four columns' scales and zero points cost a step of occupancy there).
    constexpr bool QUADS = ROWS >= 8;
    constexpr int OWN = QUADS ? 4 : 1;                 // columns of a thread
    constexpr int RROWS = ROWS < 8 ? ROWS : 8;         // activation rows per LDS round
    constexpr int RSUMS = QUADS ? RROWS / 4 : ROWS;    // rows of a thread per round
    constexpr int PSUMS = QUADS ? ROWS / 4 : ROWS;     // rows of a thread
    // One and two rows that are stored or added meet column by column: the few lanes that write leave the banks free either way,
    // and the order of the pieces below cost a step of occupancy with one step per wave.  us per launch at M = 2, by pieces -> by
    // columns, groups of 32: 4096 -> 24576 behind SwiGLU into the residual stream 18.2 -> 17.4.  (The rotary launches take fewer
    // registers by pieces, and those behind a norm lose 0.1 to 0.2 us by columns and the test below.)
    constexpr bool BY_COLUMNS = ROWS <= 2 && PRO != kProPreNorm && EPI != kEpiQkRope && !FINE;

    __shared__ __attribute__((aligned(16))) float red[WAVES][2][RROWS][kHalfCols];
    __shared__ __attribute__((aligned(16))) float xs_red[WAVES][ROWS < 4 ? 4 : ROWS];
    __shared__ uint32_t s_word[3];
    __shared__ __attribute__((aligned(16))) uint16_t s_fscale[FINE ? WAVES * KS : 1][FINE ? kTileCols : 8];
    __shared__ uint32_t s_fzero[FINE ? WAVES * KS : 1][FINE ? kTileCols / 8 : 1];
    __shared__ __attribute__((aligned(16))) uint16_t s_x[STAGED ? ROWS : 1][STAGED ? XPITCH : 8];
    __shared__ float s_inv[PRO == kProPreNorm ? ROWS : 1];

    const int tid = threadIdx.x;
    const int wave = FINE ? __builtin_amdgcn_readfirstlane(tid / kWave) : tid / kWave;
    const int lane = tid % kWave;
    const int c = lane % 16;  // column slot: word pair c of the tile, MFMA column c
    const int b = lane / 16;  // k block inside the step, D row block
    // By number column tiles run fastest, so neighbours in time are neighbours in N; where workgroups finish a tile together, in
    // groups of at most eight, so that they start within 8 * ktiles of each other.  By XCD (grid.order) those of a tile lie
    // anywhere in the grid: grids that finish together are sized to be resident whole, and their wait is bounded.
    Tile tile{static_cast<int>(blockIdx.z * grid.side + blockIdx.x), static_cast<int>(blockIdx.y)};
    const int ktiles = grid.ktiles;
    if (grid.order.run) tile = tile_of_workgroup(grid.order, (blockIdx.z * ktiles + blockIdx.y) * grid.side + blockIdx.x, static_cast<uint32_t>(ktiles));
    const int ct = tile.ct;
    const int kt = tile.kt;
    const int nw = N >> 3;

    // first row of the block that is loaded next, and how many blocks the workgroup has
    int kblock = kt * KB * (WALK ? grid.run : 1);
    const int blocks = WALK ? min(grid.run, (K - kblock + KB - 1) / KB) : 1;

    // ---- operands of the activation prologue go out first: they are small, mostly cached, and the prologue
    // should run while the weights are still on their way ----
    // Piece e = tid + i * THREADS of the workgroup is (row e / KPIECES, elements 8 (e % KPIECES) .. + 7 of
    // the block); addresses are clamped, what a clamped load brings is replaced by zeros.
    uint4 pa[STAGED ? PPT : 1], pb[PRO == kProSwiGLU ? PPT : 1];  // gate or row; up, or the norm's gain, which all rows share
    float tile_ss[PRO == kProPreNorm ? (ROWS + WAVES - 1) / WAVES : 1];
    if constexpr (PRO == kProPreNorm) {
        // wave w adds the tiles of rows w, w + WAVES, ...: lane = tile
#pragma unroll
        for (int rr = 0; rr < (ROWS + WAVES - 1) / WAVES; rr++) {
            const int m = wave + rr * WAVES;
            const int mc = m < M ? m : M - 1;
            const f32x4 qs = reinterpret_cast<const f32x4*>(fi.sumsq)[static_cast<size_t>(mc) * fi.sumsq_parts +
                                                                      (lane < fi.sumsq_parts ? lane : fi.sumsq_parts - 1)];
            tile_ss[rr] = ((qs.x + qs.y) + qs.z) + qs.w;  // the order that defines a tile's sum
        }
    }

    // ---- loads of a block, all issued before anything is consumed ----
    // Every load is unconditional: an address that would fall outside is clamped to one inside, and
    // what it brings is either masked (activations) or lands in outputs that are never stored
    // (columns past N).  A load under a condition becomes a branch with a full wait behind it, and
    // a chain of those is a chain of memory round trips.
    //
    // Scales and zero points of the columns this thread will own after the LDS round, one set per wave of the workgroup (whose
    // steps share a quantisation group, FINE aside; waves that share one read the same address).
    const int own_piece = tid % 32;
    const int own_half = tid / 128;
    const int own_row = tid / 32 % 4;
    const int own_col = ct * kTileCols + (QUADS ? 16 * (own_piece / 2) + 8 * own_half + 4 * (own_piece % 2) : tid);  // the first
    const int own_ld = own_col < N ? own_col : N - OWN;
    typename ScaleBits<OWN>::type s_bits[WAVES];
    uint32_t z_word[WAVES];
    // FINE: the scales and zero points of the workgroup's steps go through LDS, eight columns (a word) of a step per piece; a lane
    // reads those of the columns whose sums it keeps, packed as they go to LDS: its sixteen columns at sixteen rows, eight
    // (word half b / 2) at eight, four (piece b % 2 of it) below.
    constexpr int FSTEPS = WAVES * KS;
    constexpr int FPIECES = FSTEPS * 32 / THREADS;  // pieces a thread stages
    constexpr int FCOLS = ROWS >= 8 ? 8 : 4;
    u32x4 f_scale[FINE ? FPIECES : 1];
    uint32_t f_zero[FINE ? FPIECES : 1];
    // The A operand: row c of the activations, whether or not column slot c holds weights.  Rows
    // past M and steps past K (K is a multiple of 32: a step is all in or all out) are zeros.
    uint4 xa[KS];
    const int x_row = c < M ? c : M - 1;
    // The lane's two word columns, eight rows per step, both words in one load, of four-byte alignment where the
    // number of words is odd; the last lane's one word then comes as the second of its pair and is moved over.
    using word_pair = typename WordPair<LONE>::type;
    uint32_t w[KS][8][2];
    const int wc_first = ct * 32 + 2 * c;
    const int wc0 = max(0, min(wc_first, nw - 2));
    const bool lone_word = wc_first == nw - 1;
    auto load_operands = [&] {
        if constexpr (STAGED) {
            int thread = tid;
            if constexpr (SHORT_OF_REGISTERS) asm volatile("" : "+v"(thread));
#pragma unroll
            for (int i = 0; i < PPT; i++) {
                const int pm = thread / KPIECES + i * (THREADS / KPIECES);
                const int k = kblock + 8 * (thread % KPIECES);
                const int mc = pm < M ? pm : M - 1;
                const int kc = k < K ? k : K - 8;
                const size_t at = static_cast<size_t>(mc) * fi.ld + kc;
                pa[i] = *reinterpret_cast<const uint4*>(fi.a + at);
                if constexpr (PRO == kProSwiGLU) pb[i] = *reinterpret_cast<const uint4*>(fi.b + at);
                else if (i == 0) pb[0] = *reinterpret_cast<const uint4*>(fi.gain + kc);
            }
        }
        if constexpr (!STAGED) {
#pragma unroll
            for (int ks = 0; ks < KS; ks++) {
                const int kstep = kblock + wave * WROWS + ks * kStepRows;
                const int kld = kstep < K ? kstep : K - kStepRows;
                const uint4 got = *reinterpret_cast<const uint4*>(x + static_cast<size_t>(x_row) * K + kld + 8 * b);
                const bool live = FINE || (c < M && kstep < K);  // FINE masks at the product: here it waited in front of the weights' loads
                xa[ks] = make_uint4(live ? got.x : 0u, live ? got.y : 0u, live ? got.z : 0u, live ? got.w : 0u);
            }
        }
    };
    auto load_weights = [&] {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            const int kstep = kblock + wave * WROWS + ks * kStepRows;
            const int k0 = (kstep < K ? kstep : K - kStepRows) + 8 * b;  // first of the lane's eight rows
            const uint32_t* wp = qweight + static_cast<size_t>(k0) * nw + wc0;
#pragma unroll
            for (int r = 0; r < 8; r++) {
                const u32x2 v = __builtin_nontemporal_load(reinterpret_cast<const word_pair*>(wp + static_cast<size_t>(r) * nw));
                w[ks][r][0] = v.x;
                w[ks][r][1] = v.y;
            }
        }
    };
    auto load_scales = [&] {
        if constexpr (FINE) {
#pragma unroll
            for (int i = 0; i < FPIECES; i++) {
                const int e = tid + i * THREADS;
                const int kstep = kblock + e / 32 * kStepRows;
                const int step = (kstep < K ? kstep : K - 1) / kStepRows;  // rows past K meet zero activations
                const int quotient = static_cast<int>(__umulhi(static_cast<uint32_t>(step), grid.group_magic));
                const int g = grid.group_magic ? quotient : step;  // as group_of_step(), without a branch between the loads
                const int word = ct * 32 + e % 32 < nw ? ct * 32 + e % 32 : nw - 1;
                f_scale[i] = *reinterpret_cast<const u32x4*>(scales + static_cast<size_t>(g) * N + 8 * word);
                f_zero[i] = qzeros[static_cast<size_t>(g) * nw + word];
            }
            return;
        }
#pragma unroll
        for (int wv = 0; wv < WAVES; wv++) {
            const int krow = kblock + wv * WROWS;
            const int g = group_of_step(grid, (krow < K ? krow : K - 1) / kStepRows);  // rows past K meet zero activations
            s_bits[wv] = *reinterpret_cast<const typename ScaleBits<OWN>::type*>(scales + static_cast<size_t>(g) * N + own_ld);
            z_word[wv] = qzeros[static_cast<size_t>(g) * nw + (own_ld >> 3)];
        }
    };
    if constexpr (!STAGED) load_scales();
    load_operands();
    if constexpr (STAGED) load_scales();
    if constexpr (FINE && PRO == kProPreNorm) __builtin_amdgcn_sched_barrier(1);  // no load of them moves behind the weights
    load_weights();
    __builtin_amdgcn_sched_barrier(0);
#if defined(KX_ABLATE) && KX_ABLATE == 2
    if (!STAGED && ktiles > 1) {  // profiling build: loads only - fold what arrived into one word and leave
        uint32_t f = 0;
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            f ^= xa[ks].x ^ xa[ks].y ^ xa[ks].z ^ xa[ks].w;
#pragma unroll
            for (int r = 0; r < 8; r++) f ^= w[ks][r][0] ^ w[ks][r][1];
        }
#pragma unroll
        for (int wv = 0; wv < WAVES; wv++) {
            if constexpr (FINE) f ^= f_zero[0];
            else f ^= s_bits[wv][0] ^ z_word[wv];
        }
        if (f == 0x9E3779B9u) partials[tid] = 1.0f;
        return;
    }
#endif

    if constexpr (PRO == kProPreNorm) {
        // lane rr takes the total of row wave + rr * WAVES: one square root and division for all rows of the wave
        constexpr int NORM_ROWS = (ROWS + WAVES - 1) / WAVES;
        float mine = 0.0f;
#pragma unroll
        for (int rr = 0; rr < NORM_ROWS; rr++) {
            const float total = wave_sum(lane < fi.sumsq_parts ? tile_ss[rr] : 0.0f);
            mine = lane == rr ? total : mine;
        }
        const float inv = 1.0f / sqrtf(mine / static_cast<float>(K) + fi.eps);
        if (lane < NORM_ROWS && wave + lane * WAVES < ROWS) s_inv[wave + lane * WAVES] = inv;
        lds_barrier();
    }
    if constexpr (FINE) {
#pragma unroll
        for (int i = 0; i < FPIECES; i++) {
            const int e = tid + i * THREADS;
            // a step past K adds nothing: its sums are zeros, but zero times an infinite scale is not
            const uint32_t keep = kblock + e / 32 * kStepRows < K ? 0xffffffffu : 0u;
            *reinterpret_cast<u32x4*>(&s_fscale[e / 32][8 * (e % 32)]) = f_scale[i] & keep;
            s_fzero[e / 32][e % 32] = f_zero[i];
        }
        if constexpr (!STAGED) lds_barrier();  // otherwise the barrier behind the produced activations serves
    }
    FloatsOf<OWN> psum[PSUMS];
    for (int block = 0; block < blocks; block++) {
        // ---- the activation prologue: produce the staged rows, then read the A operand back ----
        if constexpr (STAGED) {
#pragma unroll
            for (int i = 0; i < PPT; i++) {
                const int pm = tid / KPIECES + i * (THREADS / KPIECES);  // a row's distance from the first is known when compiling
                const int kp = tid % KPIECES;
                if (PIECES % THREADS == 0 || pm < ROWS) {
                    // Vector instructions bound the prologue (every column tile produces its rows anew), so two elements share a
                    // conversion, the norm's gain is loaded and the inverse worked out once, and the words of a dead piece are
                    // masked at the end: a select per element had become a branch per element.  us per launch at M = 8 / 16:
                    // 4096 -> 24576 behind a norm 20.2 / 23.0 -> 19.6 / 21.0, q|k|v 10.1 / 12.0 -> 10.0 / 11.3.
                    const uint32_t aw[4] = {pa[i].x, pa[i].y, pa[i].z, pa[i].w};
                    const uint4 second = pb[PRO == kProSwiGLU ? i : 0];
                    const uint32_t bw[4] = {second.x, second.y, second.z, second.w};
                    const uint32_t keep = pm < M && kblock + 8 * kp < K ? 0xffffffffu : 0u;  // K is a multiple of eight: all in or all out
                    const float inv = PRO == kProPreNorm ? s_inv[pm] : 0.0f;
                    uint32_t out[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float lo = low_bf16(aw[j]), hi = high_bf16(aw[j]);
                        const uint32_t act = PRO == kProSwiGLU ? f32x2_to_bf16x2(silu(lo), silu(hi)) : f32x2_to_bf16x2(lo * inv, hi * inv);
                        out[j] = f32x2_to_bf16x2(low_bf16(act) * low_bf16(bw[j]), high_bf16(act) * high_bf16(bw[j])) & keep;
                    }
                    *reinterpret_cast<uint4*>(&s_x[pm][8 * kp]) = make_uint4(out[0], out[1], out[2], out[3]);
                }
            }
            lds_barrier();
            const int s_row = c < ROWS ? c : ROWS - 1;
#pragma unroll
            for (int ks = 0; ks < (THREE ? 0 : KS); ks++) {
                const uint4 got = *reinterpret_cast<const uint4*>(&s_x[s_row][(wave * KS + ks) * kStepRows + 8 * b]);
                const bool live = c < M;  // rows M .. ROWS-1 and elements past K were staged as zeros
                xa[ks] = make_uint4(live ? got.x : 0u, live ? got.y : 0u, live ? got.z : 0u, live ? got.w : 0u);
            }
        }

        // ---- matrix products ----
        const bf16x8 ones = as_bf16x8(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u);
        const f32x4v zero4 = {0.0f, 0.0f, 0.0f, 0.0f};
        f32x4v xs;
        f32x4v acc[2][8];  // [word h][nibble p]
        // FINE: scaled sums, [word h][nibble p] at sixteen rows, [nibble p] of word b / 2 at eight (rows 4 (b % 2) + v), and
        // [column of the piece] below (rows v)
        f32x4v fine[FINE ? (ROWS == 16 ? 16 : FCOLS) : 1];
        const uint32_t magic = opaque_bf16_128_pair();
        // sixteen rows that are scaled per step take the word halves one after the other: both at once spill 80 registers
        constexpr int PASSES = FINE && ROWS == 16 ? 2 : 1;
#pragma unroll
        for (int i = 0; i < KS * PASSES; i++) {
            const int ks = i % KS, h0 = PASSES == 2 ? i / KS : 0, h1 = PASSES == 2 ? h0 + 1 : 2;
            if constexpr (LONE) {
#pragma unroll
                for (int r = 0; r < 8 && i < KS; r++) w[ks][r][0] = lone_word ? w[ks][r][1] : w[ks][r][0];
            }
            if constexpr (FINE && !STAGED) {
                const uint32_t keep = c < M && kblock + wave * WROWS + ks * kStepRows < K ? 0xffffffffu : 0u;
                xa[ks] = make_uint4(xa[ks].x & keep, xa[ks].y & keep, xa[ks].z & keep, xa[ks].w & keep);
            }
            if constexpr (STAGED && THREE) {  // the others read all steps' operands at once
                const uint4 got = *reinterpret_cast<const uint4*>(&s_x[c < ROWS ? c : ROWS - 1][(wave * KS + ks) * kStepRows + 8 * b]);
                const bool live = c < M;
                xa[ks] = make_uint4(live ? got.x : 0u, live ? got.y : 0u, live ? got.z : 0u, live ? got.w : 0u);
            }
            const bf16x8 a_op = as_bf16x8(xa[ks].x, xa[ks].y, xa[ks].z, xa[ks].w);
            xs = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_op, ones, ks == 0 || FINE ? zero4 : xs, 0, 0, 0);
#pragma unroll
            for (int h = h0; h < h1; h++) {
                if constexpr (THREE) {  // four nibbles at a time: half the operands in registers
#pragma unroll
                    for (int q = 0; q < 8; q += 4) {
                        uint32_t bop[4][4];  // [nibble][row pair]
#pragma unroll
                        for (int rp = 0; rp < 4; rp++) {
                            const uint32_t v = __builtin_amdgcn_perm(w[ks][2 * rp + 1][h], w[ks][2 * rp][h], q ? 0x07060302u : 0x05040100u);
#pragma unroll
                            for (int p = 0; p < 4; p++) bop[p][rp] = code_pair_to_bf16(p == 0 ? v : v >> (4 * p), magic);
                        }
#pragma unroll
                        for (int p = 0; p < 4; p++) {
                            acc[h][q + p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                a_op, as_bf16x8(bop[p][0], bop[p][1], bop[p][2], bop[p][3]), ks == 0 ? zero4 : acc[h][q + p], 0, 0, 0);
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                } else {
                    uint32_t bop[8][4];  // [nibble p][row pair]
#pragma unroll
                    for (int rp = 0; rp < 4; rp++) {
                        const uint32_t wa = w[ks][2 * rp][h];      // row 2rp   -> low half
                        const uint32_t wb = w[ks][2 * rp + 1][h];  // row 2rp+1 -> high half
                        const uint32_t lo = __builtin_amdgcn_perm(wb, wa, 0x05040100u);  // nibbles 0..3, both rows
                        const uint32_t hi = __builtin_amdgcn_perm(wb, wa, 0x07060302u);  // nibbles 4..7
#pragma unroll
                        for (int p = 0; p < 4; p++) {
                            bop[p][rp] = code_pair_to_bf16(p == 0 ? lo : lo >> (4 * p), magic);
                            bop[4 + p][rp] = code_pair_to_bf16(p == 0 ? hi : hi >> (4 * p), magic);
                        }
                    }
#pragma unroll
                    for (int p = 0; p < 8; p++) {
                        acc[h][p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            a_op, as_bf16x8(bop[p][0], bop[p][1], bop[p][2], bop[p][3]), ks == 0 || FINE ? zero4 : acc[h][p], 0, 0, 0);
                    }
                }
                if constexpr (FINE && ROWS == 16) {
                    float zoff[8];
                    zero_offsets(s_fzero[wave * KS + ks][2 * c + h], zoff);
                    const auto scale = *reinterpret_cast<const typename ScaleBits<8>::type*>(&s_fscale[wave * KS + ks][16 * c + 8 * h]);
#pragma unroll
                    for (int p = 0; p < 8; p++) {
                        const float sc = f16_bits_to_f32(scale[order_of(p)]);
#pragma unroll
                        for (int v = 0; v < 4; v++) {
                            const float part = __builtin_fmaf(-zoff[p], xs[v], acc[h][p][v]);
                            fine[8 * h + p][v] = ks == 0 ? sc * part : __builtin_fmaf(sc, part, fine[8 * h + p][v]);
                        }
                    }
                }
            }
            if constexpr (FINE && ROWS == 8) {
                float zoff[8], row_sum[4];
                zero_offsets(s_fzero[wave * KS + ks][2 * c + b / 2], zoff);
                const auto scale = *reinterpret_cast<const typename ScaleBits<8>::type*>(&s_fscale[wave * KS + ks][16 * c + 8 * (b / 2)]);
#pragma unroll
                for (int v = 0; v < 4; v++) row_sum[v] = half_wave_pack(xs[v], xs[v], 0);
#pragma unroll
                for (int p = 0; p < 8; p++) {
                    const float sc = f16_bits_to_f32(scale[order_of(p)]);
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const float part = __builtin_fmaf(-zoff[p], row_sum[v], half_wave_pack(acc[0][p][v], acc[1][p][v], 0));
                        fine[p][v] = ks == 0 ? sc * part : __builtin_fmaf(sc, part, fine[p][v]);
                    }
                }
            }
            if constexpr (FINE && ROWS <= 4) {
                float zoff[8];
                zero_offsets(s_fzero[wave * KS + ks][2 * c + b / 2] >> (8 * (b % 2)), zoff);
                const auto scale = *reinterpret_cast<const typename ScaleBits<4>::type*>(&s_fscale[wave * KS + ks][16 * c + 4 * b]);
#pragma unroll
                for (int v = 0; v < ROWS; v++) {
                    const float twice = quarter_wave_pack(xs[v], xs[v]);
                    const float row_sum = half_wave_pack(twice, twice, 0);
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const int e = nibble_of(q);  // of the piece's column q; two further up in the second piece
                        const float part = __builtin_fmaf(-zoff[e], row_sum,
                                                          half_wave_pack(quarter_wave_pack(acc[0][e][v], acc[0][e + 2][v]),
                                                                         quarter_wave_pack(acc[1][e][v], acc[1][e + 2][v]), 0));
                        const float sc = f16_bits_to_f32(scale[q]);
                        fine[q][v] = ks == 0 ? sc * part : __builtin_fmaf(sc, part, fine[q][v]);
                    }
                }
            }
            if constexpr (FINE) {
                // A step's sums are scaled in the step; the compiler had put that off until all steps' sums were there, which
                // took the registers of all of them (at sixteen rows 76 were spilled, and 5472 -> 9000 took 30.3 us, not 18.0).
#pragma unroll
                for (int q = PASSES == 2 ? 8 * h0 : 0; q < (PASSES == 2 ? 8 * h1 : FCOLS); q++) asm volatile("" : "+v"(fine[q]));
            }
            // a step is worked through while the loads of the later steps are still in flight
            __builtin_amdgcn_sched_barrier(0);
        }

        // scales, and 128 + zero point, of the columns of the thread's pieces: nibbles 0, 4, 1, 5 of a word, or one byte up
        FloatsOf<OWN> sc[WAVES], zc[WAVES];
        auto convert_scales = [&](int wv) {
            const uint32_t zeros = z_word[wv] >> (QUADS ? 8 * (own_piece % 2) : 4 * nibble_of(own_col & 7));
            const uint32_t even = (zeros & 0x000F000Fu) | 0x00800080u, odd = ((zeros >> 4) & 0x000F000Fu) | 0x00800080u;
#pragma unroll
            for (int j = 0; j < OWN; j++) {
                sc[wv][j] = f16_bits_to_f32(s_bits[wv][j]);
                const uint32_t both = j < 2 ? even : odd;
                zc[wv][j] = static_cast<float>(j % 2 ? (both >> 16) & 0xFFu : both & 0xFFu);
            }
        };
        if constexpr (!FINE && !SHORT_OF_REGISTERS) {
#pragma unroll
            for (int wv = 0; wv < WAVES; wv++) convert_scales(wv);
        }
        auto load_next = [&] {
            if (block + 1 < blocks) {
                kblock += KB;
                load_operands();
                if constexpr (STAGED) load_scales();
                load_weights();
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if constexpr (WALK && AHEAD) load_next();

        // ---- waves meet in LDS; every thread then owns its columns ----
        // D rows 4b .. 4b+3 of the lane; its sixteen columns are 16c .. 16c+15, those of word h eight of them.  A round writes
        // with all lanes: eight rows fill half of them, and the word halves are packed side by side.
        const int piece0 = BY_COLUMNS ? 8 * c : 4 * red_piece(2 * c), piece1 = BY_COLUMNS ? 8 * c + 4 : 4 * red_piece(2 * c + 1);
#pragma unroll
        for (int rd = 0; rd < ROWS / RROWS; rd++) {
            if (rd > 0 || block > 0) lds_barrier();  // the previous round has been read
            if constexpr (!BY_COLUMNS) {
                if (rd == 0 && c == 0 && 4 * b < ROWS) *reinterpret_cast<f32x4v*>(&xs_red[wave][4 * b]) = xs;
            }
#pragma unroll
            for (int v = 0; v < (ROWS < 4 ? ROWS : 4); v++) {
                if constexpr (ROWS >= 8) {
                    float m[8];
#pragma unroll
                    for (int q = 0; q < 8; q++) {
                        if constexpr (!FINE) m[q] = half_wave_pack(acc[0][q][v], acc[1][q][v], rd);
                        else if constexpr (ROWS == 16) m[q] = half_wave_pack(fine[q][v], fine[8 + q][v], rd);
                        else m[q] = fine[q][v];
                    }
                    float* dst = &red[wave][b / 2][4 * (b % 2) + v][0];
                    *reinterpret_cast<f32x4*>(dst + piece0) = f32x4{m[0], m[4], m[1], m[5]};
                    *reinterpret_cast<f32x4*>(dst + piece1) = f32x4{m[2], m[6], m[3], m[7]};
                } else if constexpr (FINE) {
                    *reinterpret_cast<f32x4*>(&red[wave][b / 2][v][b % 2 ? piece1 : piece0]) = f32x4{fine[0][v], fine[1][v], fine[2][v], fine[3][v]};
                } else if constexpr (ROWS == 4) {  // a quarter of the lanes: every lane takes one of the four pieces of sixteen columns
                    float m[4];
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const int e = q / 2 + 4 * (q % 2);  // nibble of the piece's column q; two further up in the second piece
                        m[q] = half_wave_pack(quarter_wave_pack(acc[0][e][v], acc[0][e + 2][v]), quarter_wave_pack(acc[1][e][v], acc[1][e + 2][v]), 0);
                    }
                    *reinterpret_cast<f32x4*>(&red[wave][b / 2][v][b % 2 ? piece1 : piece0]) = f32x4{m[0], m[1], m[2], m[3]};
                } else if (b == 0) {
                    if (BY_COLUMNS && c == 0) xs_red[wave][v] = xs[v];
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        float* dst = &red[wave][h][v][0];
                        *reinterpret_cast<f32x4*>(dst + piece0) = f32x4{acc[h][0][v], acc[h][4][v], acc[h][1][v], acc[h][5][v]};
                        *reinterpret_cast<f32x4*>(dst + piece1) = f32x4{acc[h][2][v], acc[h][6][v], acc[h][3][v], acc[h][7][v]};
                    }
                }
            }
            lds_barrier();
            FloatsOf<OWN> qv[RSUMS][WAVES];
            float xv[RSUMS][WAVES];
#pragma unroll
            for (int i = 0; i < RSUMS; i++) {
                const int row = QUADS ? own_row + 4 * i : i;
                const int at = QUADS ? 4 * red_piece(own_piece)
                                     : (BY_COLUMNS ? tid / 16 * 8 + tid % 8 : 4 * red_piece(tid / 16 * 2 + tid / 4 % 2) + tid % 4);
#pragma unroll
                for (int wv = 0; wv < WAVES; wv++) {
                    qv[i][wv] = *reinterpret_cast<const FloatsOf<OWN>*>(&red[wv][QUADS ? own_half : tid / 8 % 2][row][at]);
                    xv[i][wv] = xs_red[wv][rd * RROWS + row];
                }
            }
            if constexpr (SHORT_OF_REGISTERS) {
#pragma unroll
                for (int wv = 0; wv < WAVES; wv++) {
                    asm volatile("" : "+v"(z_word[wv]));
                    convert_scales(wv);
                }
            }
#pragma unroll
            for (int i = 0; i < RSUMS; i++) {
#pragma unroll
                for (int j = 0; j < OWN; j++) {
                    float total = 0.0f;
#pragma unroll
                    for (int wv = 0; wv < WAVES; wv++) {
                        total += FINE ? qv[i][wv][j] : sc[wv][j] * __builtin_fmaf(-zc[wv][j], xv[i][wv], qv[i][wv][j]);
                    }
                    float& sum = psum[rd * RSUMS + i].v[j];
                    sum = WALK && block > 0 ? sum + total : total;
                }
            }
        }
        if constexpr (WALK && !AHEAD) load_next();
        if constexpr (WALK && !STAGED) {  // the next block's operands are out: what its sums need comes last, where registers are free
            if (block + 1 < blocks) load_scales();
        }
    }

#if defined(KX_ABLATE) && KX_ABLATE >= 1 && KX_ABLATE <= 3
    if (ktiles > 1) {  // profiling build: no exchange - every workgroup leaves its partial sums and is done
        if (own_col < N) partials[static_cast<size_t>(kt) * M * N + own_col] = psum[0][0];
        return;
    }
#endif
    // ---- the finished rows, by slices: activation row m of half a tile (128 columns, one head of a q|k|v row);
    // a lane holds columns lane and lane + 64 of the half ----
    struct Operands {
        uint16_t a, b, c, d;
        int pos;
    };
    auto request = [&](int m, int half) {
        Operands o{};
        const int ca = ct * kTileCols + half * kSliceCols + lane;
        if constexpr (EPI == kEpiResidual) {
            const size_t row = static_cast<size_t>(m) * N;
            o.a = res.in[row + (ca < N ? ca : N - 1)];
            o.b = res.in[row + (ca + kWave < N ? ca + kWave : N - 1)];
        }
        if constexpr (EPI == kEpiQkRope) {
            // both gains, then a select of values (a select between pointers ends up as a table in private memory)
            o.pos = rope.pos[m];
            o.a = rope.q_gain[lane];
            o.b = rope.q_gain[lane + 64];
            o.c = rope.k_gain[lane];
            o.d = rope.k_gain[lane + 64];
        }
        return o;
    };
    auto finish = [&](int m, int half, float a, float b, const Operands& o) {
        const int ca = ct * kTileCols + half * kSliceCols + lane;
        const int cb = ca + kWave;
        // the projection's output is a bf16 tensor, whatever follows
        const uint16_t oa = f32_to_bf16(a), ob = f32_to_bf16(b);
        if constexpr (EPI == kEpiStore) {
            uint16_t* row = y + static_cast<size_t>(m) * N;
            if (ca < N) row[ca] = oa;
            if (cb < N) row[cb] = ob;
        } else if constexpr (EPI == kEpiResidual) {
            const uint16_t ra = f32_to_bf16(bf16_to_f32(o.a) + bf16_to_f32(oa));
            const uint16_t rb = f32_to_bf16(bf16_to_f32(o.b) + bf16_to_f32(ob));
            uint16_t* row = res.out + static_cast<size_t>(m) * N;
            if (ca < N) row[ca] = ra;
            if (cb < N) row[cb] = rb;
            const float va = ca < N ? bf16_to_f32(ra) : 0.0f, vb = cb < N ? bf16_to_f32(rb) : 0.0f;
            const float qa = wave_sum(va * va), qb = wave_sum(vb * vb);  // quarters of the tile; past N: 0
            if (lane == 0) {
                float* dst = res.sumsq + (static_cast<size_t>(m) * grid.coltiles + ct) * (kTileCols / kWave) + 2 * half;
                dst[0] = qa;
                dst[1] = qb;
            }
        } else {
            const int head = ct * (kTileCols / kHeadDim) + half;
            const bool q_head = head < rope.n_q;
            RopeTarget t = rope;
            t.q_out += static_cast<size_t>(m) * rope.n_q * kHeadDim;
            t.k_cache += static_cast<size_t>(m) * cache_stride;
            t.v_cache += static_cast<size_t>(m) * cache_stride;
            qk_norm_rope_head_with(oa, ob, head, lane, t, o.pos, q_head ? o.a : o.c, q_head ? o.b : o.d);
        }
    };
    static_assert(THREADS == kTileCols && kSliceCols == kHeadDim, "one thread per tile column, a slice is a head");
    float* s_sum = &red[0][0][0][0];  // a tile of finished rows, where one workgroup holds them all: the reduction buffer, free again
    static_assert(WAVES * 2 * RROWS * kHalfCols >= ROWS * kTileCols, "the reduction buffer holds a tile of finished rows");
    // Wave w finishes slices w, w + WAVES, ...; what they need besides the sums is asked for together, ahead of the barrier.
    constexpr int PER_WAVE = (2 * ROWS + WAVES - 1) / WAVES;
    Operands early[PER_WAVE];
    auto request_all = [&] {
        if constexpr (EPI != kEpiStore) {
#pragma unroll
            for (int j = 0; j < PER_WAVE; j++) {
                const int i = min(wave + j * WAVES, 2 * M - 1);
                early[j] = request(i >> 1, i & 1);
            }
        }
    };
    auto finish_from_lds = [&] {
        __syncthreads();
#pragma unroll
        for (int j = 0; j < PER_WAVE; j++) {
            const int i = wave + j * WAVES;
            const float* src = s_sum + (i >> 1) * kTileCols + (i & 1) * kSliceCols + lane;
            if (i < 2 * M) finish(i >> 1, i & 1, src[0], src[kWave], early[j]);
        }
    };
    const auto row_of = [&](int i) { return QUADS ? own_row + 4 * i : i; };  // row of psum[i]
    constexpr bool STORES_FEW = ROWS <= 2 && PRO != kProPreNorm && EPI == kEpiStore;
    if (ktiles == 1) {
        if constexpr (EPI == kEpiStore) {  // a thread stores its own columns: nothing to hand over
#pragma unroll
            for (int i = 0; i < PSUMS; i++) {
                const int r = row_of(i);
                if (r < M && own_col < N) {
                    uint16_t* dst = y + static_cast<size_t>(r) * N + own_col;
                    if constexpr (QUADS) {
                        *reinterpret_cast<u32x2*>(dst) = u32x2{f32x2_to_bf16x2(psum[i][0], psum[i][1]), f32x2_to_bf16x2(psum[i][2], psum[i][3])};
                    } else {
                        *dst = f32_to_bf16(psum[i][0]);
                    }
                }
            }
        } else {
            request_all();
            __syncthreads();
#pragma unroll
            for (int i = 0; i < PSUMS; i++) *reinterpret_cast<FloatsOf<OWN>*>(&s_sum[row_of(i) * kTileCols + own_col - ct * kTileCols]) = psum[i];
            finish_from_lds();
        }
        if constexpr (!STORES_FEW) return;
    }
    // One and two stored rows: a test of its own rather than the other branch of the one above, whose values the compiler would
    // carry through the exchange.  us per launch at M = 2, branch -> test: 12288 -> 4096 11.28 -> 11.02, behind SwiGLU 11.30 -> 11.01,
    // 3072 -> 1024 with groups of 32 6.43 -> 6.26.  More rows lose by it (1536 -> 4096 at M = 16 7.45 -> 7.65).
    if constexpr (STORES_FEW) {
        int tiles = ktiles;
        asm volatile("" : "+s"(tiles));
        if (tiles == 1) return;
    }
    if constexpr (ROWS <= 2) {
        float own[ROWS], sum[ROWS];
#pragma unroll
        for (int r = 0; r < ROWS; r++) own[r] = psum[r][0];
        if constexpr (EPI == kEpiQkRope) {
            if (!splitk_exchange_sum<ROWS>(own, sum, 0, M, N, ct, kt, ktiles, ct, partials, counters, s_word)) return;
            request_all();
#pragma unroll
            for (int r = 0; r < ROWS; r++) s_sum[r * kTileCols + tid] = sum[r];
            finish_from_lds();
        } else {
            // every wave of 64 columns finishes for itself: the epilogue needs nothing from the other waves
            uint16_t rin[ROWS];
            if constexpr (EPI == kEpiResidual) {
#pragma unroll
                for (int r = 0; r < ROWS; r++) rin[r] = res.in[static_cast<size_t>(r < M ? r : M - 1) * N + (own_col < N ? own_col : N - 1)];
            }
            if (!splitk_exchange_sum_per_wave_rows<ROWS>(own, sum, M, N, ct, kt, ktiles, partials, counters)) return;
            const bool col_ok = own_col < N;
#pragma unroll
            for (int r = 0; r < ROWS; r++) {
                const uint16_t o = f32_to_bf16(sum[r]);
                if constexpr (EPI == kEpiStore) {
                    if (col_ok && r < M) y[static_cast<size_t>(r) * N + own_col] = o;
                } else {
                    const uint16_t rbits = f32_to_bf16(bf16_to_f32(rin[r]) + bf16_to_f32(o));
                    if (col_ok && r < M) res.out[static_cast<size_t>(r) * N + own_col] = rbits;
                    const float rv = col_ok ? bf16_to_f32(rbits) : 0.0f;
                    const float q = wave_sum(rv * rv);
                    if (lane == 0 && r < M) res.sumsq[(static_cast<size_t>(r) * grid.coltiles + ct) * (kTileCols / kWave) + wave] = q;
                }
            }
        }
    } else {
        // this workgroup's partial sums, sixteen bytes per lane and a row's 128 columns of a word half side by side
        const __amdgpu_buffer_rsrc_t rsrc = partials_buffer(partials, static_cast<size_t>(ktiles) * M * N);
#pragma unroll
        for (int i = 0; i < PSUMS; i++) {
            const int r = row_of(i);
            if (r < M && own_col < N) {
                if constexpr (!QUADS) store_agent(partials + (static_cast<size_t>(kt) * M + r) * N + own_col, psum[i][0]);
                else store_partial_quad(rsrc, partial_column(own_col, N) + r * N, static_cast<uint32_t>(kt) * M * static_cast<uint32_t>(N), psum[i].v);
            }
        }
        if constexpr (ROWS >= 8) {
            if (TRIO || grid.sliced) {  // every TRIO plan is
                splitk_exchange_sliced<ROWS>(M, N, ct, kt, ktiles, partials, counters, s_word, grid.wait_ticks, request,
                                             finish);
                return;
            }
        }
        // the wide read-back hands out two columns and half of the rows per thread
        constexpr int HALF = ROWS / 2;
        float lo[HALF], hi[HALF];
        if (!splitk_exchange_sum_wide<ROWS, RUNS>(lo, hi, M, N, ct, ktiles, partials, counters, s_word, request_all, grid.run)) {
            return;
        }
        // Where they go is worked out anew: kept over the read-back it took the registers of sixteen rows past three workgroups
        // per compute unit (185 with two steps per wave).  us per launch, kept, at two workgroups -> anew, groups of 64, M = 9 / 16:
        // 2048 -> 24576 behind SwiGLU 14.9 / 15.5 -> 13.8 / 14.3, behind a norm 15.2 / 16.0 -> 13.9 / 14.6.
        int thread = tid;
        asm volatile("" : "+v"(thread));
        const int row0 = (thread / (kTileCols / 2)) * HALF;
        const int pair = 2 * (thread % (kTileCols / 2));
        if constexpr (EPI == kEpiStore) {
#pragma unroll
            for (int i = 0; i < HALF; i++) {
                if (row0 + i < M && ct * kTileCols + pair < N) {
                    *reinterpret_cast<uint32_t*>(y + static_cast<size_t>(row0 + i) * N + ct * kTileCols + pair) = f32x2_to_bf16x2(lo[i], hi[i]);
                }
            }
        } else {
#pragma unroll
            for (int i = 0; i < HALF; i++) *reinterpret_cast<f32x2*>(&s_sum[(row0 + i) * kTileCols + pair]) = f32x2{lo[i], hi[i]};
            finish_from_lds();
        }
    }
}

template <int WAVES, int KS, int MC, int ROUNDS, int PRO = kProNone, int EPI = kEpiStore, bool LONE = false, bool WALK = false, bool FINE = false,
          bool TRIO = false>
inline void launch_awq_gemv_mfma(const uint16_t* x, const int32_t* qweight, const uint16_t* scales,
                                 const int32_t* qzeros, uint16_t* y, float* partials, uint32_t* counters,
                                 int M, int K, int N, const MfmaGrid& split,
                                 hipStream_t stream, const FusedInput& fi = FusedInput{},
                                 const ResidualTarget& res = ResidualTarget{}, const RopeTarget& rope = RopeTarget{},
                                 size_t cache_stride = 0) {

    const dim3 grid(split.side, split.ktiles, split.coltiles / split.side);
    dim3 block(WAVES * kWave, 1, 1);
    MfmaGrid ordered = split;
    const bool by_number = split.sliced ? split.run == 1 && together_by_number(M, KS, N, split.coltiles, split.ktiles)
                                        : alone_by_number(M, KS, split.coltiles, split.ktiles);
    if (!by_number) ordered.order = packed_tile_order(qweight, N, split.coltiles, split.ktiles);
    hipLaunchKernelGGL((awq_gemv_mfma_kernel<WAVES, KS, MC, ROUNDS, PRO, EPI, LONE, WALK, FINE, TRIO>), grid, block, 0, stream, x,
                       reinterpret_cast<const uint32_t*>(qweight), scales,
                       reinterpret_cast<const uint32_t*>(qzeros), y, partials, counters, M, K, N,
                       ordered, fi, res, rope, cache_stride);
}

}  // namespace kx

#endif  // KX_AWQ_GEMV_MFMA_KERNEL_H
