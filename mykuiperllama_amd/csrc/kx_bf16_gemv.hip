// BF16 GEMV fallback for gfx950: y[m,n] = sum_k x[m,k] * W[n,k], W bf16 row-major [N, K].
//
// One or two activation rows: one wave per output row, the 64 lanes walk the row in 16-byte pieces
// (eight bf16 each), pairs along K go through the packed bf16 dot instruction with an fp32
// accumulator, and the lanes meet in a wave-wide sum at the end.  Rows are contiguous, so every load
// is a full 1 KiB per wave.  Several rows: matrix cores, the activations held in registers while a workgroup walks over
// blocks of output rows (third kernel below), or, for K > 8192, sixteen output rows per workgroup (second kernel).
#include <type_traits>

#include "kx_common.h"
#include "kx_internal.h"

namespace kx {
namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float dot2_bf16(uint32_t a, uint32_t b, float c) {
    bf16x2 va, vb;
    __builtin_memcpy(&va, &a, 4);
    __builtin_memcpy(&vb, &b, 4);
    return __builtin_amdgcn_fdot2_f32_bf16(va, vb, c, false);
}

constexpr int kRowsPerBlock = 4;  // one wave each
// 16-byte weight loads in flight per lane: a row of 4096 in one sweep (four measured slower for
// every M, also where several activation rows compete for the registers)
constexpr int kUnroll = 8;

template <int MB>
__global__ __launch_bounds__(kRowsPerBlock * kWave) void bf16_gemv_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, uint16_t* __restrict__ y,
    int M, int K, int N, int m0) {
    const int lane = threadIdx.x % kWave;
    const int n = blockIdx.x * kRowsPerBlock + threadIdx.x / kWave;
    // A wave past the last row works on the last row again and stores nothing: no wave leaves
    // early, no load sits under a condition.
    const int n_ld = n < N ? n : N - 1;
    const int chunks = K >> 3;  // 16-byte pieces per row
    const u32x4* wrow = reinterpret_cast<const u32x4*>(w + static_cast<size_t>(n_ld) * K);
    const uint4* xrow[MB];
#pragma unroll
    for (int m = 0; m < MB; m++) {
        const int mr = m0 + m < M ? m0 + m : M - 1;  // rows past M repeat the last one, never stored
        xrow[m] = reinterpret_cast<const uint4*>(x + static_cast<size_t>(mr) * K);
    }

    float acc[MB];
#pragma unroll
    for (int m = 0; m < MB; m++) acc[m] = 0.0f;

    // Full sweeps of kUnroll pieces per lane, then the rest of the row two pieces per lane at a time
    // (K = 5120: one full sweep and one short one).  Inside a sweep the loads are straight-line code
    // and all in flight together; a load under a condition becomes a branch with a full wait behind it.
    auto consume = [&](const u32x4& wv, int c, bool live) {
        const uint32_t w0 = live ? wv.x : 0u, w1 = live ? wv.y : 0u;
        const uint32_t w2 = live ? wv.z : 0u, w3 = live ? wv.w : 0u;
#pragma unroll
        for (int m = 0; m < MB; m++) {
            const uint4 xv = xrow[m][c];
            acc[m] = dot2_bf16(w0, xv.x, acc[m]);
            acc[m] = dot2_bf16(w1, xv.y, acc[m]);
            acc[m] = dot2_bf16(w2, xv.z, acc[m]);
            acc[m] = dot2_bf16(w3, xv.w, acc[m]);
        }
    };
    int base = 0;  // first piece of the sweep, the same in every lane
    for (; base + kWave * kUnroll <= chunks; base += kWave * kUnroll) {
        u32x4 wv[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; u++) wv[u] = __builtin_nontemporal_load(wrow + base + lane + u * kWave);
        __builtin_amdgcn_sched_barrier(0);  // every weight load is out before the first is waited for
#pragma unroll
        for (int u = 0; u < kUnroll; u++) consume(wv[u], base + lane + u * kWave, true);
    }
    constexpr int kTail = 2;
    for (; base < chunks; base += kWave * kTail) {
        // clamped addresses, masked weights
        u32x4 wv[kTail];
#pragma unroll
        for (int u = 0; u < kTail; u++) {
            const int c = base + lane + u * kWave;
            wv[u] = __builtin_nontemporal_load(wrow + (c < chunks ? c : chunks - 1));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < kTail; u++) {
            const int c = base + lane + u * kWave;
            consume(wv[u], c < chunks ? c : chunks - 1, c < chunks);
        }
    }
#pragma unroll
    for (int m = 0; m < MB; m++) acc[m] = wave_sum(acc[m]);
    if (lane == 0 && n < N) {
#pragma unroll
        for (int m = 0; m < MB; m++) {
            // a plain store: one wave owns one column, and two-byte write-through stores from 150 000 waves cost
            // the lm_head launch 8 us
            if (m0 + m < M) y[static_cast<size_t>(m0 + m) * N + n] = f32_to_bf16(acc[m]);
        }
    }
}

// Three to sixteen activation rows, K > 8192 (up to there bf16_gemv_held_kernel serves): matrix cores, one pass over W
// whatever M is.
// v_mfma_f32_16x16x32_bf16 with A = the activations (row m = lane % 16, zero rows past M) and
// B = sixteen rows of W (column n = lane % 16): lane (c, b) supplies x[c][32 s + 8 b .. + 7] and
// W[n0 + c][32 s + 8 b .. + 7], sixteen contiguous bytes each, and receives y[4 b + v][n0 + c].
// A workgroup owns kMfmaBlocks blocks of sixteen output columns, which share every A operand.  One block
// with eight steps in flight serves up to eight rows (12288 -> 151936 925 / 930 / 1004 us at M = 3 / 5 / 8, 4.0 to 3.7 TB/s;
// 12288 -> 4096 27.8 / 29.2 / 32.3); from nine rows on four blocks with four steps in flight each (924 / 947 us at M = 9 /
// 16; 74 / 80), so that the activation rows come out of L2 once per 64 columns instead of once per 16 - at sixteen rows they
// are as many bytes as the sixteen rows of W they meet, and with one block the L2 traffic for x equals the HBM traffic for
// W (4096 -> 151936, one block against four: 370 / 299 us at M = 16, 270 / 297 at M = 3).  Its four waves take the
// 32-element steps of K in turn (step s goes to wave s % 4; runs of consecutive steps per wave measured
// slower) in sweeps of UNROLL steps with all loads of a sweep in flight together, and meet in LDS.  Addresses are clamped, what lies past K or M is zeroed
// in both operands; per output the additions run in the same order whatever kMfmaBlocks is.
constexpr int kMfmaWaves = 4;

template <int kMfmaBlocks, int kMfmaUnroll>
__global__ __launch_bounds__(kMfmaWaves * kWave) void bf16_gemv_mfma_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, uint16_t* __restrict__ y, int M, int K, int N) {
    __shared__ float red[kMfmaWaves][kMfmaBlocks][4][kWave];
    const int lane = threadIdx.x % kWave;
    const int wave = threadIdx.x / kWave;
    const int c = lane % 16;
    const int b = lane / 16;
    const int n0 = blockIdx.x * 16 * kMfmaBlocks;
    const int m_ld = c < M ? c : M - 1;
    const uint16_t* wrow[kMfmaBlocks];
#pragma unroll
    for (int j = 0; j < kMfmaBlocks; j++) {
        const int n = n0 + 16 * j + c;
        wrow[j] = w + static_cast<size_t>(n < N ? n : N - 1) * K;
    }
    const uint16_t* xrow = x + static_cast<size_t>(m_ld) * K;
    const bool row_live = c < M;
    const int k_last = K - 8;  // K is a multiple of eight

    f32x4v acc[kMfmaBlocks];
#pragma unroll
    for (int j = 0; j < kMfmaBlocks; j++) acc[j] = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
    constexpr int kSweep = 32 * kMfmaWaves * kMfmaUnroll;  // elements of K a workgroup covers per sweep
    for (int k0 = 32 * wave; k0 < K; k0 += kSweep) {
        u32x4 wv[kMfmaUnroll][kMfmaBlocks], xv[kMfmaUnroll];
#pragma unroll
        for (int u = 0; u < kMfmaUnroll; u++) {
            const int k = k0 + 32 * kMfmaWaves * u + 8 * b;
            xv[u] = *reinterpret_cast<const u32x4*>(xrow + (k < K ? k : k_last));
        }
#pragma unroll
        for (int u = 0; u < kMfmaUnroll; u++) {
            const int k = k0 + 32 * kMfmaWaves * u + 8 * b;
#pragma unroll
            for (int j = 0; j < kMfmaBlocks; j++) {
                wv[u][j] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wrow[j] + (k < K ? k : k_last)));
            }
        }
        __builtin_amdgcn_sched_barrier(0);  // every load of the sweep is out before the first is waited for
#pragma unroll
        for (int u = 0; u < kMfmaUnroll; u++) {
            const bool live = k0 + 32 * kMfmaWaves * u + 8 * b < K;
            const bool a_live = live && row_live;
            const bf16x8 a_op = as_bf16x8(a_live ? xv[u].x : 0u, a_live ? xv[u].y : 0u, a_live ? xv[u].z : 0u,
                                          a_live ? xv[u].w : 0u);
#pragma unroll
            for (int j = 0; j < kMfmaBlocks; j++) {
                const bf16x8 b_op = as_bf16x8(live ? wv[u][j].x : 0u, live ? wv[u][j].y : 0u, live ? wv[u][j].z : 0u,
                                              live ? wv[u][j].w : 0u);
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_op, b_op, acc[j], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < kMfmaBlocks; j++) {
#pragma unroll
        for (int v = 0; v < 4; v++) red[wave][j][v][lane] = acc[j][v];
    }
    __syncthreads();
    // wave j finishes block j
    static_assert(kMfmaBlocks <= kMfmaWaves, "one wave per block of sixteen columns in the final sum");
    const int n = n0 + 16 * wave + c;
    if (wave < kMfmaBlocks && n < N) {
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int m = 4 * b + v;
            const float sum = (red[0][wave][v][lane] + red[1][wave][v][lane]) + (red[2][wave][v][lane] + red[3][wave][v][lane]);
            if (m < M) y[static_cast<size_t>(m) * N + n] = f32_to_bf16(sum);
        }
    }
}

// Two to sixteen activation rows, K <= 8192: one workgroup per compute unit walks over blocks of sixteen output columns, and
// PARTS of its waves split K between them (the others take further blocks side by side).  What bounded the kernel above was
// not W but everything round it: the activation rows came out of L2 anew for every 64 columns, and an MFMA operand fetched
// straight from memory asks for 64 bytes of sixteen rows at a time, which the memory system answers at three quarters of its
// rate.  Here the A operands of a wave's part of K stay in registers for the life of the workgroup, and W goes through LDS: a
// unit is UNIT elements of the block's sixteen rows, loaded straight into the wave's own ring, so that no barrier and no
// register stands between the stream and the MFMAs and 128 KB per compute unit are in flight.  (Eight waves and units of 512
// leave a wave one slot: there it reads its unit into registers, 64 of them, before it asks for the next, and only the other waves'
// units are in flight meanwhile.)  The waves of a block meet in LDS, two buffers in turn, one barrier per block that leaves loads
// alone.  K is cut into whole units, as evenly as they go: a part has UNITS of them or one less.
// A row of a unit is stored with its 16-byte pieces permuted by the low bits of the row (the lane that loads piece j of
// row r fetches piece j ^ (r & 7)), so that the sixteen rows that an operand read touches lie in different banks.
// Where rows start on memory lines, units of 128 elements, 256 bytes of a row, which are two lines; rows that do not start on
// lines would have such a piece touch three, and longer units cost them less (held_form).  us per launch at M = 3 / 8 / 16, eight
// waves of equal parts of K rounded up to 1024 -> now: rows on lines 151936 x 4096 181 / 187 / 202 -> 180 / 182 / 189, 151936 x 5120
// 222 / 235 / 252 -> 221 / 224 / 233, 32000 x 768 12.3 / 12.6 / 12.9 -> 10.4 / 10.6 / 11.3; others 144453 x 3144 165 / 178 / 194 -> 136 /
// 139 / 150, 101754 x 2336 84 / 88 / 98 -> 74 / 75 / 79, 79438 x 1240 44.5 / 45.9 / 49.9 -> 35.8 / 37.2 / 38.2, 69572 x 4688 114 / 118 /
// 125 -> 103 / 106 / 109 (W alone at the read rate of a large buffer: 173, 216, 6.8; 126, 66, 27, 91).  Cached loads instead of streaming ones lose 10 % on lines and win 2 % off them.
constexpr int kRingBytes = 131072;

template <int WAVES, int UNIT, int UNITS, int PARTS, bool RUNS>
__global__ __launch_bounds__(WAVES * kWave, WAVES / 4) void bf16_gemv_held_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, uint16_t* __restrict__ y, int M, int K, int N, int blocks) {
    constexpr int SIDE = WAVES / PARTS;          // blocks a workgroup works on side by side
    constexpr int STEPS = UNIT / 32;
    constexpr int PIECES = UNIT / 8;             // 16-byte pieces of a row of a unit
    constexpr int ROWS = kWave / PIECES;         // rows a load brings
    constexpr int LOADS = 16 / ROWS;
    constexpr int RING = kRingBytes / WAVES / (32 * UNIT);
    __shared__ __attribute__((aligned(1024))) char ring[WAVES][RING][32 * UNIT];
    __shared__ __attribute__((aligned(16))) float red[2][WAVES][4][kWave];
    const int tid = threadIdx.x;
    const int lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int part = wave % PARTS;
    const int c = lane % 16;
    const int b = lane / 16;
    const int units = (K + UNIT - 1) / UNIT;
    const int unit0 = part * units / PARTS;                // the wave's first unit of K
    const int mine = (part + 1) * units / PARTS - unit0;   // UNITS, or one less
    const int kw = UNIT * unit0;
    // RUNS: a workgroup takes four blocks in a row as long as there are whole rounds of that, so that the 64 outputs of a line of
    // y come from one XCD; the rest, and without RUNS all, go round one by one.
    constexpr int RUN = RUNS && SIDE < 4 ? 4 / SIDE : 1;
    const int wgs = gridDim.x, wg = blockIdx.x;
    const int in_runs = (blocks + SIDE - 1) / SIDE / (RUN * wgs) * RUN;
    auto block_of = [&](int turn) { return SIDE * (turn < in_runs ? turn / RUN * RUN * wgs + wg * RUN + turn % RUN : turn * wgs + wg); };

    bf16x8 held[UNITS][STEPS];
    const uint16_t* xrow = x + static_cast<size_t>(min(c, M - 1)) * K;
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
#pragma unroll
        for (int q = 0; q < STEPS; q++) {
            const int k = kw + UNIT * u + 32 * q + 8 * b;
            const bool in = k < K;
            const u32x4 v = *reinterpret_cast<const u32x4*>(xrow + (in ? k : 0));
            const bool live = in && c < M;
            held[u][q] = as_bf16x8(live ? v.x : 0u, live ? v.y : 0u, live ? v.z : 0u, live ? v.w : 0u);
        }
    }

    // Loads unit u of a block into a ring slot: load i brings rows ROWS * i + lane / PIECES.
    auto fetch = [&](int block, int u, int slot) {
#pragma unroll
        for (int i = 0; i < LOADS; i++) {
            const int r = ROWS * i + lane / PIECES;
            const int k = kw + UNIT * u + 8 * (lane % PIECES ^ (r & 7));
            const uint16_t* src = w + static_cast<size_t>(min(16 * block + r, N - 1)) * K + min(k, K - 8);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                             (__attribute__((address_space(3))) void*)(&ring[wave][slot][i * 1024]), 16, 0, 2);
        }
    };
    // Where the lane finds its operand of step q: row c, piece 4 q + b; steps 2 and 3 lie 128 bytes behind 0 and 1.
    const uint32_t ring0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
        (__attribute__((address_space(3))) char*)(&ring[wave][0][0])));
    const uint32_t at0 = ring0 + c * (2 * UNIT) + ((b ^ (c & 7)) * 16);
    const uint32_t at1 = ring0 + c * (2 * UNIT) + (((4 + b) ^ (c & 7)) * 16);

    // the unit that is fetched next, and how many are on their way or waiting in the ring
    const int side_of_wave = wave / PARTS;
    int fetch_turn = 0, fetch_block = block_of(0) + side_of_wave, fetch_unit = 0, ahead = 0;
    auto fetch_next = [&](int slot) {
        if (mine == 0 || fetch_block >= blocks) return;
        fetch(fetch_block, fetch_unit, slot);
        ahead++;
        if (++fetch_unit == mine) {
            fetch_unit = 0;
            fetch_block = block_of(++fetch_turn) + side_of_wave;
        }
    };
#pragma unroll
    for (int j = 0; j < RING; j++) fetch_next(j);
    int slot = 0;
    for (int turn = 0, row; row = block_of(turn), row < blocks; turn++) {
        const int block = row + side_of_wave;
        f32x4v acc[2];
        acc[0] = acc[1] = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
        if (SIDE == 1 || block < blocks) {
#pragma unroll
            for (int u = 0; u < UNITS; u++) {
                if (u < mine) {
                    // Loads return in order: with the ring full, RING - 1 units may still be on their way when this one has arrived.
                    if (ahead == RING) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS * (RING - 1)) : "memory");
                    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    u32x4 v[STEPS];
                    const uint32_t s0 = at0 + slot * (32 * UNIT), s1 = at1 + slot * (32 * UNIT);
                    // in assembly, because the compiler would wait for every load in flight ahead of a read of the ring
#pragma unroll
                    for (int q = 0; q < STEPS; q += 4) {
                        asm volatile("ds_read_b128 %0, %4 offset:%6\n\tds_read_b128 %1, %5 offset:%6\n\tds_read_b128 %2, %4 offset:%7\n\t"
                                     "ds_read_b128 %3, %5 offset:%7\n\ts_waitcnt lgkmcnt(0)"
                                     : "=&v"(v[q]), "=&v"(v[q + 1]), "=&v"(v[q + 2]), "=&v"(v[q + 3])
                                     : "v"(s0), "v"(s1), "n"(64 * q), "n"(64 * q + 128)
                                     : "memory");
                    }
                    ahead--;
                    fetch_next(slot);
                    if (kw + UNIT * u + UNIT > K) {  // the last unit of a K that is no multiple of a unit
#pragma unroll
                        for (int q = 0; q < STEPS; q++) {
                            const bool live = kw + UNIT * u + 32 * q + 8 * b < K;
                            v[q] = u32x4{live ? v[q].x : 0u, live ? v[q].y : 0u, live ? v[q].z : 0u, live ? v[q].w : 0u};
                        }
                    }
#pragma unroll
                    for (int q = 0; q < STEPS; q++) {
                        acc[q & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(held[u][q], as_bf16x8(v[q].x, v[q].y, v[q].z, v[q].w), acc[q & 1], 0, 0, 0);
                    }
                    slot = (slot + 1) % RING;
                }
            }
        }
        if constexpr (PARTS == 1) {
            const int n = 16 * block + c;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int m = 4 * b + v;
                if (m < M && n < N && block < blocks) y[static_cast<size_t>(m) * N + n] = f32_to_bf16(acc[0][v] + acc[1][v]);
            }
            continue;
        }
#pragma unroll
        for (int v = 0; v < 4; v++) red[turn % 2][wave][v][lane] = acc[0][v] + acc[1][v];
        lds_barrier();
        // thread (v, lane): row 4 (lane / 16) + v of column lane % 16
#pragma unroll
        for (int e = 0; e < SIDE; e += WAVES / 4) {
            const int side = e + tid / (4 * kWave);
            if (SIDE % (WAVES / 4) != 0 && side >= SIDE) break;
            const float* src = &red[turn % 2][side * PARTS][0][0] + tid % (4 * kWave);
            float sum[PARTS];
#pragma unroll
            for (int u = 0; u < PARTS; u++) sum[u] = src[u * 4 * kWave];
#pragma unroll
            for (int d = 1; d < PARTS; d *= 2) {
#pragma unroll
                for (int u = 0; u < PARTS; u += 2 * d) sum[u] += sum[u + d];
            }
            const int m = 4 * b + wave % 4;
            const int n = 16 * (row + side) + c;
            if (m < M && n < N) y[static_cast<size_t>(m) * N + n] = f32_to_bf16(sum[0]);
        }
    }
}

constexpr int kHeldMostK = 8192;
constexpr int kComputeUnits = 256;

// Which form of the kernel a launch takes.
struct HeldForm {
    int waves, unit, parts;
    int units;  // of the fullest part
    bool runs;
};

// Runs of four blocks pay with the rows of y that are written and the rounds of blocks, and cost a little with few of either.  Time in
// runs over one by one, M = 3 / 5 / 8 / 16, at 6, 12, 16 and 37 rounds: K = 3072 1.03 / 1.03 / 1.02 / 1.01, 1.04 / 1.03 / 1.02 / 1.00, 1.03 / 1.02 /
// 1.00 / 0.98 and 1.02 / 1.00 / 0.97 / 0.93; 6144 1.06 / 1.05 / 1.04 / 1.03, 1.03 / 1.02 / 1.00 / 0.99, 1.02 / 0.98 / 0.99 / 0.98 and 1.01 / 0.98 / 0.97 /
// 0.95; 3592 alike.  Rows of 4 KB, where the blocks of a round ask the same memory channels, gain from few rounds on (K = 2048 at four:
// 0.93 / 0.94 / 0.93 / 0.92).  Past K = 6144 they are lost (40000 x 8192 at M = 8 / 16 110 / 114 us -> 115 / 118); four waves gain 1 to 2 % from
// eight rows on and lose nothing before.
//
// On lines the fewest parts whose A operands fit the registers and whose last round of blocks is not emptier for it by more than it
// gains, a barrier for every PARTS-th of the blocks: time with two parts over four, M = 3 / 8 / 16, at 8 and 16 rounds, K = 1024 1.00 / 1.02 / 1.05
// and 0.95 / 0.97 / 0.98, 1280 0.96 / 1.00 / 1.04 and 0.96 / 0.98 / 1.00, 1536 1.02 / 1.06 / 1.08 and 1.01 / 1.02 / 1.04; four over eight 2048 0.94 /
// 0.95 / 1.00 and 0.93 / 0.95 / 0.98, 2560 0.99 / 0.98 / 1.02 and 0.97 / 0.98 / 1.00, 3072 1.02 / 1.03 / 1.05 and 1.00 / 1.01 / 1.05, 4096 1.01 / 1.03 /
// 1.02 and 0.99 / 1.01 / 1.02, at 37 rounds 0.96 / 1.02 / 1.03.  Few rounds leave
// compute units idle: up to four, all waves split K (4764 x 4032 at M = 16 17.6 us with four parts, 13.1 with eight).
// Off lines eight waves that all split K, in units of the length that gives the fullest wave the fewest elements (the longer one of
// two, with fewer of its pieces across a line), are ahead of four waves and units of 512.  us per launch, four waves -> eight,
// M = 3 / 14: units of 128 up to K = 1024 4010 x 776 4.06 / 4.45 -> 3.62 / 3.81, 17000 x 904 10.4 / 11.3 -> 9.8 / 10.4, 66000 x 904 27.8 /
// 29.9 -> 28.1 / 29.6 (left out from 5120 blocks on: 120000 x 904 39.6 / 41.0 -> 47.4 / 47.5, there four, two or one part: 67290 x 912 at M = 3
// 30.2 / 27.1 / 25.8); of 256 where they leave fewer than 512
// 4100 x 1400 5.46 / 6.20 -> 5.10 / 5.75, 120000 x 1400 60.1 / 62.3 -> 57.8 / 57.9, 5500 x 5000 16.6 / 16.8 -> 15.8 / 16.9 (left out past
// K = 4096 and four rounds: 17000 x 4504 31.4 / 33.2 -> 31.4 / 33.4, 120000 x 4504 177 / 178 -> 185 / 187); of 512 otherwise 4100 x 2200
// 8.85 / 10.2 -> 6.86 / 8.05, 120000 x 3000 124 / 124 -> 112 / 113, 4100 x 7800 20.4 / 22.9 -> 17.6 / 19.9, 33000 x 7800 89.3 / 93.8 -> 88.6 / 92.8.
HeldForm held_form(bool whole_lines, int M, int K, int N) {
    const int blocks = (N + 15) / 16;
    const auto fullest = [&](int unit, int parts) { return ((K + unit - 1) / unit + parts - 1) / parts; };
    const auto form = [&](int waves, int unit, int parts) {
        const bool many = waves == 4 || (whole_lines && K == 2048) ? M >= 6 : M >= 5 && static_cast<long>(M) * blocks >= 150 * kComputeUnits;
        return HeldForm{waves, unit, parts, fullest(unit, parts), K <= 6144 && many};
    };
    if (!whole_lines) {
        if (K <= 1024) {
            if (blocks < 20 * kComputeUnits) return form(8, 128, 8);
        } else if (256 * fullest(256, 8) >= 512 * fullest(512, 8)) {
            return form(8, 512, 8);
        } else if (K <= 4096 || blocks <= 4 * kComputeUnits) {
            return form(8, 256, 8);
        }
    }
    const int waves = whole_lines ? 8 : 4;
    int least = K <= 1024 ? 1 : 4;
    if (whole_lines) {
        const bool four = K <= 2560 || (K <= 4096 && M <= 4 && blocks > 15 * kComputeUnits);
        least = blocks <= 4 * kComputeUnits ? waves : (K <= 1280 ? 2 : (four ? 4 : 8));
    }
    int parts = waves;
    long best = 0;
    for (int p = waves, weight = 100 + (waves == 8 ? 9 : 6); p >= least; p /= 2, weight -= 3) {
        const int side = waves / p;
        const long rounds = ((blocks + side - 1) / side + kComputeUnits - 1) / kComputeUnits;
        const long cost = rounds * side * weight;
        if (best == 0 || cost < best) {
            best = cost;
            parts = p;
        }
    }
    return form(waves, whole_lines ? 128 : 512, parts);
}

// Two rows share the vector kernel's loads well enough where N is small, its sweeps of 128 pieces fit a short row, or the held
// kernel's last round of blocks would be nearly empty.  us, vector -> held: 47090 x 776 17.2 -> 16.6, 53553 x 1176 33.5 -> 28.2, 101754 x
// 2336 96.7 -> 82.8, 46389 x 3912 71.6 -> 64.7, 69572 x 4688 122 -> 110, 151936 x 4096 195 -> 193, 17672 x 7064 53.4 -> 50.8; what the line
// leaves out: 32000 x 1024 13.2 -> 13.8, 28732 x 2696 31.7 -> 32.9, 83762 x 896 29.4 -> 29.4, 4361 x 1080 5.1 -> 5.7, 5573 x 3736 11.0 -> 12.7.
// Held over vector by rounds, 1.6 / 2.0 / 2.05 / 2.15 / 2.3 / 2.6 / 3.03 / 3.2 / 4.03 / 4.6: K = 3072 1.03 / 0.97 / 1.11 / 1.08 / 1.01 / 1.00 / 1.07 /
// 1.03 / 1.03 / 0.97, 4096 0.93 / 0.93 / 1.04 / 1.02 / 0.98 / 0.92 / 0.99 / 0.98 / 0.98 / 0.91, 5000 1.00 / 0.97 / 1.11 / 1.09 / 1.03 / 0.97 / 1.06 / 1.04 /
// 1.04 / 0.95; 768, a sweep for the vector kernel, 0.96 / 0.91 / 1.10 / 1.09 / 1.08 / 1.05 / 1.00 / 1.00 / 1.08 / 1.02, at 5.9 0.96.
bool takes_held(int M, int K, int N) {
    if (M == 1 || K > kHeldMostK) return false;
    if (M >= 3) return true;
    const int pieces = K / 8, swept = (pieces + 127) / 128 * 128;
    const long blocks = (static_cast<long>(N) + 15) / 16, rounds = (blocks + kComputeUnits - 1) / kComputeUnits;
    const int least_full = K < 1024 && rounds >= 3 && rounds <= 6 ? 92 : 77;  // percent of the rounds that blocks have to fill
    return N >= 6500 && (K >= 3072 || 5 * swept >= 6 * pieces) && 100 * blocks >= least_full * rounds * kComputeUnits;
}

// Launches `form` if it is one of these; UNITS are the numbers of units that the rule above gives with the others, and no
// more are compiled.
template <int WAVES, int UNIT, int PARTS, bool RUNS, int... UNITS>
bool launch_held_of(const HeldForm& form, const uint16_t* x, const uint16_t* w, uint16_t* y, int M, int K, int N, hipStream_t s) {
    if (form.waves != WAVES || form.unit != UNIT || form.parts != PARTS || form.runs != RUNS) return false;
    constexpr int SIDE = WAVES / PARTS;
    const int blocks = (N + 15) / 16, sides = (blocks + SIDE - 1) / SIDE;
    const dim3 grid(sides < kComputeUnits ? sides : kComputeUnits), block(WAVES * kWave);
    const auto launch = [&](auto units) {
        constexpr int U = decltype(units)::value;
        if (form.units != U) return false;
        hipLaunchKernelGGL((bf16_gemv_held_kernel<WAVES, UNIT, U, PARTS, RUNS>), grid, block, 0, s, x, w, y, M, K, N, blocks);
        return true;
    };
    return (launch(std::integral_constant<int, UNITS>{}) || ...);
}

int launch_held(const uint16_t* x, const uint16_t* w, uint16_t* y, int M, int K, int N, hipStream_t s) {
    const bool whole_lines = K % 64 == 0 && reinterpret_cast<uintptr_t>(w) % 128 == 0;
    const HeldForm form = held_form(whole_lines, M, K, N);
#define KX_HELD(WAVES, UNIT, PARTS, RUNS, ...) launch_held_of<WAVES, UNIT, PARTS, RUNS, __VA_ARGS__>(form, x, w, y, M, K, N, s)
    const bool launched =
        KX_HELD(8, 128, 8, false, 1, 2, 3, 4, 5, 6, 7, 8) || KX_HELD(8, 128, 8, true, 1, 2, 3, 4, 5, 6) ||
        KX_HELD(8, 128, 4, false, 1, 2, 3, 4, 5, 6, 7, 8) || KX_HELD(8, 128, 4, true, 1, 2, 3, 4, 5) ||
        KX_HELD(8, 128, 2, false, 1, 2, 3, 4, 5) || KX_HELD(8, 128, 2, true, 1, 2, 3, 4, 5) ||
        KX_HELD(8, 256, 8, false, 1, 3) || KX_HELD(8, 256, 8, true, 1) || KX_HELD(8, 512, 8, false, 1, 2) || KX_HELD(8, 512, 8, true, 1) ||
        KX_HELD(4, 512, 4, false, 1, 3) || KX_HELD(4, 512, 4, true, 1, 3) || KX_HELD(4, 512, 2, false, 1) || KX_HELD(4, 512, 2, true, 1) ||
        KX_HELD(4, 512, 1, false, 1, 2) || KX_HELD(4, 512, 1, true, 1, 2);
#undef KX_HELD
    return launched ? launch_status() : KX_ERR_BAD_SHAPE;
}

}  // namespace
}  // namespace kx

extern "C" int kx_bf16_held_form(int32_t whole_lines, int32_t M, int32_t K, int32_t N, int32_t* form) {
    if (!form || M < 1 || M > KX_MAX_BATCH || K < 8 || K % 8 != 0 || N < 1 || !kx::takes_held(M, K, N)) return 0;
    const kx::HeldForm f = kx::held_form(whole_lines != 0, M, K, N);
    const int32_t fields[5] = {f.waves, f.unit, f.units, f.parts, f.runs};
    for (int i = 0; i < 5; i++) form[i] = fields[i];
    return 1;
}

extern "C" int kx_gemv_bf16(const uint16_t* x, const uint16_t* w, uint16_t* y, int32_t M, int32_t K,
                            int32_t N, void* workspace, size_t workspace_bytes, void* stream) {
    (void)workspace;
    (void)workspace_bytes;
    if (!x || !w || !y) return KX_ERR_NULL_POINTER;
    if (M < 1 || M > KX_MAX_BATCH || K < 8 || (K % 8) != 0 || N < 1) return KX_ERR_BAD_SHAPE;
    if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(w) % 16 ||
        reinterpret_cast<uintptr_t>(y) % 2) {
        return KX_ERR_ALIGNMENT;
    }
    hipStream_t s = kx::as_stream(stream);
    if (kx::takes_held(M, K, N)) return kx::launch_held(x, w, y, M, K, N, s);
    if (M >= 3) {
        // K > 8192: the activations of a wave's part do not fit its registers
        if (M <= 8) {
            hipLaunchKernelGGL((kx::bf16_gemv_mfma_kernel<1, 8>), dim3((N + 15) / 16), dim3(kx::kMfmaWaves * kx::kWave), 0,
                               s, x, w, y, M, K, N);
        } else {
            hipLaunchKernelGGL((kx::bf16_gemv_mfma_kernel<4, 4>), dim3((N + 63) / 64), dim3(kx::kMfmaWaves * kx::kWave), 0,
                               s, x, w, y, M, K, N);
        }
        return kx::launch_status();
    }
    const dim3 grid((N + kx::kRowsPerBlock - 1) / kx::kRowsPerBlock);
    const dim3 block(kx::kRowsPerBlock * kx::kWave);
    if (M == 1) {
        hipLaunchKernelGGL((kx::bf16_gemv_kernel<1>), grid, block, 0, s, x, w, y, M, K, N, 0);
    } else {
        hipLaunchKernelGGL((kx::bf16_gemv_kernel<2>), grid, block, 0, s, x, w, y, M, K, N, 0);
    }
    return kx::launch_status();
}
