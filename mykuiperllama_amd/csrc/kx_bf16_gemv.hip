// BF16 GEMV fallback for gfx950: y[m,n] = sum_k x[m,k] * W[n,k], W bf16 row-major [N, K].
//
// One or two activation rows: one wave per output row, the 64 lanes walk the row in 16-byte pieces
// (eight bf16 each), pairs along K go through the packed bf16 dot instruction with an fp32
// accumulator, and the lanes meet in a wave-wide sum at the end.  Rows are contiguous, so every load
// is a full 1 KiB per wave.  Several rows: matrix cores, the activations held in registers while a workgroup walks over
// blocks of output rows (third kernel below), or, for K > 8192, sixteen output rows per workgroup (second kernel).
#include "kx_common.h"

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

// Two to sixteen activation rows, K <= 1024 * UNITS: one workgroup per compute unit walks over blocks of sixteen output
// columns, and its eight waves split K.  What bounded the kernel above was not W but everything round it: the
// activation rows came out of L2 anew for every 64 columns, and an MFMA operand fetched straight from memory asks for
// 64 bytes of sixteen rows at a time, which the memory system answers at three quarters of its rate.  Here the A operands
// of a wave's part of K stay in registers for the life of the workgroup, and W goes through LDS: a unit is 128 elements
// of the block's sixteen rows (4 KB, four loads of 4 rows x 256 bytes), loaded straight into the wave's own ring of
// kRing units, so that no barrier and no register stands between the stream and the MFMAs and 128 KB per compute unit
// are in flight.  The waves of a block meet in LDS, two buffers in turn, one barrier per block that leaves loads alone.
// A row of a unit is stored with its 16-byte pieces permuted by the low bits of the row (the lane that loads piece j of
// row r fetches piece j ^ (r & 7)), so that the sixteen rows that an operand read touches lie in different banks.
// us at M = 3 / 8 / 16, kernel above -> this one: lm_head 151936 x 4096 273 / 308 / 297 -> 182 / 189 / 199 (W alone at the
// read rate of a large buffer: 171), 151936 x 5120 382 / 447 / 405 -> 231 / 240 / 254, 4096 x 4096 11.4 / 12.1 / 26.3 ->
// 9.1 / 9.2 / 10.5.
// EXACT: K is 1024 * UNITS; otherwise what lies past K is zeroed in both operands.
constexpr int kHeldWaves = 8;
constexpr int kRing = 4;
constexpr int kUnitBytes = 16 * 256;

template <int UNITS, bool EXACT>
__global__ __launch_bounds__(kHeldWaves * kWave, 2) void bf16_gemv_held_kernel(
    const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, uint16_t* __restrict__ y, int M, int K, int N, int blocks) {
    __shared__ __attribute__((aligned(1024))) char ring[kHeldWaves][kRing][kUnitBytes];
    __shared__ __attribute__((aligned(16))) float red[2][kHeldWaves][4][kWave];
    const int tid = threadIdx.x;
    const int lane = tid % kWave;
    const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int c = lane % 16;
    const int b = lane / 16;
    const int kw = wave * 128 * UNITS;  // the wave's first element of K
    const int stride = gridDim.x;

    bf16x8 held[UNITS][4];
    const uint16_t* xrow = x + static_cast<size_t>(min(c, M - 1)) * K;
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int k = kw + 128 * u + 32 * q + 8 * b;
            const bool in = EXACT || k < K;
            const u32x4 v = *reinterpret_cast<const u32x4*>(xrow + (in ? k : 0));
            const bool live = in && c < M;
            held[u][q] = as_bf16x8(live ? v.x : 0u, live ? v.y : 0u, live ? v.z : 0u, live ? v.w : 0u);
        }
    }

    // Loads unit u of a block into a ring slot: load i brings rows 4 i + lane / 16.
    auto fetch = [&](int block, int u, int slot) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int r = 4 * i + b;
            const int k = kw + 128 * u + 8 * (c ^ (r & 7));
            const uint16_t* src = w + static_cast<size_t>(min(16 * block + r, N - 1)) * K + (EXACT || k < K ? k : 0);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                             (__attribute__((address_space(3))) void*)(&ring[wave][slot][i * 1024]), 16, 0, 2);
        }
    };
    // Where the lane finds its operand of step q: row c, piece 4 q + b; steps 2 and 3 lie 128 bytes behind 0 and 1.
    const uint32_t ring0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
        (__attribute__((address_space(3))) char*)(&ring[wave][0][0])));
    const uint32_t at0 = ring0 + c * 256 + ((b ^ (c & 7)) * 16);
    const uint32_t at1 = ring0 + c * 256 + (((4 + b) ^ (c & 7)) * 16);

    const int first = blockIdx.x;
#pragma unroll
    for (int j = 0; j < kRing; j++) {
        const int block = first + (j / UNITS) * stride;
        if (block < blocks) fetch(block, j % UNITS, j);
    }
    int slot = 0, turn = 0;
    for (int block = first; block < blocks; block += stride, turn ^= 1) {
        f32x4v acc[2];
        acc[0] = acc[1] = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            // The unit kRing places further on will take this slot.  Loads return in order: with it to come, kRing - 1
            // units may still be on their way when this one has arrived; in the last ring, wait for everything.
            const int next = block + ((u + kRing) / UNITS) * stride;
            const int held_back = block + ((u + kRing - 1) / UNITS) * stride;
            if (held_back < blocks) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (kRing - 1)) : "memory");
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            u32x4 v[4];
            const uint32_t s0 = at0 + slot * kUnitBytes, s1 = at1 + slot * kUnitBytes;
            // in assembly, because the compiler would wait for every load in flight ahead of a read of the ring
            asm volatile("ds_read_b128 %0, %4\n\tds_read_b128 %1, %5\n\tds_read_b128 %2, %4 offset:128\n\tds_read_b128 %3, %5 offset:128\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
                         : "v"(s0), "v"(s1)
                         : "memory");
            if (next < blocks) fetch(next, (u + kRing) % UNITS, slot);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                u32x4 p = v[q];
                if constexpr (!EXACT) {
                    const bool live = kw + 128 * u + 32 * q + 8 * b < K;
                    p = u32x4{live ? p.x : 0u, live ? p.y : 0u, live ? p.z : 0u, live ? p.w : 0u};
                }
                acc[q & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(held[u][q], as_bf16x8(p.x, p.y, p.z, p.w), acc[q & 1], 0, 0, 0);
            }
            slot = (slot + 1) % kRing;
        }
#pragma unroll
        for (int v = 0; v < 4; v++) red[turn][wave][v][lane] = acc[0][v] + acc[1][v];
        lds_barrier();
        if (tid < 4 * kWave) {  // thread (v, lane): row 4 (lane / 16) + v of column lane % 16
            const float* src = &red[turn][0][0][0] + tid;
            float part[kHeldWaves];
#pragma unroll
            for (int u = 0; u < kHeldWaves; u++) part[u] = src[u * 4 * kWave];
            const float sum = ((part[0] + part[1]) + (part[2] + part[3])) + ((part[4] + part[5]) + (part[6] + part[7]));
            const int m = 4 * b + tid / kWave;
            const int n = 16 * block + c;
            if (m < M && n < N) y[static_cast<size_t>(m) * N + n] = f32_to_bf16(sum);
        }
    }
}

}  // namespace
}  // namespace kx

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
    constexpr int kReach = 128 * kx::kHeldWaves;  // elements of K that a unit of every wave covers
    // Two rows share the vector kernel's loads well enough where W is small; with eight blocks per compute unit and rows of
    // 8 KB its wave sums no longer hide.  us, vector -> held, 151936 outputs: K = 1024 50.9 -> 56.1, 2048 99 -> 99, 4096 204
    // -> 187, 5120 269 -> 230, 8192 439 -> 380; 32768 outputs: 1024 13.4 -> 15.2, 2048 24.1 -> 25.8, 4096 46.4 -> 44.0, 8192
    // 97.8 -> 85.2; 4096 outputs: 4096 9.0 -> 9.4, 8192 15.4 -> 15.5.  The line is on the safe side: K = 1536, 2560, 3072 and
    // 3584 (6 to 15 % ahead from 32768 outputs on) and 16384 outputs from K = 4096 on (5 to 12 %) stay with the vector kernel.
    if ((M >= 3 || (M == 2 && K >= 4096 && N >= 32768)) && K <= 8 * kReach) {
        const int blocks = (N + 15) / 16;
        const dim3 grid(blocks < 256 ? blocks : 256), block(kx::kHeldWaves * kx::kWave);
#define KX_HELD(U)                                                                                                      \
    do {                                                                                                                \
        if (K == U * kReach) hipLaunchKernelGGL((kx::bf16_gemv_held_kernel<U, true>), grid, block, 0, s, x, w, y, M, K, N, blocks); \
        else hipLaunchKernelGGL((kx::bf16_gemv_held_kernel<U, false>), grid, block, 0, s, x, w, y, M, K, N, blocks);     \
    } while (0)
        switch ((K + kReach - 1) / kReach) {
            case 1: KX_HELD(1); break;
            case 2: KX_HELD(2); break;
            case 3: KX_HELD(3); break;
            case 4: KX_HELD(4); break;
            case 5: KX_HELD(5); break;
            case 6: KX_HELD(6); break;
            case 7: KX_HELD(7); break;
            default: KX_HELD(8); break;
        }
#undef KX_HELD
        return kx::launch_status();
    }
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
