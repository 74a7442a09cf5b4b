// Host side of the fused INT4 AWQ dequantise + GEMV: shape checks, launch plan, C ABI.
#include "kx_awq_gemv_kernel.h"
#include "kx_awq_gemv_mfma_kernel.h"
#include "kx_internal.h"

#include <mutex>


namespace kx {
namespace {

struct AwqPlan {
    bool mfma;     // matrix-core kernel or the VALU kernel
    int run;       // MFMA kernel: blocks of K whose sums are added up before they join the others'
    bool walks;    // MFMA kernel: a workgroup walks over such a run; otherwise the read-back adds in that order
    bool fine;     // MFMA kernel: the steps of a wave lie in groups of their own
    bool sliced;   // MFMA kernel: all workgroups of a column tile finish it together
    bool trio;     // MFMA kernel, plain: the form of which three fit a compute unit
    int waves;     // waves per workgroup stacked along K (4, 8 or 16)
    int rt;        // VALU kernel: consecutive rows per lane (8 or 16); MFMA kernel: 32-row steps per wave
    int mb;        // activation rows per workgroup (1, 2, 4 or 8)
    int coltiles;  // tiles of 256 output columns
    int ktiles;    // workgroups along K that share a column tile
    int mtiles;    // ceil(M / mb)
};

inline int rows_per_block(int waves, int rt) {
    return waves * kSlotsPerWave * rt;
}

constexpr int kComputeUnits = 256;  // MI355X
constexpr int kExchangeRows = 8;    // what a K tile's share of the split-K exchange costs, in rows of K streamed

// MFMA kernel: four waves per workgroup, each walking `ks` consecutive 32-row steps, in one quantisation group or (below) across
// them.  What it costs besides the weights is the exchange of partial sums, M KB per K tile and column tile.
//   M <= 4   one workgroup (or wave) of a column tile reads all of them back, sixteen K tiles in flight: two steps per
//            wave, or four where that brings the K tiles down to one such batch and gives the busiest compute unit no
//            more rows to stream (or saves three rows and more a nearly full second batch), on at most two workgroups per
//            compute unit.  us per launch at M = 2 / 3 / 4, two steps -> four: 5120 -> 5120 (200 workgroups of four) 8.5 /
//            9.6 / 9.6 -> 7.6 / 8.5 / 8.5, 5120 -> 10240 (400) 11.8 / 13.2 / 13.3 -> 11.0 / 11.8 / 11.8, 8192 -> 5120 (320)
//            at M = 3 / 4 11.1 / 11.2 -> 10.8 / 11.0.  What the rule leaves out: 5120 -> 1024 (40) 6.8 / 7.8 / 7.9 -> 7.0 /
//            7.8 / 7.9, 6400 -> 5120 (260) 8.6 / 9.8 / 9.8 -> 9.3 / 10.2 / 10.2, 5120 -> 8192 (320) 9.6 / 10.7 / 10.8 ->
//            10.7 / 11.5 / 11.6, 6400 -> 10240 (520) 12.3 / 13.3 / 13.7 -> 14.0 / 14.8 / 14.9, 5120 -> 51200 (2000) behind a
//            norm 31.9 / 33.9 / 34.4 -> 34.8 / 37.2 / 37.8.
//   M >= 5   every workgroup of a column tile finishes a share (splitk_exchange_sliced), provided that they are on the
//            chip together: at most two per compute unit.  The shortest run of steps that leaves one workgroup per
//            compute unit and sixteen K tiles (fewer workgroups idle against more partial sums: 1024 -> 2048 ks = 1, q ks
//            = 2, q|k|v and down ks = 4).  Against the single reader, us per launch at M = 8 / 16: k 4096 -> 1024
//            7.6 / 10.2 -> 6.9 / 8.1, q 4096 -> 4096 8.2 / 10.7 -> 7.5 / 8.9, q|k|v 9.2 / 11.0 -> 8.6 / 9.8, down
//            12288 -> 4096 15.4 / 18.9 -> 12.6 / 14.7, gate 4096 -> 12288 12.1 / 14.3 -> 12.0 / 12.6, 5120 -> 10240
//            17.4 / 17.4 -> 12.9 / 14.1.  Where that leaves two per compute unit and K ends in the first half of a block,
//            half the run may need no more of them: behind a norm at M = 5 / 8 / 9 / 16 1152 -> 23040 (270 workgroups of
//            four steps, 450 of two) 12.3 / 13.0 / 15.8 / 16.9 -> 10.0 / 10.2 / 12.4 / 13.8, 2304 -> 13824 (270, 486) 12.7 /
//            12.6 / 15.5 / 16.5 -> 10.1 / 10.4 / 12.9 / 13.7, 3328 -> 9984 (273, 507) 12.7 / 12.9 / 15.6 / 16.6 -> 10.8 / 11.0 /
//            13.4 / 14.6; with K a multiple of 512 there is no such case, and from two steps to one (groups of 64, 1664 ->
//            9344 at M = 11 / 16 10.7 / 11.3 -> 11.2 / 11.9) it loses.  A K that one workgroup covers stays with one, which
//            has nothing to exchange (512 -> 17920 at M = 8 / 16 8.1 / 10.7 -> 6.1 / 7.3, 512 -> 1280 6.6 / 8.3 -> 5.5 /
//            6.7; into the residual stream 512 -> 4096 6.6 / 8.6 -> 7.1 / 9.0).  Larger grids, whose workgroups
//            come in rounds, keep the single reader: with shares the early ones would hold the places the late ones need
//            (gate|up 4096 -> 24576 at M = 16: 19.7 against 21.5 us), and so do their column-tile-fastest order and 256 /
//            512 rows per workgroup.
//            Up to three per compute unit where that many of the form fit (kThreePerUnit, four steps, at most sixteen K
//            tiles).  Behind a norm always: the figures stand there.  A plain launch of nine and more rows from ten K tiles on,
//            M = 9 / 16, single reader and two per compute unit -> shares and three: 5120 -> 15360 (600 workgroups, ten K
//            tiles) 19.1 / 20.2 -> 16.1 / 17.6, 8192 -> 10240 (640, sixteen) 20.3 / 21.2 -> 17.8 / 20.0; left out 4096 -> 24576
//            (768, eight) 18.3 / 19.3 -> 18.0 / 19.6, 2048 -> 40960 (640, four) 18.1 / 19.2 -> 17.6 / 19.9, and at six rows 8192 ->
//            10240 17.0 -> 17.5.  (Five to eight rows with two steps per wave would gain by four and shares, 4096 -> 24576
//            behind a norm 18.6 -> 16.1, but add their K tiles in another order then: after five layers the logits
//            of a step are 0.005 apart.)
//            Unless K is long as well, more than 16 blocks of 512 rows (32 up to eight rows): then the partial sums
//            outweigh that, and a workgroup walks over as many blocks as bring the grid down to two per compute unit.  us
//            per launch, single reader -> walk, M = 5 / 8 / 9 / 16: 14336 -> 5120 (28 blocks) 18.4 / 18.8 / 25.0 / 26.5
//            -> 19.2 / 19.4 / 21.7 / 22.4, 16384 -> 5120 (32) 18.6 / 19.0 / 25.4 / 26.7 -> 20.1 / 20.2 / 22.1 / 22.7,
//            18432 -> 5120 (36) 21.1 / 21.7 / 28.0 / 29.3 -> 21.1 / 20.8 / 22.8 / 23.6, 25600 -> 5120 (50) 27.1 / 27.7 /
//            36.1 / 36.6 -> 22.2 / 22.4 / 24.1 / 24.3; M = 9 / 16: 8192 -> 10240 (16) 21.7 / 22.2 -> 22.5 / 23.7, 8704 ->
//            10240 (17) 24.1 / 24.7 -> 23.2 / 24.1, 12288 -> 8192 (24) 24.1 / 25.0 -> 22.8 / 23.1.
//            Behind SwiGLU nine and more rows cannot load the next block's operands ahead, and walk past 32 blocks only,
//            over no more of them than there would be rounds of workgroups (a line drawn while a walking block still waited
//            for spilled addresses; without them 18432 -> 5120 takes 24.1 / 24.5): M = 9 / 16 14336 -> 5120 27.3 / 28.9 -> 28.4 /
//            30.3, 16384 -> 5120 28.1 / 29.0 -> 29.4 / 30.9, 18432 -> 5120 30.7 / 31.7 -> 30.3 / 31.9, 20480 -> 5120 (40)
//            34.2 / 35.5 -> 30.9 / 32.3; 24576 -> 16384 (six, for six rounds) 72.2 / 77.4 -> 69.7 / 73.4, 17408 -> 8192 (three,
//            for three) 38.0 / 40.2 -> 35.2 / 38.0, 20096 -> 9616 (four, for three) 51.7 / 54.1 -> 58.7 / 61.9, 17920 -> 14592
//            (five, for four) 50.7 / 53.0 -> 55.6 / 59.4.
//
// What a launch does to its activations and its result decides whether its workgroups walk, but not how the sums are
// added: K tiles, steps per wave and the runs of blocks that are added up ahead of the others depend on M, K, N and the
// group size alone, so that the launches of a shape return the same bits (one that does not walk leaves the runs to the
// read-back, splitk_sum_runs: 14336 -> 5120 behind SwiGLU at M = 16 30.3 us with K tiles in order, 29.9 in runs).
// `may_walk`: the kernel exists in a form that walks; `produced_x`: its activations are produced on the way in.
enum LaunchEnds { kPlainEnds, kNormEnds, kOtherEnds };  // a row in and out; normed on the way in; anything else
inline AwqPlan make_mfma_plan(int M, int K, int N, int group, bool may_walk = true, bool produced_x = false,
                              bool may_cross_groups = true, LaunchEnds ends = kPlainEnds) {
    AwqPlan p;
    p.mfma = true;
    p.fine = false;
    p.coltiles = (N / 8 + kWC - 1) / kWC;
    p.mb = M;
    p.mtiles = 1;
    p.waves = 4;
    const auto ktiles_with = [&](int ks) { return (K + p.waves * ks * kStepRows - 1) / (p.waves * ks * kStepRows); };
    const auto allowed = [&](int ks) { return group % (ks * kStepRows) == 0 && (ks == 1 || p.waves * ks * kStepRows <= K); };
    int ks = (M >= 9 || (M >= 5 && K >= 8192)) ? 4 : 2;
    const auto rounds_with = [&](int c) { return (p.coltiles * ktiles_with(c) + kComputeUnits - 1) / kComputeUnits; };
    if (M <= 4 && ktiles_with(2) > 16 && ktiles_with(2) <= 32 && rounds_with(4) <= 2 &&
        (2 * rounds_with(4) <= rounds_with(2) || (M >= 3 && ktiles_with(2) >= 30))) {
        ks = 4;
    }
    // Groups that leave a wave one or two steps make a K tile of every 128 or 256 rows.  Where there are many of them, four
    // steps across groups, scaled step by step, cost less than the exchange; few of them are better met by the shorter
    // run.  us per launch, inside a group -> across: groups of 32 5472 -> 9000 (43 tiles) at M = 4 / 6 / 11 / 16 19.0 / 24.0 /
    // 32 / 34 -> 15.9 / 16.8 / 17.1 / 17.9, 12288 -> 4096 behind SwiGLU at M = 2 / 4 / 6 / 16 14.5 / 17.9 / 26.5 / 45 -> 13.2 /
    // 15.0 / 15.9 / 17.8, 4096 -> 12288 (32) at M = 6 / 16 16.5 / 24.5 -> 12.6 / 13.7, 1536 -> 17920 (groups of 96, 12) 11.9 /
    // 18.7 -> 10.7 / 13.6, 3072 -> 5120 (24, 480 workgroups) 10.2 / 12.0 -> 9.6 / 11.3; groups of 64 16384 -> 4096 (64) at
    // M = 2 / 4 / 6 / 16 13.5 / 15.2 / 21.8 / 33.5 -> 12.3 / 14.0 / 14.9 / 16.2, 5120 -> 5120 (20, 400) at M = 6 / 16 11.5 / 12.7
    // -> 10.5 / 12.1.  What the rule leaves out: groups of 32 at M = 2 / 4 3072 -> 5120 7.5 / 8.5 -> 7.9 / 9.1; 2560 -> 4096
    // (20, 320) at M = 6 / 11 9.9 / 10.1 -> 10.2 / 12.1, 3072 -> 1024 (24, 96) 7.4 / 7.7 -> 8.8 / 9.6, 1280 -> 10240 (10, 400)
    // at M = 6 / 16 8.9 / 11.2 -> 10.3 / 12.7; groups of 64 4096 -> 12288 (16) at M = 2 / 4 / 8 9.5 / 10.2 / 12.2 -> 11.0 /
    // 12.3 / 13.3, 9728 -> 512 (38, 76) at M = 6 9.0 -> 9.8.
    const int inside = allowed(2) ? 2 : 1;
    const int inside_kt = ktiles_with(inside);
    const int line = inside == 2 ? (M <= 2 ? 60 : (M <= 4 ? 52 : (M <= 8 ? 16 : 8))) : (M <= 2 ? 48 : (M <= 4 ? 32 : 8));
    const bool crosses = may_cross_groups && !allowed(4) && p.waves * 4 * kStepRows <= K && inside_kt > line &&
                         (inside_kt > 48 || 8 * p.coltiles * inside_kt > (inside_kt < 20 ? 16 : 11) * kComputeUnits);
    if (crosses) ks = 4;
    else while (!allowed(ks)) ks /= 2;
    p.sliced = p.walks = p.trio = false;
    p.run = 1;
    if (M >= 5) {
        int best = 0;  // the longest run that is allowed, or a shorter one that is short enough
        for (int c = 4; c >= 1; c /= 2) {
            if (best > 0 && ktiles_with(best) == 1) break;  // nothing to exchange
            if ((!allowed(c) && !(crosses && c == 4)) || (best > 0 && ktiles_with(c) > 16)) continue;
            // one workgroup per compute unit, or two where twice the run leaves two as well (its last block mostly idle)
            if (best == 0 || rounds_with(c) == 1 || (best == 4 && rounds_with(c) == 2 && rounds_with(best) == 2)) best = c;
        }
        const int kt = ktiles_with(best);
        if (kt == 1 || (kt <= kSliceMaxKTiles && p.coltiles * kt <= 2 * kComputeUnits)) {
            p.sliced = kt > 1;
            ks = best;
        } else if (ks == 4 && best == 4 && allowed(4) && kt <= 16 && p.coltiles * kt <= 3 * kComputeUnits) {
            p.trio = ends == kPlainEnds && M >= 9 && kt >= 10;
            p.sliced = p.trio || ends == kNormEnds;
        } else if (allowed(4) && ktiles_with(4) > (M >= 9 ? 16 : 32)) {
            const int blocks = ktiles_with(4);
            int walk = 2;
            while (walk < blocks && p.coltiles * ((blocks + walk - 1) / walk) > 2 * kComputeUnits) walk++;
            const int left = (blocks + walk - 1) / walk;
            if (left > 1 && left <= kSliceMaxKTiles && p.coltiles * left <= 2 * kComputeUnits) {
                p.run = (blocks + left - 1) / left;
                const int rounds = (p.coltiles * blocks + 2 * kComputeUnits - 1) / (2 * kComputeUnits);  // without the walk
                p.walks = p.sliced = may_walk && (M <= 8 || !produced_x || (blocks > 32 && p.run <= rounds));
                ks = 4;
            }
        }
    }
    p.rt = ks;  // steps per wave
    p.fine = group % (ks * kStepRows) != 0;
    p.ktiles = p.walks ? (ktiles_with(ks) + p.run - 1) / p.run : ktiles_with(ks);
    return p;
}

inline AwqPlan make_valu_plan(int M, int K, int N, bool allow_long_rows = true, bool allow_12_waves = true) {
    AwqPlan p;
    p.mfma = p.sliced = p.trio = p.walks = p.fine = false;
    p.run = 1;
    p.coltiles = (N / 8 + kWC - 1) / kWC;
    p.mb = M >= 8 ? 8 : (M >= 4 ? 4 : (M >= 2 ? 2 : 1));
    p.mtiles = (M + p.mb - 1) / p.mb;
    // Three shapes of workgroup: eight waves of sixteen rows per lane (256 rows of K), eight waves of
    // 32 rows per lane (512 rows, half the partial sums to exchange) and twelve waves of sixteen
    // rows (384 rows).  What a launch costs, in rows of K streamed by the busiest compute unit, is
    // the number of workgroups that compute unit gets (all of them resident together or not) times
    // the rows of a workgroup, plus about eight rows' worth per K tile for the exchange.  Measured,
    // us per launch at M = 1 (256 / 512 / 384 rows): q 4096->4096 5.7 / 6.2 / -, gate 4096->12288
    // 8.6 / 9.3 / -, q|k|v 4096->6144 6.8 / 6.6 / -, gate|up 4096->24576 15.7 / 13.8 / -, down
    // 12288->4096 10.0 / - / 9.1, 32B-shaped q|k|v 5120->10240 10.6 / 9.8 / -, o 8192->5120
    // 9.1 / 9.3 / -: the minimum of that cost picks the faster one every time.
    // (Twelve waves of 32 rows, 768 rows per workgroup and one workgroup per compute unit on down
    // 12288->4096, are faster still on the plain launch, 9.0 -> 8.6 us, but slower with the SwiGLU
    // prologue of the decode step, whose latency then has no second workgroup to hide behind.  Eight
    // waves of eight rows, 128 rows per workgroup, for projections too narrow to give every compute
    // unit a workgroup — k 4096->1024 has 64 — are slower as well, 5.07 -> 5.48 us: twice the K tiles
    // to exchange cost more than the idle compute units.)
    // Twelve waves: one activation row, plain or SwiGLU input, plain or residual output only (the
    // other prologues and epilogues are laid out for 4 or 8 waves).  Shorter K than 256 takes fewer
    // waves so that no workgroup is mostly idle.
    p.rt = 16;
    p.waves = 8;
    if (K >= rows_per_block(8, 16)) {
        const struct { int waves, rt; bool allowed; } shapes[3] = {
            {8, 16, true}, {8, 32, allow_long_rows}, {12, 16, allow_12_waves && M == 1}};
        long best = -1;
        for (const auto& c : shapes) {
            const int rows = rows_per_block(c.waves, c.rt);
            if (!c.allowed || ((c.waves != 8 || c.rt != 16) && K % rows != 0)) continue;
            const long kt = (K + rows - 1) / rows;
            const long blocks = static_cast<long>(p.coltiles) * p.mtiles * kt;
            const long cost = (blocks + kComputeUnits - 1) / kComputeUnits * rows + kExchangeRows * kt;
            if (best < 0 || cost < best) {
                best = cost;
                p.waves = c.waves;
                p.rt = c.rt;
                p.ktiles = static_cast<int>(kt);
            }
        }
        return p;
    }
    while (p.waves > 4 && rows_per_block(p.waves, p.rt) > K) p.waves /= 2;
    if (rows_per_block(p.waves, p.rt) > K) p.rt = 8;
    const int kb = rows_per_block(p.waves, p.rt);
    p.ktiles = (K + kb - 1) / kb;
    return p;
}

// One activation row, plain store, the K tiles meeting in fixed point (splitk_exchange_store_fixed): that
// exchange costs about half of the one above per K tile, which moves the choice towards smaller workgroups -
// four waves of sixteen rows (128 rows of K, 256 threads) join the candidates.  Measured, us per launch with
// 128 / 256 / 512 / 384 rows per workgroup: k 4096->1024 3.65 / 3.85 / 4.72 / -, q 4096->4096 4.47 / 4.55 /
// 5.10 / -, q|k|v 4096->6144 5.19 / 5.52 / 5.38 / -, gate 4096->12288 8.16 / 7.63 / 8.34 / -, gate|up
// 4096->24576 13.67 / 12.81 / 12.82 / -, down 12288->4096 - / 7.75 / 8.61 / 7.28, 32B-shaped o 8192->5120
// - / 7.10 / 8.03 / -.  ktiles == 1 in the result means that the exchange does not apply (a single K tile, more
// K tiles than the slot's arrival count holds, or more columns than the zeroed area has slots for).
constexpr int kFixedExchangeRows = 4;

inline AwqPlan make_fixed_plan(int K, int N) {
    AwqPlan p{};
    p.mfma = p.sliced = p.trio = p.walks = p.fine = false;
    p.run = 1;
    p.coltiles = (N / 8 + kWC - 1) / kWC;
    p.mb = 1;
    p.mtiles = 1;
    p.waves = 8;
    p.rt = 16;
    p.ktiles = 1;
    if (static_cast<size_t>(N) * 16 > kCounterBytes) return p;  // a slot and a mask word per column
    const struct { int waves, rt; } shapes[4] = {{8, 16}, {4, 16}, {8, 32}, {12, 16}};
    long best = -1;
    for (const auto& c : shapes) {
        const int rows = rows_per_block(c.waves, c.rt);
        if (K < rows || ((c.waves != 8 || c.rt != 16) && K % rows != 0)) continue;
        const long kt = (K + rows - 1) / rows;
        if (kt < 2 || kt > kFixedMaxKTiles) continue;
        const long blocks = static_cast<long>(p.coltiles) * kt;
        const long cost = (blocks + kComputeUnits - 1) / kComputeUnits * rows + kFixedExchangeRows * kt;
        if (best < 0 || cost < best) {
            best = cost;
            p.waves = c.waves;
            p.rt = c.rt;
            p.ktiles = static_cast<int>(kt);
        }
    }
    return p;
}

// Several activation rows go to the matrix cores, where a lane loads two words of a row.  With an odd number of words and groups
// that leave a wave one step, two rows past K = 2048 and narrow matrices past K = 8192 stay on the vector kernel, which served
// them first and whose sums are the more exact ones (its codes carry an offset of 16, not 128, that cancels in fp32: the error
// of the sum against float64 is 1.3 to 4 times as large on the matrix cores, 12288 -> 1288 with groups of 32 and x of mean 0 and
// 1: of 20608 outputs at M = 16 and mean 1, 1 against 9 are not the correctly rounded sum).  us per launch, vector kernel / matrix
// cores, groups of 32: M = 2 3072 -> 5128 7.8 / 8.7, 5472 -> 9000 15.0 / 15.7, 8224 -> 1288 9.1 / 10.1, -> 5128 14.5 / 14.9, 12288 ->
// 10248 28.9 / 26.7 (2080 -> 3000 6.9 / 6.9); M = 3 9216 -> 520 9.6 / 10.8, 12288 -> 1032 10.0 / 11.3, -> 1288 13.5 / 11.5; M = 4 / 16
// 9216 -> 520 12.0 / 19.5 against 11.0 / 12.0, 12288 -> 1288 13.6 / 35.0 against 11.7 / 13.3, groups of 96 16512 -> 824 at M = 10 39.0
// against 13.8: what the exactness costs.  Behind SwiGLU 10240 -> 24 at M = 6 / 16 8.8 / 9.6 against 9.9 / 10.9.
inline bool rows_on_mfma(int M, int K, int N, int group) {
    if (M < 2 || N < 16) return false;
    const bool odd = N % 16 != 0, one_step = group % (2 * kStepRows) != 0;
    return !(odd && one_step && (M == 2 ? K > 2048 : K > 8192 && N <= 2048));
}

inline AwqPlan make_plan(int M, int K, int N, int group, int mode) {
    // One activation row stays on the vector kernel: with the fixed-point exchange it is ahead of the MFMA kernel on
    // every measured shape (kx_gemv_awq_bf16_policy decides that before it comes here), and the launches with an
    // activation prologue or an epilogue live in it.
    const bool mfma = mode >= KX_POLICY_MFMA ? N >= 16 : mode == KX_POLICY_BY_SHAPE && rows_on_mfma(M, K, N, group);
    return mfma ? make_mfma_plan(M, K, N, group) : make_valu_plan(M, K, N);
}

inline MfmaGrid mfma_grid(const AwqPlan& p, int group) {
    const uint32_t gs = static_cast<uint32_t>(group / kStepRows);
    MfmaGrid g{};
    g.coltiles = p.coltiles;
    g.ktiles = p.ktiles;
    g.side = p.sliced ? tile_group(p.coltiles) : p.coltiles;
    g.sliced = p.sliced;
    g.run = p.run;
    g.wait_ticks = kSliceWaitTicks;
    g.group_magic = gs == 1 ? 0u : static_cast<uint32_t>(((1ull << 32) + gs - 1) / gs);
    return g;
}

template <int WAVES, int RT>
void launch_mb(const AwqPlan& p, const uint16_t* x, const int32_t* qweight, const uint16_t* scales,
               const int32_t* qzeros, uint16_t* y, float* partials, uint32_t* counters, int M,
               int K, int N, int group, hipStream_t stream) {
#define KX_ARGS x, qweight, scales, qzeros, y, partials, counters, M, K, N, group, p.coltiles, p.ktiles, p.mtiles, stream
    switch (p.mb) {
        case 1: launch_awq_gemv<WAVES, RT, 1>(KX_ARGS); break;
        case 2: launch_awq_gemv<WAVES, RT, 2>(KX_ARGS); break;
        case 4: launch_awq_gemv<WAVES, RT, 4>(KX_ARGS); break;
        default: launch_awq_gemv<WAVES, RT, 8>(KX_ARGS); break;
    }
#undef KX_ARGS
}

// Launches with an activation prologue are built for the decode step (M = 1); larger M is served
// two activation rows per workgroup.
inline AwqPlan make_fused_plan(int M, int K, int N, bool allow_12_waves) {
    AwqPlan p = make_valu_plan(M, K, N, true, allow_12_waves);
    p.mb = M >= 2 ? 2 : 1;
    p.mtiles = (M + p.mb - 1) / p.mb;
    return p;
}

// One activation row, add + RMSNorm on the way in, per-head norm + rotation + cache append on the way out.
template <int PRO>
void launch_qkv(const AwqPlan& p, const FusedInput& fi, const RopeTarget& rope, const int32_t* qweight,
                const uint16_t* scales, const int32_t* qzeros, float* partials, uint32_t* counters, int K, int N,
                int group, hipStream_t stream) {
#define KX_ARGS nullptr, qweight, scales, qzeros, nullptr, partials, counters, 1, K, N, group, p.coltiles, p.ktiles, 1, stream, fi, rope
    if (p.rt == 32) launch_awq_gemv<8, 32, 1, PRO, kEpiQkRope>(KX_ARGS);
    else if (p.waves == 8) launch_awq_gemv<8, 16, 1, PRO, kEpiQkRope>(KX_ARGS);
    else if (p.rt == 16) launch_awq_gemv<4, 16, 1, PRO, kEpiQkRope>(KX_ARGS);
    else launch_awq_gemv<4, 8, 1, PRO, kEpiQkRope>(KX_ARGS);
#undef KX_ARGS
}

template <int PRO>
void launch_fused(const AwqPlan& p, const FusedInput& fi, const int32_t* qweight, const uint16_t* scales,
                  const int32_t* qzeros, uint16_t* y, float* partials, uint32_t* counters, int M, int K,
                  int N, int group, hipStream_t stream) {
#define KX_ARGS nullptr, qweight, scales, qzeros, y, partials, counters, M, K, N, group, p.coltiles, p.ktiles, p.mtiles, stream, fi
#define KX_BY_MB(W, R)                                                  \
    do {                                                                \
        if (p.mb == 1) launch_awq_gemv<W, R, 1, PRO>(KX_ARGS);          \
        else launch_awq_gemv<W, R, 2, PRO>(KX_ARGS);                    \
    } while (0)
    if constexpr (PRO == kProSwiGLU) {
        if (p.waves == 12) {  // one activation row by construction of the plan
            launch_awq_gemv<12, 16, 1, PRO>(KX_ARGS);
            return;
        }
    }
    if (p.rt == 32) KX_BY_MB(8, 32);
    else if (p.waves == 8) KX_BY_MB(8, 16);
    else if (p.rt == 16) KX_BY_MB(4, 16);
    else KX_BY_MB(4, 8);
#undef KX_BY_MB
#undef KX_ARGS
}

// The matrix-core kernel with an activation prologue and / or the residual epilogue, 2 <= M <= 16.
template <int PRO, int EPI, bool LONE = false>
void launch_mfma_fused(const AwqPlan& p, const FusedInput& fi, const ResidualTarget& res, const uint16_t* x,
                       const int32_t* qweight, const uint16_t* scales, const int32_t* qzeros, uint16_t* y,
                       float* partials, uint32_t* counters, int M, int K, int N, int group, hipStream_t stream,
                       const RopeTarget& rope = RopeTarget{}, size_t cache_stride = 0) {
    const MfmaGrid grid = mfma_grid(p, group);
#define KX_MARGS x, qweight, scales, qzeros, y, partials, counters, M, K, N, grid, stream, fi, res, rope, cache_stride
#define KX_MFMA_BY_M(KS)                                                             \
    do {                                                                             \
        if (M <= 2) launch_awq_gemv_mfma<4, KS, 2, 1, PRO, EPI, LONE>(KX_MARGS);     \
        else if (M <= 4) launch_awq_gemv_mfma<4, KS, 4, 1, PRO, EPI, LONE>(KX_MARGS); \
        else if (M <= 8) launch_awq_gemv_mfma<4, KS, 8, 1, PRO, EPI, LONE>(KX_MARGS); \
        else launch_awq_gemv_mfma<4, KS, 8, 2, PRO, EPI, LONE>(KX_MARGS);            \
    } while (0)
    if constexpr (PRO == kProNone && EPI == kEpiStore) {
        if (p.trio) {
            launch_awq_gemv_mfma<4, 4, 8, 2, PRO, EPI, LONE, false, false, true>(KX_MARGS);
            return;
        }
    }
    if constexpr (PRO != kProPreNorm && EPI != kEpiQkRope && !LONE) {
        if (p.walks) {
            if (M <= 8) launch_awq_gemv_mfma<4, 4, 8, 1, PRO, EPI, false, true>(KX_MARGS);
            else launch_awq_gemv_mfma<4, 4, 8, 2, PRO, EPI, false, true>(KX_MARGS);
            return;
        }
    }
    if (p.fine) {
        if (M <= 2) launch_awq_gemv_mfma<4, 4, 2, 1, PRO, EPI, LONE, false, true>(KX_MARGS);
        else if (M <= 4) launch_awq_gemv_mfma<4, 4, 4, 1, PRO, EPI, LONE, false, true>(KX_MARGS);
        else if (M <= 8) launch_awq_gemv_mfma<4, 4, 8, 1, PRO, EPI, LONE, false, true>(KX_MARGS);
        else launch_awq_gemv_mfma<4, 4, 8, 2, PRO, EPI, LONE, false, true>(KX_MARGS);
        return;
    }
    if (p.rt == 4) KX_MFMA_BY_M(4);
    else if (p.rt == 2) KX_MFMA_BY_M(2);
    else KX_MFMA_BY_M(1);
#undef KX_MFMA_BY_M
#undef KX_MARGS
}

inline bool aligned_to(const void* p, size_t a) {
    return reinterpret_cast<uintptr_t>(p) % a == 0;
}

// Checks shared by every AWQ entry point; `x` stands for whichever tensors feed the activations.
inline int check_awq_weights(const int32_t* qweight, const uint16_t* scales, const int32_t* qzeros,
                             const uint16_t* y, int M, int K, int N, int group_size, bool stores_y = true) {
    if (!qweight || !scales || !qzeros || (stores_y && !y)) return KX_ERR_NULL_POINTER;
    if (M < 1 || M > KX_MAX_BATCH || K < 1 || N < 8 || (N % 8) != 0) return KX_ERR_BAD_SHAPE;
    if (group_size < 32 || (group_size % 32) != 0 || (K % group_size) != 0) return KX_ERR_BAD_SHAPE;
    if (reinterpret_cast<uintptr_t>(scales) % 16 || reinterpret_cast<uintptr_t>(qweight) % 4 ||
        reinterpret_cast<uintptr_t>(qzeros) % 4 || (stores_y && reinterpret_cast<uintptr_t>(y) % 8)) {
        return KX_ERR_ALIGNMENT;
    }
    return KX_OK;
}

// The launches with an activation prologue address the packed weights with 32-bit offsets.
inline bool weights_fit_buffer_loads(int K, int N) {
    return static_cast<size_t>(K) * N / 2 < (static_cast<size_t>(1) << 31);
}

// Do the byte ranges [a, a + abytes) and [b, b + bbytes) share a byte?  Null pointers overlap nothing.
inline bool ranges_overlap(const void* a, size_t abytes, const void* b, size_t bbytes) {
    if (!a || !b || abytes == 0 || bbytes == 0) return false;
    const uintptr_t a0 = reinterpret_cast<uintptr_t>(a), b0 = reinterpret_cast<uintptr_t>(b);
    return a0 < b0 + bbytes && b0 < a0 + abytes;
}

// Splits the workspace into counters and partial sums when the plan shares column tiles.
inline int resolve_workspace(const AwqPlan& p, int M, int N, void* workspace, size_t workspace_bytes,
                             float** partials, uint32_t** counters) {
    *partials = nullptr;
    *counters = nullptr;
    if (p.ktiles <= 1) return KX_OK;
    if (!workspace) return KX_ERR_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(workspace) % 256) return KX_ERR_ALIGNMENT;
    const size_t partial_bytes = static_cast<size_t>(p.ktiles) * M * N * sizeof(float);
    if (partial_bytes >= (static_cast<size_t>(1) << 32)) return KX_ERR_BAD_SHAPE;  // 32-bit offsets in the read-back
    const size_t need = kCounterBytes + partial_bytes;
    if (workspace_bytes < need) return KX_ERR_WORKSPACE;
    if (p.coltiles * p.mtiles > kMaxTiles) return KX_ERR_BAD_SHAPE;
    *counters = static_cast<uint32_t*>(workspace);
    *partials = reinterpret_cast<float*>(static_cast<char*>(workspace) + kCounterBytes);
    return KX_OK;
}

__global__ void fill_zero_u32(uint32_t* p, size_t n) {
    size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

}  // namespace
}  // namespace kx

extern "C" size_t kx_gemv_workspace_bytes(int32_t M, int32_t K, int32_t N) {
    if (M < 1 || M > KX_MAX_BATCH || K < 1 || N < 8) return 0;
    // Either kernel may serve a shape (the group size and M decide); size for the larger exchange.
    const int kt_valu = kx::make_valu_plan(M, K, N, true, false).ktiles;  // the entry points that keep 8 waves exchange more
    const int kt_mfma = kx::make_mfma_plan(M, K, N, 32, true, false, false).ktiles;  // one step per wave gives the most K tiles
    size_t ktiles = static_cast<size_t>(kt_valu > kt_mfma ? kt_valu : kt_mfma);
    if (M == 1) {
        const size_t kt_fixed = static_cast<size_t>(kx::make_fixed_plan(K, N).ktiles);  // its slow path parks partial sums there
        if (kt_fixed > ktiles) ktiles = kt_fixed;
    }
    return kx::kCounterBytes + ktiles * M * static_cast<size_t>(N) * sizeof(float);
}

extern "C" int kx_shared_line_tile(int32_t coltiles, int32_t ktiles, int32_t id, int32_t* ct, int32_t* kt) {
    const kx::TileOrder order = kx::tile_order_of(static_cast<uint32_t>(coltiles), static_cast<uint32_t>(ktiles));
    if (!order.run) return 0;
    const kx::Tile tile = kx::tile_of_workgroup(order, static_cast<uint32_t>(id), static_cast<uint32_t>(ktiles));
    *ct = tile.ct;
    *kt = tile.kt;
    return 1;
}

extern "C" int kx_tiles_by_number(int32_t M, int32_t steps, int32_t N, int32_t coltiles, int32_t ktiles, int32_t together) {
    return together ? kx::together_by_number(M, steps, N, coltiles, ktiles) : kx::alone_by_number(M, steps, coltiles, ktiles);
}

extern "C" int kx_workspace_init(void* workspace, size_t workspace_bytes, void* stream) {
    if (!workspace) return KX_ERR_NULL_POINTER;
    if (workspace_bytes < kx::kCounterBytes) return KX_ERR_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(workspace) % 256) return KX_ERR_ALIGNMENT;
    // A fill kernel rather than hipMemsetAsync, so that the call may sit inside a captured graph.
    size_t n = kx::kCounterBytes / sizeof(uint32_t);
    hipLaunchKernelGGL(kx::fill_zero_u32, dim3((n + 255) / 256), dim3(256), 0, kx::as_stream(stream),
                       static_cast<uint32_t*>(workspace), n);
    return kx::launch_status();
}

// ---- the entry point that allocates nothing ----
// The split-K workspace of kx_gemv_awq_bf16_static: arrival counters, then partial sums.  Every GPU the
// library runs on holds its own copy of this array until the process ends.
namespace {

constexpr size_t kStaticPartialBytes = static_cast<size_t>(8) << 20;
constexpr size_t kStaticScratchBytes = kx::kCounterBytes + kStaticPartialBytes;
constexpr int kMaxDevices = 64;

static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

struct StaticScratch {
    std::mutex mu;
    void* ptr[kMaxDevices] = {};  // device address of `scratch` on each device, null until first use there
};

StaticScratch g_static_scratch;

// Device address of the current device's copy of `scratch`; on the first call on a device the address is
// looked up and the arrival counters are zeroed on `stream` (a kernel, so that a capturing stream records
// it like any other launch).  In host code the array's name is not a device address: only the pointer
// obtained here is ever handed to a kernel.
int static_scratch_for_current_device(void** out, hipStream_t stream) {
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return static_cast<int>(e);
    if (dev < 0 || dev >= kMaxDevices) return KX_ERR_BAD_SHAPE;
    std::lock_guard<std::mutex> lock(g_static_scratch.mu);
    if (!g_static_scratch.ptr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return static_cast<int>(e);
        if (!p || reinterpret_cast<uintptr_t>(p) % 256) return KX_ERR_ALIGNMENT;
        const size_t n = kx::kCounterBytes / sizeof(uint32_t);
        hipLaunchKernelGGL(kx::fill_zero_u32, dim3((n + 255) / 256), dim3(256), 0, stream, static_cast<uint32_t*>(p), n);
        const int rc = kx::launch_status();
        if (rc != KX_OK) return rc;
        g_static_scratch.ptr[dev] = p;
    }
    *out = g_static_scratch.ptr[dev];
    return KX_OK;
}

}  // namespace

extern "C" size_t kx_gemv_awq_static_scratch_bytes(void) {
    return kStaticScratchBytes;
}

extern "C" int kx_gemv_awq_bf16_static(const uint16_t* x, const int32_t* qweight, const uint16_t* scales,
                                       const int32_t* qzeros, uint16_t* y, int32_t M, int32_t K, int32_t N,
                                       int32_t group_size, void* stream) {
    // argument errors first, so that a rejected call touches nothing
    if (!x) return KX_ERR_NULL_POINTER;
    int rc = kx::check_awq_weights(qweight, scales, qzeros, y, M, K, N, group_size);
    if (rc != KX_OK) return rc;
    if (reinterpret_cast<uintptr_t>(x) % 16) return KX_ERR_ALIGNMENT;
    if (kx_gemv_workspace_bytes(M, K, N) > kStaticScratchBytes) return KX_ERR_WORKSPACE;  // larger than the static array
    void* ws = nullptr;
    rc = static_scratch_for_current_device(&ws, kx::as_stream(stream));
    if (rc != KX_OK) return rc;
    return kx_gemv_awq_bf16_policy(x, qweight, scales, qzeros, y, M, K, N, group_size, ws, kStaticScratchBytes, stream,
                                   KX_POLICY_BY_SHAPE);
}

extern "C" int kx_gemv_awq_bf16(const uint16_t* x, const int32_t* qweight, const uint16_t* scales,
                                const int32_t* qzeros, uint16_t* y, int32_t M, int32_t K, int32_t N,
                                int32_t group_size, void* workspace, size_t workspace_bytes,
                                void* stream) {
    return kx_gemv_awq_bf16_policy(x, qweight, scales, qzeros, y, M, K, N, group_size, workspace, workspace_bytes,
                                   stream, KX_POLICY_BY_SHAPE);
}

extern "C" int kx_gemv_awq_bf16_policy(const uint16_t* x, const int32_t* qweight, const uint16_t* scales,
                                       const int32_t* qzeros, uint16_t* y, int32_t M, int32_t K, int32_t N,
                                       int32_t group_size, void* workspace, size_t workspace_bytes,
                                       void* stream, int32_t policy) {
    if (policy < KX_POLICY_BY_SHAPE || policy > KX_POLICY_MFMA_NO_WAIT) return KX_ERR_BAD_SHAPE;
    if (!x) return KX_ERR_NULL_POINTER;
    int rc = kx::check_awq_weights(qweight, scales, qzeros, y, M, K, N, group_size);
    if (rc != KX_OK) return rc;
    if (reinterpret_cast<uintptr_t>(x) % 16) return KX_ERR_ALIGNMENT;
    float* partials = nullptr;
    uint32_t* counters = nullptr;
    hipStream_t s = kx::as_stream(stream);
    if (M == 1 && policy == KX_POLICY_BY_SHAPE) {
        // one activation row, plain store: the K tiles of a column meet in a 64-bit fixed-point word
        const kx::AwqPlan fp = kx::make_fixed_plan(K, N);
        if (fp.ktiles > 1) {
            rc = kx::resolve_workspace(fp, 1, N, workspace, workspace_bytes, &partials, &counters);
            if (rc != KX_OK) return rc;
#define KX_FARGS x, qweight, scales, qzeros, y, partials, counters, 1, K, N, group_size, fp.coltiles, fp.ktiles, 1, s
            if (fp.rt == 32) kx::launch_awq_gemv<8, 32, 1, kx::kProNone, kx::kEpiStoreFixed>(KX_FARGS);
            else if (fp.waves == 12) kx::launch_awq_gemv<12, 16, 1, kx::kProNone, kx::kEpiStoreFixed>(KX_FARGS);
            else if (fp.waves == 8) kx::launch_awq_gemv<8, 16, 1, kx::kProNone, kx::kEpiStoreFixed>(KX_FARGS);
            else kx::launch_awq_gemv<4, 16, 1, kx::kProNone, kx::kEpiStoreFixed>(KX_FARGS);
#undef KX_FARGS
            return kx::launch_status();
        }
    }
    kx::AwqPlan p = kx::make_plan(M, K, N, group_size, policy);
    rc = kx::resolve_workspace(p, M, N, workspace, workspace_bytes, &partials, &counters);
    if (rc != KX_OK) return rc;
    if (p.mfma) {
        kx::MfmaGrid grid = kx::mfma_grid(p, group_size);
        if (policy == KX_POLICY_MFMA_NO_WAIT) grid.wait_ticks = 0;
#define KX_MARGS x, qweight, scales, qzeros, y, partials, counters, M, K, N, grid, s
#define KX_MFMA_WALK(LONE)                                                                                         \
    do {                                                                                                            \
        if (M <= 8) kx::launch_awq_gemv_mfma<4, 4, 8, 1, kx::kProNone, kx::kEpiStore, LONE, true>(KX_MARGS);        \
        else kx::launch_awq_gemv_mfma<4, 4, 8, 2, kx::kProNone, kx::kEpiStore, LONE, true>(KX_MARGS);               \
    } while (0)
        if (p.walks) {
            if (N % 16) KX_MFMA_WALK(true);
            else KX_MFMA_WALK(false);
            return kx::launch_status();
        }
#undef KX_MFMA_WALK
        if (p.trio) {
            if (N % 16) kx::launch_awq_gemv_mfma<4, 4, 8, 2, kx::kProNone, kx::kEpiStore, true, false, false, true>(KX_MARGS);
            else kx::launch_awq_gemv_mfma<4, 4, 8, 2, kx::kProNone, kx::kEpiStore, false, false, false, true>(KX_MARGS);
            return kx::launch_status();
        }
#define KX_MFMA_FINE(LONE)                                                                                          \
    do {                                                                                                             \
        if (M == 1) kx::launch_awq_gemv_mfma<4, 4, 1, 1, kx::kProNone, kx::kEpiStore, LONE, false, true>(KX_MARGS);  \
        else if (M == 2) kx::launch_awq_gemv_mfma<4, 4, 2, 1, kx::kProNone, kx::kEpiStore, LONE, false, true>(KX_MARGS); \
        else if (M <= 4) kx::launch_awq_gemv_mfma<4, 4, 4, 1, kx::kProNone, kx::kEpiStore, LONE, false, true>(KX_MARGS); \
        else if (M <= 8) kx::launch_awq_gemv_mfma<4, 4, 8, 1, kx::kProNone, kx::kEpiStore, LONE, false, true>(KX_MARGS); \
        else kx::launch_awq_gemv_mfma<4, 4, 8, 2, kx::kProNone, kx::kEpiStore, LONE, false, true>(KX_MARGS);         \
    } while (0)
        if (p.fine) {
            if (N % 16) KX_MFMA_FINE(true);
            else KX_MFMA_FINE(false);
            return kx::launch_status();
        }
#undef KX_MFMA_FINE
#define KX_MFMA_ROWS(KS, LONE)                                                                                \
    do {                                                                                                       \
        if (M == 1) kx::launch_awq_gemv_mfma<4, KS, 1, 1, kx::kProNone, kx::kEpiStore, LONE>(KX_MARGS);        \
        else if (M == 2) kx::launch_awq_gemv_mfma<4, KS, 2, 1, kx::kProNone, kx::kEpiStore, LONE>(KX_MARGS);   \
        else if (M <= 4) kx::launch_awq_gemv_mfma<4, KS, 4, 1, kx::kProNone, kx::kEpiStore, LONE>(KX_MARGS);   \
        else if (M <= 8) kx::launch_awq_gemv_mfma<4, KS, 8, 1, kx::kProNone, kx::kEpiStore, LONE>(KX_MARGS);   \
        else kx::launch_awq_gemv_mfma<4, KS, 8, 2, kx::kProNone, kx::kEpiStore, LONE>(KX_MARGS);               \
    } while (0)
#define KX_MFMA_BY_M(KS)                        \
    do {                                        \
        if (N % 16) KX_MFMA_ROWS(KS, true);     \
        else KX_MFMA_ROWS(KS, false);           \
    } while (0)
        if (p.rt == 4) KX_MFMA_BY_M(4);
        else if (p.rt == 2) KX_MFMA_BY_M(2);
        else KX_MFMA_BY_M(1);
#undef KX_MFMA_ROWS
#undef KX_MFMA_BY_M
#undef KX_MARGS
        return kx::launch_status();
    }
#define KX_ARGS p, x, qweight, scales, qzeros, y, partials, counters, M, K, N, group_size, s
    if (p.rt == 32) {
        kx::launch_mb<8, 32>(KX_ARGS);
    } else if (p.waves == 12) {  // one activation row by construction of the plan
        kx::launch_awq_gemv<12, 16, 1>(x, qweight, scales, qzeros, y, partials, counters, M, K, N, group_size, p.coltiles,
                                       p.ktiles, p.mtiles, s);
    } else if (p.waves == 8) {
        kx::launch_mb<8, 16>(KX_ARGS);
    } else if (p.rt == 16) {
        kx::launch_mb<4, 16>(KX_ARGS);
    } else {
        kx::launch_mb<4, 8>(KX_ARGS);
    }
#undef KX_ARGS
    return kx::launch_status();
}

extern "C" int kx_gemv_awq_swiglu_bf16(const uint16_t* gate, const uint16_t* up, int32_t act_ld,
                                       const int32_t* qweight, const uint16_t* scales,
                                       const int32_t* qzeros, uint16_t* y, int32_t M, int32_t K,
                                       int32_t N, int32_t group_size, void* workspace,
                                       size_t workspace_bytes, void* stream) {
    if (!gate || !up) return KX_ERR_NULL_POINTER;
    int rc = kx::check_awq_weights(qweight, scales, qzeros, y, M, K, N, group_size);
    if (rc != KX_OK) return rc;
    if (!kx::weights_fit_buffer_loads(K, N)) return KX_ERR_BAD_SHAPE;
    if (act_ld < K) return KX_ERR_BAD_SHAPE;
    if (reinterpret_cast<uintptr_t>(gate) % 2 || reinterpret_cast<uintptr_t>(up) % 2) return KX_ERR_ALIGNMENT;
    kx::FusedInput fi{};
    fi.a = gate;
    fi.b = up;
    fi.ld = act_ld;
    // Several rows go where kx_gemv_awq_bf16 takes them, when gate and up can be read 16 bytes at a time
    if (kx::rows_on_mfma(M, K, N, group_size) && kx::aligned_to(gate, 16) && kx::aligned_to(up, 16) && (act_ld % 8) == 0) {
        const bool lone = N % 16 != 0;
        const kx::AwqPlan mp = kx::make_mfma_plan(M, K, N, group_size, !lone, true, true, kx::kOtherEnds);
        float* partials = nullptr;
        uint32_t* counters = nullptr;
        rc = kx::resolve_workspace(mp, M, N, workspace, workspace_bytes, &partials, &counters);
        if (rc != KX_OK) return rc;
#define KX_MARGS mp, fi, kx::ResidualTarget{}, nullptr, qweight, scales, qzeros, y, partials, counters, M, K, N, group_size, kx::as_stream(stream)
        if (lone) kx::launch_mfma_fused<kx::kProSwiGLU, kx::kEpiStore, true>(KX_MARGS);
        else kx::launch_mfma_fused<kx::kProSwiGLU, kx::kEpiStore>(KX_MARGS);
#undef KX_MARGS
        return kx::launch_status();
    }
    const kx::AwqPlan p = kx::make_fused_plan(M, K, N, true);
    float* partials = nullptr;
    uint32_t* counters = nullptr;
    rc = kx::resolve_workspace(p, M, N, workspace, workspace_bytes, &partials, &counters);
    if (rc != KX_OK) return rc;
    kx::launch_fused<kx::kProSwiGLU>(p, fi, qweight, scales, qzeros, y, partials, counters, M, K, N, group_size,
                                     kx::as_stream(stream));
    return kx::launch_status();
}

extern "C" int kx_gemv_awq_addnorm_bf16(const uint16_t* residual, const uint16_t* delta, const uint16_t* gain,
                                        float eps, uint16_t* residual_out, const int32_t* qweight,
                                        const uint16_t* scales, const int32_t* qzeros, uint16_t* y,
                                        int32_t M, int32_t K, int32_t N, int32_t group_size,
                                        void* workspace, size_t workspace_bytes, void* stream) {
    if (!residual || !gain) return KX_ERR_NULL_POINTER;
    int rc = kx::check_awq_weights(qweight, scales, qzeros, y, M, K, N, group_size);
    if (rc != KX_OK) return rc;
    if (!kx::weights_fit_buffer_loads(K, N)) return KX_ERR_BAD_SHAPE;
    if (reinterpret_cast<uintptr_t>(residual) % 16 || reinterpret_cast<uintptr_t>(delta) % 16 ||
        reinterpret_cast<uintptr_t>(gain) % 2 || reinterpret_cast<uintptr_t>(residual_out) % 2) {
        return KX_ERR_ALIGNMENT;
    }
    // every workgroup reads the whole incoming rows while the first column tile writes the outgoing ones
    {
        const size_t row_bytes = static_cast<size_t>(M) * K * sizeof(uint16_t);
        if (kx::ranges_overlap(residual_out, row_bytes, residual, row_bytes) ||
            kx::ranges_overlap(residual_out, row_bytes, delta, row_bytes) ||
            kx::ranges_overlap(residual_out, row_bytes, gain, static_cast<size_t>(K) * sizeof(uint16_t))) {
            return KX_ERR_ALIAS;
        }
    }
    const kx::AwqPlan p = kx::make_fused_plan(M, K, N, false);
    // a thread holds kNormChunks 16-byte pieces of the row for the sum of squares
    if ((K >> 3) > kx::kNormChunks * p.waves * kx::kWave) return KX_ERR_BAD_SHAPE;
    float* partials = nullptr;
    uint32_t* counters = nullptr;
    rc = kx::resolve_workspace(p, M, N, workspace, workspace_bytes, &partials, &counters);
    if (rc != KX_OK) return rc;
    kx::FusedInput fi{};
    fi.a = residual;
    fi.b = delta;
    fi.gain = gain;
    fi.r_out = residual_out;
    fi.ld = K;
    fi.eps = eps;
    if ((K >> 3) <= p.waves * kx::kWave) {
        kx::launch_fused<kx::kProAddNorm>(p, fi, qweight, scales, qzeros, y, partials, counters, M, K, N,
                                          group_size, kx::as_stream(stream));
    } else {
        kx::launch_fused<kx::kProAddNormLong>(p, fi, qweight, scales, qzeros, y, partials, counters, M, K, N,
                                              group_size, kx::as_stream(stream));
    }
    return kx::launch_status();
}

extern "C" int kx_gemv_awq_qkv_rope_bf16(const uint16_t* residual, const uint16_t* delta, const uint16_t* gain,
                                         float eps, uint16_t* residual_out, const int32_t* qweight,
                                         const uint16_t* scales, const int32_t* qzeros, const uint16_t* q_gain,
                                         const uint16_t* k_gain, uint16_t* q_out, uint16_t* k_cache,
                                         uint16_t* v_cache, int32_t n_q_heads, int32_t n_kv_heads,
                                         int32_t head_dim, const int32_t* pos, int32_t cache_positions,
                                         float rope_theta, float qk_eps,
                                         int32_t K, int32_t group_size, void* workspace,
                                         size_t workspace_bytes, void* stream) {
    if (!residual || !gain || !q_gain || !k_gain || !q_out || !k_cache || !v_cache || !pos) {
        return KX_ERR_NULL_POINTER;
    }
    if (head_dim != kx::kHeadDim || n_q_heads < 1 || n_kv_heads < 1 || cache_positions < 1 || !(rope_theta > 1.0f)) {
        return KX_ERR_BAD_SHAPE;
    }
    // a column tile of 256 must hold whole heads
    if ((n_q_heads + 2 * n_kv_heads) % (kx::kTileCols / kx::kHeadDim) != 0) return KX_ERR_BAD_SHAPE;
    const int N = (n_q_heads + 2 * n_kv_heads) * kx::kHeadDim;
    int rc = kx::check_awq_weights(qweight, scales, qzeros, q_out, 1, K, N, group_size);
    if (rc != KX_OK) return rc;
    if (!kx::weights_fit_buffer_loads(K, N)) return KX_ERR_BAD_SHAPE;
    if (reinterpret_cast<uintptr_t>(residual) % 16 || reinterpret_cast<uintptr_t>(delta) % 16 ||
        reinterpret_cast<uintptr_t>(gain) % 2 || reinterpret_cast<uintptr_t>(residual_out) % 2) {
        return KX_ERR_ALIGNMENT;
    }
    {
        const size_t row_bytes = static_cast<size_t>(K) * sizeof(uint16_t);
        if (kx::ranges_overlap(residual_out, row_bytes, residual, row_bytes) ||
            kx::ranges_overlap(residual_out, row_bytes, delta, row_bytes) ||
            kx::ranges_overlap(residual_out, row_bytes, gain, row_bytes)) {
            return KX_ERR_ALIAS;
        }
    }
    const kx::AwqPlan p = kx::make_fused_plan(1, K, N, false);
    if ((K >> 3) > kx::kNormChunks * p.waves * kx::kWave) return KX_ERR_BAD_SHAPE;
    float* partials = nullptr;
    uint32_t* counters = nullptr;
    rc = kx::resolve_workspace(p, 1, N, workspace, workspace_bytes, &partials, &counters);
    if (rc != KX_OK) return rc;
    kx::FusedInput fi{};
    fi.a = residual;
    fi.b = delta;
    fi.gain = gain;
    fi.r_out = residual_out;
    fi.ld = K;
    fi.eps = eps;
    const kx::RopeTarget rope{q_gain, k_gain, q_out, k_cache, v_cache, pos, cache_positions, n_q_heads, n_kv_heads,
                              log2f(rope_theta), qk_eps};
    if ((K >> 3) <= p.waves * kx::kWave) {
        kx::launch_qkv<kx::kProAddNorm>(p, fi, rope, qweight, scales, qzeros, partials, counters, K, N, group_size,
                                        kx::as_stream(stream));
    } else {
        kx::launch_qkv<kx::kProAddNormLong>(p, fi, rope, qweight, scales, qzeros, partials, counters, K, N,
                                            group_size, kx::as_stream(stream));
    }
    return kx::launch_status();
}

extern "C" int kx_gemv_awq_attn_merge_bf16(const void* attn_workspace, size_t attn_workspace_bytes,
                                           int32_t n_q_heads, int32_t n_kv_heads, int32_t head_dim,
                                           int32_t max_positions, const int32_t* qweight, const uint16_t* scales,
                                           const int32_t* qzeros, uint16_t* y, int32_t N, int32_t group_size,
                                           void* workspace, size_t workspace_bytes, void* stream) {
    if (!attn_workspace) return KX_ERR_NULL_POINTER;
    if (head_dim != kx::kHeadDim || n_q_heads < 1 || n_kv_heads < 1 || (n_q_heads % n_kv_heads) != 0 ||
        max_positions < 1) {
        return KX_ERR_BAD_SHAPE;
    }
    const int K = n_q_heads * kx::kHeadDim;
    int rc = kx::check_awq_weights(qweight, scales, qzeros, y, 1, K, N, group_size);
    if (rc != KX_OK) return rc;
    if (!kx::weights_fit_buffer_loads(K, N)) return KX_ERR_BAD_SHAPE;
    const int nchunks = kx::attn_chunks_of(max_positions);
    // a thread holds kMergeHold values of each of its elements: longer contexts take the separate merge
    if (nchunks > kx::kMergeParts * kx::kMergeHold) return KX_ERR_BAD_SHAPE;
    const size_t need = static_cast<size_t>(nchunks) * n_q_heads * (kx::kHeadDim + 2) * sizeof(float);
    if (attn_workspace_bytes < need) return KX_ERR_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(attn_workspace) % 16) return KX_ERR_ALIGNMENT;
    kx::AwqPlan p = kx::make_valu_plan(1, K, N, false, false);
    p.mb = 1;
    p.mtiles = 1;
    float* partials = nullptr;
    uint32_t* counters = nullptr;
    rc = kx::resolve_workspace(p, 1, N, workspace, workspace_bytes, &partials, &counters);
    if (rc != KX_OK) return rc;
    kx::FusedInput fi{};
    fi.part_out = static_cast<const float*>(attn_workspace);
    fi.part_ml = fi.part_out + static_cast<size_t>(nchunks) * n_q_heads * kx::kHeadDim;
    fi.nchunks = nchunks;
    fi.heads_per_kv = n_q_heads / n_kv_heads;
    hipStream_t s = kx::as_stream(stream);
#define KX_ARGS nullptr, qweight, scales, qzeros, y, partials, counters, 1, K, N, group_size, p.coltiles, p.ktiles, 1, s, fi
#define KX_MERGE(PRO) \
    if (p.waves == 8 && nchunks <= kx::kMergeParts * kx::merge_hold(PRO)) kx::launch_awq_gemv<8, 16, 1, PRO>(KX_ARGS)
    KX_MERGE(kx::kProAttnMerge32);
    else KX_MERGE(kx::kProAttnMerge48);
    else KX_MERGE(kx::kProAttnMerge64);
    else KX_MERGE(kx::kProAttnMerge);
#undef KX_MERGE
    else kx::launch_awq_gemv<4, 16, 1, kx::kProAttnMerge>(KX_ARGS);  // K = 128: one head
#undef KX_ARGS
    return kx::launch_status();
}

namespace kx {
namespace {

template <int PRO, int EPI>
void launch_chain(const AwqPlan& p, const FusedInput& fi, const RopeTarget& rope, const ResidualTarget& res,
                  const uint16_t* x, const int32_t* qweight, const uint16_t* scales, const int32_t* qzeros,
                  uint16_t* y, float* partials, uint32_t* counters, int K, int N, int group, hipStream_t stream) {
#define KX_ARGS x, qweight, scales, qzeros, y, partials, counters, 1, K, N, group, p.coltiles, p.ktiles, 1, stream, fi, rope, res
    constexpr bool MERGE = merges_attention(PRO);
    if constexpr (!MERGE) {
        if (p.rt == 32) {
            launch_awq_gemv<8, 32, 1, PRO, EPI>(KX_ARGS);
            return;
        }
    }
    if constexpr ((PRO == kProNone || PRO == kProSwiGLU) && (EPI == kEpiStore || EPI == kEpiResidual)) {
        if (p.waves == 12) {
            launch_awq_gemv<12, 16, 1, PRO, EPI>(KX_ARGS);
            return;
        }
    }
    if (p.waves == 8) launch_awq_gemv<8, 16, 1, PRO, EPI>(KX_ARGS);
    else if (p.rt == 16) launch_awq_gemv<4, 16, 1, PRO, EPI>(KX_ARGS);
    else if constexpr (!MERGE) launch_awq_gemv<4, 8, 1, PRO, EPI>(KX_ARGS);
#undef KX_ARGS
}

}  // namespace
}  // namespace kx

extern "C" int kx_gemv_awq_chain_bf16(const kx_chain_desc* d, const int32_t* qweight, const uint16_t* scales,
                                      const int32_t* qzeros, int32_t K, int32_t N, int32_t group_size,
                                      void* workspace, size_t workspace_bytes, void* stream) {
    if (!d) return KX_ERR_NULL_POINTER;
    kx::FusedInput fi{};
    kx::RopeTarget rope{};
    kx::ResidualTarget res{};
    const uint16_t* x = nullptr;
    uint16_t* y = nullptr;
    bool long_rows = true;
    const int rows = d->rows > 0 ? d->rows : 1;
    if (rows > KX_MAX_BATCH || K < 1 || N < 8) return KX_ERR_BAD_SHAPE;
    const int act_ld = d->act_ld > 0 ? d->act_ld : K;
    if (act_ld < K) return KX_ERR_BAD_SHAPE;
    if (rows > 1) {
        // several rows: the matrix-core kernel, which produces activations 16 bytes at a time
        if (d->in_kind == KX_IN_ATTN) return KX_ERR_BAD_SHAPE;
        if ((N % 16) != 0 || (act_ld % 8) != 0) return KX_ERR_BAD_SHAPE;
    }

    // where the activations come from
    switch (d->in_kind) {
        case KX_IN_ROW:
            if (!d->x) return KX_ERR_NULL_POINTER;
            if (reinterpret_cast<uintptr_t>(d->x) % 16) return KX_ERR_ALIGNMENT;
            x = d->x;
            break;
        case KX_IN_SWIGLU:
            if (!d->gate || !d->up) return KX_ERR_NULL_POINTER;
            if (reinterpret_cast<uintptr_t>(d->gate) % 2 || reinterpret_cast<uintptr_t>(d->up) % 2) return KX_ERR_ALIGNMENT;
            if (rows > 1 && (!kx::aligned_to(d->gate, 16) || !kx::aligned_to(d->up, 16))) return KX_ERR_ALIGNMENT;
            fi.a = d->gate;
            fi.b = d->up;
            fi.ld = act_ld;
            break;
        case KX_IN_ATTN: {
            if (!d->attn_workspace) return KX_ERR_NULL_POINTER;
            if (d->n_q_heads < 1 || d->n_kv_heads < 1 || (d->n_q_heads % d->n_kv_heads) != 0 || d->max_positions < 1 ||
                K != d->n_q_heads * kx::kHeadDim) {
                return KX_ERR_BAD_SHAPE;
            }
            const int nchunks = kx::attn_chunks_of(d->max_positions);
            if (nchunks > kx::kMergeParts * kx::kMergeHold) return KX_ERR_BAD_SHAPE;
            const size_t need = static_cast<size_t>(nchunks) * d->n_q_heads * (kx::kHeadDim + 2) * sizeof(float);
            if (d->attn_workspace_bytes < need) return KX_ERR_WORKSPACE;
            if (reinterpret_cast<uintptr_t>(d->attn_workspace) % 16) return KX_ERR_ALIGNMENT;
            fi.part_out = static_cast<const float*>(d->attn_workspace);
            fi.part_ml = fi.part_out + static_cast<size_t>(nchunks) * d->n_q_heads * kx::kHeadDim;
            fi.nchunks = nchunks;
            fi.heads_per_kv = d->n_q_heads / d->n_kv_heads;
            long_rows = false;  // the merge covers at most 256 rows of K per workgroup
            break;
        }
        case KX_IN_NORM:
            if (!d->norm_row || !d->norm_sumsq || !d->norm_gain) return KX_ERR_NULL_POINTER;
            if (d->norm_parts != (K + kx::kTileCols - 1) / kx::kTileCols || d->norm_parts > kx::kWave) return KX_ERR_BAD_SHAPE;
            if (reinterpret_cast<uintptr_t>(d->norm_row) % 2 || reinterpret_cast<uintptr_t>(d->norm_sumsq) % 16 ||
                reinterpret_cast<uintptr_t>(d->norm_gain) % 2) {
                return KX_ERR_ALIGNMENT;  // the four quarter sums of a tile are read as one 16-byte piece
            }
            if (rows > 1 && (!kx::aligned_to(d->norm_row, 16) || !kx::aligned_to(d->norm_gain, 16))) return KX_ERR_ALIGNMENT;
            fi.a = d->norm_row;
            fi.gain = d->norm_gain;
            fi.eps = d->norm_eps;
            fi.sumsq = d->norm_sumsq;
            fi.sumsq_parts = d->norm_parts;
            fi.ld = act_ld;
            break;
        default: return KX_ERR_BAD_SHAPE;
    }

    // where the result goes
    const uint16_t* out_probe = nullptr;  // any output pointer, for the shared checks
    switch (d->out_kind) {
        case KX_OUT_ROW:
            if (!d->y) return KX_ERR_NULL_POINTER;
            y = d->y;
            out_probe = d->y;
            break;
        case KX_OUT_RESIDUAL:
            if (!d->residual_in || !d->residual_out || !d->sumsq_out) return KX_ERR_NULL_POINTER;
            if (reinterpret_cast<uintptr_t>(d->residual_in) % 2 || reinterpret_cast<uintptr_t>(d->residual_out) % 2 ||
                reinterpret_cast<uintptr_t>(d->sumsq_out) % 4) {
                return KX_ERR_ALIGNMENT;
            }
            {
                // Workgroups of other column tiles still read the activations while the tile that finishes
                // first already writes its 256 columns of the outgoing row: the two must not share a byte.
                // (residual_out may be residual_in itself: a column is read and written by one thread.)
                const size_t out_bytes = static_cast<size_t>(rows) * N * sizeof(uint16_t);
                const size_t in_bytes = (static_cast<size_t>(rows - 1) * act_ld + K) * sizeof(uint16_t);
                if (kx::ranges_overlap(d->residual_out, out_bytes, d->in_kind == KX_IN_NORM ? d->norm_row : nullptr, in_bytes) ||
                    kx::ranges_overlap(d->residual_out, out_bytes, d->in_kind == KX_IN_ROW ? d->x : nullptr, in_bytes) ||
                    kx::ranges_overlap(d->residual_out, out_bytes, d->in_kind == KX_IN_SWIGLU ? d->gate : nullptr, in_bytes) ||
                    kx::ranges_overlap(d->residual_out, out_bytes, d->in_kind == KX_IN_SWIGLU ? d->up : nullptr, in_bytes)) {
                    return KX_ERR_ALIAS;
                }
                if (d->residual_out != d->residual_in &&
                    kx::ranges_overlap(d->residual_out, out_bytes, d->residual_in, out_bytes)) {
                    return KX_ERR_ALIAS;  // a shifted overlap: another thread's column would be overwritten
                }
            }
            res.in = d->residual_in;
            res.out = d->residual_out;
            res.sumsq = d->sumsq_out;
            out_probe = d->residual_out;
            break;
        case KX_OUT_QKV_ROPE:
            if (!d->q_gain || !d->k_gain || !d->q_out || !d->k_cache || !d->v_cache || !d->pos) return KX_ERR_NULL_POINTER;
            if (d->rope_n_q_heads < 1 || d->rope_n_kv_heads < 1 || d->cache_positions < 1 || !(d->rope_theta > 1.0f) ||
                N != (d->rope_n_q_heads + 2 * d->rope_n_kv_heads) * kx::kHeadDim ||
                (d->rope_n_q_heads + 2 * d->rope_n_kv_heads) % (kx::kTileCols / kx::kHeadDim) != 0) {
                return KX_ERR_BAD_SHAPE;
            }
            // several rows are several sequences, each with a cache pair of its own
            if (rows > 1 && d->cache_stride < static_cast<size_t>(d->cache_positions) * d->rope_n_kv_heads * kx::kHeadDim) {
                return KX_ERR_BAD_SHAPE;
            }
            rope = kx::RopeTarget{d->q_gain, d->k_gain, d->q_out, d->k_cache, d->v_cache, d->pos, d->cache_positions,
                                  d->rope_n_q_heads, d->rope_n_kv_heads, log2f(d->rope_theta), d->qk_eps};
            out_probe = d->q_out;
            break;
        default: return KX_ERR_BAD_SHAPE;
    }
    // 8-byte alignment is what the plain store asks of y; the other outputs are written per element
    int rc = kx::check_awq_weights(qweight, scales, qzeros, out_probe, rows, K, N, group_size, d->out_kind == KX_OUT_ROW);
    if (rc != KX_OK) return rc;
    if (d->in_kind != KX_IN_ROW && !kx::weights_fit_buffer_loads(K, N)) return KX_ERR_BAD_SHAPE;
    if (d->in_kind == KX_IN_ATTN && (K % kx::kHeadDim) != 0) return KX_ERR_BAD_SHAPE;

    if (rows > 1) {
        const kx::AwqPlan mp = kx::make_mfma_plan(rows, K, N, group_size,
                                                   d->in_kind != KX_IN_NORM && d->out_kind != KX_OUT_QKV_ROPE,
                                                   d->in_kind != KX_IN_ROW, true,
                                                   d->out_kind != KX_OUT_ROW || d->in_kind == KX_IN_SWIGLU
                                                       ? kx::kOtherEnds : (d->in_kind == KX_IN_NORM ? kx::kNormEnds : kx::kPlainEnds));
        float* partials = nullptr;
        uint32_t* counters = nullptr;
        rc = kx::resolve_workspace(mp, rows, N, workspace, workspace_bytes, &partials, &counters);
        if (rc != KX_OK) return rc;
        hipStream_t s = kx::as_stream(stream);
#define KX_MCHAIN(PRO, EPI) kx::launch_mfma_fused<PRO, EPI>(mp, fi, res, x, qweight, scales, qzeros, y, partials, counters, rows, K, N, group_size, s, rope, d->cache_stride)
#define KX_MBY_OUT(PRO)                                                               \
    do {                                                                              \
        if (d->out_kind == KX_OUT_ROW) KX_MCHAIN(PRO, kx::kEpiStore);                 \
        else if (d->out_kind == KX_OUT_RESIDUAL) KX_MCHAIN(PRO, kx::kEpiResidual);    \
        else KX_MCHAIN(PRO, kx::kEpiQkRope);                                          \
    } while (0)
        switch (d->in_kind) {
            case KX_IN_ROW: KX_MBY_OUT(kx::kProNone); break;
            case KX_IN_SWIGLU: KX_MBY_OUT(kx::kProSwiGLU); break;
            default: KX_MBY_OUT(kx::kProPreNorm); break;
        }
#undef KX_MBY_OUT
#undef KX_MCHAIN
        return kx::launch_status();
    }

    const bool plain_ends = (d->in_kind == KX_IN_ROW || d->in_kind == KX_IN_SWIGLU) &&
                            (d->out_kind == KX_OUT_ROW || d->out_kind == KX_OUT_RESIDUAL);
    kx::AwqPlan p = kx::make_valu_plan(1, K, N, long_rows, plain_ends);
    p.mb = 1;
    p.mtiles = 1;
    float* partials = nullptr;
    uint32_t* counters = nullptr;
    rc = kx::resolve_workspace(p, 1, N, workspace, workspace_bytes, &partials, &counters);
    if (rc != KX_OK) return rc;
    hipStream_t s = kx::as_stream(stream);

#define KX_CHAIN(PRO, EPI) kx::launch_chain<PRO, EPI>(p, fi, rope, res, x, qweight, scales, qzeros, y, partials, counters, K, N, group_size, s)
#define KX_BY_OUT(PRO)                                                                   \
    do {                                                                                 \
        if (d->out_kind == KX_OUT_ROW) KX_CHAIN(PRO, kx::kEpiStore);                     \
        else if (d->out_kind == KX_OUT_RESIDUAL) KX_CHAIN(PRO, kx::kEpiResidual);        \
        else KX_CHAIN(PRO, kx::kEpiQkRope);                                              \
    } while (0)
    switch (d->in_kind) {
        case KX_IN_ROW: KX_BY_OUT(kx::kProNone); break;
        case KX_IN_SWIGLU: KX_BY_OUT(kx::kProSwiGLU); break;
        case KX_IN_ATTN:
            if (fi.nchunks <= kx::kMergeParts * kx::merge_hold(kx::kProAttnMerge32)) KX_BY_OUT(kx::kProAttnMerge32);
            else if (fi.nchunks <= kx::kMergeParts * kx::merge_hold(kx::kProAttnMerge48)) KX_BY_OUT(kx::kProAttnMerge48);
            else if (fi.nchunks <= kx::kMergeParts * kx::merge_hold(kx::kProAttnMerge64)) KX_BY_OUT(kx::kProAttnMerge64);
            else KX_BY_OUT(kx::kProAttnMerge);
            break;
        default: KX_BY_OUT(kx::kProPreNorm); break;
    }
#undef KX_BY_OUT
#undef KX_CHAIN
    return kx::launch_status();
}
