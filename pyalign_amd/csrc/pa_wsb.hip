// pa_wsb.hip -- general gap costs (Waterman-Smith-Beyer, solver.h:3047-3184)
// in blocks: scores and one optimal path.
//
// D(i, j) folds the diagonal, the whole column above (D(k, j) + ws(i - k))
// and the whole row to the left (D(i, k) + wt(j - k)): O(n m (n + m))
// candidates, one add and half a max3 each where folds may take any order
// (the caller has checked that: finite values, no -0, see wsb_any_order in
// pa_api.cpp).  The matrix is cut into blocks of 16 x 16 cells and computed
// one block anti-diagonal per launch.  A wave takes four neighbouring blocks
// of one problem's anti-diagonal, 16 lanes each, and
//
// 1. folds the finished blocks above (16 lanes = 16 columns, 16 rows in
//    registers) and to the left (lanes = rows, columns in registers, read from
//    a transposed copy of D): a (max, +) product with a Toeplitz matrix, 256
//    candidates a lane from 16 loaded values and 31 costs.  The costs depend
//    on the distance of the blocks only, which is the same for all four
//    blocks, so they are scalars;
// 2. solves the blocks: lane r owns row r and at step s computes column
//    s - r, then pushes the new value into its row's later cells (registers)
//    and, through DPP row shifts, into the cells below it.
//
// The folds of (1) are split over the waves of a workgroup and reduced through
// LDS.  Where a few long problems leave most of the GPU idle (wsb_plan's
// `carry`), a block does not fold everything before it: once solved, its
// values are pushed on into sums carried per block, by workgroups beside those
// that solve the next anti-diagonal, so a launch's critical path is two folds
// and the solve.
//
// (1) takes 1.5 instructions per candidate and (2) 1,300 per four blocks, and a
// launch at least 8 us (dependent loads and the serial solve): that, and each
// launch's longest workgroup, bounds both below (0.31 VALU instructions per SIMD
// in four cycles over the first's launches).  Measured: 1,024 pairs of 100 to 300 (local, 20
// symbols) 1.6 ms and their paths 0.18 ms, one global pair of 1,200 x 1,000
// 1.6 ms (3.5 ms without carried sums) and 0.23 ms.  The cell-by-cell kernel
// (pa_wsb_kernel: two 4-byte loads, an add, a compare and two selects per
// candidate) takes 17.4 ms and 146 ms; it still serves what this one does not:
// all-optimal lists, Solution matrices, and values whose folds depend on the
// order.
#include "pa_kernels.h"

#include <algorithm>
#include <utility>

namespace pa {

namespace {

constexpr int B = WSB_TILE;
static_assert(B == 16, "a block's row is one DPP row");
constexpr int TS = B + 1;          // LDS row stride of a block
constexpr int TILE = B * TS;       // floats per block
constexpr int KS = 2 * B + 1;      // LDS row stride of a solved block (by row and step)
constexpr int WAVE_LDS = 4 * TILE; // a wave's four blocks
constexpr int MIN_LDS = 4 * B * KS;

// lane r of a row of 16 <- lane r - M; lanes r < M read 0
template <int M>
__device__ __forceinline__ float row_shr0(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x110 + M, 0xf, 0xf, true));
}
// lane r <- lane r - 1; lane 0 <- first
__device__ __forceinline__ int row_shr1(int first, int x) {
    return __builtin_amdgcn_update_dpp(first, x, 0x111, 0xf, 0xf, false);
}
// lane 0 of a row <- lane S (S = 0: itself); beyond the row: unspecified
template <int S>
__device__ __forceinline__ int row_first(int x) {
    if constexpr (S == 0 || S >= B) return x;
    else return __builtin_amdgcn_update_dpp(x, x, 0x100 + S, 0xf, 0xf, false);
}

template <class F, int... K>
__device__ __forceinline__ void static_for(std::integer_sequence<int, K...>, F &&f) {
    (f(std::integral_constant<int, K>{}), ...);
}

// 16 values of a block, one row (column) of 16 lanes each
__device__ __forceinline__ void load_block(const float *p, int64_t stride, float (&v)[B]) {
#pragma unroll
    for (int k = 0; k < B; ++k) v[k] = p[k * stride];
}

// acc[r] folds v[k] + w[r - k], k = 0 .. 15: a block's candidates for the block
// whose distance w points to
template <int DIR>
__device__ __forceinline__ void fold_block(const float (&v)[B], const float *__restrict__ w, float (&acc)[B]) {
#pragma unroll
    for (int k = 0; k < B; k += 2)
#pragma unroll
        for (int r = 0; r < B; ++r) acc[r] = opt<DIR>(opt<DIR>(acc[r], v[k] + w[r - k]), v[k + 1] + w[r - k - 1]);
}

// Folds the blocks at distances x = first, first + step, ... <= count (this
// lane's; `most`, the wave's largest, bounds the loop), src(x) their first
// row.  The next block's values are loaded before this one's are folded.
template <int DIR, class Src>
__device__ __forceinline__ void fold_blocks(int first, int step, int count, int most, Src &&src, int64_t stride,
                                            const float *__restrict__ w, float (&acc)[B]) {
    if (first > most) return;
    float v[2][B];
    if (first <= count) load_block(src(first), stride, v[0]);
    for (int x = first;;) {
        if (x + step <= count) load_block(src(x + step), stride, v[1]);
        if (x <= count) fold_block<DIR>(v[0], w + B * x, acc);
        x += step;
        if (x > most) break;
        if (x + step <= count) load_block(src(x + step), stride, v[0]);
        if (x <= count) fold_block<DIR>(v[1], w + B * x, acc);
        x += step;
        if (x > most) break;
    }
}

// the largest value over a wave's four rows of 16 lanes (each uniform)
__device__ __forceinline__ int wave_most(int x) {
    return max(max(__builtin_amdgcn_readlane(x, 0), __builtin_amdgcn_readlane(x, B)),
               max(__builtin_amdgcn_readlane(x, 2 * B), __builtin_amdgcn_readlane(x, 3 * B)));
}

template <int FORM>
__device__ __forceinline__ float similarity(const KArgs &a, const Prob &pr, int i, int j) {
    if constexpr (FORM == F_DENSE) {
        return a.dense[pr.off_s + int64_t(i) * pr.si + int64_t(j) * pr.sj];
    } else if constexpr (FORM == F_TABLE) {
        const int x = ((const uint8_t *)a.codes_s)[pr.off_s + i];
        const int y = ((const uint8_t *)a.codes_t)[pr.off_t + j];
        return a.table[x * a.K1 + y];
    } else if constexpr (FORM == F_TABLE_G) {
        // codes beyond the table read its pad row / column
        const int x = min(int(((const uint16_t *)a.codes_s)[pr.off_s + i]), a.K1 - 1);
        const int y = min(int(((const uint16_t *)a.codes_t)[pr.off_t + j]), a.K1 - 1);
        return a.table[int64_t(x) * a.K1 + y];
    } else {
        const uint32_t x = ((const uint32_t *)a.codes_s)[pr.off_s + i];
        const uint32_t y = ((const uint32_t *)a.codes_t)[pr.off_t + j];
        return x == y ? a.eq : a.ne;
    }
}

// Carried sums (problems of `carry`): a block's candidates so far, 16 x 16 for
// the columns above (lane = column) and 16 x 16 for the rows to the left (lane
// = row), behind the problem's planes.
__device__ __forceinline__ float *carried(const KArgs &a, const Prob &pr, int64_t block) {
    return a.dvals + pr.tb_off + block * (2 * B * B);
}

// The blocks of anti-diagonal diag - 1 pushed into the blocks two or more
// below and to the right of them (those next to them fold them themselves).
// A unit is four neighbouring blocks, one direction and WSB_PUSHES distances; a
// wave takes the problem's units from `first` on, `step` apart (a long pair has
// more than a grid has rows: 16,383 symbols a side 262,000 on one
// anti-diagonal).
template <int DIR>
__device__ __forceinline__ void push_blocks(const KArgs &a, const Prob &pr, const float *__restrict__ ws,
                                            const float *__restrict__ wt, int diag, int first, int step, int lane) {
    const int ls = pr.len_s, lt = pr.len_t;
    const int nbs = (ls + B - 1) / B, nbt = (lt + B - 1) / B, src = diag - 1;
    const int lo = max(0, src - nbt + 1), hi = min(src, nbs - 1);
    if (lo > hi) return;
    const int groups = (hi - lo + 4) / 4;
    // distances 2 .. the farthest of the anti-diagonal's blocks, in either direction
    const int farthest = max(nbs - 1 - lo, nbt - 1 - (src - hi));
    const int units = farthest < 2 ? 0 : groups * 2 * ((farthest - 1 + WSB_PUSHES - 1) / WSB_PUSHES);
    const int q = lane >> 4, l = lane & (B - 1);
    const int64_t cells = int64_t(ls) * lt;
    const float *D = a.dvals + pr.dv_off, *DT = D + cells;
    for (int unit = first; unit < units; unit += step) {
        const int g = unit % groups, down = unit / groups % 2, x0 = 2 + unit / groups / 2 * WSB_PUSHES;
        const int bi = lo + 4 * g + q, bj = src - bi;
        const int reach = bi > hi ? 0 : (down ? nbs - 1 - bi : nbt - 1 - bj);  // blocks below / to the right
        if (x0 > reach) continue;
        const bool start = (down ? bi : bj) == 0;  // the target's first candidates
        float v[B];
        if (down) load_block(D + int64_t(B) * bi * lt + min(B * bj + l, lt - 1), lt, v);
        else load_block(DT + int64_t(B) * bj * ls + min(B * bi + l, ls - 1), ls, v);
        for (int x = x0; x < x0 + WSB_PUSHES && x <= reach; ++x) {
            float *acc_at = carried(a, pr, down ? int64_t(bi + x) * nbt + bj : int64_t(bi) * nbt + bj + x) +
                            (down ? 0 : B * B) + l;
            float acc[B];
#pragma unroll
            for (int r = 0; r < B; ++r) acc[r] = start ? worst<DIR>() : acc_at[r * B];
            if (down) fold_block<DIR>(v, ws + B * x, acc);
            else fold_block<DIR>(v, wt + B * x, acc);
#pragma unroll
            for (int r = 0; r < B; ++r) acc_at[r * B] = acc[r];
        }
    }
}

// Block anti-diagonal `diag` of the problems [0, problems), sorted by their
// number of anti-diagonals, most first.  A workgroup takes four blocks:
// neighbours of one problem (across = 0), or the same place of four problems
// of similar shape (across = 1: no lane waits for a block that is further
// from the border).  carry: each block folds its two neighbours and the sums
// carried for it; the workgroups from blockIdx.y = groups on push the previous
// anti-diagonal on.  ws / wt hold w(k) * sgn and WSB_TILE readable floats past
// their ends.
template <int LOC, int DIR, int FORM>
__global__ __launch_bounds__(512) void pa_wsb_block_kernel(KArgs a, const float *__restrict__ ws,
                                                           const float *__restrict__ wt, int diag, int problems,
                                                           int groups, int across, int carry) {
    constexpr float W = worst<DIR>();
    const int wave = __builtin_amdgcn_readfirstlane(int(threadIdx.x) / WAVE);
    const int waves = int(blockDim.x) / WAVE;
    const int lane = int(threadIdx.x) & (WAVE - 1);
    if (int(blockIdx.y) >= groups) {
        push_blocks<DIR>(a, a.probs[blockIdx.x], ws, wt, diag, (int(blockIdx.y) - groups) * waves + wave,
                         (int(gridDim.y) - groups) * waves, lane);
        return;
    }
    const int q = lane >> 4, l = lane & (B - 1);
    const Prob &pr = a.probs[across ? min(4 * int(blockIdx.x) + q, problems - 1) : int(blockIdx.x)];
    const int ls = pr.len_s, lt = pr.len_t;
    const int nbs = (ls + B - 1) / B, nbt = (lt + B - 1) / B;
    const int last = min(diag, nbs - 1);
    const int at = max(0, diag - nbt + 1) + (across ? int(blockIdx.y) : 4 * int(blockIdx.y) + q);
    const bool has = at <= last && (!across || 4 * int(blockIdx.x) + q < problems);
    if (__ballot(has) == 0) return;  // (the same for every wave of the workgroup)
    const int bi = min(at, last), bj = diag - bi;  // (a lane without a block repeats the last, unstored)
    const int64_t cells = int64_t(ls) * lt;
    float *D = a.dvals + pr.dv_off;
    float *DT = D + cells;
    const int i_l = min(B * bi + l, ls - 1), j_l = min(B * bj + l, lt - 1);  // this lane's row / column
    float *tile = pa_dyn_lds + wave * WAVE_LDS + q * TILE;

    // the block's similarities, lane l = row l, step s = column s - l (used by
    // the first wave; loaded first, to arrive during the folds)
    constexpr int STEPS = 2 * B - 1;
    float S[STEPS];
    if (wave == 0) {
#pragma unroll
        for (int s = 0; s < STEPS; ++s) S[s] = similarity<FORM>(a, pr, i_l, min(max(B * bj + s - l, 0), lt - 1));
    }

    // ---- the finished blocks above (lane = column, rows in registers) and to
    // the left (lane = row, columns in registers), and the borders; with
    // several waves, even ones take the columns above and odd ones the rows
    const int step = waves > 1 ? waves / 2 : 1, from = 1 + (waves > 1 ? wave / 2 : 0);
    float acc[B];
    if (waves == 1 || wave % 2 == 0) {
#pragma unroll
        for (int r = 0; r < B; ++r) acc[r] = W;
        if (wave == 0) {  // k = -1
            const float bt = a.border_t[j_l + 1];
#pragma unroll
            for (int r = 0; r < B; ++r) acc[r] = bt + ws[min(B * bi + r, ls - 1) + 1];
            if (carry && bi >= 2) {
                const float *c = carried(a, pr, int64_t(bi) * nbt + bj) + l;
#pragma unroll
                for (int r = 0; r < B; ++r) acc[r] = opt<DIR>(acc[r], c[r * B]);
            }
        }
        const int count = carry ? min(bi, 1) : bi;
        fold_blocks<DIR>(from, step, count, wave_most(count),
                         [&](int x) { return D + int64_t(B) * (bi - x) * lt + j_l; }, lt, ws, acc);
#pragma unroll
        for (int r = 0; r < B; ++r) tile[r * TS + l] = acc[r];
    }
    if (waves == 1) {
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    if (waves == 1 || wave % 2 == 1) {
#pragma unroll
        for (int c = 0; c < B; ++c) acc[c] = waves == 1 ? tile[l * TS + c] : W;
        if (wave <= 1) {
            const float bs = a.border_s[i_l + 1];
#pragma unroll
            for (int c = 0; c < B; ++c) acc[c] = opt<DIR>(acc[c], bs + wt[min(B * bj + c, lt - 1) + 1]);
            if (carry && bj >= 2) {
                const float *p = carried(a, pr, int64_t(bi) * nbt + bj) + B * B + l;
#pragma unroll
                for (int c = 0; c < B; ++c) acc[c] = opt<DIR>(acc[c], p[c * B]);
            }
        }
        const int count = carry ? min(bj, 1) : bj;
        fold_blocks<DIR>(from, step, count, wave_most(count),
                         [&](int x) { return DT + int64_t(B) * (bj - x) * ls + i_l; }, ls, wt, acc);
#pragma unroll
        for (int c = 0; c < B; ++c) tile[l * TS + c] = acc[c];
    }
    if (waves > 1) {
        __syncthreads();
        for (int e = int(threadIdx.x); e < WAVE_LDS; e += int(blockDim.x)) {
            float v = pa_dyn_lds[e];
            for (int p = 1; p < waves; ++p) v = opt<DIR>(v, pa_dyn_lds[p * WAVE_LDS + e]);
            pa_dyn_lds[e] = v;
        }
        __syncthreads();
        if (wave != 0) return;
    } else {
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }

    // ---- the block itself: lane l = row l, step s = column s - l ------------
    float A[STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) A[s] = tile[l * B + s];  // = row l, column s - l where that is in the block
    // D(row above, column l - 1) and D(row l - 1, column to the left)
    float top, left;
    {
        const int u = B * bi - 1, v = min(B * bj + l, lt) - 1;
        top = u < 0 ? a.border_t[v + 1] : (v < 0 ? a.border_s[u + 1] : D[int64_t(u) * lt + v]);
        const int y = min(B * bi + l, ls) - 1, x = B * bj - 1;
        left = x < 0 ? a.border_s[y + 1] : (y < 0 ? a.border_t[x + 1] : DT[int64_t(x) * ls + y]);
    }
    float wv[B], wh[B];  // costs of the pushes down (lane l reaches lane l + m) and along the row
    const float wt_l = wt[l];
#pragma unroll
    for (int m = 1; m < B; ++m) {
        wv[m] = l >= m ? ws[m] : W;
        wh[m] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wt_l), m));  // (a scalar)
    }
    // the block's values go to LDS by row and step (one wave's LDS accesses
    // stay in order; rows KS apart, a cell (r, c) at step r + c)
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    float *out = pa_dyn_lds + q * B * KS;
    float D1 = W, D2 = W;  // the last two steps' values
    static_for(std::make_integer_sequence<int, STEPS>{}, [&](auto step) {
        constexpr int s = decltype(step)::value;
        float dg = __int_as_float(row_shr1(row_first<s>(__float_as_int(top)), __float_as_int(D2)));
        if constexpr (s < B) dg = l == s ? left : dg;
        float v = opt<DIR>(dg + S[s], A[s]);
        if constexpr (LOC == LOC_LOCAL) v = opt<DIR>(v, 0.0f);
        if constexpr (s < B - 1) v = l <= s ? v : W;  // (columns past the block feed only their like)
        out[l * KS + s] = v;
        static_for(std::make_integer_sequence<int, B - 1>{}, [&](auto mm) {
            constexpr int m = decltype(mm)::value + 1;
            if constexpr (s + m < STEPS)
                A[s + m] = opt<DIR>(opt<DIR>(A[s + m], v + wh[m]), row_shr0<m>(v) + wv[m]);
        });
        D2 = D1;
        D1 = v;
    });
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (!has) return;
    const bool row_in = B * bi + l < ls, col_in = B * bj + l < lt;
    float bv = W;  // local: the block's best cell, the lowest row and then the last column of equals
    int br = -1, bc = l;
#pragma unroll
    for (int r = 0; r < B; ++r) {
        const float v = out[r * KS + r + l];
        if (B * bi + r < ls && col_in) {
            D[int64_t(B * bi + r) * lt + B * bj + l] = v;
            if (LOC == LOC_LOCAL && !better<DIR>(bv, v)) {
                bv = v;
                br = r;
            }
        }
    }
#pragma unroll
    for (int c = 0; c < B; ++c)
        if (row_in && B * bj + c < lt) DT[int64_t(B * bj + c) * ls + B * bi + l] = out[l * KS + l + c];
    if constexpr (LOC == LOC_LOCAL) {
#pragma unroll
        for (int m = 1; m < B; m <<= 1) {
            const float ov = __shfl_xor(bv, m, B);
            const int orow = __shfl_xor(br, m, B), oc = __shfl_xor(bc, m, B);
            if (orow >= 0 &&
                (br < 0 || better<DIR>(ov, bv) || (ov == bv && (orow > br || (orow == br && oc > bc))))) {
                bv = ov;
                br = orow;
                bc = oc;
            }
        }
        if (l == 0) {
            float *best = a.dvals + pr.rb_off + 2 * (int64_t(bi) * nbt + bj);
            best[0] = bv;
            best[1] = __int_as_float(br * B + bc);
        }
    }
}

// One wave per problem: the seed in the reference's visiting order
// (solver.h:2042-2057, 2179-2187, 2273-2293), the score and, with `path`, the
// one-optimal path (build_path, solver.h:858-935).  A cell's move is the first
// candidate in push order equal to its value: lane m tests whether the cell m
// moves on along the diagonal came from its diagonal, a ballot gives the run's
// length; at the run's end the lanes compare SCAN x 64 origins of a gap at a
// time.
constexpr int SCAN = 4;
template <int LOC, int DIR, int FORM>
__global__ __launch_bounds__(WAVE) void pa_wsb_finish_kernel(KArgs a, const float *__restrict__ ws,
                                                             const float *__restrict__ wt, int32_t *path,
                                                             const int64_t *path_off, int32_t *path_len) {
    constexpr float W = worst<DIR>();
    const Prob &pr = a.probs[blockIdx.x];
    const int ls = pr.len_s, lt = pr.len_t, lane = int(threadIdx.x);
    int32_t *P = path ? path + 2 * path_off[pr.out] : nullptr;
    if (ls <= 0 || lt <= 0) {
        if (lane == 0) {
            write_empty<LOC, DIR>(a, pr);
            if (path) {
                const int si = a.seeds[2 * pr.out], sj = a.seeds[2 * pr.out + 1];
                if (si != NO_SEED) {
                    P[0] = si;
                    P[1] = sj;
                }
                path_len[pr.out] = si == NO_SEED ? -1 : 1;
            }
        }
        return;
    }
    const int64_t cells = int64_t(ls) * lt;
    const float *D = a.dvals + pr.dv_off, *DT = D + cells;
    int si = ls - 1, sj = lt - 1;
    float score;
    if constexpr (LOC == LOC_GLOBAL) {
        score = D[cells - 1];
    } else {
        // (value, visiting position): local the last of equals by rows, then
        // columns; semiglobal the last row, then the last column.  Cells that
        // do not beat the worst value never seed.
        float bv = W;
        int64_t bp = -1;
        auto fold = [&](float v, int64_t p) {
            const bool earlier = LOC == LOC_LOCAL ? p > bp : p < bp;
            if (p >= 0 && better<DIR>(v, W) && (bp < 0 || better<DIR>(v, bv) || (v == bv && earlier))) {
                bv = v;
                bp = p;
            }
        };
        if constexpr (LOC == LOC_LOCAL) {
            const int nbs = (ls + B - 1) / B, nbt = (lt + B - 1) / B;
            const float *best = a.dvals + pr.rb_off;
            for (int64_t k = lane; k < int64_t(nbs) * nbt; k += WAVE) {
                const int rc = __float_as_int(best[2 * k + 1]);
                if (rc >= 0) fold(best[2 * k], (k / nbt * B + rc / B) * lt + k % nbt * B + rc % B);
            }
        } else {
            for (int64_t p = lane; p < int64_t(lt) + ls; p += WAVE)
                fold(p < lt ? D[int64_t(ls - 1) * lt + p] : D[(p - lt) * lt + (lt - 1)], p);
        }
        for (int m = 1; m < WAVE; m <<= 1) {
            const float ov = __shfl_xor(bv, m, WAVE);
            const int64_t op = __shfl_xor(bp, m, WAVE);
            fold(ov, op);
        }
        score = bp < 0 ? W : bv;
        if (bp < 0) {
            si = NO_SEED;
            sj = 0;
        } else if (LOC == LOC_LOCAL) {
            si = int(bp / lt);
            sj = int(bp % lt);
        } else {
            si = bp < lt ? ls - 1 : int(bp - lt);
            sj = bp < lt ? int(bp) : lt - 1;
        }
    }
    si = __builtin_amdgcn_readfirstlane(si);
    sj = __builtin_amdgcn_readfirstlane(sj);
    if (lane == 0) {
        a.scores[pr.out] = score;
        a.seeds[2 * pr.out] = si;
        a.seeds[2 * pr.out + 1] = sj;
    }
    if (!path) return;
    if (si == NO_SEED) {
        if (lane == 0) path_len[pr.out] = -1;
        return;
    }
    auto Dv = [&](int i, int j) -> float {  // D with its borders
        if (i < 0) return a.border_t[j + 1];
        if (j < 0) return a.border_s[i + 1];
        return D[int64_t(i) * lt + j];
    };
    int u = si, v = sj, cnt = 1;
    if (lane == 0) {
        P[0] = u;
        P[1] = v;
    }
    while (u >= 0 && v >= 0) {
        const int i = u - lane, j = v - lane;
        bool live = i >= 0 && j >= 0, diag = false;
        float x = W;
        if (live) {
            x = D[int64_t(i) * lt + j];
            diag = Dv(i - 1, j - 1) + similarity<FORM>(a, pr, i, j) == x;
            // Local stops where D is not above zero (solver.h:2117-2127)
            if constexpr (LOC == LOC_LOCAL) live = better<DIR>(x, 0.0f);
        }
        const uint64_t stays = __ballot(live && diag);
        const int n = ~stays == 0 ? WAVE : __builtin_ctzll(~stays);
        if (lane < n) {
            P[2 * (cnt + lane)] = i - 1;
            P[2 * (cnt + lane) + 1] = j - 1;
        }
        cnt += n;
        u -= n;
        v -= n;
        if (n == WAVE) continue;
        if (!((__ballot(live) >> n) & 1u)) break;
        x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), n));
        // the first origin k = -1 .. end - 1 whose candidate equals x
        auto origin = [&](float border, const float *base, const float *w, int end) -> int {
            for (int k0 = -1; k0 < end; k0 += SCAN * WAVE) {
                bool eq[SCAN];
#pragma unroll
                for (int c = 0; c < SCAN; ++c) {
                    const int k = k0 + c * WAVE + lane, kc = min(k, end - 1);
                    const float from = base[max(kc, 0)];
                    eq[c] = k < end && (kc < 0 ? border : from) + w[end - kc] == x;
                }
#pragma unroll
                for (int c = 0; c < SCAN; ++c) {
                    const uint64_t hit = __ballot(eq[c]);
                    if (hit) return k0 + c * WAVE + __builtin_ctzll(hit);
                }
            }
            return -2;
        };
        bool vertical = true;
        int to = origin(a.border_t[v + 1], DT + int64_t(v) * ls, ws, u);
        if (to == -2) {
            vertical = false;
            to = origin(a.border_s[u + 1], D + int64_t(u) * lt, wt, v);
        }
        if (to == -2) break;  // (every value is one of its candidates)
        if (vertical) u = to;
        else v = to;
        if (lane == 0) {
            P[2 * cnt] = u;
            P[2 * cnt + 1] = v;
        }
        ++cnt;
    }
    if (lane == 0) path_len[pr.out] = cnt;
}

template <int LOC, int DIR, int FORM>
hipError_t launch_blocks(const KArgs &a, const WsbPlan &plan, const float *ws, const float *wt, int32_t *path,
                         const int64_t *path_off, int32_t *path_len, hipStream_t st) {
    for (size_t d = 0; d < plan.diags.size(); ++d) {
        const WsbPlan::Diag &g = plan.diags[d];
        const int x = plan.across ? (g.problems + 3) / 4 : g.problems;
        hipLaunchKernelGGL((pa_wsb_block_kernel<LOC, DIR, FORM>),
                           dim3(unsigned(x), unsigned(g.groups + g.pushes)), dim3(unsigned(g.waves * WAVE)),
                           std::max(size_t(g.waves) * WAVE_LDS, size_t(MIN_LDS)) * 4, st, a, ws, wt, int(d),
                           int(g.problems), int(g.groups), int(plan.across), int(plan.carry));
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL((pa_wsb_finish_kernel<LOC, DIR, FORM>), dim3(unsigned(plan.n)), dim3(WAVE), 0, st, a, ws, wt,
                       path, path_off, path_len);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_wsb_blocks(int loc, int dir, int form, const KArgs &a, const WsbPlan &plan, const float *ws,
                             const float *wt, int32_t *path, const int64_t *path_off, int32_t *path_len,
                             hipStream_t st) {
    if (plan.n == 0) return hipSuccess;
#define PA_WSB(LC, DR, FM) return launch_blocks<LC, DR, FM>(a, plan, ws, wt, path, path_off, path_len, st)
#define PA_WSB_F(LC, DR)                                        \
    do {                                                        \
        if (form == F_DENSE) PA_WSB(LC, DR, F_DENSE);           \
        if (form == F_TABLE) PA_WSB(LC, DR, F_TABLE);           \
        if (form == F_TABLE_G) PA_WSB(LC, DR, F_TABLE_G);       \
        if (form == F_BINARY) PA_WSB(LC, DR, F_BINARY);         \
        return hipErrorInvalidValue;                            \
    } while (0)
    const bool mx = dir == DIR_MAX;
    switch (loc) {
        case LOC_LOCAL: if (mx) PA_WSB_F(LOC_LOCAL, DIR_MAX); else PA_WSB_F(LOC_LOCAL, DIR_MIN); break;
        case LOC_GLOBAL: if (mx) PA_WSB_F(LOC_GLOBAL, DIR_MAX); else PA_WSB_F(LOC_GLOBAL, DIR_MIN); break;
        default: if (mx) PA_WSB_F(LOC_SEMI, DIR_MAX); else PA_WSB_F(LOC_SEMI, DIR_MIN); break;
    }
#undef PA_WSB_F
#undef PA_WSB
}

}  // namespace pa
