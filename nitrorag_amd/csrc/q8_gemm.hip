// Q8_0 products over many activation rows (prompts) for gfx950 (MI355X):
// out[b][i] = sum_k w[i][k] * x[b][k], full rows, at fp32 accuracy on the bf16
// matrix cores, with the residual add, SwiGLU and RoPE + K/V append folded in
// as in the other Q8 kernels (src/model_q8.cpp:382-420, :447-557).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "bf16_split.hpp"
#include "q8_group.hpp"

namespace nitro {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// q8_gemm_kernel: a workgroup of 4 waves owns 128 batch rows x 16 NT weight
// rows (128 or 64); wave w owns batch rows 32w..32w+31 and all the weight rows,
// as 2 x NT tiles of v_mfma_f32_16x16x32_bf16 (lane l: A = batch row l%16, B =
// weight row l%16, k = 8*(l/16) .. +8 of a 32-k block).
//  - x, as the exact sum of three bf16 parts: a wave alone reads its rows, so
//    they go to registers and not through LDS.  PRE: the parts were written
//    in operand order where x was made, 1 KB per load instruction;
//    otherwise the wave splits its rows itself, once per 16 NT weight rows.
//    (Split per 16 weight rows, as q8_mma_kernel does, and read again from L2
//    each time, x cost more than the products.)
//  - weights: a block of the rows is converted to bf16 (exact) into LDS, shared
//    by the waves; two buffers, one barrier per block.  A row's four 16-byte
//    runs are swizzled by (row / 2) % 4, so that 8 lanes reading or writing
//    consecutive rows hit distinct banks (no conflict cycles in wq/wk/wv and
//    q8_matmul; 0.05 per LDS instruction in the others, from their epilogues).
//  - per block and tile, three products (lo, mid, hi parts) from zero give
//    sum_k q*x, which is scaled into the accumulators by the lane's own weight
//    row's scale.  Every GEMM_FLUSH blocks the accumulators are added to sums in
//    LDS, so that no chain of fp32 adds is longer than GEMM_FLUSH + n / (32
//    GEMM_FLUSH): error against 64 bits 0.78e-7 / 0.97e-7 / 1.2e-7 / 1.75e-7
//    (2-norm) at n = 768 / 2048 / 4096 / 11008, as q8_mma_kernel's 0.80 / 0.97
//    / 1.2 / 1.74, which adds eight waves' chains; one chain gave 1.0e-7 at 768.
// Bound by the matrix cores and, at n = 768, by the first and last blocks of a
// tile: w1/w3 of 5520 rows at 768 x 2048 370 -> 117 us with hb written split
// (0.89 PFLOP/s of bf16 products, three per multiply), wq/wk/wv 216 -> 89, wo
// 99 -> 39, w2 251 -> 78.  The matrix cores are busy in 45% of the CUs' cycles in
// w1/w3, 36% in wq/wk/wv, wo and w2, 37 and 29% in q8_matmul of 1024 rows at 4096 x
// 11008 (w1, w2), where a plain 8192^3 bf16 product has 73%.  Prompts of 8 users,
// 110M-parameter shapes: 11.96 -> 4.5 ms; q8_matmul of 1024 rows, 4096 x 11008,
// three products: 5.18 -> 1.08 ms.
constexpr int GEMM_WAVES = 4;
constexpr int GEMM_BM = 32 * GEMM_WAVES;
constexpr int GEMM_MT = 2;            // 16-row batch tiles per wave
constexpr int GEMM_FLUSH = 8;

// The 16-byte run c (8 k) of a row in an LDS weight buffer (64 bytes a row).
__device__ __forceinline__ int w_at(int row, int c) { return row * 32 + ((c ^ (row >> 1)) & 3) * 8; }

// A model's launches (all but Store) read its matrices in the tile layout and x in
// split form (PRE); q8_matmul's have neither.
template <Q8Epilogue EPI, int GEMM_NT>
__global__ __launch_bounds__(64 * GEMM_WAVES, GEMM_NT == 8 ? 2 : 3) void q8_gemm_kernel(Q8Group grp, const void* __restrict__ xin,
                                                                     int batch, int n, int col_tiles, Q8Norm nm, Q8Resid resid,
                                                                     Q8SplitOut out, Q8Rope rope) {
    constexpr bool TILED = EPI != Q8Epilogue::Store, PRE = TILED;
    constexpr int GEMM_BN = 16 * GEMM_NT;
    constexpr bool NORM = EPI == Q8Epilogue::SwiGlu || EPI == Q8Epilogue::Rope;
    constexpr bool SWIGLU = EPI == Q8Epilogue::SwiGlu;
    constexpr int MROWS = SWIGLU ? GEMM_BN / 2 : GEMM_BN;  // rows of a member per workgroup
    __shared__ __attribute__((aligned(16))) uint16_t wlds[2][GEMM_BN * 32];
    __shared__ f32x4 sums[GEMM_WAVES][GEMM_MT * GEMM_NT][64];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int lr = lane & 15, lg = lane >> 4;

    // Work order: column tiles fastest, XCD i taking the i-th eighth of it, so
    // an XCD's workgroups share a few panels of x and the weights in its L2.
    int wg = blockIdx.x;
    {
        const int total = gridDim.x, per = total >> 3, rem = total & 7, xcd = wg & 7;
        wg = xcd * per + min(xcd, rem) + (wg >> 3);
    }
    const int b0 = wg / col_tiles * GEMM_BM + wave * 32;  // this wave's first batch row
    int ct = wg % col_tiles, member = 0;
    if constexpr (EPI == Q8Epilogue::Rope) {  // the column tiles of wq, then wk, then wv
        for (; member < 2; member++) {
            const int t = (grp.d[member] + GEMM_BN - 1) / GEMM_BN;
            if (ct < t) break;
            ct -= t;
        }
    }
    const int row0 = ct * MROWS;  // first weight row (of each member with SwiGLU)
    const int d = grp.d[member];
    const int nb = n / Q8_BLOCK;

    // 32-bit byte offsets from bases that are the same for the workgroup (the
    // launcher keeps each matrix and x under 2^32 bytes).
    auto wrow_of = [&](int r) { return min(row0 + (SWIGLU ? r % MROWS : r), d - 1); };
    constexpr uint32_t BSTEP = TILED ? Q8_TILE_BYTES : Q8_BLOCK_BYTES;
    // Staging units: 8 weights of one row, UNITS per thread (a wave's unit is of
    // one member's rows).
    constexpr int THREADS = 64 * GEMM_WAVES;
    constexpr int UNITS = GEMM_BN * 4 / THREADS;
    auto base_of = [&](int m) { return TILED ? grp.wt[m] : grp.w[m]; };
    const uint8_t* wbase[UNITS];
    uint32_t woff[UNITS];
    int wdst[UNITS];
#pragma unroll
    for (int u = 0; u < UNITS; u++) {
        const int e = threadIdx.x + u * THREADS;
        const int r = TILED ? e / 64 * 16 + e % 16 : e / 4;
        const int c = TILED ? e % 64 / 16 : e % 4;
        const uint32_t row = wrow_of(r);
        wbase[u] = base_of(__builtin_amdgcn_readfirstlane(SWIGLU ? r / MROWS : member));
        woff[u] = TILED ? row / 16 * nb * Q8_TILE_BYTES + 64 + 8 * (row % 16 + 16 * c)
                        : row * nb * Q8_BLOCK_BYTES + 4 + 8 * c;
        wdst[u] = w_at(r, c);
    }
    // A block's scales, one per lane of each 64 weight rows: a tile's are handed
    // to its lanes by a permute.  (Loaded per tile, 16 rows by each of 4 lane
    // groups, they took twice the address slots of row-major x: three products of
    // 1024 rows at 4096 x 11008 1.70 -> 1.10 ms, 8 prompts of the 110M-parameter
    // shapes 4.72 -> 4.56 ms.)
    constexpr int SC = GEMM_NT / 4;
    const uint8_t* sbase[SC];
#pragma unroll
    for (int u = 0; u < SC; u++) {
        const int rr = 64 * u + lane;
        const uint32_t row = wrow_of(rr);
        sbase[u] = base_of(SWIGLU ? rr / MROWS : member) +
                   (TILED ? row / 16 * nb * Q8_TILE_BYTES + 4 * (row % 16) : row * nb * Q8_BLOCK_BYTES);
    }
    // x of the wave's two 16-row tiles: their planes (PRE; tiles clamped), or the
    // batch rows this lane feeds (clamped: never stored).
    uint32_t xoff[GEMM_MT];
#pragma unroll
    for (int m = 0; m < GEMM_MT; m++)
        xoff[m] = PRE ? (uint32_t)min(b0 / 16 + m, (batch - 1) / 16) * nb * Q8_SPLIT_BYTES + 16 * lane
                      : ((uint32_t)min(b0 + 16 * m + lr, batch - 1) * n + 8 * lg) * 4;
    constexpr uint32_t XSTEP = PRE ? Q8_SPLIT_BYTES : Q8_BLOCK * 4;

    // The i-th block (past the end: the last).  Every workgroup walks the blocks in
    // the same order, so equal rows give equal bits wherever they lie.  (Starting
    // at different blocks for row-major x, whose rows sit on one L2 channel when
    // they are a multiple of 4 KB apart, gained 1.2% at 192 and 256 rows of 4096 x
    // 11008 and lost up to 1.9% elsewhere.)
    auto walk = [&](int i) __attribute__((always_inline)) { return min(i, nb - 1); };
    // A block's loads.  None is behind a branch (a block past the end rereads
    // the last), so that each wait counts exactly the loads it needs.
    struct WRound {
        uint32_t q[UNITS][2];
    };
    struct XRound {
        u32x4 v[GEMM_MT][PRE ? 3 : 2];  // PRE: hi, mid, lo; else 8 floats
        float sc[SC];
    };
    auto load_w = [&](WRound& R, int blk) __attribute__((always_inline)) {
        const size_t step = (size_t)((uint32_t)walk(blk) * BSTEP);
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            const uint8_t* p = wbase[u] + step + woff[u];
            if constexpr (TILED) {
                const uint2 v = *reinterpret_cast<const uint2*>(p);
                R.q[u][0] = v.x, R.q[u][1] = v.y;
            } else {
                R.q[u][0] = reinterpret_cast<const uint32_t*>(p)[0];
                R.q[u][1] = reinterpret_cast<const uint32_t*>(p)[1];
            }
        }
    };
    auto load_x = [&](XRound& R, int blk) __attribute__((always_inline)) {
        blk = walk(blk);
        const char* xb = static_cast<const char*>(xin) + (size_t)((uint32_t)blk * XSTEP);
#pragma unroll
        for (int m = 0; m < GEMM_MT; m++)
#pragma unroll
            for (int i = 0; i < (PRE ? 3 : 2); i++)
                R.v[m][i] = *reinterpret_cast<const u32x4*>(xb + xoff[m] + (PRE ? 1024 : 16) * i);
#pragma unroll
        for (int u = 0; u < SC; u++) R.sc[u] = *reinterpret_cast<const float*>(sbase[u] + (size_t)((uint32_t)blk * BSTEP));
    };
    auto stage_w = [&](const WRound& R, int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            u32x4 v;
#pragma unroll
            for (int i = 0; i < 4; i++)
                v[i] = bf16_pair(q8_value(R.q[u][i >> 1], 2 * (i & 1)), q8_value(R.q[u][i >> 1], 2 * (i & 1) + 1));
            *reinterpret_cast<u32x4*>(&wlds[buf][wdst[u]]) = v;
        }
    };
    f32x4 acc[GEMM_MT][GEMM_NT];
#pragma unroll
    for (int m = 0; m < GEMM_MT; m++)
#pragma unroll
        for (int t = 0; t < GEMM_NT; t++) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Sums of the two weight tiles last multiplied, not yet scaled in.
    f32x4 late[GEMM_MT][2];
    float late_sc[2] = {0.f, 0.f};
#pragma unroll
    for (int m = 0; m < GEMM_MT; m++) late[m][0] = late[m][1] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Block blk: its x and scales in xc, the next one's weights in wn.  The
    // next x and scales go out first.  Two weight tiles at a time: the next
    // two tiles' weights are read from LDS, then the products (lo, mid, hi parts
    // from zero) issue with the scaling of the two tiles before them, and the
    // next block's staging, between them.
    auto step = [&](int blk, XRound& xc, XRound& xn, WRound& wn) __attribute__((always_inline)) {
        __syncthreads();  // block blk is staged; the other buffer's readers are done
        const uint16_t* wb = wlds[blk & 1];
        bf16x8 w[GEMM_NT];
        auto read_w = [&](int t) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < 2; u++) w[t + u] = *reinterpret_cast<const bf16x8*>(&wb[w_at(16 * (t + u) + lr, lg)]);
        };
        read_w(0);
        load_x(xn, blk + 1);
        __builtin_amdgcn_sched_barrier(0);  // (left free, the scheduler sinks the loads to the block's end)
        bf16x8 xp[GEMM_MT][3];  // x of this block: hi, mid, lo
#pragma unroll
        for (int m = 0; m < GEMM_MT; m++) {
            if constexpr (PRE) {
#pragma unroll
                for (int p = 0; p < 3; p++) xp[m][p] = __builtin_bit_cast(bf16x8, xc.v[m][p]);
            } else {
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; i++) v[i] = __uint_as_float(xc.v[m][i >> 2][i & 3]);
                split3(v, xp[m][0], xp[m][1], xp[m][2]);
            }
        }
#pragma unroll
        for (int t = 0; t < GEMM_NT; t += 2) {
            if (t + 2 < GEMM_NT) read_w(t + 2);
            f32x4 s[GEMM_MT][2];
#pragma unroll
            for (int p = 2; p >= 0; p--)
#pragma unroll
                for (int m = 0; m < GEMM_MT; m++)
#pragma unroll
                    for (int u = 0; u < 2; u++)
                        s[m][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            xp[m][p], w[t + u], p == 2 ? f32x4{0.f, 0.f, 0.f, 0.f} : s[m][u], 0, 0, 0);
            constexpr int LAST = GEMM_NT - 2;
            const int tl = t ? t - 2 : LAST;  // the tiles of `late`
#pragma unroll
            for (int m = 0; m < GEMM_MT; m++)
#pragma unroll
                for (int u = 0; u < 2; u++) {
#pragma unroll
                    for (int i = 0; i < 4; i++) acc[m][tl + u][i] = fmaf(late_sc[u], late[m][u][i], acc[m][tl + u][i]);
                    late[m][u] = s[m][u];
                }
#pragma unroll
            for (int u = 0; u < 2; u++)
                late_sc[u] = __int_as_float(
                    __builtin_amdgcn_ds_bpermute(4 * (16 * ((t + u) % 4) + lr), __float_as_int(xc.sc[t / 4])));
            if (t == 0) stage_w(wn, (blk + 1) & 1);
            if (t == 2) load_w(wn, blk + 3);
            if (t + 2 < GEMM_NT) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);  // LDS reads
#pragma unroll
            for (int i = 0; i < 12; i++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);               // a product
                __builtin_amdgcn_sched_group_barrier(0x002, 3, 0);  // VALU
            }
        }
    };
    // The last two tiles' sums into their accumulators.
    auto scale_late = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int m = 0; m < GEMM_MT; m++)
#pragma unroll
            for (int u = 0; u < 2; u++) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    acc[m][GEMM_NT - 2 + u][i] = fmaf(late_sc[u], late[m][u][i], acc[m][GEMM_NT - 2 + u][i]);
                late[m][u] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        late_sc[0] = late_sc[1] = 0.f;
    };
    // (late sums included, after the other tiles: every tile's chains hold the
    // same blocks)
    auto flush = [&](bool first) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < GEMM_NT; t++) {
            if (t == GEMM_NT - 2) scale_late();
#pragma unroll
            for (int m = 0; m < GEMM_MT; m++) {
                f32x4& slot = sums[wave][m * GEMM_NT + t][lane];
                slot = first ? acc[m][t] : slot + acc[m][t];
                acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
    };
    WRound wa, wb;
    XRound xa, xb;
    load_w(wb, 0);
    load_x(xa, 0);
    load_w(wa, 1);
    stage_w(wb, 0);
    load_w(wb, 2);
    float inv = 1.0f;  // 1/rms of batch row b0 + lane % 32
    if constexpr (NORM) {  // lanes l and l + 32 add a row's even and odd partials
        float ss = partial_sum_unbranched<16>(nm, min(b0 + (lane & 31), batch - 1), lane >> 5, 2);
        ss += __shfl_xor(ss, 32);
        inv = inv_rms(ss, n);
    }
    static_assert(GEMM_FLUSH % 2 == 0, "blocks in pairs");
    int blk = 0;
    for (int end = GEMM_FLUSH; end <= nb; end += GEMM_FLUSH) {
#pragma unroll 1
        for (; blk < end; blk += 2) {
            step(blk, xa, xb, wa);
            step(blk + 1, xb, xa, wb);
        }
        flush(end == GEMM_FLUSH);
    }
#pragma unroll 1
    for (; blk + 1 < nb; blk += 2) {
        step(blk, xa, xb, wa);
        step(blk + 1, xb, xa, wb);
    }
    if (blk < nb) step(blk, xa, xb, wa);
    scale_late();
    if (nb >= GEMM_FLUSH) {
#pragma unroll
        for (int m = 0; m < GEMM_MT; m++)
#pragma unroll
            for (int t = 0; t < GEMM_NT; t++) acc[m][t] += sums[wave][m * GEMM_NT + t][lane];
    }

    // The next norm's weights of the lane's split columns, loaded before any store.
    float out_w[EPI == Q8Epilogue::Residual ? GEMM_BN / 32 : 1][8];
    if constexpr (EPI == Q8Epilogue::Residual) {
        if (out.planes && out.weight) {  // uniform
#pragma unroll
            for (int j = 0; j < GEMM_BN / 32; j++)
#pragma unroll
                for (int i = 0; i < 8; i++) out_w[j][i] = out.weight[min(row0 + 32 * j + 8 * lg, d - 8) + i];
        }
    }

    // Lane l holds out[b0 + 16m + 4*(l/16) + i][16t + l%16] in acc[m][t][i].
#pragma unroll
    for (int m = 0; m < GEMM_MT; m++) {
        const int bm = b0 + 16 * m + 4 * lg;
        if constexpr (NORM) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float f = __shfl(inv, 16 * m + 4 * lg + i);
#pragma unroll
                for (int t = 0; t < GEMM_NT; t++) acc[m][t][i] *= f;
            }
        }
        // The wave's 16 x COLS outputs of tile m through LDS (rows 4 floats
        // apart in banks) into split form, one run of 8 columns per lane.
        constexpr int COLS = SWIGLU ? GEMM_BN / 2 : GEMM_BN;
        float* const rows = reinterpret_cast<float*>(&sums[wave][0][0]);
        static_assert(16 * (COLS + 4) <= GEMM_MT * GEMM_NT * 256, "the outputs fit the wave's sums");
        // Lanes read what other lanes of the wave wrote there, and write where others
        // read: no access may pass another between them.
        auto exchange = []() __attribute__((always_inline)) {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        };
        auto write_split = [&]() __attribute__((always_inline)) {
            exchange();
            if (b0 + 16 * m >= batch) return;  // wave-uniform
#pragma unroll
            for (int j = 0; j < COLS / 32; j++) {
                const int k = row0 + 32 * j + 8 * lg;
                if (row0 + 32 * j >= d) break;  // uniform (d is a multiple of 32)
                const float* src = rows + lr * (COLS + 4) + 32 * j + 8 * lg;
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; i++) v[i] = EPI == Q8Epilogue::Residual && out.weight ? src[i] * out_w[j][i] : src[i];
                bf16x8 p[3];
                split3(v, p[0], p[1], p[2]);
                char* dst = out.planes + split_at(b0 + 16 * m + lr, k, out.nb);
#pragma unroll
                for (int i = 0; i < 3; i++) *reinterpret_cast<bf16x8*>(dst + 1024 * i) = p[i];
            }
        };
        if constexpr (SWIGLU || EPI == Q8Epilogue::Residual) exchange();
        if constexpr (SWIGLU) {
            // the first half of the tiles are w1's rows, the second the same rows of w3
#pragma unroll
            for (int t = 0; t < GEMM_NT / 2; t++) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float h = acc[m][t][i];
                    h *= 1.0f / (1.0f + expf(-h));
                    h *= acc[m][t + GEMM_NT / 2][i];
                    rows[(4 * lg + i) * (COLS + 4) + 16 * t + lr] = h;
                }
            }
            write_split();
        } else if constexpr (EPI == Q8Epilogue::Residual) {
            // x += product; the squares of the new entries are added over each
            // 16-row tile's 16 lanes (one partial per batch row and tile)
            // (every x is loaded before the first store: a load behind a store
            // that may alias it waits its turn, one round trip per tile)
            float xv[GEMM_NT][4];
#pragma unroll
            for (int t = 0; t < GEMM_NT; t++)
#pragma unroll
                for (int i = 0; i < 4; i++)
                    xv[t][i] = grp.out[0][(size_t)min(bm + i, batch - 1) * d + min(row0 + 16 * t + lr, d - 1)];
#pragma unroll
            for (int t = 0; t < GEMM_NT; t++) {
                const int row = row0 + 16 * t + lr;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float v = xv[t][i] + acc[m][t][i];
                    const bool ok = bm + i < batch && row < d;
                    if (ok) grp.out[0][(size_t)(bm + i) * d + row] = v;
                    rows[(4 * lg + i) * (COLS + 4) + 16 * t + lr] = v;
                    float sq = ok ? v * v : 0.0f;
#pragma unroll
                    for (int msk = 8; msk > 0; msk >>= 1) sq += __shfl_xor(sq, msk, 16);
                    if (lr == 0 && ok) resid.ss[(size_t)(row >> 4) * resid.ss_stride + bm + i] = sq;
                }
            }
            if (out.planes) write_split();  // uniform
        } else if constexpr (EPI == Q8Epilogue::Rope) {
            // RoPE pairs are adjacent weight rows, so adjacent lanes; the rows'
            // slots and angles are loaded before the first store, as above
            RopeRow rr[4];
            float cs[4][GEMM_NT], sn[4][GEMM_NT];
#pragma unroll
            for (int i = 0; i < 4; i++) rr[i] = rope_row(rope, min(bm + i, batch - 1));
            if (member < 2) {  // uniform
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int t = 0; t < GEMM_NT; t++) {
                        const size_t f = (size_t)rr[i].pos * (rope.head_dim >> 1) + ((row0 + 16 * t + lr) % rope.head_dim >> 1);
                        cs[i][t] = rope.freq_real[f];
                        sn[i][t] = rope.freq_imag[f];
                    }
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int b = bm + i;
#pragma unroll
                for (int t = 0; t < GEMM_NT; t++) {
                    const int row = row0 + 16 * t + lr;
                    const float mine = acc[m][t][i], other = __shfl_xor(mine, 1);
                    if (b >= batch || row >= d) continue;
                    float v = mine;
                    if (member < 2)  // rotate_pair's (x*c - y*sn, x*sn + y*c)
                        v = row & 1 ? other * sn[i][t] + mine * cs[i][t] : mine * cs[i][t] - other * sn[i][t];
                    if (member == 0) {
                        grp.out[0][(size_t)b * d + row] = v;
                    } else if (rr[i].page_ok) {
                        float* pool = member == 1 ? rope.k_pool : rope.v_pool;
                        pool[(size_t)rr[i].page * rope.page_stride + rope.layer_off + (size_t)rr[i].in_page * d + row] = v;
                    } else if (member == 1 && row == 0) {
                        atomicAdd(rope.bad_pages, 1);  // once per row
                    }
                }
            }
        } else {
#pragma unroll
            for (int t = 0; t < GEMM_NT; t++) {
                const int row = row0 + 16 * t + lr;
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (bm + i < batch && row < d) grp.out[0][(size_t)(bm + i) * d + row] = acc[m][t][i];
            }
        }
    }
}

// fp32 activations to split form: workgroup (tile, group) takes 16 rows x 16
// blocks, wave w blocks w, w + 4, ..; a lane reads a run of 8 k and writes it as
// three bf16 runs.
__global__ __launch_bounds__(256) void q8_split_kernel(const float* __restrict__ x, char* __restrict__ out, int rows,
                                                       int n) {
    const int nb = n / Q8_BLOCK;
    const int lane = threadIdx.x & 63;
    const int row = blockIdx.x * 16 + (lane & 15);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int blk = blockIdx.y * 16 + 4 * i + (threadIdx.x >> 6);
        if (blk >= nb) break;  // wave-uniform
        const int k = blk * Q8_BLOCK + 8 * (lane >> 4);
        const float4* src = reinterpret_cast<const float4*>(x + (size_t)min(row, rows - 1) * n + k);
        const float4 a = src[0], b = src[1];
        const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        bf16x8 p[3];
        split3(v, p[0], p[1], p[2]);
        char* dst = out + split_at(row, k, nb);
#pragma unroll
        for (int j = 0; j < 3; j++) *reinterpret_cast<bf16x8*>(dst + 1024 * j) = p[j];
    }
}

template <Q8Epilogue EPI, int NT>
void launch(dim3 grid, hipStream_t stream, const Q8Group& grp, const void* x, int batch, int n, int cols,
            const Q8Norm& nm, const Q8Resid& resid, const Q8SplitOut& out, const Q8Rope& rope) {
    hipLaunchKernelGGL((q8_gemm_kernel<EPI, NT>), grid, dim3(64 * GEMM_WAVES), 0, stream, grp, x, batch, n, cols, nm,
                       resid, out, rope);
}

}  // namespace

namespace {
int members_of(Q8Epilogue e) { return e == Q8Epilogue::Rope ? 3 : e == Q8Epilogue::SwiGlu ? 2 : 1; }

// Column tiles of `rows` weight rows (with SwiGLU, of w1 and w3 in equal parts).
int columns(Q8Epilogue e, const int* d, int rows) {
    if (e == Q8Epilogue::SwiGlu) return (d[0] + rows / 2 - 1) / (rows / 2);
    int c = 0;
    for (int m = 0; m < members_of(e); m++) c += (d[m] + rows - 1) / rows;
    return c;
}
}  // namespace

int q8_gemm_tile(Q8Epilogue epilogue, const int* d, int batch, int n) {
    const int members = members_of(epilogue);
    const bool pre = epilogue != Q8Epilogue::Store;
    const int dmax = epilogue == Q8Epilogue::Rope ? std::max(d[0], std::max(d[1], d[2])) : d[0];
    if (q8_tiled_bytes(dmax, n) >= (1ull << 32) || q8_split_bytes(batch, n) >= (1ull << 32)) return 0;
    // 128 or 64 weight rows per workgroup: whichever fills its dispatch rounds
    // better (two or three workgroups per CU; a round costs about the same
    // however full it is).  wo at 5520 x 768: 264 wide workgroups 51 us, 528
    // narrow 39; at 1600 x 4096, 416 wide ones fit a round and 832 narrow ones
    // do not: 4.20 ms per pass against 4.38.  Where a wave splits x itself, it
    // does so twice as often with 64, hence the 0.75 (also from an earlier form).
    const long long cus = device_cus();
    const long long panels = (batch + GEMM_BM - 1) / GEMM_BM;
    const long long wide = panels * columns(epilogue, d, 128), slim = panels * columns(epilogue, d, 64);
    const long long wide_rounds = (wide + 2 * cus - 1) / (2 * cus), slim_rounds = (slim + 3 * cus - 1) / (3 * cus);
    const double wide_fill = (double)wide / (wide_rounds * 2 * cus), slim_fill = (double)slim / (slim_rounds * 3 * cus);
    const bool narrow = slim_fill * (pre ? 1.0 : 0.75) > wide_fill;
    // From how many outputs per dispatch round this kernel is taken.  The line was
    // fitted to an earlier form of it and is cautious for the present one: no
    // product measured goes to this kernel where the small-batch one is faster, but
    // the 64-row tile would win sooner and more often.  One product, small-batch /
    // 64 rows / 128 rows, us (the rule's choice in brackets): 256 rows of 2048 x
    // 2048 [47] / 42 / 66, of 4096 x 4096 [169] / 84 / 131; 64 rows of 11008 x 4096
    // [128] / 79 / 128, 128 rows 232 / 84 / [130]; 512 rows of 4096 x 4096 335 / 87 /
    // [131], of 2048 x 768 [31] / 19 / 29; 1024 of 2048 x 768 59 / 20 / [29].
    double outputs = 0;
    for (int m = 0; m < members; m++) outputs += (double)batch * d[epilogue == Q8Epilogue::SwiGlu ? 0 : m];
    if ((narrow ? slim : wide) > (1ll << 30) || outputs < (narrow ? 830e3 * slim_rounds : 1080e3 * wide_rounds)) return 0;
    return narrow ? 64 : 128;
}

int q8_tile_rows(int launch, int batch, int n, int d, int d_kv) {
    const Q8Epilogue epilogue[] = {Q8Epilogue::Store, Q8Epilogue::Residual, Q8Epilogue::SwiGlu, Q8Epilogue::Rope};
    const int ds[3] = {d, d_kv, d_kv};
    return batch > Q8_GEMV_MAX_BATCH && use_mma() ? q8_gemm_tile(epilogue[launch], ds, batch, n) : 0;
}

bool launch_q8_gemm(Q8Epilogue epilogue, const Q8Group& grp, const float* x, const Q8Split& split, int batch, int n,
                    const Q8Norm& nm, const Q8Resid& resid, const Q8Rope& rope, hipStream_t stream) {
    const bool pre = epilogue != Q8Epilogue::Store;
    if (pre)
        for (int m = 0; m < members_of(epilogue); m++)
            if (!grp.wt[m]) return false;
    if (pre && !split.in && (!split.scratch || nm.weight)) return false;
    if (epilogue == Q8Epilogue::SwiGlu && !split.out.planes) return false;
    const int rows = q8_gemm_tile(epilogue, grp.d, batch, n);
    if (rows == 0) return false;
    const int cols = columns(epilogue, grp.d, rows);
    const dim3 grid((unsigned)((batch + GEMM_BM - 1) / GEMM_BM * cols));
    const void* in = x;
    if (pre && split.in) {
        in = split.in;
    } else if (pre) {
        hipLaunchKernelGGL(q8_split_kernel, dim3((unsigned)((batch + 15) / 16), (unsigned)((n / Q8_BLOCK + 15) / 16)),
                           dim3(256), 0, stream, x, static_cast<char*>(split.scratch), batch, n);
        in = split.scratch;
    }
    const auto run = [&](auto nt) {
        constexpr int NT = decltype(nt)::value;
        switch (epilogue) {
            case Q8Epilogue::Store: launch<Q8Epilogue::Store, NT>(grid, stream, grp, in, batch, n, cols, nm, resid, split.out, rope); break;
            case Q8Epilogue::Residual: launch<Q8Epilogue::Residual, NT>(grid, stream, grp, in, batch, n, cols, nm, resid, split.out, rope); break;
            case Q8Epilogue::SwiGlu: launch<Q8Epilogue::SwiGlu, NT>(grid, stream, grp, in, batch, n, cols, nm, resid, split.out, rope); break;
            case Q8Epilogue::Rope: launch<Q8Epilogue::Rope, NT>(grid, stream, grp, in, batch, n, cols, nm, resid, split.out, rope); break;
        }
    };
    if (rows == 64)
        run(std::integral_constant<int, 4>{});
    else
        run(std::integral_constant<int, 8>{});
    return true;
}

}  // namespace nitro
