// What the Q8 product kernels share: the matrices of a launch and the pieces
// of their epilogues.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "bf16_split.hpp"
#include "device_pool.hpp"

namespace nitro {

constexpr int Q8_BLOCK = 32;         // weights per block
constexpr int Q8_BLOCK_BYTES = 36;   // float scale + 32 int8
constexpr int Q8_TILE_BYTES = 576;   // a (16 rows, one block) record of the tile layout

// Up to 3 matrices sharing x (same n); out[m] is [batch][d[m]]; wt[m] the
// same matrix in the tile layout (or null).
struct Q8Group {
    const uint8_t* w[3];
    float* out[3];
    int d[3];
    const uint8_t* wt[3];
};

// Weight j (0..3) of a word of int8 weights, as a float.
__device__ __forceinline__ float q8_value(uint32_t w, int j) { return (float)(int)(int8_t)(w >> (8 * j)); }

__device__ __forceinline__ float inv_rms(float ss, int n) { return 1.0f / sqrtf(ss / (float)n + 1e-5f); }

// Partials first, first + step, ... of batch row b, added in that order, with
// no branch around the loads: an index past the end rereads the last partial
// and adds 0, so all L loads of a round go out together, behind any loads
// issued before.
template <int L>
__device__ __forceinline__ float partial_sum_unbranched(const Q8Norm& nm, int b, int first, int step) {
    float s = 0.0f;
    for (int p0 = first; p0 < nm.nparts; p0 += L * step) {
        float v[L];
#pragma unroll
        for (int i = 0; i < L; i++) v[i] = nm.ss[(size_t)min(p0 + i * step, nm.nparts - 1) * nm.ss_stride + b];
#pragma unroll
        for (int i = 0; i < L; i++) s += p0 + i * step < nm.nparts ? v[i] : 0.0f;
    }
    return s;
}

// Where batch row b's K/V goes and the position it rotates with.
struct RopeRow {
    int pos, page, in_page;
    bool page_ok;
};

__device__ __forceinline__ RopeRow rope_row(const Q8Rope& rp, int b) {
    const int w = b < rp.split ? 0 : 1;
    const int i = w ? b - rp.split : b;
    RopeRow r;
    r.pos = rp.pos[w][i];
    const int slot = rp.slot[w][i];
    r.page = slot >> 4;
    r.in_page = slot & 15;
    r.page_ok = r.page >= 0 && r.page < rp.num_pages;
    return r;
}

// (x, y) rotated by the angle of pair f of position pos: the reference's
// (x*fcr - y*fci, x*fci + y*fcr) (src/model_q8.cpp:600-612).
__device__ __forceinline__ float2 rotate_pair(const Q8Rope& rp, int pos, int feature, float x, float y) {
    const int f = (feature % rp.head_dim) >> 1;
    const float c = rp.freq_real[(size_t)pos * (rp.head_dim >> 1) + f];
    const float sn = rp.freq_imag[(size_t)pos * (rp.head_dim >> 1) + f];
    return make_float2(x * c - y * sn, x * sn + y * c);
}

// Byte offset of (row, column k)'s part 0 in split form (part p: + 1024 p).
__device__ __forceinline__ size_t split_at(int row, int k, int nb) {
    return ((size_t)(row >> 4) * nb + (k >> 5)) * Q8_SPLIT_BYTES + ((row & 15) + 16 * ((k >> 3) & 3)) * 16 + (k & 7) * 2;
}

// One value of a product's output in split form.
__device__ __forceinline__ void store_split(const Q8SplitOut& o, int row, int k, float v) {
    if (o.weight) v *= o.weight[k];
    uint16_t hi, mid, lo;
    split_parts(v, hi, mid, lo);
    char* dst = o.planes + split_at(row, k, o.nb);
    *reinterpret_cast<uint16_t*>(dst) = hi;
    *reinterpret_cast<uint16_t*>(dst + 1024) = mid;
    *reinterpret_cast<uint16_t*>(dst + 2048) = lo;
}

// What a large product does with its sums.
enum class Q8Epilogue { Store, Residual, SwiGlu, Rope };

// Compute units of the current device (256 where there is none).
int device_cus();

// Whether NITRO_Q8_MMA leaves the bf16 matrix-core kernels in use.
bool use_mma();

// Weight rows per workgroup (128 or 64) with which the large-batch kernel takes a
// launch over matrices of d[] rows (wq, wk, wv; w1, w3 of d[0]; or one), 0 where it
// does not.
int q8_gemm_tile(Q8Epilogue epilogue, const int* d, int batch, int n);

// The large-batch product (q8_gemm.hip): true if launched, false where the
// shapes are not its own (the caller takes another kernel).
bool launch_q8_gemm(Q8Epilogue epilogue, const Q8Group& grp, const float* x, const Q8Split& split, int batch, int n,
                    const Q8Norm& nm, const Q8Resid& resid, const Q8Rope& rope, hipStream_t stream);

}  // namespace nitro
