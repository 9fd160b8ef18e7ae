// Prefill GEMMs whose tiles do not fill the CUs in whole rounds: the K split of the remaining tiles and the sum of their
// partials (shared by the bf16 and the INT8 MFMA kernels).
#pragma once
#include "mfma_tile.hpp"

namespace qe_tile {

enum Out : int { kOutF32 = 0, kOutBF16 = 1, kOutGLU = 2 };
constexpr int kMaxSplit = 16;
// the most partial-sum workspace a split may take: one 256 x 256 fp32 tile per CU (64 MB)
inline size_t max_split_bytes() { return (size_t)qe_num_cus() * 256 * 256 * 4; }

// Split tiles: the tiles from `ndirect` on run as `ks` K ranges of whole 128-k groups each (the last, partly filled
// round, or every tile when they do not fill one round); their fp32 partials go to
// part [(tile - ndirect) * ks + split][BM][BN] and splitk_reduce_kernel adds them
struct SplitArgs {
    int ndirect = 1 << 30;
    int ks = 1;
    float* part = nullptr;
};

// Block j of the split part -> (tile index from ndirect, K range z); false for blocks past the last item. Ranges
// outermost in bands per XCD (block j runs on XCD j % 8): consecutive items of a band read the same K range of one X
// tile.
__device__ __forceinline__ bool split_item(int j, int nsplit, int ks, int& ts, int& z) {
    const int items = nsplit * ks, per = (items + 7) >> 3, it = (j & 7) * per + (j >> 3);
    if ((j >> 3) >= per || it >= items) return false;
    z = it / nsplit;
    ts = it - z * nsplit;
    return true;
}
// blocks of the split part
inline unsigned split_blocks(int nsplit, int ks) { return 8u * (unsigned)((nsplit * ks + 7) / 8); }

// Tile number -> (token block, weight-column tile): CG = 0: token blocks outer, columns inner; CG > 0: groups of CG
// column tiles, inside a group token blocks outer and columns inner
template <int CG>
__device__ __forceinline__ void tile_place(int tile, int nbn, int nbt, int& tb, int& cb) {
    if constexpr (CG == 0) {
        tb = tile / nbn;
        cb = tile % nbn;
    } else {
        const int full = nbn / CG, cg = tile / (nbt * CG);
        const int w = cg < full ? CG : nbn - full * CG, r = tile - cg * nbt * CG;
        tb = r / w;
        cb = cg * CG + r % w;
    }
}

// Split tiles' partials -> outputs: one thread per (split tile, token row, 4 input columns; GLU: 4 gate columns and
// the 4 up columns 8 to the right); the ks partials are added in split order (fixed order: the result does not depend
// on timing), then the epilogue of the GEMM. Reads are 16 bytes a lane, consecutive lanes consecutive.
template <int BM, int BN, int CG, bool GLU>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(const float* __restrict__ part, int ks, int ndirect,
                                                            int nsplit, int nbn, int nbt, int T, int N,
                                                            void* __restrict__ c, int ldc, int out) {
    constexpr int CB = GLU ? BN / 8 : BN / 4;  // threads per row
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)nsplit * BM * CB) return;
    const int st = (int)(idx / ((size_t)BM * CB)), r = (int)((idx / CB) % BM), cb = (int)(idx % CB);
    int tb, tc;
    tile_place<CG>(ndirect + st, nbn, nbt, tb, tc);
    const int col = GLU ? 16 * (cb >> 1) + 4 * (cb & 1) : 4 * cb;
    const int tok = tb * BM + r, n = tc * BN + col;
    if (tok >= T || n >= N) return;
    const float* p = part + ((size_t)st * ks * BM + r) * BN + col;
    f32x4_v v{0.f, 0.f, 0.f, 0.f}, u{0.f, 0.f, 0.f, 0.f};
    for (int z = 0; z < ks; z++, p += (size_t)BM * BN) {
        const f32x4_v a = *reinterpret_cast<const f32x4_v*>(p);
#pragma unroll
        for (int j = 0; j < 4; j++) v[j] += a[j];
        if constexpr (GLU) {
            const f32x4_v b = *reinterpret_cast<const f32x4_v*>(p + 8);
#pragma unroll
            for (int j = 0; j < 4; j++) u[j] += b[j];
        }
    }
    if constexpr (GLU) {
        uint16_t* o = reinterpret_cast<uint16_t*>(c) + (size_t)tok * ldc + (n >> 4) * 8 + (n & 7);
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = f32_to_bf16(silu_f32(v[j]) * u[j]);
    } else if (out == kOutBF16) {
        uint16_t* o = reinterpret_cast<uint16_t*>(c) + (size_t)tok * ldc + n;
        if (((ldc & 3) | ((uintptr_t)c & 7)) == 0) {
            *reinterpret_cast<uint2*>(o) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++) o[j] = f32_to_bf16(v[j]);
        }
    } else {
        float* o = reinterpret_cast<float*>(c) + (size_t)tok * ldc + n;
#pragma unroll
        for (int j = 0; j < 4; j++) o[j] = v[j];
    }
}

template <int BM, int BN, int CG>
void launch_splitk_reduce(const float* part, int ks, int ndirect, int nsplit, int nbn, int nbt, int t, int n, void* c, int ldc,
                          int out, hipStream_t st) {
    const bool glu = out == kOutGLU;
    const size_t threads = (size_t)nsplit * BM * (BN / (glu ? 8 : 4));
    const dim3 grid((unsigned)((threads + 255) / 256));
    if (glu) splitk_reduce_kernel<BM, BN, CG, true><<<grid, dim3(256), 0, st>>>(part, ks, ndirect, nsplit, nbn, nbt, t, n, c,
                                                                                ldc, out);
    else splitk_reduce_kernel<BM, BN, CG, false><<<grid, dim3(256), 0, st>>>(part, ks, ndirect, nsplit, nbn, nbt, t, n, c,
                                                                                ldc, out);
    HIP_CHECK(hipGetLastError());
}

}  // namespace qe_tile
