// Prefill GEMM on the W4 / W8 layouts for gfx950: C[t][n] = sum_k X[t][k] * W[n][k], bf16 MFMA, fp32 accumulate.
//
// The weights are dequantized once per block tile, in registers, to the reference's bf16 operand
// (bf16_rn((u - 8) * s) for INT4, bf16_rn(w * s) for INT8; reference gemm.cu:68-77) and staged in LDS next to the
// activation tile; v_mfma_f32_32x32x16_bf16 consumes both from LDS.
//   block: 512 threads = 8 waves in 2 (tokens) x 4 (weight rows); wave tile WMT x WNT MFMA tiles of 32 x 32;
//          block tile BM = 64 WMT tokens x BN = 128 WNT rows, BK = 64 (one W4 chunk)
//   LDS: two stages of X [BM][64] and W [BN][64] bf16, rows of 128 B with the 16-byte chunks XOR-swizzled by
//        (row % 8) so the MFMA fragment reads (32 rows x 16 B per half-wave) spread over the banks
//   pipeline, per k step: the MFMAs of step k read stage k % 2 while the same waves dequantize step k + 1 into the
//        other stage; the activations of step k + 1 arrive there by LDS DMA issued at the top of step k. The raw
//        records of step k + 2 are DMA'd to LDS at the top of step k and dequantized from LDS a step later. Every
//        step ends with vmcnt(0), lgkmcnt(0) and one barrier: each load gets a step of MFMA time to arrive, and the
//        VALU dequantization overlaps the matrix pipe.
//   grid: one block per output tile, tiles ordered so that the 8 XCDs (blockIdx % 8) each sweep a contiguous band
//        of tiles (their L2 keeps the shared X / W tiles).
#include "mfma_tile.hpp"
#include "gemm_split.hpp"
#include "gemm_tune.hpp"

#include <algorithm>
#include <optional>
#include <mutex>
#include <type_traits>
#include <vector>

namespace {

using namespace qe_tile;
constexpr int BK = 64, NTH = 512;

enum Fmt : int { kFmtW4 = 0, kFmtW8G = 1, kFmtW8C = 2, kFmtQ8 = 3 };

template <int WMT, int WNT>
struct Cfg {
    static constexpr int BM = 64 * WMT, BN = 128 * WNT;
    static constexpr int kStage = (BM + BN) * BK * 2;
    static constexpr int XDMA = BM / 64;         // 1 KB X DMA loads per wave and step (INT4 path)
    // INT4 path: raw W records of one k step (BN / 16 tiles x 512 B) and the scales of one group (BN / 16 x 32 B),
    // both double-buffered after the two stages
    static constexpr int kRaw = BN * 32, kSc = BN * 2;
    static constexpr int kLdsW4 = 2 * kStage + 2 * kRaw + 2 * kSc;
    // INT8: the records of one k step are twice as long; the scales stay in registers (256 x 256 tiles fill the 160 KB)
    static constexpr int kRaw8 = BN * 64;
    static constexpr int kLdsW8 = 2 * kStage + 2 * kRaw8;
};

template <int FMT, int SDT, int WMT, int WNT>
__global__ void __launch_bounds__(NTH) gemm_kernel(const uint4* __restrict__ q, const uint16_t* __restrict__ s,
                                                   int N, int K, const uint16_t* __restrict__ x, int ldx, int T,
                                                   void* __restrict__ c, int ldc, int out, int sdt, int nbn, int nbt,
                                                   SplitArgs sp) {
    using C = Cfg<WMT, WNT>;
    constexpr int BM = C::BM, BN = C::BN;
    constexpr bool W4 = FMT == kFmtW4;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned lds32 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)lds);  // LDS byte address of lds[]
    // XCD-aware tile order: block b runs on XCD b % 8; XCD j takes tiles [j * per, (j + 1) * per) of the
    // n-major tile sequence (consecutive tiles share the X tile, a band of them shares W tiles)
    int n0, t0;
    int kt0 = 0, KTL = K / BK;  // this block's k steps [kt0, kt0 + KTL)
    int split_slot = -1;        // >= 0: a split tile's part, stored raw to sp.part
    // tiles [0, sp.ndirect): whole K, XCD bands; tiles [sp.ndirect, ntiles): split into sp.ks K ranges whose
    // fp32 partials splitk_reduce_kernel sums (the blocks of the otherwise partly idle last round)
    const int ntiles = nbn * nbt, per = (sp.ndirect + 7) >> 3;
    const int b = blockIdx.x;
    int tile;
    if (b < 8 * per) {
        tile = (b & 7) * per + (b >> 3);
        if (tile >= sp.ndirect) return;
    } else {
        const int j = b - 8 * per;
        int ts, z;
        if (!split_item(j, ntiles - sp.ndirect, sp.ks, ts, z)) return;
        const int groups = K >> 7;
        tile = sp.ndirect + ts;
        kt0 = 2 * (z * groups / sp.ks);
        KTL = 2 * ((z + 1) * groups / sp.ks) - kt0;
        split_slot = ts * sp.ks + z;
    }
    n0 = (tile % nbn) * BN;
    t0 = (tile / nbn) * BM;
    const int G = K >> 7;

    // ---- X (every format): LDS DMA (global_load_lds_dwordx4), 1 KB = 8 rows per wave instruction. Lane i lands at
    //      LDS slot i of the 8-row block, so it loads the chunk that the swizzle puts there. Rows past T re-read
    //      row T - 1 (their outputs are not stored).
    auto dma_x = [&](int kt, unsigned xt) {  // xt: LDS offset of the X tile from lds[]
#pragma unroll
        for (int i = 0; i < C::XDMA; i++) {
            const int r0 = (wave * C::XDMA + i) * 8, row = r0 + (lane >> 3);
            const int ch = (lane & 7) ^ swz_f(row);
            const int tok = t0 + row < T ? t0 + row : T - 1;
            dma16(x + (size_t)tok * ldx + kt * BK + ch * 8, lds32 + xt + r0 * 128);
        }
    };
    // ---- W, INT4 path. Raw records go to LDS by DMA: a 1 KB wave load covers two 16-row tiles; lane i holds record
    //      (tile 2 u + (i / 8) % 2, g = i % 8, t = i / 16), so that a job's reads below hit 64 distinct banks. A job =
    //      k step j (16 k) of the row pair (g, g + 8) of a tile: word j of the tile's 4 records (g, t = 0..3) ->
    //      4 full 16-byte chunks of the bf16 tile (rows g and g + 8, chunks 2 j and 2 j + 1).
    constexpr int NJOB = BN * 2;
    const bool jactive = tid < NJOB;
    const int jj = tid & 3, jg = (tid >> 2) & 7, jtr = (tid >> 5) & (BN / 16 - 1);  // (threads without a job: another's)
    const int ntile_last = (N >> 4) - 1;
    // record (tile tl, 64-k step kt) and scales (tile tl, group grp)
    auto w_rec = [&](int tl, int kt) -> const uint4* { return q + ((size_t)tl * (K >> 6) + kt) * 32; };
    auto w_sc = [&](int tl, int grp) -> const uint16_t* { return s + ((size_t)tl * G + grp) * 16; };
    auto dma_w4 = [&](int kt, unsigned raw) {  // raw: LDS offset of the raw record buffer
        if (wave < BN / 32) {
            const int tl = min((n0 >> 4) + 2 * wave + ((lane >> 3) & 1), ntile_last);
            dma16(w_rec(tl, kt) + 4 * (lane & 7) + (lane >> 4), lds32 + raw + wave * 1024);
        }
    };
    auto dma_sc = [&](int grp, unsigned sc) {  // [BN / 16 tiles][16] scales of group grp; lane i: dword i % 8 of tile i / 8
        if (wave < BN / 128) {
            const int tl = min((n0 >> 4) + 8 * wave + (lane >> 3), ntile_last);
            dma4(w_sc(tl, grp) + 2 * (lane & 7), lds32 + sc + wave * 256);
        }
    };
    // dequantize half h (0: row g, 1: row g + 8) of this thread's job from the raw records into the W tile
    auto store_w4 = [&](char* wtile, const char* raw, const char* sc, int h) {
        if constexpr (NJOB < NTH) {
            if (!jactive) return;
        }
        const uint32_t* rw = reinterpret_cast<const uint32_t*>(raw + (jtr >> 1) * 1024) + (8 * (jtr & 1) + jg) * 4 + jj;
        const float scl = scale_rt<SDT>(reinterpret_cast<const uint16_t*>(sc)[jtr * 16 + jg + 8 * h], sdt);
        // h = 1 keeps its nibbles high (v = 16 u): qe_tile::dq_pair's s / 16, -72 s
        const float sv = h ? scl * 0.0625f : scl, bv = h ? -72.f * scl : -1032.f * scl;
        const uint32_t msk = h ? 0xF0F0F0F0u : nib_mask();
        uint32_t lo[4], hi[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const uint32_t u = rw[64 * t] & msk;  // bytes: k0, k0+8, k0+1, k0+9
            lo[t] = dq_pair(magic_f16<kSel02>(u), sv, bv);
            hi[t] = dq_pair(magic_f16<kSel13>(u), sv, bv);
        }
        const int row = jtr * 16 + jg + 8 * h;
        *reinterpret_cast<u32x4_v*>(wtile + swz(row, 2 * jj)) = u32x4_v{lo[0], lo[1], lo[2], lo[3]};
        *reinterpret_cast<u32x4_v*>(wtile + swz(row, 2 * jj + 1)) = u32x4_v{hi[0], hi[1], hi[2], hi[3]};
    };

    // ---- W, INT8 formats: raw records by LDS DMA too. A step holds two slabs of 32 k, a slab 512 B a tile; a 1 KB wave
    //      load covers two tiles of a slab, lanes placed as above. A job = dword d of the row pair (g, g + 8) of a tile
    //      in both slabs: that dword of the 4 records (g, t = 0..3) is 2 full 16-byte chunks. W8: dword d = bytes
    //      (row g: k, k + 1; row g + 8: k, k + 1) at k = 8 d + 2 t: chunk d of rows g and g + 8. Q8: word d = row
    //      g + 8 (d % 2), bytes at k0 + {0, 8, 1, 9}, k0 = 16 (d / 2) + 2 t: chunks 2 (d / 2) and + 1 of that row.
    auto dma_w8 = [&](int kt, unsigned raw) {
        if (wave < BN / 32) {
            const int tl = min((n0 >> 4) + 2 * wave + ((lane >> 3) & 1), ntile_last);
            const uint4* p = q + ((size_t)tl * (K >> 5) + 2 * kt) * 32 + 4 * (lane & 7) + (lane >> 4);
            dma16(p, lds32 + raw + wave * 1024);
            dma16(p + 32, lds32 + raw + BN * 32 + wave * 1024);
        }
    };
    const int jtl = min((n0 >> 4) + jtr, ntile_last);
    // raw scales of rows g and g + 8 of this thread's tile for global step kt
    auto load_s8 = [&](int kt, uint16_t (&r)[2]) {
        const uint16_t* p = FMT == kFmtW8C ? s + (size_t)jtl * 16 : s + ((size_t)jtl * G + (kt >> 1)) * 16;
        r[0] = p[jg];
        r[1] = p[jg + 8];
    };
    // unit (slab, t) of the dequantization: word t of the job -> one bf16 pair of either chunk; after t = 3 the stores
    auto unit_w8 = [&](char* wtile, uint32_t word, const float (&sc)[2], int slab, int t, uint32_t (&lo)[4], uint32_t (&hi)[4]) {
        const uint32_t x = word ^ 0x80808080u;  // w + 128
        if constexpr (FMT == kFmtQ8) {
            const float v = (jj & 1) ? sc[1] : sc[0], bs = -1152.f * v;  // qe_tile::dq_pair's W8 bias
            lo[t] = dq_pair(magic_f16<kSel02>(x), v, bs);
            hi[t] = dq_pair(magic_f16<kSel13>(x), v, bs);
        } else {
            lo[t] = dq_pair(magic_f16<kSel01>(x), sc[0], -1152.f * sc[0]);
            hi[t] = dq_pair(magic_f16<kSel23>(x), sc[1], -1152.f * sc[1]);
        }
        if (t == 3 && (NJOB >= NTH || jactive)) {
            const int row = jtr * 16 + jg, ch = 4 * slab;
            const int r0 = FMT == kFmtQ8 ? row + 8 * (jj & 1) : row, c0 = FMT == kFmtQ8 ? ch + 2 * (jj >> 1) : ch + jj;
            const int r1 = FMT == kFmtQ8 ? r0 : row + 8, c1 = FMT == kFmtQ8 ? c0 + 1 : c0;
            *reinterpret_cast<u32x4_v*>(wtile + swz(r0, c0)) = u32x4_v{lo[0], lo[1], lo[2], lo[3]};
            *reinterpret_cast<u32x4_v*>(wtile + swz(r1, c1)) = u32x4_v{hi[0], hi[1], hi[2], hi[3]};
        }
    };

    // ---- MFMA tiles: wave (wm, wn) owns tokens wm * 32 WMT .. , rows wn * 32 WNT ..
    const int wm = wave >> 2, wn = wave & 3;
    f32x16_v acc[WMT][WNT];
#pragma unroll
    for (int a = 0; a < WMT; a++)
#pragma unroll
        for (int bb = 0; bb < WNT; bb++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[a][bb][r] = 0.f;

    // one k step: MFMAs on stage kt % 2 while the next step's tiles go into the other stage
    int lane_off[BK / 16];  // swz(l % 32, 2 ks + l / 32) of this lane
#pragma unroll
    for (int ks = 0; ks < BK / 16; ks++) lane_off[ks] = swz(lane & 31, 2 * ks + (lane >> 5));
    // pre() runs after the first fragment reads, between(slot) after each row of WNT MFMAs (slot = ks * WMT + row).
    // pin: nothing is scheduled across those calls, so the work placed in them keeps its place among the MFMAs
    // (the INT4 dequantization: left to the scheduler it clusters into one VALU block per k16 step, during which
    // the wave issues no MFMA).
    auto mfma_step = [&](const char* xt, const char* wt, auto&& pre, auto&& between, auto pin) {
        // fragments of lane l: row l % 32, k = 16 ks + 8 (l / 32) .. + 8 -> chunk 2 ks + l / 32; the reads of k16
        // step ks + 1 are issued before the MFMAs of step ks
        // (every fragment row block is 32-aligned, so the swizzled offset is a per-lane part + a constant)
        bf16x8_v af[2][WMT], bfr[2][WNT];
        auto read_frags = [&](int ks, int buf) {
            const char* xl = xt + lane_off[ks];
            const char* wl = wt + lane_off[ks];
#pragma unroll
            for (int a = 0; a < WMT; a++)
                af[buf][a] = *reinterpret_cast<const bf16x8_v*>(xl + (wm * 32 * WMT + a * 32) * 128);
#pragma unroll
            for (int bb = 0; bb < WNT; bb++)
                bfr[buf][bb] = *reinterpret_cast<const bf16x8_v*>(wl + (wn * 32 * WNT + bb * 32) * 128);
        };
        auto fence = [&] {
            if constexpr (decltype(pin)::value) __builtin_amdgcn_sched_barrier(0);
        };
        read_frags(0, 0);
        pre();
        fence();
#pragma unroll
        for (int ks = 0; ks < BK / 16; ks++) {
            if (ks + 1 < BK / 16) read_frags(ks + 1, (ks + 1) & 1);
#pragma unroll
            for (int a = 0; a < WMT; a++) {
#pragma unroll
                for (int bb = 0; bb < WNT; bb++)
                    acc[a][bb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bfr[ks & 1][bb], af[ks & 1][a], acc[a][bb], 0, 0, 0);
                between(ks * WMT + a);
                fence();
            }
        }
    };

    if constexpr (W4) {
        // Every global load is an LDS DMA issued at the top of a step, so the compiler tracks none of them and
        // inserts no waits inside the step; each step ends with vmcnt(0) (its DMAs landed), lgkmcnt(0) and the
        // barrier that publishes them. Step kt: DMA X of step kt + 1 into the other stage and the raw W of step
        // kt + 2 (plus the scales of its group when it starts one), then the MFMAs of step kt with the dequantization
        // of step kt + 1 (raw records published by the previous step) into the other stage: this thread's 4 raw
        // words and 2 scales are read at the top, and its 8 (row half, word) units run one after every
        // NSLOT / 8-th MFMA row, each half's two 16-byte stores after its last unit. The last step, which has no
        // next step to dequantize, is a separate instance, so the steps before it are one basic block (measured on
        // C2: 41-42 % -> 44-46 % of the bf16 peak against the dequantization left to the scheduler after a branch;
        // matrix pipes busy 51 % -> 61 % of the busy cycles).
        constexpr unsigned kRawOff = 2 * C::kStage, kScOff = kRawOff + 2 * C::kRaw;
        char* raw = lds + kRawOff;
        char* scb = lds + kScOff;
        // buffers by the local step kt, addresses by the global step kt0 + kt (kt0 is even: group aligned)
        dma_x(kt0, 0);
        dma_w4(kt0, kRawOff);
        dma_w4(kt0 + 1, kRawOff + C::kRaw);
        dma_sc(kt0 >> 1, kScOff);
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        store_w4(lds + BM * BK * 2, raw, scb, 0);
        store_w4(lds + BM * BK * 2, raw, scb, 1);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        constexpr int NSLOT = (BK / 16) * WMT, STRIDE = NSLOT >= 8 ? NSLOT / 8 : 1;
        static_assert(NSLOT >= 8, "eight dequantization units per k step");
        auto kstep = [&](int kt, auto more) {
            constexpr bool MORE = decltype(more)::value;
            char* wnext = lds + ((kt + 1) & 1) * C::kStage + BM * BK * 2;
            if (MORE) dma_x(kt0 + kt + 1, ((kt + 1) & 1) * C::kStage);
            if (kt + 2 < KTL) {
                dma_w4(kt0 + kt + 2, kRawOff + (kt & 1) * C::kRaw);
                if (((kt + 2) & 1) == 0) dma_sc((kt0 + kt + 2) >> 1, kScOff + (((kt + 2) >> 1) & 1) * C::kSc);
            }
            const char* rnext = raw + ((kt + 1) & 1) * C::kRaw;
            const uint16_t* snext = reinterpret_cast<const uint16_t*>(scb + (((kt + 1) >> 1) & 1) * C::kSc);
            const uint32_t* rw = reinterpret_cast<const uint32_t*>(rnext + (jtr >> 1) * 1024) + (8 * (jtr & 1) + jg) * 4 + jj;
            uint32_t wd[4], lo[2][4], hi[2][4];
            float scl[2];
            const char* xt = lds + (kt & 1) * C::kStage;
            mfma_step(xt, xt + BM * BK * 2, [&] {
                if constexpr (MORE) {
#pragma unroll
                    for (int t = 0; t < 4; t++) wd[t] = rw[64 * t];
#pragma unroll
                    for (int h = 0; h < 2; h++) scl[h] = scale_rt<SDT>(snext[jtr * 16 + jg + 8 * h], sdt);
                }
            }, [&](int slot) {
                if constexpr (MORE) {
                    if (slot % STRIDE != STRIDE - 1 || slot / STRIDE >= 8) return;
                    // unit (h, t): word t, nibbles of row g + 8 h -> bf16 pairs at k0 (lo) and k0 + 8 (hi)
                    const int un = slot / STRIDE, h = un >> 2, t = un & 3;
                    // h = 1 keeps its nibbles high (v = 16 u): qe_tile::dq_pair's s / 16, -72 s
                    const float sv = h ? scl[h] * 0.0625f : scl[h], bv = h ? -72.f * scl[h] : -1032.f * scl[h];
                    const uint32_t u = wd[t] & (h ? 0xF0F0F0F0u : nib_mask());  // bytes: k0, k0+8, k0+1, k0+9
                    lo[h][t] = dq_pair(magic_f16<kSel02>(u), sv, bv);
                    hi[h][t] = dq_pair(magic_f16<kSel13>(u), sv, bv);
                    if (t == 3 && (NJOB >= NTH || jactive)) {
                        const int row = jtr * 16 + jg + 8 * h;
                        *reinterpret_cast<u32x4_v*>(wnext + swz(row, 2 * jj)) = u32x4_v{lo[h][0], lo[h][1], lo[h][2], lo[h][3]};
                        *reinterpret_cast<u32x4_v*>(wnext + swz(row, 2 * jj + 1)) = u32x4_v{hi[h][0], hi[h][1], hi[h][2], hi[h][3]};
                    }
                }
            }, std::true_type{});
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        };
        for (int kt = 0; kt + 1 < KTL; kt++) kstep(kt, std::true_type{});
        kstep(KTL - 1, std::false_type{});
    } else {
        // As the INT4 path: X and the raw records by LDS DMA at the top of a step, a thread's 2 x 4 words read there, its
        // 8 (slab, word) units pinned after every NSLOT / 8-th MFMA row. The two scales a thread needs are loaded to
        // registers two steps ahead and converted right after the step's wait (nothing else is in flight there).
        // Against the records in registers, transposed across quads by DPP, and the units left to the scheduler:
        // 8192 x 2048, t = 4096 155 -> 137 us, 14176 x 2304, t = 1500 143 -> 124 us, 3760 x 5120, t = 200 30.8 -> 25.2.
        constexpr unsigned kRawOff = 2 * C::kStage;
        char* raw = lds + kRawOff;
        constexpr int NSLOT = (BK / 16) * WMT, STRIDE = NSLOT / 8;
        static_assert(NSLOT >= 8 && NSLOT % 8 == 0, "eight dequantization units per k step");
        uint16_t sr[2];
        float sc[2];
        auto cvt = [&] {
#pragma unroll
            for (int h = 0; h < 2; h++) sc[h] = scale_rt<SDT>(sr[h], sdt);
        };
        dma_x(kt0, 0);
        dma_w8(kt0, kRawOff);
        dma_w8(kt0 + 1, kRawOff + C::kRaw8);
        load_s8(kt0, sr);
        asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        cvt();
        auto words = [&](const char* r, uint32_t (&wd)[2][4]) {
#pragma unroll
            for (int sl = 0; sl < 2; sl++) {
                const uint32_t* rw = reinterpret_cast<const uint32_t*>(r + sl * BN * 32 + (jtr >> 1) * 1024) +
                                     (8 * (jtr & 1) + jg) * 4 + jj;
#pragma unroll
                for (int t = 0; t < 4; t++) wd[sl][t] = rw[64 * t];
            }
        };
        {
            uint32_t wd[2][4], lo[4], hi[4];
            words(raw, wd);
#pragma unroll
            for (int un = 0; un < 8; un++) unit_w8(lds + BM * BK * 2, wd[un >> 2][un & 3], sc, un >> 2, un & 3, lo, hi);
        }
        if constexpr (FMT != kFmtW8C) load_s8(kt0 + 1, sr);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if constexpr (FMT != kFmtW8C) cvt();
        auto kstep = [&](int kt, auto more) {
            constexpr bool MORE = decltype(more)::value;
            char* wnext = lds + ((kt + 1) & 1) * C::kStage + BM * BK * 2;
            if (MORE) dma_x(kt0 + kt + 1, ((kt + 1) & 1) * C::kStage);
            if (kt + 2 < KTL) {
                dma_w8(kt0 + kt + 2, kRawOff + (kt & 1) * C::kRaw8);
                if constexpr (FMT != kFmtW8C) load_s8(kt0 + kt + 2, sr);
            }
            uint32_t wd[2][4], lo[2][4], hi[2][4];
            const char* xt = lds + (kt & 1) * C::kStage;
            mfma_step(xt, xt + BM * BK * 2, [&] {
                if constexpr (MORE) words(raw + ((kt + 1) & 1) * C::kRaw8, wd);
            }, [&](int slot) {
                if constexpr (MORE) {
                    if (slot % STRIDE != STRIDE - 1) return;
                    const int un = slot / STRIDE;
                    unit_w8(wnext, wd[un >> 2][un & 3], sc, un >> 2, un & 3, lo[un >> 2], hi[un >> 2]);
                }
            }, std::true_type{});
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            if constexpr (FMT != kFmtW8C) cvt();
        };
        for (int kt = 0; kt + 1 < KTL; kt++) kstep(kt, std::true_type{});
        kstep(KTL - 1, std::false_type{});
    }

    // ---- epilogue. The MFMAs take the W fragments as A and the X fragments as B, so each 32 x 32 tile holds C^T:
    //      lane l holds token l % 32 and weight rows (output columns) 8 (r / 4) + 4 (l / 32) + r % 4, i.e. 4
    //      consecutive output columns per r / 4 -> one 8-byte (bf16) or 16-byte (fp32) store, or scalar stores where
    //      ldc / c are not aligned for them. GLU: gate row g and up row g + 8 of a 16-row tile are registers r and
    //      r + 4 of the same lane.
    const int cj = lane & 31, ci = 4 * (lane >> 5);
    if (split_slot >= 0) {
        // raw fp32 partial of the BM x BN tile, [token][row] (rows past N included, tokens past T not)
        static_assert(NTH / 64 * 32 * out_pitch<kOutF32, WNT>() <= 2 * C::kStage, "one buffer per wave in the stages");
        store_rows<kOutF32>(acc, lds + wave * 32 * out_pitch<kOutF32, WNT>(), lane, wm * 32 * WMT, T - t0,
                            wn * 32 * WNT, BN, sp.part + (size_t)split_slot * BM * BN, BN,
                            [](int bb, int rb) { return 32 * bb + 8 * rb; });
        return;
    }
    if ((ldc & (out == kOutF32 ? 3 : 7)) == 0 && ((uintptr_t)c & 15) == 0) {
        auto rows = [&](auto o) {
            constexpr int OUT = decltype(o)::value;
            store_rows<OUT>(acc, lds + wave * 32 * out_pitch<OUT, WNT>(), lane, t0 + wm * 32 * WMT, T,
                            n0 + wn * 32 * WNT, N, c, ldc, [](int bb, int rb) { return 32 * bb + 8 * rb; });
        };
        if (out == kOutGLU) rows(std::integral_constant<int, kOutGLU>{});
        else if (out == kOutBF16) rows(std::integral_constant<int, kOutBF16>{});
        else rows(std::integral_constant<int, kOutF32>{});
        return;
    }
    const bool vec = (ldc & 3) == 0 && ((uintptr_t)c & (out == kOutF32 ? 15u : 7u)) == 0;
    auto st4 = [&](uint16_t* p, float v0, float v1, float v2, float v3) {  // 4 consecutive bf16
        if (vec) {
            *reinterpret_cast<uint2*>(p) = uint2{pack_bf16x2(v0, v1), pack_bf16x2(v2, v3)};
        } else {
            p[0] = f32_to_bf16(v0);
            p[1] = f32_to_bf16(v1);
            p[2] = f32_to_bf16(v2);
            p[3] = f32_to_bf16(v3);
        }
    };
#pragma unroll
    for (int a = 0; a < WMT; a++)
#pragma unroll
        for (int bb = 0; bb < WNT; bb++) {
            const int tok = t0 + wm * 32 * WMT + a * 32 + cj;
            if (tok >= T) continue;
#pragma unroll
            for (int rb = 0; rb < 4; rb++) {
                const int n = n0 + wn * 32 * WNT + bb * 32 + 8 * rb + ci;  // first of the 4 columns
                const f32x16_v& v = acc[a][bb];
                if (out == kOutGLU) {
                    if (rb & 1) continue;  // rows 8 (rb + 1) + ..: the up rows of this gate block
                    float g[4];
#pragma unroll
                    for (int j = 0; j < 4; j++) g[j] = silu_f32(v[4 * rb + j]) * v[4 * rb + 4 + j];
                    if (n < N)
                        st4(reinterpret_cast<uint16_t*>(c) + (size_t)tok * ldc + (n >> 4) * 8 + (n & 7), g[0], g[1],
                            g[2], g[3]);
                } else if (n < N) {
                    if (out == kOutBF16) {
                        st4(reinterpret_cast<uint16_t*>(c) + (size_t)tok * ldc + n, v[4 * rb], v[4 * rb + 1],
                            v[4 * rb + 2], v[4 * rb + 3]);
                    } else {
                        float* p = reinterpret_cast<float*>(c) + (size_t)tok * ldc + n;
                        if (vec) {
                            *reinterpret_cast<f32x4_v*>(p) = f32x4_v{v[4 * rb], v[4 * rb + 1], v[4 * rb + 2], v[4 * rb + 3]};
                        } else {
#pragma unroll
                            for (int j = 0; j < 4; j++) p[j] = v[4 * rb + j];
                        }
                    }
                }
            }
        }
}

// tile configurations: 0 = 256 tokens x 256 rows (WMT 4, WNT 2), 1 = 256 x 128 (4, 1), 2 = 128 x 256 (2, 2),
// 3 = 128 x 128 (2, 1; two blocks per CU)
constexpr int kNumCfg = 4;
template <int CFG>
struct CfgOf;
template <>
struct CfgOf<0> {
    static constexpr int WMT = 4, WNT = 2;
};
template <>
struct CfgOf<1> {
    static constexpr int WMT = 4, WNT = 1;
};
template <>
struct CfgOf<2> {
    static constexpr int WMT = 2, WNT = 2;
};
template <>
struct CfgOf<3> {
    static constexpr int WMT = 2, WNT = 1;
};

struct GemmGeom {
    int nbn, nbt, ntiles, ndirect, nsplit, ks;
    size_t ws_bytes;
};
struct CfgDims {
    int BM, BN, slots;  // tile and how many of its blocks the device holds at once (LDS: one per CU, two of 128 x 128)
};
CfgDims cfg_dims(int cfg) {
    return CfgDims{cfg < 2 ? 256 : 128, (cfg & 1) ? 128 : 256, qe_num_cus() * (cfg == 3 ? 2 : 1)};
}
// tiles of configuration cfg and, for ks > 1, the split of the last partial round (stream-K): whole rounds of
// tiles run directly, the remaining tiles (all of them when they do not fill one round) as ks K ranges; false when
// that split does not apply (no partial round, fewer 128-k groups than ranges, too much workspace)
bool gemm_geom(int cfg, int n, int k, int t, int ks, GemmGeom& g) {
    const CfgDims d = cfg_dims(cfg);
    g.nbn = (n + d.BN - 1) / d.BN;
    g.nbt = (t + d.BM - 1) / d.BM;
    g.ntiles = g.nbn * g.nbt;
    g.ks = ks;
    g.ndirect = g.ntiles;
    g.nsplit = 0;
    g.ws_bytes = 0;
    if (ks == 1) return true;
    const int tail = g.ntiles % d.slots;
    const size_t bytes = (size_t)tail * ks * d.BM * d.BN * 4;
    if (tail == 0 || k / 128 < ks || bytes > max_split_bytes()) return false;
    g.ndirect = g.ntiles - tail;
    g.nsplit = tail;
    g.ws_bytes = bytes;
    return true;
}

// Predicted time in us of a choice: the k steps of the fullest CU at a measured cost per step, which falls when only
// part of the CUs run (clock, shared caches), plus the partial sums written and read again. Fitted to sweeps of every
// (configuration, ks <= 16) on (n, k) from 1280 x 4224 to 34816 x 5120, t = 70..4000 (MI355X; INT4 26 shapes 5.4 % rms,
// INT8, whose dequantization is a little longer, 20 shapes 5.7 % rms): the lowest prediction is within 9 % of the best
// measured choice at every one of them. What it replaces for shapes whose tiles leave CUs idle (256 x 128
// tiles, one K range): 5120 x 17408, t = 200 (40 tiles) 240 -> 58 us with 20 tiles of 256 x 256 in 12 ranges;
// 34816 x 5120 GLU, t = 200 (272 tiles, two rounds) 163 -> 108 us with the last 16 tiles in 10 ranges; 5120 x 17408,
// t = 1000 272 -> 174 us; 2976 x 7936, t = 75 114 -> 22 us; INT8 1280 x 7168, t = 100 104 -> 20 us.
double gemm_cost_us(bool w8, int cfg, int n, int k, int t, const GemmGeom& g) {
    static const double kFull[2][kNumCfg] = {{1.652, 1.014, 1.027, 1.112}, {1.832, 1.069, 1.128, 1.197}};
    static const double kPart[2][kNumCfg] = {{1.216, 0.797, 0.807, 0.649}, {1.343, 0.814, 0.824, 0.660}};
    const double full_us = kFull[w8][cfg], part_us = kPart[w8][cfg];  // per 64-k step: every slot filled, few
    const CfgDims d = cfg_dims(cfg);
    auto phase = [&](int blocks, int steps) {
        const int full = blocks / d.slots, rem = blocks % d.slots;
        double us = full * (steps * full_us + 1.2);
        if (rem) {
            const double u = cfg == 3 ? (2 * rem > d.slots ? 1.0 : 0.0) : (double)rem / d.slots;  // 3: two per CU
            us += steps * (u * full_us + (1.0 - u) * part_us) + 1.2;
        }
        return us;
    };
    double us = 4.3 + phase(g.ndirect, k / BK);
    if (g.nsplit > 0) {
        us += phase(g.nsplit * g.ks, 2 * ((k / 128 + g.ks - 1) / g.ks));
        us += 4.0 + 0.245e-6 * g.nsplit * g.ks * ((double)t / g.nbt) * d.BN * 4;
    }
    return us;
}

}  // namespace

void gemm_reserve(size_t bytes, hipStream_t st) {
    ws_reserve(kWsSplit, bytes, st);
}

namespace {

template <int FMT, int SDT, int CFG>
void launch_cfg(const uint4* q, const uint16_t* s, int n, int k, const uint16_t* x, int ldx, int t, void* c, int ldc,
                int out, int sdt, const GemmGeom& g, float* part, hipStream_t st) {
    constexpr int WMT = CfgOf<CFG>::WMT, WNT = CfgOf<CFG>::WNT;
    using C = Cfg<WMT, WNT>;
    SplitArgs sp;
    sp.ndirect = g.ndirect;
    sp.ks = g.ks;
    sp.part = part;
    const int per = (g.ndirect + 7) / 8;
    const unsigned blocks = (unsigned)(8 * per) + split_blocks(g.nsplit, g.ks);
    gemm_kernel<FMT, SDT, WMT, WNT><<<dim3(blocks), dim3(NTH), FMT == kFmtW4 ? C::kLdsW4 : C::kLdsW8, st>>>(
        q, s, n, k, x, ldx, t, c, ldc, out, sdt, g.nbn, g.nbt, sp);
    HIP_CHECK(hipGetLastError());
    if (g.nsplit > 0) {
        launch_splitk_reduce<C::BM, C::BN, 0>(part, g.ks, g.ndirect, g.nsplit, g.nbn, g.nbt, t, n, c, ldc, out, st);
    }
}

// untuned choice: 256 x 256 tiles when they fill the CUs at least once (else 256 x 128), with the last partial round
// split in two K ranges when it is at most half full, unless the cost model puts another choice at least 6 % lower
// (its error; below that the larger tile stays). maxparts: the largest split allowed (0: any).
// The last choices of a thread are kept: 64 cost evaluations take about as long as a launch.
GemmChoice gemm_model_choice(bool w8, int n, int k, int t, int maxparts) {
    const int cus = qe_num_cus();
    struct Kept {
        int n = 0, k = 0, t = 0, maxparts = 0, cus = 0;
        bool w8 = false;
        GemmChoice ch;
    };
    static thread_local Kept kept[64];
    Kept& slot = kept[((unsigned)n * 31u + (unsigned)k * 17u + (unsigned)t * 7u + (unsigned)maxparts) >> 4 & 63u];
    if (slot.n == n && slot.k == k && slot.t == t && slot.maxparts == maxparts && slot.cus == cus && slot.w8 == w8) return slot.ch;
    const long tiles_big = (long)((n + 255) / 256) * ((t + 255) / 256);
    GemmChoice ch{tiles_big >= cus ? 0 : 1, 1};
    GemmGeom g;
    if (ch.cfg == 0 && maxparts != 1 && k / BK % 4 == 0 && gemm_geom(0, n, k, t, 2, g) && 2 * g.nsplit <= cus) ch.ks = 2;
    else if (ch.cfg == 0) {
        const long rounds = (tiles_big + cus - 1) / cus;
        if ((double)tiles_big / (rounds * cus) < 0.9) ch.cfg = 1;
    }
    gemm_geom(ch.cfg, n, k, t, ch.ks, g);
    const double base = gemm_cost_us(w8, ch.cfg, n, k, t, g);
    double best = 0.94 * base;
    for (int cfg = 0; cfg < kNumCfg; cfg++)
        for (int ks = 1; ks <= kMaxSplit && (maxparts <= 0 || ks <= maxparts); ks++) {
            if (!gemm_geom(cfg, n, k, t, ks, g)) continue;
            const double us = gemm_cost_us(w8, cfg, n, k, t, g);
            if (us < best) {
                best = us;
                ch = GemmChoice{cfg, ks};
            }
        }
    slot = Kept{n, k, t, maxparts, cus, w8, ch};
    return ch;
}

template <int FMT, int SDT>
void run_choice(int cfg, int ks, const uint4* q, const uint16_t* s, int n, int k, const uint16_t* x, int ldx, int t,
                void* c, int ldc, int out, int sdt, hipStream_t st) {
    GemmGeom g;
    float* part = nullptr;
    std::optional<WsHold> hold;  // until the sum of the partials is launched
    if (ks > 1) {
        // no such split: these tiles unsplit; no workspace for it (memory; a graph capture on a stream that was not
        // sized before): the best unsplit configuration
        if (!gemm_geom(cfg, n, k, t, ks, g)) ks = 1;
        else if ((part = static_cast<float*>(hold.emplace(st).get(kWsSplit, g.ws_bytes))) == nullptr) {
            ks = 1;
            cfg = gemm_model_choice(FMT != kFmtW4, n, k, t, 1).cfg;
        }
    }
    if (ks == 1) gemm_geom(cfg, n, k, t, 1, g);
    if (cfg == 0) launch_cfg<FMT, SDT, 0>(q, s, n, k, x, ldx, t, c, ldc, out, sdt, g, part, st);
    else if (cfg == 1) launch_cfg<FMT, SDT, 1>(q, s, n, k, x, ldx, t, c, ldc, out, sdt, g, part, st);
    else if (cfg == 2) launch_cfg<FMT, SDT, 2>(q, s, n, k, x, ldx, t, c, ldc, out, sdt, g, part, st);
    else launch_cfg<FMT, SDT, 3>(q, s, n, k, x, ldx, t, c, ldc, out, sdt, g, part, st);
}

// timed choice: the candidates (the eight the cost model puts lowest, beside 256 x 256 and 256 x 128 tiles with splits
// 1, 2 and 4) once untimed, then 5 rounds in rotating order, the median; outside graph capture only (during capture:
// the cost model)
template <int FMT, int SDT>
GemmChoice gemm_tune_choice(int n, int k, const uint16_t* x, int ldx, int t, void* c, int ldc, int out, int sdt,
                            const uint4* q, const uint16_t* s, hipStream_t st) {
    std::vector<GemmChoice> cl;
    std::vector<std::pair<double, GemmChoice>> all;
    for (int cfg = 0; cfg < kNumCfg; cfg++)
        for (int ks = 1; ks <= kMaxSplit; ks++) {
            GemmGeom g;
            if (gemm_geom(cfg, n, k, t, ks, g)) all.emplace_back(gemm_cost_us(FMT != kFmtW4, cfg, n, k, t, g), GemmChoice{cfg, ks});
        }
    std::stable_sort(all.begin(), all.end(), [](const auto& a, const auto& b) { return a.first < b.first; });
    for (size_t i = 0; i < all.size(); i++) {
        const GemmChoice& ch = all[i].second;
        if (i < 8 || (ch.cfg < 2 && (ch.ks == 1 || ch.ks == 2 || ch.ks == 4))) cl.push_back(ch);
    }
    hipEvent_t e0, e1;
    HIP_CHECK(hipEventCreate(&e0));
    HIP_CHECK(hipEventCreate(&e1));
    auto time1 = [&](const GemmChoice& ch) {
        HIP_CHECK(hipEventRecord(e0, st));
        run_choice<FMT, SDT>(ch.cfg, ch.ks, q, s, n, k, x, ldx, t, c, ldc, out, sdt, st);
        HIP_CHECK(hipEventRecord(e1, st));
        HIP_CHECK(hipEventSynchronize(e1));
        float ms = 0.f;
        HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
        return ms;
    };
    for (const auto& ch : cl) time1(ch);
    constexpr int kReps = 5;
    std::vector<std::vector<float>> ts(cl.size());
    for (int r = 0; r < kReps; r++)
        for (size_t j = 0; j < cl.size(); j++) {
            const size_t i = (j + r) % cl.size();
            ts[i].push_back(time1(cl[i]));
        }
    size_t best = 0;
    float best_ms = 1e30f;
    for (size_t j = 0; j < cl.size(); j++) {
        std::sort(ts[j].begin(), ts[j].end());
        if (ts[j][kReps / 2] < best_ms) {
            best_ms = ts[j][kReps / 2];
            best = j;
        }
    }
    HIP_CHECK(hipEventDestroy(e0));
    HIP_CHECK(hipEventDestroy(e1));
    return cl[best];
}

// a stored or tuned split, halved until qe_gemm_set_sk_maxparts allows it
int capped_split(int ks) {
    const int cap = gemm_sk_maxparts();
    while (cap > 0 && ks > cap) ks /= 2;
    return ks < 1 ? 1 : ks;
}

template <int FMT, int SDT>
void launch_gemm(const uint4* q, const uint16_t* s, int n, int k, const uint16_t* x, int ldx, int t, void* c, int ldc,
                 int out, int sdt, bool tuned, hipStream_t st) {
    GemmChoice ch;
    const GemmKey key{FMT, n, k, gemm_bucket(t), out == kOutGLU ? 1 : 0};
    if (gemm_table_find(key, ch)) {
        // a stored split that the cap takes away, or that does not apply at this t of its bucket, leaves large tiles that
        // fill few CUs (1280 x 8192, t = 200: 173 us unsplit at 256 x 256, 94 at 128 x 128): the model's choice instead
        GemmGeom g;
        if (ch.ks > 1 && (capped_split(ch.ks) == 1 || !gemm_geom(ch.cfg, n, k, t, capped_split(ch.ks), g)))
            ch = gemm_model_choice(FMT != kFmtW4, n, k, t, gemm_sk_maxparts());
    } else {
        hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
        HIP_CHECK(hipStreamIsCapturing(st, &cs));
        if ((tuned || qe_config().gemm_tune) && cs == hipStreamCaptureStatusNone) {
            ch = gemm_tune_choice<FMT, SDT>(n, k, x, ldx, t, c, ldc, out, sdt, q, s, st);
            gemm_table_add(key, ch);
        } else {
            ch = gemm_model_choice(FMT != kFmtW4, n, k, t, gemm_sk_maxparts());
        }
    }
    run_choice<FMT, SDT>(ch.cfg, capped_split(ch.ks), q, s, n, k, x, ldx, t, c, ldc, out, sdt, st);
}

void gemm_check(int n, int k, const void* x, int ldx, int ldc, int t, bool glu) {
    CHECK(n > 0 && k > 0 && n % 16 == 0 && k % 128 == 0 && t >= 1, "gemm %d %d %d", n, k, t);
    CHECK(ldx >= k && ldx % 8 == 0 && ((uintptr_t)x & 15) == 0, "gemm ldx %d (multiple of 8, x 16-byte aligned)", ldx);
    CHECK(ldc >= (glu ? n / 2 : n), "gemm ldc %d", ldc);
    CHECK((long)((n + 127) / 128) * ((t + 255) / 256) < (1L << 31) / 8, "gemm t %d n %d", t, n);
}

}  // namespace

void gemm_w4(const W4& w, const uint16_t* x, int ldx, void* c, int ldc, int t, bool out_bf16, hipStream_t st,
             bool tuned) {
    gemm_check(w.n, w.k, x, ldx, ldc, t, w.glu);
    if (qe_config().gemm_h16) {  // the reference's fp16-accumulate numerics (its QE_GEMM_H16 with W4A8 off)
        gemm_w4h(w, x, ldx, c, ldc, t, out_bf16, st);
        return;
    }
    const int out = w.glu ? kOutGLU : out_bf16 ? kOutBF16 : kOutF32;
    if (w.sdt == kScaleF16) launch_gemm<kFmtW4, kScaleF16>(w.q, w.s, w.n, w.k, x, ldx, t, c, ldc, out, w.sdt, tuned, st);
    else launch_gemm<kFmtW4, kScaleBF16>(w.q, w.s, w.n, w.k, x, ldx, t, c, ldc, out, w.sdt, tuned, st);
}

void gemm_w4_choice(const W4& w, const uint16_t* x, int ldx, void* c, int ldc, int t, bool out_bf16, int cfg, int ks,
                    hipStream_t st) {
    gemm_check(w.n, w.k, x, ldx, ldc, t, w.glu);
    CHECK(cfg >= 0 && cfg < kNumCfg && ks >= 1 && ks <= kMaxSplit, "gemm choice cfg %d ks %d", cfg, ks);
    const int out = w.glu ? kOutGLU : out_bf16 ? kOutBF16 : kOutF32;
    if (w.sdt == kScaleF16) run_choice<kFmtW4, kScaleF16>(cfg, ks, w.q, w.s, w.n, w.k, x, ldx, t, c, ldc, out, w.sdt, st);
    else run_choice<kFmtW4, kScaleBF16>(cfg, ks, w.q, w.s, w.n, w.k, x, ldx, t, c, ldc, out, w.sdt, st);
}

bool gemm_split_applies(int cfg, int n, int k, int t, int ks) {
    GemmGeom g;
    return gemm_geom(cfg, n, k, t, ks, g) && g.nsplit > 0;
}

void gemm_w8(const W8& w, const uint16_t* x, int ldx, void* c, int ldc, int t, bool out_bf16, hipStream_t st,
             bool tuned) {
    gemm_check(w.n, w.k, x, ldx, ldc, t, w.glu);
    CHECK(!w.glu || w.q8, "gemm_w8: GLU is for Q8 matrices");
    const int out = w.glu ? kOutGLU : out_bf16 ? kOutBF16 : kOutF32;
    if (w.q8) launch_gemm<kFmtQ8, -1>(w.q, w.s, w.n, w.k, x, ldx, t, c, ldc, out, w.sdt, tuned, st);
    else if (w.per_channel) launch_gemm<kFmtW8C, -1>(w.q, w.s, w.n, w.k, x, ldx, t, c, ldc, out, w.sdt, tuned, st);
    else launch_gemm<kFmtW8G, -1>(w.q, w.s, w.n, w.k, x, ldx, t, c, ldc, out, w.sdt, tuned, st);
}

void matmul_w4(const W4& w, const uint16_t* x, int ldx, void* y, int ldy, int m, bool out_bf16, hipStream_t st) {
    if (m > kMatmulGemvRows) {
        gemm_w4(w, x, ldx, y, ldy, m, out_bf16, st);
        return;
    }
    // 17..64 rows: one pass over the weights (wdec.hip) where the shape fits it and it is the faster choice, unless
    // every row must keep the bits it has alone (batch_invariant)
    if (m > kMaxGemvRows && !qe_config().batch_invariant && wdec_w4_pick(w, x, ldx, m)) {
        wdec_w4(w, x, ldx, y, ldy, m, out_bf16, st);
        return;
    }
    // row blocks: 32 rows per launch (the skinny kernel's wide variant) while more than 16 remain and the rows are
    // 16-byte aligned, else 16; a row's bits do not depend on the block it falls in
    const size_t esz = (w.glu || out_bf16) ? 2 : 4;
    const bool aligned = ((uintptr_t)x & 15) == 0 && ldx % 8 == 0;
    for (int r0 = 0; r0 < m;) {
        const int left = m - r0;
        char* yr = reinterpret_cast<char*>(y) + (size_t)r0 * ldy * esz;
        if (aligned && left > kMaxGemvRows) {
            const int mm = left < kWideRows ? left : kWideRows;
            skinny_w4_wide(w, x + (size_t)r0 * ldx, ldx, yr, ldy, mm, out_bf16, st);
            r0 += mm;
        } else {
            const int mm = left < kMaxGemvRows ? left : kMaxGemvRows;
            gemv_w4(w, x + (size_t)r0 * ldx, ldx, yr, ldy, mm, out_bf16, st);
            r0 += mm;
        }
    }
}
