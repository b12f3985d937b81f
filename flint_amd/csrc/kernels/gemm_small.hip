// GEMMs whose output has few tiles: tiles of 32 x 32 to 128 x 64, one per
// workgroup, for every layout, epilogue and size the entry points take.
//
// A product with a few hundred rows leaves gemm_pipe.hip's 128 x 192 tiles on
// 4 to 48 of the 256 CUs, and each of those then streams its whole k-range at
// one CU's load rate. What bounds such a product is the bytes that one CU has
// to stream (its tile's two operand strips) and the latency of the first of
// them, so the tile here is as small as the MFMA's 32 x 32 allows:
//  * WM x WN waves each own one 32 x 32 block. Either they issue the operand
//    loads as well, or (LD) four more waves do: a load holds its wave for
//    about 33 cycles, as long as an MFMA takes, so that on a CU with one tile
//    the MFMA wave's own loads cost it half its time (NT 256 x 768 x 3072 9.6
//    -> 7.4 us with the loader waves, NN 11.3 -> 9.3; with eight of them 7.8).
//    Where several tiles share a CU the extra waves only get in the way.
//  * k-steps of 64 through S LDS stages by direct-to-LDS buffer loads, S steps
//    in flight, in groups of U steps with one barrier each. The fragments of
//    the next group are read while a group's MFMAs run, which also frees its
//    stages for the loads of the group S / U further on at the same barrier.
//  * Each 32 x 32 block is one chain of v_mfma_f32_32x32x16_f16 over k in
//    ascending order from a zero accumulator, as in the other GEMM kernels:
//    the same sums, bit for bit, whichever kernel a shape runs on.
//  * The epilogue's inputs (bias, residual, pre, the old y) load before the
//    k-loop; the sums go through LDS once so that every thread finishes 4 or 8
//    consecutive columns of a row.
//  * Ragged sizes: rows and columns past the operands read zeros or values
//    that only reach outputs that are not stored; a k tail (k % 64) reads
//    zeros from both operands.
//  * Larger tiles (32 x 64 to 128 x 64) take over as the tile count passes the
//    CUs, until gemm_pipe.hip's tiles fill the GPU: gemm_small_plan compares
//    all of them by their estimated times.
// Measured (one MI355X, operands rotated past the caches, launch included,
// against the kernels before these): NT 64 x 768 x 3072 22.4 -> 7.2 us, 256 x
// 768 x 768 9.5 -> 4.6, 1024 x 768 x 3072 25 -> 12.2; NN 256 x 768 x 50304 518
// -> 177; TN 768 x 768 x 256 9.0 -> 4.9; ragged NT 1000 x 200 x 800 14.0 ->
// 4.6, TN 768 x 768 x 1000 60 -> 7.2. What bounds a tile alone on its CU: the
// chain of dependent MFMAs (32 cycles each, 4 a k-step and block) and one
// exposed LDS read per group; with the operand loads returning nothing at all
// it takes as long. With several tiles a CU, the direct-to-LDS load rate
// (about 32 B a cycle with four waves) and the fragment reads.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <type_traits>

#include "common/common.h"
#include "common/tuning.h"
#include "kernels/gemm_common.h"
#include "kernels/kernels.h"

namespace flint {
namespace {

constexpr int kStep = 64;   // k per step

// A split TN's sum of its partials: a launch of its own (us).
constexpr double kSplitSumUs = 3.0;

// A buffer offset past every resource: the load returns zeros.
constexpr unsigned kOutside = 0xfffffff0u;

// The FP32 value itself, however it was formed: a conversion that follows
// rounds it and not the exact product behind it.
__device__ __forceinline__ float settled(float x) {
    asm("" : "+v"(x));
    return x;
}

template <int WM, int WN, int NW, int S, int U, bool LD, Layout L, Store ST, bool HV = false>
__global__ void __launch_bounds__(NW * 64) gemm_small(Operands op, TileArgs ta) {
    // The host pass only needs a kernel to emit a launch stub for.
#if defined(__HIP_DEVICE_COMPILE__)
    static_assert(WM * WN <= NW, "at most one block per wave");
    static_assert(S % U == 0 && S / U >= 2, "a group in use, one landing");
    constexpr int T = NW * 64;
    constexpr int BM = 32 * WM, BN = 32 * WN;
    // x (rows m, the MFMA's B operand) and w (rows n, its A operand) are
    // k-major ([64 k][rows] in LDS) or row-major ([rows][64 k]).
    constexpr bool kXM = L == Layout::kTN;
    constexpr bool kWM = L != Layout::kNT;
    using XFrag = std::conditional_t<kXM, TrFrag, f16x8>;
    using WFrag = std::conditional_t<kWM, TrFrag, f16x8>;
    constexpr bool kBias =
        ST == Store::kBias || ST == Store::kBiasGelu || ST == Store::kBiasResidual;
    constexpr bool kF32 = ST == Store::kBiasResidual || ST == Store::kTn;
    // A step's 1 KB loads, x's first, dealt to the waves in turn.
    constexpr int NL = LD ? NW - WM * WN : NW;   // waves that load
    constexpr int kLoadsA = BM / 8, kLoads = (BM + BN) / 8, PER = kLoads / NL;
    static_assert(kLoads % NL == 0 && S * PER < 64, "whole loads per wave, vmcnt range");
    constexpr int kGroupLoads = U * PER;
    constexpr int kStage = (BM + BN) * kStep;
    constexpr int kLd = BN + 4;                       // staged sums: floats a row
    static_assert(BM * kLd * 2 <= S * kStage, "the sums reuse the stages");
    __shared__ __attribute__((aligned(16))) _Float16 lds[S * kStage];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m = op.m, n = op.n, K = op.k;
    const bool loads = !LD || wave >= WM * WN;
    const int lw = LD ? max(wave - WM * WN, 0) : wave;   // among the loading waves
    const bool split = ST == Store::kTn && op.partials != nullptr;

    // ---- this workgroup's tile
    int slice, tm, tn;
    if (op.causal && L != Layout::kNT) {
        // A tile's k-range grows (NN) or shrinks (TN) with its row block:
        // longest first.
        const unsigned per_row = unsigned(ta.slices) * unsigned(ta.tiles_n);
        const int d = int(blockIdx.x / per_row);
        const unsigned rem = blockIdx.x % per_row;
        tm = L == Layout::kNN ? ta.tiles_m - 1 - d : d;
        slice = int(rem / unsigned(ta.tiles_n));
        tn = int(rem % unsigned(ta.tiles_n));
    } else {
        map_tile(ta, blockIdx.x, &slice, &tm, &tn);
    }
    const int m0 = tm * BM, n0 = tn * BN;
    if (L == Layout::kNT && op.causal && n0 >= m0 + BM) return;   // above the diagonal
    int k_begin = 0, k_end = K;
    if (L == Layout::kNN && op.causal) k_end = min(K, (m0 + BM + kStep - 1) / kStep * kStep);
    if (L == Layout::kTN && op.causal) k_begin = m0 / kStep * kStep;
    const _Float16* xs = op.x;
    const _Float16* ws = op.w;
    size_t y_off = 0;
    if (split) {
        k_begin = slice * ta.split_len;
        k_end = min(K, k_begin + ta.split_len);
        y_off = size_t(slice) * m * n;
    } else if (ta.slices > 1) {
        xs += size_t(slice) * m * K;
        ws += HV ? head_view_offset(op.wv, slice) : size_t(slice) * n * K;
        y_off = HV ? head_view_offset(op.yv, slice) : size_t(slice) * m * n;
    }
    const int a_ld = kXM ? m : K;
    const int b_ld = kWM ? (HV ? op.wv.ld : n) : K;
    const size_t y_ld = HV ? op.yv.ld : n;

    // ---- operand loads. Row-major: a resource over the tile's valid rows,
    // the k-step in the scalar offset, chunks past k_end sent outside.
    // k-major: a resource from the step's first k row to the operand's end.
    // Offsets within a tile fit in 32 bits: the entry points take k up to 65,536
    // (kGemmMaxK) and m and n up to 8,388,480 (kGemmMaxMN).
    const _Float16* const a = kXM ? xs + m0 : xs + size_t(m0) * K;
    const _Float16* const b = kWM ? ws + n0 : ws + size_t(n0) * K;
    const size_t a_bytes = kXM ? (size_t(K) * m - m0) * 2 : size_t(min(BM, m - m0)) * K * 2;
    const size_t b_bytes = kWM ? (size_t(K - 1) * b_ld + n - n0) * 2
                               : size_t(min(BN, n - n0)) * K * 2;
    // Load v = q NL + lw of a step fills LDS bytes [v KB, v KB + 1 KB) of its
    // stage (x's region, then w's); lane l writes bytes 16 l .. + 15 of it.
    unsigned voff[PER];
    int kofs[PER];   // row-major: the lane's k within a step
    auto of_x = [&](int q) {
        return kLoadsA % NL == 0 ? q < kLoadsA / NL : q * NL + lw < kLoadsA;
    };
    auto place = [&](int q, bool kmajor, int rows, int u, int ld) {
        if (kmajor) {
            const int cpr = rows / 8;                 // chunks per k row
            const int c = u * 64 + lane;
            const int r = c / cpr;
            const int chunk = rows >= 64 ? (c % cpr) ^ kmajor_key(r) : c % cpr;
            voff[q] = unsigned(r) * unsigned(ld) * 2u + unsigned(chunk) * 16u;
            kofs[q] = 0;
        } else {
            const int row = u * 8 + lane / 8;
            const int chunk = (lane % 8) ^ row_key<kStep>(row);
            voff[q] = unsigned(row) * unsigned(ld) * 2u + unsigned(chunk) * 16u;
            kofs[q] = chunk * 8;
        }
    };
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int v = q * NL + lw;
        if (of_x(q)) place(q, kXM, BM, v, a_ld);
        else place(q, kWM, BN, v - kLoadsA, b_ld);
    }
    auto clamp32 = [](size_t v) { return v < 0xffffffffu ? unsigned(v) : 0xffffffffu; };
    // Loads step k0 into stage st. Steps past the last one load nothing (an
    // empty resource), so that every wait counts the same loads.
    auto issue = [&](int k0, int st) {
        if (!loads) return;
        const bool live = k0 < k_end;
        const size_t ka = kXM ? size_t(k0) * a_ld : 0, kb = kWM ? size_t(k0) * b_ld : 0;
        const auto ra = __builtin_amdgcn_make_buffer_rsrc(
            uniform_ptr(a + ka), 0, live ? clamp32(a_bytes - ka * 2) : 0u, 0x00020000);
        const auto rb = __builtin_amdgcn_make_buffer_rsrc(
            uniform_ptr(b + kb), 0, live ? clamp32(b_bytes - kb * 2) : 0u, 0x00020000);
        const int left = k_end - k0;
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int v = q * NL + lw;
            lds_half* dst = (lds_half*)(lds + st * kStage + v * 512);
            auto load = [&](const auto& rsrc, bool kmajor) {
                const unsigned off = kmajor || kofs[q] < left ? voff[q] : kOutside;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    rsrc, (__attribute__((address_space(3))) void*)dst, 16, off,
                    kmajor ? 0u : unsigned(k0) * 2u, 0, 0);
            };
            if (of_x(q)) load(ra, kXM);
            else load(rb, kWM);
        }
    };

    // ---- the epilogue's chunks: kCh consecutive columns of a row, each
    // thread kChunks of them; their inputs load now.
    constexpr int kCh = BM * BN >= 8 * T ? 8 : 4;
    constexpr int kCpr = BN / kCh, kTileChunks = BM * BN / kCh;
    constexpr int kChunks = (kTileChunks + T - 1) / T;
    // Whole chunks only, unless n leaves a partial one (NT alone; others have
    // n % 8 == 0).
    const bool whole = L != Layout::kNT || n % kCh == 0;
    const bool accumulate = ST == Store::kTn && !split && op.accumulate;
    float aux[kF32 || ST == Store::kDGelu ? kChunks : 1][kCh];
    float bias[kBias ? kChunks : 1][kCh];
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
        const int c = i * T + tid;
        const int row = c < kTileChunks ? m0 + c / kCpr : m, col = n0 + c % kCpr * kCh;
        const int cols = row < m ? n - col : 0;       // valid columns from col on
        const size_t at = y_off + size_t(row) * y_ld + col;
        if constexpr (kBias) {
            if (whole) {
#pragma unroll
                for (int e = 0; e < kCh; e += 4) {
                    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
                    if (cols > 0) v = *reinterpret_cast<const f32x4*>(op.bias + col + e);
#pragma unroll
                    for (int j = 0; j < 4; ++j) bias[i][e + j] = v[j];
                }
            } else {
#pragma unroll
                for (int e = 0; e < kCh; ++e) bias[i][e] = e < cols ? op.bias[col + e] : 0.0f;
            }
        }
        if constexpr (kF32) {
            const float* src = ST == Store::kTn ? static_cast<const float*>(op.y)
                                                : static_cast<const float*>(op.aux);
            const bool reads = ST == Store::kBiasResidual || accumulate;
            if (whole) {
#pragma unroll
                for (int e = 0; e < kCh; e += 4) {
                    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
                    if (reads && cols > 0) v = *reinterpret_cast<const f32x4*>(src + at + e);
#pragma unroll
                    for (int j = 0; j < 4; ++j) aux[i][e + j] = v[j];
                }
            } else {
#pragma unroll
                for (int e = 0; e < kCh; ++e) aux[i][e] = reads && e < cols ? src[at + e] : 0.0f;
            }
        }
        if constexpr (ST == Store::kDGelu) {
            const _Float16* src = static_cast<const _Float16*>(op.aux) + at;
#pragma unroll
            for (int e = 0; e < kCh; e += 4) {
                f16x4 v = {};
                if (cols > 0) v = *reinterpret_cast<const f16x4*>(src + e);
#pragma unroll
                for (int j = 0; j < 4; ++j) aux[i][e + j] = float(v[j]);
            }
        }
    }

    // ---- k-loop
    const bool computes = wave < WM * WN;
    const int wm = wave / WN, wn = wave % WN;
    const int fr = lane & 31, fc = lane >> 5;
    f32x16 acc = {};
    // Fragment of operand rows r0 .. r0 + 31, k16 sub-step kk: lane l gets row
    // r0 + l % 32, k 8 (l / 32) .. + 8.
    auto frag_rowmajor = [&](const _Float16* region, int r0, int kk) {
        const int row = r0 + fr;
        return *reinterpret_cast<const f16x8*>(region + row * kStep +
                                               (((kk * 2 + fc) ^ row_key<kStep>(row)) * 8));
    };
    // Two transposing reads (inline asm: see gemm_pipe.hip). Their results are
    // not there until wait_frags; every use comes after one, and so does every
    // way out of the loop. A 32-row region's rows are 64 bytes: the four that
    // 32 lanes read are consecutive, so it needs no swizzle.
    auto frag_kmajor = [&](const _Float16* region, auto rows_c, int r0, int kk) {
        constexpr int rows = decltype(rows_c)::value;
        const int j = lane & 15;
        const int col = r0 + 16 * ((lane >> 4) & 1) + 4 * (j & 3);
        const int key = rows >= 64 ? kmajor_key(j >> 2) : 0;
        const int chunk = ((col >> 3) ^ key) * 8 + (col & 4);
        const int k = kk * 16 + 8 * fc + (j >> 2);
        const unsigned a0 =
            unsigned(reinterpret_cast<uintptr_t>((lds_half*)(region + k * rows + chunk)));
        TrFrag f;
        asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(f.lo) : "v"(a0));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(f.hi) : "v"(a0), "i"(4 * rows * 2));
        return f;
    };
    // Waits for a step's fragments. The empty asm uses the transposing reads'
    // registers, so that they stay theirs while the reads are in flight, also
    // where nothing uses the values (after the last step).
    auto wait_frags = [&](const XFrag (&x)[4 * U], const WFrag (&w)[4 * U]) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int kk = 0; kk < 4 * U; ++kk) {
            if constexpr (kXM) asm volatile("" ::"v"(x[kk].lo), "v"(x[kk].hi));
            if constexpr (kWM) asm volatile("" ::"v"(w[kk].lo), "v"(w[kk].hi));
        }
    };
    // Fragments of a batch of kBatch steps: a whole group's, where groups have
    // two steps, else a step's.
    constexpr int kBatch = U, kFrags = 4 * kBatch;
    XFrag xf[2][kFrags];
    WFrag wf[2][kFrags];
    // Fragment q of the batch whose first stage is st.
    auto read_frag = [&](int st, int q, XFrag& x, WFrag& w) {
        const _Float16* s0 = lds + (st + q / 4) * kStage;
        const int kk = q % 4;
        if constexpr (kXM) x = frag_kmajor(s0, std::integral_constant<int, BM>{}, wm * 32, kk);
        else x = frag_rowmajor(s0, wm * 32, kk);
        if constexpr (kWM)
            w = frag_kmajor(s0 + BM * kStep, std::integral_constant<int, BN>{}, wn * 32, kk);
        else w = frag_rowmajor(s0 + BM * kStep, wn * 32, kk);
    };

    // Groups of U steps; a last group's steps past k_end add zeros.
    const int groups = (k_end - k_begin + U * kStep - 1) / (U * kStep);
    int k0 = k_begin;
#pragma unroll
    for (int j = 0; j < S; ++j, k0 += kStep) issue(k0, j);
    wait_vmcnt<(S / U - 1) * kGroupLoads>();
    block_sync();
    if (computes) {
#pragma unroll
        for (int q = 0; q < kFrags; ++q) read_frag(0, q, xf[0][q], wf[0][q]);
        wait_frags(xf[0], wf[0]);
    }
    int st = 0;   // the first stage of the group whose fragments are in registers
    // One group: its MFMAs with the next group's fragment reads between them
    // (a burst of reads before the MFMAs cost a third of a step). Before the
    // reads the next group has landed for every wave, and every wave holds
    // this group's fragments, so its stages take the loads of the group S / U
    // further on; the first MFMA runs under that barrier. One wait per group
    // for the fragments: at the end of every step, it exposed the last read's
    // latency each time.
    auto group = [&](XFrag (&x)[kFrags], WFrag (&w)[kFrags], XFrag (&xn)[kFrags],
                     WFrag (&wn_)[kFrags]) {
        auto mfma = [&](int q) {
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(as_f16x8(w[q]), as_f16x8(x[q]), acc, 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        if (computes) mfma(0);
        wait_vmcnt<(S / U - 2) * kGroupLoads>();
        block_sync();
#pragma unroll
        for (int j = 0; j < U; ++j, k0 += kStep) issue(k0, st + j);
        st = st + U == S ? 0 : st + U;
        if (computes) {
            __builtin_amdgcn_sched_barrier(0);
            read_frag(st, 0, xn[0], wn_[0]);
#pragma unroll
            for (int q = 1; q < kFrags; ++q) {
                read_frag(st, q, xn[q], wn_[q]);
                __builtin_amdgcn_sched_barrier(0);
                mfma(q);
            }
            wait_frags(xn, wn_);
        }
    };
    for (int g = 0; g < groups; g += 2) {
        group(xf[0], wf[0], xf[1], wf[1]);
        if (g + 1 < groups) group(xf[1], wf[1], xf[0], wf[0]);
    }

    // ---- epilogue: the sums through LDS (the stages, once every load into
    // them has landed), then whole chunks.
    wait_vmcnt<0>();
    block_sync();
    float* const sums = reinterpret_cast<float*>(lds);
    if (computes) {
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
            const f32x4 v = {acc[g4 * 4 + 0], acc[g4 * 4 + 1], acc[g4 * 4 + 2], acc[g4 * 4 + 3]};
            *reinterpret_cast<f32x4*>(sums + (wm * 32 + fr) * kLd + wn * 32 + g4 * 8 + fc * 4) = v;
        }
    }
    block_sync();
#pragma unroll
    for (int i = 0; i < kChunks; ++i) {
        const int c = i * T + tid;
        const int r = c / kCpr, cc = c % kCpr * kCh;
        const int row = m0 + r, col = n0 + cc;
        if (c >= kTileChunks || row >= m || col >= n) continue;
        float v[kCh];
#pragma unroll
        for (int e = 0; e < kCh; e += 4) {
            const f32x4 s4 = *reinterpret_cast<const f32x4*>(sums + r * kLd + cc + e);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[e + j] = s4[j];
        }
        const size_t at = y_off + size_t(row) * y_ld + col;
        const int cols = n - col;
        typedef _Float16 hch __attribute__((ext_vector_type(kCh)));
        auto store_half = [&](void* out, const hch& h) {
            _Float16* p = static_cast<_Float16*>(out) + at;
            if (whole) {
                *reinterpret_cast<hch*>(p) = h;
            } else {
#pragma unroll
                for (int e = 0; e < kCh; ++e)
                    if (e < cols) p[e] = h[e];
            }
        };
        if constexpr (kF32) {
            if constexpr (ST == Store::kBiasResidual) {
#pragma unroll
                for (int e = 0; e < kCh; ++e) v[e] = aux[i][e] + (v[e] + bias[i][e]);
            } else if (accumulate) {
#pragma unroll
                for (int e = 0; e < kCh; ++e) v[e] = aux[i][e] + v[e];
            }
            float* p = (split ? op.partials : static_cast<float*>(op.y)) + at;
            if (whole) {
#pragma unroll
                for (int e = 0; e < kCh; e += 4)
                    *reinterpret_cast<f32x4*>(p + e) = f32x4{v[e], v[e + 1], v[e + 2], v[e + 3]};
            } else {
#pragma unroll
                for (int e = 0; e < kCh; ++e)
                    if (e < cols) p[e] = v[e];
            }
        } else {
            hch h;
            if constexpr (kBias) {
#pragma unroll
                for (int e = 0; e < kCh; ++e) v[e] = settled(v[e] + bias[i][e]);
            }
            if constexpr (ST == Store::kScale) {
#pragma unroll
                for (int e = 0; e < kCh; ++e) v[e] = settled(v[e] * op.scale);
            }
            if constexpr (ST == Store::kDGelu) {
#pragma unroll
                for (int e = 0; e < kCh; ++e) v[e] = settled(v[e] * gelu_grad(aux[i][e]));
            }
#pragma unroll
            for (int e = 0; e < kCh; ++e) h[e] = _Float16(v[e]);
            store_half(ST == Store::kBiasGelu ? op.aux : op.y, h);
            if constexpr (ST == Store::kBiasGelu) {
#pragma unroll
                for (int e = 0; e < kCh; ++e) h[e] = _Float16(settled(gelu(v[e])));
                store_half(op.y, h);
            }
        }
    }
#endif
}

// A configuration and its cost in us: `alone` is a k-step of a tile that has
// its CU to itself, `shared` a tile's k-step where the CU runs several, `fixed`
// a tile's prologue and epilogue. Each per layout NT, NN, TN (FP32 stores).
// Fitted, together with gemm_pipe_estimate's constants, to measured times of
// products of 16 to 8,192 rows, widths 64 to 50,304 and k 16 to 50,304, batched
// ones among them (one MI355X, operands rotated past the caches). Of 1,047 drawn
// ones timed on every kernel and tile, the choice (with the charges and limits
// below) is within 7% of the fastest for 929, at worst 1.65 times it, 2.6% in the
// geometric mean.
struct SmallConfig {
    int bm, bn, waves, stages, unit;
    int resident;   // workgroups a CU holds
    double alone[3], shared[3], fixed[3];
};
constexpr SmallConfig kSmallConfigs[] = {
    // Least to stream per CU, four loader waves beside the MFMA wave: the
    // smallest products.
    {32, 32, 5, 8, 2, 2, {0.052, 0.100, 0.172}, {0.128, 0.196, 0.195}, {1.0, 0.571, 1.02}},
    // The same for up to twice the tiles.
    {32, 64, 4, 6, 2, 2, {0.080, 0.170, 0.190}, {0.138, 0.185, 0.208}, {0.99, 0.291, 0.955}},
    // One tile a CU, four loader waves: long k-ranges.
    {64, 64, 8, 6, 2, 1, {0.098, 0.187, 0.193}, {0.250, 0.318, 0.308}, {1.35, 0.351, 1.15}},
    // Two tiles a CU.
    {64, 64, 4, 4, 1, 2, {0.178, 0.254, 0.235}, {0.234, 0.277, 0.314}, {1.03, 0.226, 0.776}},
    // The fewest operand bytes per output: many tiles.
    {128, 64, 8, 3, 1, 2, {0.263, 0.347, 0.410}, {0.393, 0.499, 0.630}, {1.12, 0.198, 0.645}},
};

// The pipeline's workgroups store one tile while they load the next; here a
// tile's stores are waited for before its CU's place is free. Over 1,050 drawn
// products (16 to 16,384 rows, k from 8) the choice without this and the limit
// below was slower than the kernel before by more than 3% for 65, up to 1.74
// times, all of a round of pipeline tiles or more or of short k (TN 1472 x 50304 x 64
// 61 -> 103 us, batched NT 38 x 640 x 640 x 64 10.9 -> 18.1); with them for 17, ten
// of them of ragged k, where gemm.hip's kernels now and then are the fastest (NT +
// residual 1391 x 1536 x 5192 71 us and 90; in the geometric mean over ragged k the
// choice takes 0.55 of their time).
constexpr double kStoreMbPerUs = 6.0;
constexpr double kMostPipeLoad = 1.25;

// Bytes a product writes per output value.
double out_bytes(Epilogue e) {
    return e == Epilogue::kBiasGelu || e == Epilogue::kBiasResidual || e == kTnFloat ? 4.0 : 2.0;
}

// Up to how many rounds of 128 x 64 tiles these kernels are faster than
// gemm.hip's, which run what the pipeline does not take. Up to five: nearly
// everywhere (NN 512 x 17000 x 65536, past 2^31 bytes, 3175 -> 2372 us; NT 64 x
// 50301 x 7744 245 -> 183). Past that gemm.hip's larger tiles read less: TN 50304 x
// 768 x 24576 2645 us against 4095, NN 24576 x 768 x 50304 2372 against 3316,
// batched NT 96 x 1000 x 1000 x 520 231 against 278. Two exceptions: odd widths
// (gemm.hip stores them value by value) while k is short (NT 8190 x 24001 x 768
// 769 us and 646 here, x 1536 1035 and 1180; with bias 768 730 and 788; GELU's
// second output moves the line to 2,048), and batched TN of ragged k (200 x 520 x
// 520 x 520 672 and 188, 96 x 1000 x 1000 x 520 250 and 273). Either was measured
// up to 96 rounds (NT 8192 x 50257 x 768, 196 of them: 1486 us and 1592).
double most_rounds(GemmLayout l, Epilogue e, size_t n, size_t k) {
    const size_t odd_k = e == Epilogue::kBiasGelu ? 2048
                         : e == Epilogue::kNone || e == Epilogue::kScale ? 1280
                                                                         : 640;
    const bool batched_tn = l == GemmLayout::kTN && e == Epilogue::kNone;
    return batched_tn || (n % 8 != 0 && k <= odd_k) ? 96.0 : 5.0;
}

int layout_index(GemmLayout l) { return l == GemmLayout::kNT ? 0 : (l == GemmLayout::kNN ? 1 : 2); }

// Estimated us (past a launch's own) of `tiles` tiles of `steps` k-steps.
double small_cost(const SmallConfig& c, GemmLayout l, double tiles, double steps, int cus) {
    const int i = layout_index(l);
    const double load = tiles / cus;
    if (load <= 1.0) return c.fixed[i] + steps * c.alone[i];
    if (c.resident == 1) return std::ceil(load) * (c.fixed[i] + steps * c.shared[i]);
    // Tiles that share a CU overlap one another's prologues. The last round is
    // as long as its fullest CU, but runs faster where the others are empty.
    const double full = 0.5 * (load + std::ceil(load));
    return std::max(1.0, load - 0.5) * c.fixed[i] +
           steps * std::max(c.alone[i], full * c.shared[i]);
}

// A launch holds fewer than 2^32 threads along x.
bool fits_a_launch(double tiles, int waves) { return tiles * waves * 64 <= double(0xffffffffu); }

double small_tiles(const SmallConfig& c, size_t slices, size_t m, size_t n) {
    return double((m + c.bm - 1) / c.bm) * double((n + c.bn - 1) / c.bn) * double(slices);
}

// The "gemm_small" override: "0" turns these kernels off,
// "bm,bn,waves,stages,unit" takes that configuration for every product.
bool small_forced(SmallConfig* out, bool* disabled) {
    *disabled = false;
    const char* e = tuning(Tune::kGemmSmall);
    if (e == nullptr) return false;
    if (e[0] == '0' && e[1] == '\0') {
        *disabled = true;
        return false;
    }
    SmallConfig c{};
    if (std::sscanf(e, "%d,%d,%d,%d,%d", &c.bm, &c.bn, &c.waves, &c.stages, &c.unit) != 5)
        return false;
    for (const SmallConfig& k : kSmallConfigs) {
        if (k.bm == c.bm && k.bn == c.bn && k.waves == c.waves && k.stages == c.stages &&
            k.unit == c.unit) {
            *out = k;
            return true;
        }
    }
    return false;
}

template <Layout L, Store ST, bool HV>
hipError_t launch(const SmallPlan& c, const Operands& op, size_t slices, hipStream_t stream) {
    TileArgs ta{};
    ta.tiles_m = (op.m + c.bm - 1) / c.bm;
    ta.tiles_n = (op.n + c.bn - 1) / c.bn;
    const size_t per = size_t(ta.tiles_m) * size_t(ta.tiles_n);
    if (!fits_a_launch(double(per) * double(slices), c.waves)) return hipErrorInvalidValue;
    ta.tiles_per_slice = int(per);
    ta.slices = int(slices);
    ta.group_m = 8;
    ta.split_len = c.split_len;
    const dim3 grid(unsigned(per * slices));
#define FLINT_SMALL_CASE(BM_, BN_, NW_, S_, U_, LD_)                                               \
    if (c.bm == BM_ && c.bn == BN_ && c.waves == NW_ && c.stages == S_ && c.unit == U_) {          \
        hipLaunchKernelGGL((gemm_small<BM_ / 32, BN_ / 32, NW_, S_, U_, LD_, L, ST, HV>), grid,    \
                           dim3(NW_ * 64), 0, stream, op, ta);                                     \
        return hipGetLastError();                                                                  \
    }
    FLINT_SMALL_CASE(32, 32, 5, 8, 2, true)
    FLINT_SMALL_CASE(32, 64, 4, 6, 2, false)
    FLINT_SMALL_CASE(64, 64, 8, 6, 2, true)
    FLINT_SMALL_CASE(64, 64, 4, 4, 1, false)
    FLINT_SMALL_CASE(128, 64, 8, 3, 1, false)
#undef FLINT_SMALL_CASE
    return hipErrorInvalidValue;
}

}  // namespace

// Whether these kernels take a product, and with which tile and TN split:
// where the cheapest configuration costs less than gemm_pipe.hip's choice, by
// the estimates of both (gemm_pipe_estimate; infinite where the pipeline does
// not take the shape). Either side gives the same sums, so the line only has
// to be about right.
bool gemm_small_plan(GemmLayout l, Epilogue e, size_t slices, size_t m, size_t n, size_t k,
                     int max_splits, SmallPlan* plan, bool views) {
    SmallConfig forced;
    bool disabled = false;
    const bool force = small_forced(&forced, &disabled);
    if (disabled || m == 0 || n == 0 || k == 0) return false;
    // A forced pipeline tile means the pipeline, and no pipeline gemm.hip.
    if (!force && gemm_pipe_override(l, e, m, n, k, views)) return false;
    int cus = 256;
    if (device_cus(&cus) != hipSuccess) return false;
    const PipeEstimate pipe =
        force ? PipeEstimate{} : gemm_pipe_estimate(l, e, slices, m, n, k, max_splits, views);
    // From a round and a quarter of the pipeline's tiles on they are the faster
    // ones, whatever the estimates say (kMostPipeLoad).
    if (pipe.load > kMostPipeLoad) return false;
    double best = pipe.us;
    if (best == kNoEstimate && !force &&
        small_tiles(kSmallConfigs[4], slices, m, n) > most_rounds(l, e, n, k) * cus)
        return false;
    // Only for a clear gain, so that no product gets slower by an estimate's
    // error (NN 1500 x 2272 x 568: 11.7 us here, 10.3 in the pipeline).
    if (best != kNoEstimate) best *= 0.9;
    const double out_mb = double(slices) * double(m) * double(n) * out_bytes(e) / 1e6;
    bool taken = false;
    for (const SmallConfig& c : kSmallConfigs) {
        if (force && (c.bm != forced.bm || c.bn != forced.bn || c.waves != forced.waves)) continue;
        const double tiles = small_tiles(c, slices, m, n);
        if (!fits_a_launch(tiles, c.waves)) continue;
        for (int sp = 1; sp <= max_splits; ++sp) {
            const size_t len = ((k + sp - 1) / sp + kStep - 1) / kStep * kStep;
            if (size_t(sp - 1) * len >= k || !fits_a_launch(tiles * sp, c.waves)) break;
            double cost = small_cost(c, l, tiles * sp, double(len / kStep), cus);
            cost += double(sp) * out_mb / kStoreMbPerUs;
            if (sp > 1) cost += kSplitSumUs + double(sp + 2) * double(m) * double(n) * 4.0 / 5e6;
            if (cost < best) {
                best = cost;
                taken = true;
                *plan = {c.bm, c.bn, c.waves, c.stages, c.unit, sp, int(len)};
            }
        }
    }
    return taken;
}

bool gemm_small_override() {
    SmallConfig forced;
    bool disabled = false;
    return small_forced(&forced, &disabled);
}

hipError_t launch_gemm_small(const SmallPlan& c, GemmLayout l, Epilogue e, void* y, const void* x,
                             const void* w, const void* bias, void* aux, float scale,
                             size_t slices, size_t m, size_t n, size_t k, bool accumulate,
                             void* partials, hipStream_t stream, bool causal, const HeadView* wv,
                             const HeadView* yv) {
    Operands op{};
    op.y = y;
    op.x = static_cast<const _Float16*>(x);
    op.w = static_cast<const _Float16*>(w);
    op.bias = static_cast<const float*>(bias);
    op.aux = aux;
    op.partials = static_cast<float*>(partials);
    op.scale = scale;
    op.accumulate = accumulate ? 1 : 0;
    op.m = int(m);
    op.n = int(n);
    op.k = int(k);
    op.causal = causal ? 1 : 0;
    const bool hv = wv != nullptr && yv != nullptr;
    if (hv) {
        op.wv = *wv;
        op.yv = *yv;
    }
    if (l == GemmLayout::kNT) {
        switch (e) {
        case Epilogue::kNone: return launch<Layout::kNT, Store::kNone, false>(c, op, slices, stream);
        case Epilogue::kBias: return launch<Layout::kNT, Store::kBias, false>(c, op, slices, stream);
        case Epilogue::kBiasGelu:
            return launch<Layout::kNT, Store::kBiasGelu, false>(c, op, slices, stream);
        case Epilogue::kBiasResidual:
            return launch<Layout::kNT, Store::kBiasResidual, false>(c, op, slices, stream);
        case Epilogue::kScale: return launch<Layout::kNT, Store::kScale, false>(c, op, slices, stream);
        default: return hipErrorInvalidValue;
        }
    }
    if (l == GemmLayout::kNN) {
        if (e == Epilogue::kDGelu) return launch<Layout::kNN, Store::kDGelu, false>(c, op, slices, stream);
        if (e != Epilogue::kNone) return hipErrorInvalidValue;
        return hv ? launch<Layout::kNN, Store::kNone, true>(c, op, slices, stream)
                  : launch<Layout::kNN, Store::kNone, false>(c, op, slices, stream);
    }
    if (e == kTnFloat) return launch<Layout::kTN, Store::kTn, false>(c, op, size_t(c.splits), stream);
    if (e != Epilogue::kNone) return hipErrorInvalidValue;
    return hv ? launch<Layout::kTN, Store::kTnHalf, true>(c, op, slices, stream)
              : launch<Layout::kTN, Store::kTnHalf, false>(c, op, slices, stream);
}

}  // namespace flint
