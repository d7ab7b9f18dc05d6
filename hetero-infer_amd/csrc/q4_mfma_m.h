// Small-M GEMV on the int8 matrix cores (up to 16 activation rows, gs 64; the
// library takes it from kMfMinRows rows, below which the streaming kernel is
// faster).
//
// The arithmetic is the reference's x86 path of kernel/q4gemv.c:232-301 for
// every row of x: x quantised to int16 once per row (:244-270), an exact
// integer dot per group of 64 (:80-111), and per output
//   acc = acc + fma(scale, xscale * (float)idot, bias * xsum[g])   (:173-180)
// in ascending group order.  Only the integer dots move to the MFMA; the fp32
// steps stay in the order above, so the result is bit-identical to the
// streaming kernel and to the reference.
//
// Integer dots.  One v_mfma_i32_16x16x64_i8 covers a group: A (16 x 64, int8)
// is one byte plane of x, B (64 x 16) the group's nibbles of 16 weight rows.
// xq = 256 * xh + xl with xh the signed high byte and xl the unsigned low
// byte; A carries xl ^ 0x80 (= xl - 128, a signed byte) and xh, and a third
// MFMA with A = 1 gives the nibbles' sum, so
//   idot = D[xl] + 256 * D[xh] + 128 * D[1]          (exact in int32)
// Up to 8 rows of x (MB = 8) both planes share one A: row 2 m + p is plane p
// of activation row m; 9..16 rows (MB = 16) take an A per plane.  Either way
// a lane of D holds both planes of its activation rows.
// A lane's 16 bytes of B are two packed words: even nibbles, odd nibbles of
// each; the order of k inside a group is free as long as A matches.
//
// Vector-memory results return in issue order, so a wave that also loads the
// x operand (1 to 4 times the bytes of its weights, from the L2) holds few
// weights in flight and waits for them behind x.  The waves of a workgroup
// therefore have separate jobs:
//   * 8 compute waves load nothing but weights, into a register ring, and
//     take everything else from LDS;
//   * one copy wave moves the x operand and the group sums into LDS by
//     global->LDS copies ahead of their window, another the scales and biases;
//   * MB / 4 chain waves add the terms in group order, a window behind.
// A workgroup owns a tile of 16 weight rows (PAIR: 16 gate rows and the same
// 16 up rows, one x operand for both) and walks K in windows of 16 groups,
// two groups per compute wave; workgroups are persistent over tiles, so the
// ring never drains between them.  A compute wave writes its groups' fp32
// terms to an LDS table (two buffers), and after the window's one barrier a
// lane per (weight row, activation row) adds the window's terms in ascending
// group order.  All the matrices of a grouped call are one launch.
//
// Measured (Qwen2.5-7B shapes, graph replays, against the earlier form: x
// operand in the register ring, a launch per matrix and per 8 rows): MLP
// block 60 -> 47 us at 3..8 rows, 114 -> 62 at 16; q/k/v at 16 rows 58 ->
// 14.5; down_proj at 16 rows 48.5 -> 23.4.  What bounds it now is a window's
// instructions and LDS traffic: with the copies and the weights' loads taken
// out it still needs 0.5 us a window (0.75 paired) where the weights alone
// need 0.43 (0.86), and the two overlap only in part across the barrier.
// Measured and not kept: 12 compute waves (24 groups a window), two
// workgroups per CU, a deeper ring.
#pragma once

#include "q4_common.h"

namespace q4k {

constexpr int kMfRowsMax = 16;               // activation rows of one launch

// x of M <= MB rows, prepared for the small-M kernel.  Grid (P, MB):
// workgroup (p, m) takes row slot m (slots >= M write zeros) and the p-th
// slice of its groups.  The fp32 steps are xprep_kernel's:
//   xa      MB = 16: per group 2 KiB, plane p (low, high) at 1024 p: lane
//           (q, m) = 16 q + m, 16 bytes; MB = 8: 1 KiB, lane 16 q + 2 m + p.
//           Word j of the group is half j & 1 of quarter q = (j >> 2) |
//           (j & 2): its even-k bytes, then its odd-k bytes.
//   xsum_t[g * MB + m], xscale[m]
// Every workgroup of a row stages the whole row in LDS by 16-byte loads all
// issued at once (one memory round trip) and takes its amax; the group sums
// and the quantisation of its slice then read LDS.
constexpr int kMfPrepMaxK = 32768;           // floats of one x row staged in LDS
template <int MB>
__global__ __launch_bounds__(1024) void xprep_mf_kernel(const float* __restrict__ x, int M, int n_in,
                                                        uint2* __restrict__ xa, float* __restrict__ xsum_t,
                                                        float* __restrict__ xscale_out) {
    extern __shared__ float4 xrow4[];                            // [n_in / 4]
    const int m = blockIdx.y;
    const int tid = threadIdx.x, nt = blockDim.x;
    const int G = n_in >> 6;
    const int gs = (G + gridDim.x - 1) / gridDim.x;              // groups per slice
    const int g0 = blockIdx.x * gs, g1 = g0 + gs < G ? g0 + gs : G;
    // the 8 bytes (even k, odd k) of word j of the row in plane p
    auto at = [&](int j, int p) -> uint2& {
        const int g = j >> 3, q = ((j >> 2) & 1) | (j & 2), s = j & 1;
        const size_t lane = MB == 16 ? static_cast<size_t>(g * 2 + p) * 64 + q * 16 + m
                                     : static_cast<size_t>(g) * 64 + q * 16 + 2 * m + p;
        return xa[lane * 2 + s];
    };
    if (m >= M) {
        for (int j = g0 * 8 + tid; j < g1 * 8; j += nt) at(j, 0) = at(j, 1) = make_uint2(0u, 0u);
        for (int g = g0 + tid; g < g1; g += nt) xsum_t[static_cast<size_t>(g) * MB + m] = 0.0f;
        if (tid == 0 && blockIdx.x == 0) xscale_out[m] = 1.0f;
        return;
    }
    __shared__ float red[16];
    __shared__ float s_inv;
    const float4* xr4 = reinterpret_cast<const float4*>(x + static_cast<size_t>(m) * n_in);
    const int n4 = n_in >> 2;

    // stage the row; amax on the way (kernel/q4gemv.c:258-259, NaN-skipping)
    float amax = 0.0f;
    constexpr int kPer = kMfPrepMaxK / 4 / 1024;                // float4 per thread at most
    float4 v[kPer];
#pragma unroll
    for (int r = 0; r < kPer; r++) {
        const int i = r * nt + tid;
        v[r] = i < n4 ? xr4[i] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int r = 0; r < kPer; r++) {
        const int i = r * nt + tid;
        if (i < n4) {
            xrow4[i] = v[r];
            const float a[4] = {v[r].x, v[r].y, v[r].z, v[r].w};
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float t = a[k] < 0 ? -a[k] : a[k];
                amax = t > amax ? t : amax;
            }
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        float o = __shfl_xor(amax, off);
        amax = o > amax ? o : amax;
    }
    if ((tid & 63) == 0) red[tid >> 6] = amax;
    __syncthreads();
    if (tid == 0) {
        float a = 0.0f;
        for (int i = 0; i < (nt >> 6); i++) a = red[i] > a ? red[i] : a;
        const float sc = a > 0.0f ? __fdiv_rn(a, 32767.0f) : 1.0f;   // :260
        if (blockIdx.x == 0) xscale_out[m] = sc;
        s_inv = __fdiv_rn(1.0f, sc);                                  // :261
    }
    for (int g = g0 + tid; g < g1; g += nt) {                    // kernel/q4gemv.c:244-248
        const float4* p = xrow4 + g * 16;
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const float4 q = p[i];
            s = __fadd_rn(s, q.x);
            s = __fadd_rn(s, q.y);
            s = __fadd_rn(s, q.z);
            s = __fadd_rn(s, q.w);
        }
        xsum_t[static_cast<size_t>(g) * MB + m] = s;
    }
    __syncthreads();
    const float inv = s_inv;
    const float* xl = reinterpret_cast<const float*>(xrow4);
    for (int j = g0 * 8 + tid; j < g1 * 8; j += nt) {
        uint32_t le = 0, lo = 0, he = 0, ho = 0;
#pragma unroll
        for (int n = 0; n < 8; n++) {
            const float a = __fmul_rn(xl[8 * j + n], inv);             // :266
            const float r = a < 0 ? __fsub_rn(a, 0.5f) : __fadd_rn(a, 0.5f);  // :267-268
            const int32_t q = to_i16_like_x86(r);
            const uint32_t xlb = static_cast<uint32_t>(q) & 0xFFu;
            const uint32_t xhb = static_cast<uint32_t>(q >> 8) & 0xFFu;
            const int sh = 8 * (n >> 1);
            if (n & 1) { lo |= xlb << sh; ho |= xhb << sh; }
            else       { le |= xlb << sh; he |= xhb << sh; }
        }
        at(j, 0) = make_uint2(le ^ 0x80808080u, lo ^ 0x80808080u);
        at(j, 1) = make_uint2(he, ho);
    }
}

typedef int mf_v4i __attribute__((ext_vector_type(4)));

// The matrices of one launch, sharing x: matrix k's 16-row tiles are tiles
// tile0[k] .. tile0[k + 1] - 1.  PAIR: gate in 0 and up in 1, n[0] rows each,
// tiles tile0[0] .. tile0[1] - 1, out[0].
struct MfMats {
    const uint32_t* w[4];
    const uint16_t* s[4];
    const uint16_t* b[4];
    float* out[4];
    int n[4];
    int tile0[5];
};

// B of one group: two packed words, each its even then its odd nibbles.
__device__ __forceinline__ mf_v4i mf_nibbles(uint32_t a, uint32_t b) {
    return {static_cast<int>(a & 0x0F0F0F0Fu), static_cast<int>((a >> 4) & 0x0F0F0F0Fu),
            static_cast<int>(b & 0x0F0F0F0Fu), static_cast<int>((b >> 4) & 0x0F0F0F0Fu)};
}

// The waves of a workgroup meet once per window.  Each makes its own LDS
// accesses and copies complete before it (a compute or chain wave its LDS
// accesses, not the weights in flight; the copy wave the copies of the next
// window), which a fence would do by waiting for everything.
__device__ __forceinline__ void mf_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}
constexpr int kMfWaitLds = 0xC07F;                               // s_waitcnt lgkmcnt(0)
constexpr int mf_wait_copies(int n) {                            // s_waitcnt vmcnt(n), at most the counter's 63
    return n > 63 ? 0xCF7F : 0x0F70 | (n & 15) | ((n >> 4) << 14);
}

// Sizes of an instance.  EVEN: an even group count and 4-byte aligned scales
// and biases, copied two groups at a time; else one at a time, zero-extended.
// The ring's depth hardly matters to a long K (the copies and the compute of a
// window set the pace, not the weights), and every slot is a copy of the
// loop's code, which runs cold in a short call: 3 rows, prep included, with 4
// and 2 windows 9.2 and 8.3 us at 896 -> 200, 11.0 and 9.4 at 896 -> 4864, 19.0
// and 17.8 at 3584 -> 18944, 18.0 and 17.4 at 18944 -> 3584 (the form before the
// wave jobs: 8.0, 10.4, 20.1, 24.3).
constexpr int kMfWaves = 8;                                       // compute waves
template <bool PAIR, int MB, bool EVEN>
struct MfShape {
    static constexpr int NM = PAIR ? 2 : 1;
    static constexpr int win = 2 * kMfWaves;                      // groups per window
    static constexpr int chain = MB / 4;                          // chain waves: 16 MB lanes
    static constexpr int threads = 64 * (kMfWaves + chain + 2);
    static constexpr int depth = 2;                               // windows of weights in a wave's ring
    static constexpr int xslots = PAIR && MB == 16 ? 2 : 3;       // windows of x in LDS (160 KB)
    static constexpr int sbslots = PAIR && MB == 16 ? 6 : 8;      // and of scales and biases
    static constexpr int xbytes = win * MB * 128;                 // x operand of a window
    static constexpr int xcopies = xbytes / 1024 + 1;             // and its group sums (up to a KiB)
    static constexpr int sbcopies = (EVEN ? 4 : 8) * NM;
    static constexpr int sbbytes = sbcopies * 256;
    static constexpr int tbytes = NM * win * 16 * MB * 4;         // terms of a window
    static constexpr int xs0 = xslots * xbytes, sb0 = xs0 + xslots * 1024, t0 = sb0 + sbslots * sbbytes;
    static constexpr int lds = t0 + 2 * tbytes;
};

// The copy wave's copies (plain device functions: the copy builtin in a
// lambda of the kernel keeps the compiler from emitting the host stub).
template <int MB, int WIN>
__device__ __forceinline__ void mf_copy_x(char* x_s, char* xs_s, const __amdgpu_buffer_rsrc_t rx,
                                          const __amdgpu_buffer_rsrc_t rxs, int t, int lane) {
    typedef __attribute__((address_space(3))) void* lds_ptr;
    constexpr int XB = WIN * MB * 128;
    const uint32_t base = static_cast<uint32_t>(t) * XB + static_cast<uint32_t>(lane) * 16u;
#pragma unroll
    for (int i = 0; i < XB / 1024; i++)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_ptr)(x_s + i * 1024), 16, base + i * 1024u, 0, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        rxs, (lds_ptr)xs_s, 16, static_cast<uint32_t>(t) * (WIN * MB * 4) + static_cast<uint32_t>(lane) * 16u, 0, 0, 0);
}

// A window's scales (copies 0 .. n/2 - 1) and biases of one tile: EVEN, word
// (group pair p, row r) at 4 (16 p + r); else word (group g, row r).
// Groups past G and rows past the tile read 0 (or, within the tile, a value
// that no term uses).
template <bool EVEN, int WIN>
__device__ __forceinline__ void mf_copy_sb(char* s_s, const __amdgpu_buffer_rsrc_t rs, const __amdgpu_buffer_rsrc_t rb,
                                           int G, int t, int lane) {
    typedef __attribute__((address_space(3))) void* lds_ptr;
    constexpr int n = EVEN ? WIN / 8 : WIN / 4, size = EVEN ? 4 : 2;
    const uint32_t off = static_cast<uint32_t>(lane & 15) * G * 2u + static_cast<uint32_t>(t) * (WIN * 2u) +
                         static_cast<uint32_t>(lane >> 4) * size;
#pragma unroll
    for (int i = 0; i < n; i++) {
        if constexpr (EVEN) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)(s_s + i * 256), 4, off + i * 16u, 0, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr)(s_s + (n + i) * 256), 4, off + i * 16u, 0, 0, 0);
        } else {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr)(s_s + i * 256), 2, off + i * 8u, 0, 0, 0);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr)(s_s + (n + i) * 256), 2, off + i * 8u, 0, 0, 0);
        }
    }
}

// Matrix of a tile (wave-uniform): a chain of selects over the arguments.
__device__ __forceinline__ int mf_matrix(const MfMats& mt, int tile) {
    return (tile >= mt.tile0[1]) + (tile >= mt.tile0[2]) + (tile >= mt.tile0[3]);
}

// out[k][m][row] for m < M (PAIR: h[m][row] = SiLU(gate) * up).  Grid: up to
// one workgroup per tile, persistent; block: MfShape::threads.
template <bool PAIR, int MB, bool EVEN>
__global__ __launch_bounds__((MfShape<PAIR, MB, EVEN>::threads)) void gemv_mfma_kernel(
    MfMats mt, int tiles, int K, int M, const uint32_t* __restrict__ xa, const float* __restrict__ xsum_t,
    const float* __restrict__ xscale) {
    using S = MfShape<PAIR, MB, EVEN>;
    constexpr int NM = S::NM, WIN = S::win, W = kMfWaves, MPL = MB / 4;   // MPL: activation rows per lane of D
    extern __shared__ __attribute__((aligned(16))) char mf_lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = K >> 6, nwin = (G + WIN - 1) / WIN;
    const int mine = (tiles - static_cast<int>(blockIdx.x) + static_cast<int>(gridDim.x) - 1) / static_cast<int>(gridDim.x);
    const int iters = mine * nwin;                               // windows of this workgroup
    const int meets = (iters + S::depth - 1) / S::depth * S::depth;   // barriers before the last
    const uint32_t rowb = static_cast<uint32_t>(K) >> 1;         // bytes of a weight row
    // rows [row0, row0 + 16) of matrix k as a buffer of `stride` bytes a row
    // (past the last tile: empty)
    auto rows_of = [&](const void* p, int k, int row0, uint32_t stride, bool live) {
        int rows = mt.n[PAIR ? 0 : k] - row0;
        rows = !live || rows < 0 ? 0 : rows > 16 ? 16 : rows;
        return buf_rsrc(static_cast<const char*>(p) + static_cast<size_t>(row0) * stride,
                        static_cast<uint32_t>(rows) * stride);
    };

    if (wave < W) {
        // ---- compute waves: groups 2 wave, 2 wave + 1 of each window
        const int q = lane >> 4, col = lane & 15;
        // xscale of the lane's activation rows, by scalar loads: a vector load
        // would count among the ring's loads in every wait of the loop.  Bit
        // masks, not selects, which become one load at a per-lane index.
        float xsc[MPL];
#pragma unroll
        for (int i = 0; i < MPL; i++) {
            uint32_t v = 0;
#pragma unroll
            for (int k = 0; k < 4; k++) v |= __float_as_uint(xscale[MPL * k + i]) & (q == k ? ~0u : 0u);
            xsc[i] = __uint_as_float(v);
        }
        uint4 ring[S::depth][NM];
        int lt = 0, ltile = blockIdx.x;                          // window and tile of the next load
        __amdgpu_buffer_rsrc_t rw[NM];                           // its rows
        auto tile_rows = [&]() {
            const bool live = ltile < tiles;
            const int k = PAIR || !live ? 0 : mf_matrix(mt, ltile);
            const int row0 = live ? (ltile - mt.tile0[k]) * 16 : 0;
#pragma unroll
            for (int e = 0; e < NM; e++) rw[e] = rows_of(mt.w[PAIR ? e : k], k, row0, rowb, live);
        };
        const uint32_t lw = static_cast<uint32_t>(col) * rowb + static_cast<uint32_t>(q) * 16u;
        auto load = [&](uint4 (&r)[NM]) {
            if (lt == 0) tile_rows();
            const int g = lt * WIN + 2 * wave;
            const uint32_t off = lw + (g < G ? static_cast<uint32_t>(g) * 32u : kOutOfRange);
            __builtin_amdgcn_sched_barrier(0);
            // default cache policy: a row's 128-byte line is shared with the
            // next wave's groups
#pragma unroll
            for (int e = 0; e < NM; e++)
                r[e] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rw[e], off, 0, 0));
            __builtin_amdgcn_sched_barrier(0);
            if (++lt == nwin) {
                lt = 0;
                ltile += gridDim.x;
            }
        };
        const mf_v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101}, zero = {};
        // the LDS operands of a window: A per group and plane, the group sums
        // of the lane's activation rows, scales and biases (fp16 words)
        struct Ops {
            mf_v4i a[2][MB / 8];
            float xs[2][MPL];
            uint32_t s[NM][EVEN ? 1 : 2], b[NM][EVEN ? 1 : 2];
        };
        int xslot = 0, sslot = 0, tslot = 0;                     // of the next operands; of the next terms
        auto operands = [&](Ops& o) {
            const char* x_s = mf_lds + xslot * S::xbytes + wave * (2 * MB * 128) + lane * 16;
            const char* xs_s = mf_lds + S::xs0 + xslot * 1024 + (2 * wave * MB + MPL * q) * 4;
            const char* s_s = mf_lds + S::sb0 + sslot * S::sbbytes + ((EVEN ? 1 : 2) * wave * 16 + col) * 4;
#pragma unroll
            for (int g = 0; g < 2; g++) {
#pragma unroll
                for (int p = 0; p < MB / 8; p++)
                    o.a[g][p] = *reinterpret_cast<const mf_v4i*>(x_s + (g * (MB / 8) + p) * 1024);
#pragma unroll
                for (int i = 0; i < MPL; i++) o.xs[g][i] = reinterpret_cast<const float*>(xs_s + g * MB * 4)[i];
            }
#pragma unroll
            for (int e = 0; e < NM; e++)
#pragma unroll
                for (int g = 0; g < (EVEN ? 1 : 2); g++) {
                    o.s[e][g] = *reinterpret_cast<const uint32_t*>(s_s + e * (S::sbbytes / NM) + g * 64);
                    o.b[e][g] = *reinterpret_cast<const uint32_t*>(s_s + e * (S::sbbytes / NM) + S::sbbytes / (2 * NM) + g * 64);
                }
            xslot = xslot + 1 == S::xslots ? 0 : xslot + 1;
            sslot = sslot + 1 == S::sbslots ? 0 : sslot + 1;
        };
        auto window = [&](const Ops& o, const uint4 (&r)[NM]) {
            // lane (row, quarter q) holds words 4q .. 4q + 3 of the pair's 16:
            // swapping the upper half of one register with the lower half of
            // another leaves one group in each, its words in the order of
            // xprep_mf_kernel
            char* t_s = mf_lds + S::t0 + tslot * S::tbytes + (2 * wave * 16 + col) * (MB * 4) + q * (MPL * 4);
#pragma unroll
            for (int e = 0; e < NM; e++) {
                const auto p0 = __builtin_amdgcn_permlane32_swap(r[e].x, r[e].z, false, false);
                const auto p1 = __builtin_amdgcn_permlane32_swap(r[e].y, r[e].w, false, false);
                mf_v4i d0[2], dh[2], d1[2];
#pragma unroll
                for (int g = 0; g < 2; g++) {
                    const mf_v4i b = mf_nibbles(p0[g], p1[g]);
                    d1[g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, b, zero, 0, 0, 0);
                    d0[g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o.a[g][0], b, zero, 0, 0, 0);
                    if constexpr (MB == 16) dh[g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o.a[g][1], b, zero, 0, 0, 0);
                }
#pragma unroll
                for (int g = 0; g < 2; g++) {
                    const float sc = h2f(static_cast<uint16_t>(EVEN ? o.s[e][0] >> (16 * g) : o.s[e][g]));
                    const float bi = h2f(static_cast<uint16_t>(EVEN ? o.b[e][0] >> (16 * g) : o.b[e][g]));
                    float term[MPL];
#pragma unroll
                    for (int i = 0; i < MPL; i++) {
                        // kernel/q4gemv.c:173-180 with xq = 256 xh + (xl' + 128)
                        const int32_t lo = MB == 16 ? d0[g][i] : d0[g][2 * (i & 1)];
                        const int32_t hi = MB == 16 ? dh[g][i] : d0[g][2 * (i & 1) + 1];
                        const int32_t idot = lo + hi * 256 + d1[g][0] * 128;
                        const float dot = __fmul_rn(xsc[i], static_cast<float>(idot));
                        term[i] = __fmaf_rn(sc, dot, __fmul_rn(bi, o.xs[g][i]));
                    }
                    char* to = t_s + (e * WIN + g) * (16 * MB * 4);
                    if constexpr (MB == 16)
                        *reinterpret_cast<float4*>(to) = make_float4(term[0], term[1], term[2], term[3]);
                    else
                        *reinterpret_cast<float2*>(to) = make_float2(term[0], term[1]);
                }
            }
            tslot ^= 1;
        };
        // whole rings, the first one only filled: the loads go out (past the
        // last window: empty) on every path, so that the waits for the ring
        // never assume a skipped load.  A window's LDS operands are read
        // while the window before is computed.  (One site for each slot's
        // load: code that runs cold costs about 0.4 us per KB.)
        Ops ops[2];
        static_assert(S::depth % 2 == 0, "the operands alternate");
#pragma unroll 1
        for (int it = -S::depth; it < iters; it += S::depth)
#pragma unroll
            for (int d = 0; d < S::depth; d++) {
                if (it >= 0) {                                   // uniform
                    if (d == 0 && it == 0) {
                        mf_barrier();                            // window 0 is in LDS
                        operands(ops[0]);
                        __builtin_amdgcn_s_waitcnt(kMfWaitLds);
                    }
                    mf_barrier();                                // window it + d + 1 is in LDS
                    operands(ops[(d + 1) & 1]);
                    __builtin_amdgcn_sched_barrier(0);
                    if (it + d < iters) window(ops[d & 1], ring[d]);
                }
                load(ring[d]);
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_waitcnt(kMfWaitLds);          // the terms are in LDS
            }
        mf_barrier();
        return;
    }

    if (wave < W + S::chain) {
        // ---- chain waves: lane (weight row col, activation row m)
        const int t = (wave - W) * 64 + lane, col = t / MB, m = t % MB;
        float acc[NM];
#pragma unroll
        for (int e = 0; e < NM; e++) acc[e] = 0.0f;
        int win = 0, tile = blockIdx.x;
        mf_barrier();
        mf_barrier();
        for (int it = 0; it < iters; it++) {
            mf_barrier();                                        // window it's terms are in the table
            const float* tp = reinterpret_cast<const float*>(mf_lds + S::t0 + (it & 1) * S::tbytes) + t;
            const int n = G - win * WIN < WIN ? G - win * WIN : WIN;
            float v[NM][WIN];
#pragma unroll
            for (int e = 0; e < NM; e++)
#pragma unroll
                for (int g = 0; g < WIN; g++) v[e][g] = tp[(e * WIN + g) * (16 * MB)];
            __builtin_amdgcn_s_waitcnt(kMfWaitLds);              // read before the next barrier
            if (n == WIN) {
#pragma unroll
                for (int g = 0; g < WIN; g++)
#pragma unroll
                    for (int e = 0; e < NM; e++) acc[e] = __fadd_rn(acc[e], v[e][g]);
            } else {
#pragma unroll
                for (int g = 0; g < WIN; g++)
#pragma unroll
                    for (int e = 0; e < NM; e++)
                        if (g < n) acc[e] = __fadd_rn(acc[e], v[e][g]);
            }
            if (++win == nwin) {
                const int k = PAIR ? 0 : mf_matrix(mt, tile);
                const int row = (tile - mt.tile0[k]) * 16 + col, N = mt.n[k];
                if (row < N && m < M) {
                    float* o = mt.out[k] + static_cast<size_t>(m) * N + row;
                    if constexpr (PAIR) *o = silu_mul(acc[0], acc[1]);
                    else *o = acc[0];
                }
                win = 0;
                tile += gridDim.x;
#pragma unroll
                for (int e = 0; e < NM; e++) acc[e] = 0.0f;
            }
        }
#pragma unroll 1
        for (int it = iters; it < meets; it++) mf_barrier();
        return;
    }

    if (wave == W + S::chain) {
        // ---- the x copy wave: a window's operand and group sums, up to
        // xslots - 1 windows ahead of its use
        const __amdgpu_buffer_rsrc_t rx = buf_rsrc(xa, static_cast<uint32_t>(G) * (MB * 128u));
        const __amdgpu_buffer_rsrc_t rxs = buf_rsrc(xsum_t, static_cast<uint32_t>(G) * (MB * 4u));
        int win = 0, slot = 0;                                   // of the next copy
        auto copy = [&]() {
            mf_copy_x<MB, WIN>(mf_lds + slot * S::xbytes, mf_lds + S::xs0 + slot * 1024, rx, rxs, win, lane);
            slot = slot + 1 == S::xslots ? 0 : slot + 1;
            win = win + 1 == nwin ? 0 : win + 1;
        };
#pragma unroll 1
        for (int it = -S::xslots; it < iters; it++) {
            if (it >= 0) {
                if (it == 0) {
                    __builtin_amdgcn_s_waitcnt(mf_wait_copies((S::xslots - 1) * S::xcopies));
                    mf_barrier();                                // window 0
                }
                __builtin_amdgcn_s_waitcnt(mf_wait_copies((S::xslots - 2) * S::xcopies));
                mf_barrier();                                    // window it + 1
            }
            copy();                                              // window it + xslots
        }
        __builtin_amdgcn_s_waitcnt(mf_wait_copies(0));           // none may land after the workgroup ends
#pragma unroll 1
        for (int it = iters; it <= meets; it++) mf_barrier();
        return;
    }

    // ---- the scale copy wave: a window's scales and biases, up to sbslots - 1
    // windows ahead (they come from HBM: in the x wave's queue they would hold back
    // the x copies, which the L2 holds)
    int win = 0, tile = blockIdx.x, slot = 0;                    // of the next copy
    __amdgpu_buffer_rsrc_t rs[NM], rb[NM];
    auto tile_rows = [&]() {
        const bool live = tile < tiles;
        const int k = PAIR || !live ? 0 : mf_matrix(mt, tile);
        const int row0 = live ? (tile - mt.tile0[k]) * 16 : 0;
#pragma unroll
        for (int e = 0; e < NM; e++) {
            rs[e] = rows_of(mt.s[PAIR ? e : k], k, row0, static_cast<uint32_t>(G) * 2u, live);
            rb[e] = rows_of(mt.b[PAIR ? e : k], k, row0, static_cast<uint32_t>(G) * 2u, live);
        }
    };
    auto copy = [&]() {
        if (win == 0) tile_rows();
#pragma unroll
        for (int e = 0; e < NM; e++)
            mf_copy_sb<EVEN, WIN>(mf_lds + S::sb0 + slot * S::sbbytes + e * (S::sbbytes / NM), rs[e], rb[e], G, win, lane);
        slot = slot + 1 == S::sbslots ? 0 : slot + 1;
        if (++win == nwin) {
            win = 0;
            tile += gridDim.x;
        }
    };
#pragma unroll 1
    for (int it = -S::sbslots; it < iters; it++) {
        if (it >= 0) {
            if (it == 0) {
                __builtin_amdgcn_s_waitcnt(mf_wait_copies((S::sbslots - 1) * S::sbcopies));
                mf_barrier();                                    // window 0
            }
            __builtin_amdgcn_s_waitcnt(mf_wait_copies((S::sbslots - 2) * S::sbcopies));
            mf_barrier();                                        // window it + 1
        }
        copy();                                                  // window it + sbslots
    }
    __builtin_amdgcn_s_waitcnt(mf_wait_copies(0));
#pragma unroll 1
    for (int it = iters; it <= meets; it++) mf_barrier();
}

}  // namespace q4k
