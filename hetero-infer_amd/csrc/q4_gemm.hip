// Prefill GEMM on the matrix cores with the 4-bit weights kept 4-bit up to
// the MFMA: out[M][N] = bf16(x)[M][K] . bf16(dequant W)[N][K]^T, fp32
// accumulation on v_mfma_f32_32x32x16_bf16.
//
// Workgroup tile BM x 256 (BM 256, 192, 128 or 64), NW waves side by side, each
// BM x 256/NW -- TM x TN MFMA tiles of 32 x 32.  One K step is 64 = one
// quantisation group, so each weight row has one scale/bias pair per step.
// Every operand reaches LDS by global->LDS copies (buffer_load ... lds, 16,
// 4 or 2 bytes a lane):
//   * A: the bf16 copy of x, BM rows x 128 bytes, a ring of three K steps;
//     16-byte chunk c of row r at r * 128 + (c ^ (r / 2 & 7)) * 16 (the XOR
//     spreads a fragment read by 32 rows over the 64 banks, which hold two
//     rows);
//   * B: the packed weights as they are in memory, 256 rows x 64 bytes: two
//     K steps at a time, two slots; chunk c of row r at c ^ (r / 4 & 3);
//   * the 256 rows' scales and biases, SG groups at a time, two slots: SG = 8
//     (16 bytes a row) where the group count and the pointers allow it, 2 (4
//     bytes), else 1 (2 bytes, zero-extended).
// What bounds the copies is their number of requests, not their bytes: with
// 32 bytes of weights and 2-byte scales and biases per row and step, those
// 2 x 256 + 256 requests of a step (A has 256, of 128 bytes) kept the L2 busy
// and the non-temporal policy fetched a row's 128-byte line once per step.
// Measured at 512 rows (graph replays, before -> after these copies, the bank
// swizzle, byte selects in the dequant and the next step's operands read under
// the last slice, in 4 waves of 64 columns): gate/up + down of a prompt chunk
// 308 -> 270 us, down 111 -> 94, o 45 -> 37, 1000 rows 546 -> 446; one 256-row
// tile per CU over K = 18944 took 2.02 us a step (MFMAs and barriers alone 1.52:
// the clock drops as the CUs fill).  8 waves of 32
// columns (the present form): a lone tile's step 1.50 -> 1.31 us at 256 rows,
// 1.25 -> 1.09 at 192; with a tile on every CU 2.0 to 2.2 (988 TFLOP/s at 2.17).
// B is dequantised in registers right before the MFMA that consumes it:
// one packed word (word ks + 4 (lane/32) of the row: a lane's four words of
// a step are one 16-byte read) is exactly one lane's 8-value B fragment of K
// slice ks, and its value is bf16(fma(q, scale, bias)) -- what
// q4_dequant_bf16_dev writes.  Staging B 4-bit keeps its LDS
// traffic a quarter of bf16's, and a dequantised word feeds TM MFMAs.
// Pipeline: step k + 2's copies are issued while step k is multiplied; at
// the top of step k each wave waits for its own copies of step k + 1, made
// a step before, and one barrier publishes everyone's, so that step k can
// read and dequantise the first operands of step k + 1 under its last MFMAs.
// Every copy goes through a buffer resource bounded to the tile's rows:
// rows past M or N and steps past the workgroup's K range read 0 and cost
// no access.  Split-K: blockIdx.z takes steps [z kt_split, (z+1) kt_split)
// and writes its partial sums to out + z M ldo.
// Paired tiles (gate/up of the MLP): the tile's 256 weight rows are rows
// [n0, n0 + 128) of the gate matrix, then the same rows of the up matrix,
// and wave w's 32 columns are gate rows n0 + 16 w .. + 16 and the same up
// rows: the epilogue brings a column's two sums into one lane and stores
// bf16(SiLU(gate) * up), the down projection's bf16 operand.
#include "q4_common.h"

namespace q4k {

typedef __bf16 gemm_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gemm_f32x16 __attribute__((ext_vector_type(16)));

// LDS: three steps of A (BM rows x 128 bytes), two slots of B (256 rows x 64
// bytes), two slots of scales, then biases (256 rows of SG values, at least a
// word, each).
__host__ __device__ constexpr int w4_row_bytes(int sg) { return sg == 8 ? 16 : 4; }
__host__ __device__ constexpr int w4_b0(int bm) { return 3 * bm * 128; }
__host__ __device__ constexpr int w4_s0(int bm) { return w4_b0(bm) + 2 * 16384; }
__host__ __device__ constexpr int w4_lds_bytes(int bm, int sg) { return w4_s0(bm) + 2 * 512 * w4_row_bytes(sg); }

__device__ __forceinline__ uint32_t w4_pack_bf16(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));
    const f32x2 p = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(p, bf16x2v));
}

// The nibbles of a packed word as bytes: even elements in lo, odd in hi.
// (Opaque to the compiler, which would fold the masks into a bit-field
// extract per value instead of the byte selects of v_cvt_f32_ubyte0..3.)
__device__ __forceinline__ void w4_bytes(uint32_t w, uint32_t& lo, uint32_t& hi) {
    lo = w & 0x0F0F0F0Fu;
    hi = (w >> 4) & 0x0F0F0F0Fu;
    asm("" : "+v"(lo), "+v"(hi));
}

// Elements 2q and 2q + 1 of a word's bytes, each bf16(fma(q_e, s, b)).
__device__ __forceinline__ uint32_t w4_dequant2(uint32_t lo, uint32_t hi, int q, float s, float b) {
    return w4_pack_bf16(__builtin_fmaf(static_cast<float>((lo >> (8 * q)) & 0xFFu), s, b),
                        __builtin_fmaf(static_cast<float>((hi >> (8 * q)) & 0xFFu), s, b));
}

// What a wave copies of one tile (M block m0, N block n0): rows of x, of W and
// of the scales or the biases, and their bytes (the bounds of the copies'
// resources).  Paired tiles: waves 0..3 copy the gate rows of W, 4..7 the up
// rows.
struct W4Tile {
    const uint16_t* x;
    const uint32_t* w;
    const uint16_t* g;
    uint32_t xbytes, wbytes, gbytes;
    int m0, n0;
};

// Copy i of the up to w4_copies that a wave makes for K step k of its range,
// `first` its first step (a plain device function: the copy builtin in a
// lambda of the kernel keeps the compiler from emitting the kernel's host
// stub).  NW waves share the copies: A in 1 KiB copies of 8 rows, B in 16
// copies of 16 rows (on even steps, for two), 64 scales (waves 0..3) or biases
// (4..7) each (every SG steps).  The step's offset is the scalar
// one.
template <int BM, int NW>
constexpr int w4_copies() { return BM / (8 * NW) + 16 / NW + 1; }

template <int BM, int NW, int SG, bool PAIR>
__device__ __forceinline__ void w4_issue(int i, char* lds, const W4Tile& t, const uint32_t* a_src, const uint32_t* b_src,
                                         uint32_t g_src, int k, int slot, bool first, int wave) {
    typedef __attribute__((address_space(3))) void* lds_ptr;
    constexpr int A_DMA = BM / (8 * NW), B_DMA = 16 / NW;
    if (i < A_DMA) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds(buf_rsrc(t.x, t.xbytes),
                                                 (lds_ptr)(lds + slot * (BM * 128) + (wave * A_DMA + i) * 1024), 16,
                                                 a_src[i], k * 128, 0, 0);
    } else if (i < A_DMA + B_DMA) {
        const int q = i - A_DMA;
        if (first || (k & 1) == 0)
            // default cache policy: a row's 128-byte line holds four steps
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                buf_rsrc(t.w, t.wbytes),
                (lds_ptr)(lds + w4_b0(BM) + (k >> 1 & 1) * 16384 + (B_DMA * wave + q) * 1024), 16, b_src[q],
                (k >> 1) * 64, 0, 0);
    } else if (first || k % SG == 0) {
        const __amdgpu_buffer_rsrc_t r = buf_rsrc(t.g, t.gbytes);
        constexpr int RB = w4_row_bytes(SG);
        const lds_ptr to = (lds_ptr)(lds + w4_s0(BM) + ((k / SG & 1) * 512 + wave * 64) * RB);
        if constexpr (SG == 8) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 16, g_src, k / 8 * 16, 0, 0);
        else if constexpr (SG == 2) __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 4, g_src, k / 2 * 4, 0, 0);
        else __builtin_amdgcn_raw_ptr_buffer_load_lds(r, to, 2, g_src, k * 2, 0, 0);
    }
}

template <int BM>
__device__ __forceinline__ W4Tile w4_tile(const uint16_t* xb, const uint32_t* w, const uint16_t* sc, const uint16_t* bi,
                                          int M, int N, int K, int mt, int nt, int wave) {
    constexpr int BN = 256;
    W4Tile t;
    t.m0 = mt * BM;
    t.n0 = nt * BN;
    const int G = K >> 6, wpr = K >> 3;
    const int mrows = M - t.m0 < BM ? M - t.m0 : BM, nrows = N - t.n0 < BN ? N - t.n0 : BN;
    t.x = xb + static_cast<size_t>(t.m0) * K;
    t.w = w + static_cast<size_t>(t.n0) * wpr;
    t.g = (wave < 4 ? sc : bi) + static_cast<size_t>(t.n0) * G;
    t.xbytes = static_cast<uint32_t>(mrows * K) * 2u;
    t.wbytes = static_cast<uint32_t>(nrows * wpr) * 4u;
    t.gbytes = static_cast<uint32_t>(nrows * G) * 2u;
    return t;
}

// A paired tile: output columns [nt 128, nt 128 + 128) of N, weight rows of
// matrix 0 (gate) and matrix 1 (up) of gm.
template <int BM>
__device__ __forceinline__ W4Tile w4_tile_pair(const uint16_t* xb, const GemmMats& gm, int M, int N, int K, int mt,
                                               int nt, int wave) {
    W4Tile t;
    t.m0 = mt * BM;
    t.n0 = nt * 128;
    const int G = K >> 6, wpr = K >> 3;
    const int mrows = M - t.m0 < BM ? M - t.m0 : BM, nrows = N - t.n0 < 128 ? N - t.n0 : 128;
    const int up = wave & 2 ? 1 : 0;                               // rows 64 (wave & 3) .. of the 256 scales or biases
    t.x = xb + static_cast<size_t>(t.m0) * K;
    t.w = (wave < 4 ? gm.w[0] : gm.w[1]) + static_cast<size_t>(t.n0) * wpr;
    t.g = (wave < 4 ? (up ? gm.s[1] : gm.s[0]) : (up ? gm.b[1] : gm.b[0])) + static_cast<size_t>(t.n0) * G;
    t.xbytes = static_cast<uint32_t>(mrows * K) * 2u;
    t.wbytes = static_cast<uint32_t>(nrows * wpr) * 4u;
    t.gbytes = static_cast<uint32_t>(nrows * G) * 2u;
    return t;
}

// Per-lane source offsets of a step's copies.  A: copy i of wave w moves rows
// 8 (w A_DMA + i) .. + 8, lane -> (row, 16-byte position p), reading chunk
// p ^ (row / 2 & 7) of the row.  B: copy q moves rows 16 (B_DMA w + q) .. +
// 16, four lanes per row, reading chunk p ^ (row / 4 & 3).  Scales / biases:
// one row per lane.
template <int BM, int NW>
struct W4Src {
    uint32_t a[BM / (8 * NW)];
    uint32_t b[16 / NW];
    uint32_t g;
};

template <int BM, int NW, bool PAIR>
__device__ __forceinline__ void w4_src(W4Src<BM, NW>& src, int K, int wave, int lane) {
    constexpr int A_DMA = BM / (8 * NW), B_DMA = 16 / NW;
    const int G = K >> 6, wpr = K >> 3;
#pragma unroll
    for (int i = 0; i < A_DMA; i++) {
        const int r = (wave * A_DMA + i) * 8 + (lane >> 3), c = lane & 7;
        src.a[i] = static_cast<uint32_t>(r * K + (c ^ (r >> 1 & 7)) * 8) * 2u;
    }
#pragma unroll
    for (int q = 0; q < B_DMA; q++) {
        const int r = (B_DMA * wave + q) * 16 + (lane >> 2);             // stage row
        src.b[q] = static_cast<uint32_t>((r & (PAIR ? 127 : 255)) * wpr) * 4u + ((lane & 3) ^ (r >> 2 & 3)) * 16u;
    }
    src.g = static_cast<uint32_t>(((PAIR ? wave & 1 : wave & 3) * 64 + lane) * G) * 2u;
}

// How NW waves split a BM x 256 tile: side by side, each the tile's BM rows
// x 256 / NW columns, TM x TN MFMA tiles of 32 x 32, so that every weight
// word is dequantised once and feeds TM MFMAs (128 rows took 1.10 us a step in
// 2 x 4 waves of 64 x 64, 0.88 side by side).  Two waves per SIMD, so that one
// dequantises while the other multiplies.
template <int BM, int NW>
struct W4Layout {
    static constexpr int RW = BM, WC = 256 / NW;
    static constexpr int TM = RW / 32, TN = WC / 32;
};

template <int BM, int NW>
using W4Acc = gemm_f32x16[W4Layout<BM, NW>::TM][W4Layout<BM, NW>::TN];

// The stage row (of 256) of a lane's column in block j of its wave: WC
// consecutive rows per wave; paired tiles (WC 32): lanes 0..15 gate rows 16
// wave .., lanes 16..31 the same up rows, 128 further.
template <bool PAIR, int WC>
__device__ __forceinline__ int w4_brow(int wave, int j, int lane) {
    static_assert(!PAIR || WC == 32, "paired tiles: 16 gate and 16 up rows a wave");
    return PAIR ? (lane & 16) * 8 + wave * 16 + (lane & 15) : wave * WC + j * 32 + (lane & 31);
}

// K steps [k0, k0 + nk) of one tile into acc (which it adds to): the copy
// pipeline starts and drains inside, and on return every wave is past its
// last LDS read and no copy is in flight, so the next segment may reuse the
// LDS.
template <int BM, int NW, int SG, bool PAIR = false>
__device__ __forceinline__ void w4_segment(W4Acc<BM, NW>& acc, char* lds, const W4Tile& t, const W4Src<BM, NW>& src,
                                           int k0, int nk, int wave, int lane) {
    using L = W4Layout<BM, NW>;
    constexpr int WC = L::WC, TM = L::TM, TN = L::TN;
    constexpr int COPIES = w4_copies<BM, NW>(), A_DMA = BM / (8 * NW);
    constexpr int NM = TM * TN, NPC = TN * 4;                      // MFMAs, dequant pieces per slice
    const int hb = lane >> 5;
    auto issue = [&](int i, int it) {
        w4_issue<BM, NW, SG, PAIR>(i, lds, t, src.a, src.b, src.g, k0 + it, it % 3, it == 0, wave);
    };
    // the operands of slice ks of step it: lane half hb takes 16-byte chunk
    // (8 values of x) and packed word 4 hb + ks of the 64
    auto a_frag = [&](int it, int ks, int i) {
        const int row = i * 32 + (lane & 31);
        const int c = (4 * hb + ks) ^ (row >> 1 & 7);
        return *reinterpret_cast<const gemm_bf16x8*>(lds + it % 3 * (BM * 128) + row * 128 + c * 16);
    };
    uint32_t bw[TN][4];                                            // the step's packed words of the lane
    float sf[TN], bf[TN];                                          // its scale and bias
    auto b_step = [&](int it) {
        const int k = k0 + it;
        const char* bs = lds + w4_b0(BM) + (k >> 1 & 1) * 16384;
        constexpr int RB = w4_row_bytes(SG);
        const char* ss = lds + w4_s0(BM) + (k / SG & 1) * (512 * RB) + k % SG * 2;
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int row = w4_brow<PAIR, WC>(wave, j, lane);
            const uint4 w = *reinterpret_cast<const uint4*>(bs + row * 64 + (((k & 1) * 2 + hb) ^ (row >> 2 & 3)) * 16);
            bw[j][0] = w.x; bw[j][1] = w.y; bw[j][2] = w.z; bw[j][3] = w.w;
            sf[j] = h2f(*reinterpret_cast<const uint16_t*>(ss + row * RB));
            bf[j] = h2f(*reinterpret_cast<const uint16_t*>(ss + 256 * RB + row * RB));
        }
    };
    gemm_bf16x8 av[2][TM], bv[2][TN];
#pragma unroll
    for (int i = 0; i < COPIES; i++) issue(i, 0);
    if (nk > 1) {
#pragma unroll
        for (int i = 0; i < COPIES; i++) issue(i, 1);
        // step 1 made at least A_DMA copies
        __builtin_amdgcn_s_waitcnt(0x0F70 | A_DMA);
    } else
        __builtin_amdgcn_s_waitcnt(0x0F70);
    __builtin_amdgcn_s_barrier();                                  // step 0 is in LDS
    b_step(0);
#pragma unroll
    for (int i = 0; i < TM; i++) av[0][i] = a_frag(0, 0, i);
#pragma unroll
    for (int j = 0; j < TN; j++) {
        uint32_t lo, hi, pk[4];
        w4_bytes(bw[j][0], lo, hi);
#pragma unroll
        for (int q = 0; q < 4; q++) pk[q] = w4_dequant2(lo, hi, q, sf[j], bf[j]);
        bv[0][j] = __builtin_bit_cast(gemm_bf16x8, make_uint4(pk[0], pk[1], pk[2], pk[3]));
    }
    for (int it = 0; it < nk; it++) {
        // step it + 1's copies, a step old, are done
        __builtin_amdgcn_s_waitcnt(0x0F70);
        // a bare barrier: every wave's copies of step it + 1 are in LDS and
        // every wave is past step it - 1, whose slots step it + 2 refills (a
        // fence would also wait for the LDS reads in flight)
        __builtin_amdgcn_s_barrier();
        const bool more = it + 2 < nk;
        // four K slices of 16; the next slice's operands (after the last, the
        // next step's first) are read while this one multiplies, and its
        // dequant is spread over the last of this slice's MFMAs (fences pin
        // the order), so the VALU work runs under the matrix core instead of
        // before it; the copies of step it + 2 go out between the first
        // slice's MFMAs.  (Past the last step the reads find old values,
        // which nothing uses.)
#pragma unroll
        for (int ks = 0; ks < 4; ks++) {
            const int cu = ks & 1, nx = cu ^ 1, kn = (ks + 1) & 3;
            if (ks == 3) b_step(it + 1);
#pragma unroll
            for (int i = 0; i < TM; i++) av[nx][i] = a_frag(ks < 3 ? it : it + 1, kn, i);
            __builtin_amdgcn_sched_barrier(0);
            uint32_t blo[TN], bhi[TN], pk[TN][4];
#pragma unroll
            for (int m = 0; m < NM; m++) {
                const int i = m / TN, j = m % TN;
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[cu][i], bv[cu][j], acc[i][j], 0, 0, 0);
                if (ks == 0 && more) {
#pragma unroll
                    for (int c = m * COPIES / NM; c < (m + 1) * COPIES / NM; c++) issue(c, it + 2);
                }
                constexpr int M0 = NPC < NM ? NM - NPC : 0, NR = NM - M0;   // pieces in the last NR MFMAs
#pragma unroll
                for (int pc = m < M0 ? 0 : (m - M0) * NPC / NR; pc < (m < M0 ? 0 : (m - M0 + 1) * NPC / NR); pc++) {
                    const int jj = pc / 4, q = pc % 4;
                    if (q == 0) w4_bytes(bw[jj][kn], blo[jj], bhi[jj]);
                    pk[jj][q] = w4_dequant2(blo[jj], bhi[jj], q, sf[jj], bf[jj]);
                    if (q == 3)
                        bv[nx][jj] = __builtin_bit_cast(gemm_bf16x8,
                                                        make_uint4(pk[jj][0], pk[jj][1], pk[jj][2], pk[jj][3]));
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    }
    __syncthreads();                                               // every wave's last LDS reads are done
}

// C tile: lane l, register v holds row 8 (v / 4) + 4 (l / 32) + v % 4,
// column l % 32.  o: a [M][ldo] block whose column 0 is column c0 of the
// product.
template <int BM, int NW>
__device__ __forceinline__ void w4_store(const W4Acc<BM, NW>& acc, float* o, const W4Tile& t, int M, int N, int ldo,
                                         int c0, int wave, int lane) {
    using L = W4Layout<BM, NW>;
    constexpr int WC = L::WC, TM = L::TM, TN = L::TN;
    const int hb = lane >> 5;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int row = t.m0 + i * 32 + 8 * (v >> 2) + 4 * hb + (v & 3);
                const int col = t.n0 + wave * WC + j * 32 + (lane & 31);
                if (row < M && col < N) o[static_cast<size_t>(row) * ldo + (col - c0)] = acc[i][j][v];
            }
}

// Part h of NP of w4_store's tiles (i TN + j in [h TM TN / NP, (h + 1) TM TN
// / NP)), into a [M][N] output; NaN in place of every value if `poison`.
template <int BM, int NW, int NP>
__device__ __forceinline__ void w4_store_rows(const W4Acc<BM, NW>& acc, float* o, const W4Tile& t, int M, int N, int h,
                                              bool poison, int wave, int lane) {
    using L = W4Layout<BM, NW>;
    constexpr int WC = L::WC, TM = L::TM, TN = L::TN;
    const int hb = lane >> 5;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++) {
            if ((i * TN + j) / (TM * TN / NP) != h) continue;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int row = t.m0 + i * 32 + 8 * (v >> 2) + 4 * hb + (v & 3);
                const int col = t.n0 + wave * WC + j * 32 + (lane & 31);
                if (row < M && col < N)
                    o[static_cast<size_t>(row) * N + col] = poison ? __builtin_nanf("") : acc[i][j][v];
            }
        }
}

template <int BM, int NW>
__device__ __forceinline__ void w4_zero(W4Acc<BM, NW>& acc) {
    constexpr int TM = W4Layout<BM, NW>::TM, TN = W4Layout<BM, NW>::TN;
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
}

// The matrix of launch block nt (uniform).
__device__ __forceinline__ int gm_mat(const GemmMats& gm, int nt) {
    int k = 0;
#pragma unroll
    for (int i = 1; i < 4; i++) k += (i < gm.count && nt >= gm.nb0[i]) ? 1 : 0;
    return __builtin_amdgcn_readfirstlane(k);
}

// Data-parallel: workgroup (mt, nt, z) computes K steps [z kt_split,
// (z+1) kt_split) of tile (mt, nt): into its matrix's output, or (part)
// into part + z M ldp at the matrix's columns.
template <int BM, int NW, int SG>
__global__ __launch_bounds__(64 * NW) void gemm_w4_kernel(const uint16_t* __restrict__ xb, GemmMats gm,
                                                          float* __restrict__ part, int M, int K, int kt_split,
                                                          int ldp) {
    extern __shared__ uint4 w4_lds[];
    char* lds = reinterpret_cast<char*>(w4_lds);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int G = K >> 6;
    const int kt0 = blockIdx.z * kt_split;
    const int nk = G - kt0 < kt_split ? G - kt0 : kt_split;
    const int k = gm_mat(gm, blockIdx.y);
    const int N = gm.n_out[k];
    const W4Tile t = w4_tile<BM>(xb, gm.w[k], gm.s[k], gm.b[k], M, N, K, blockIdx.x, blockIdx.y - gm.nb0[k],
                                  wave);
    W4Src<BM, NW> src;
    w4_src<BM, NW, false>(src, K, wave, lane);
    W4Acc<BM, NW> acc;
    w4_zero<BM, NW>(acc);
    w4_segment<BM, NW, SG>(acc, lds, t, src, kt0, nk, wave, lane);
    if (part)
        w4_store<BM, NW>(acc, part + static_cast<size_t>(blockIdx.z) * M * ldp + gm.col0[k], t, M, N, ldp, 0, wave,
                         lane);
    else
        w4_store<BM, NW>(acc, gm.out[k], t, M, N, N, 0, wave, lane);
}

// Row block i of a paired tile's outputs, h = bf16(SiLU(gate) * up), NaN if
// `poison`.  Lanes 0..15 of a half hold gate and lanes 16..31 up of the same
// 16 columns, row r in register v and r + 1 in v + 1; the swap of odd and even
// 16-lane rows leaves gate in one register and up in the other, of row r in
// lanes 0..15 and r + 1 in lanes 16..31.
__device__ __forceinline__ void w4_store_pair(const gemm_f32x16 a, uint16_t* h, const W4Tile& t, int M, int N, int i,
                                              bool poison, int wave, int lane) {
    const int col = t.n0 + wave * 16 + (lane & 15);
#pragma unroll
    for (int v = 0; v < 16; v += 2) {
        const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a[v]), __float_as_uint(a[v + 1]), false, false);
        const float o = silu_mul(__uint_as_float(s[0]), __uint_as_float(s[1]));
        const int row = t.m0 + i * 32 + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3) + (lane >> 4 & 1);
        if (row < M && col < N)
            h[static_cast<size_t>(row) * N + col] =
                poison ? static_cast<uint16_t>(0x7FC0u) : static_cast<uint16_t>(w4_pack_bf16(o, o) & 0xFFFFu);
    }
}

// Paired gate/up tiles (blockIdx.y = block of 128 output columns), every K
// step: h[r][c] = bf16(SiLU(x W_gate^T) * (x W_up^T)), rounded to nearest
// even -- the fp32 products of two gemm_w4_kernel calls through silu_mul,
// then the bf16 rounding the down projection applies to its x.
template <int BM, int NW, int SG>
__global__ __launch_bounds__(64 * NW) void gemm_w4_pair_kernel(const uint16_t* __restrict__ xb, GemmMats gm,
                                                               uint16_t* __restrict__ h, int M, int K) {
    using L = W4Layout<BM, NW>;
    constexpr int TM = L::TM;
    extern __shared__ uint4 w4_lds[];
    char* lds = reinterpret_cast<char*>(w4_lds);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int N = gm.n_out[0];
    const W4Tile t = w4_tile_pair<BM>(xb, gm, M, N, K, blockIdx.x, blockIdx.y, wave);
    W4Src<BM, NW> src;
    w4_src<BM, NW, true>(src, K, wave, lane);
    W4Acc<BM, NW> acc;
    w4_zero<BM, NW>(acc);
    w4_segment<BM, NW, SG, true>(acc, lds, t, src, 0, K >> 6, wave, lane);
#pragma unroll
    for (int i = 0; i < TM; i++) w4_store_pair(acc[i][0], h, t, M, N, i, false, wave, lane);
}

// Stream-K: the tiles (m block major) are split into nx contiguous groups,
// one per XCD, and each group's T = tiles x G (tile, K step) iterations,
// tile-major and K-minor, into P equal contiguous ranges, one per workgroup
// of that XCD.  A range splits at tile boundaries into segments: a tile's
// tail, whole tiles, the next tile's head; the workgroup runs them last to
// first.  A segment that does not reach its tile's end (only a range's last
// one can be such) is a partial: it goes to the workgroup's slot in `part`
// at device scope, then its flag is set to the launch's epoch.  The segment
// that ends a tile (its owner's) adds the partials of the workgroups before
// it in its group that cover the rest of the tile, nearest first, and
// stores the tile.  Waits point only to lower-numbered workgroups, which
// are dispatched first, and a partial is a workgroup's first segment, so an
// owner, which reaches its first segment last, rarely waits.  With at
// least as many workgroups as tiles a range is at most G iterations long
// (two segments); with fewer, each tile has at most one partial.
// Paired gate/up tiles (PAIR) take the same route, the owner's store being
// the SiLU * up epilogue of gemm_w4_pair_kernel.
//
// The epoch makes a flag mean "this launch's partial is in": every
// workgroup reads it from ctl[0] when it starts, and the last workgroup to
// leave advances it.  A flag is never lowered, so a partial that arrives
// after its owner gave up waiting (an error, its tile stored as NaN) holds
// an old epoch that no later launch waits for.  Stream-ordered launches on
// one workspace, captured ones included, each see their own epoch.
//
// A slot holds 256 x 256 floats as [block b][quad q][thread] of 16 bytes,
// block b = i TN + j of the accumulators, quad q = v / 4: every store and
// LDS read of a wave is 1 KiB contiguous.  The owner cannot add a whole
// partial in registers (the accumulators live in AGPRs, which VALU adds do
// not read), so it brings each quarter of a slot into the drained LDS ring by
// global->LDS copies and adds it from there, storing each quarter of the
// tile once its partials are in.
constexpr int kSkParts = 4;                                        // the owner adds a slot in 4 parts
constexpr int kSkFlagStride = 32;                                  // flags 128 bytes apart
constexpr long long kSkSpinTicks = 20000000;                       // 200 ms at 100 MHz
// The control words after the flags (each on its own 128-byte line): the
// epoch counter, the exit counter, the error counter.
constexpr int kSkCtlGen = 0, kSkCtlExited = 32, kSkCtlErrors = 64, kSkCtlWords = 96;
static_assert(kSkCtlWords == kSkCtlWordsHost && kSkCtlErrors == kSkCtlErrorsHost, "one layout of the control words");

// A workgroup's stream-K group: the tiles [t0, t0 + T / G) of XCD `xcd`
// (tiles m-block major, split into nx contiguous groups; workgroup i runs
// on XCD i mod nx, so an XCD's L2 holds only its group's rows of x), run
// by the P workgroups xcd, xcd + nx, .. (slots 0 .. P - 1).
struct SkGroup {
    long T;
    int P, slot, xcd, nx, t0;
    __device__ int phys(int s) const { return xcd + nx * s; }
};

// Segment [it, stop) of a stream-K range (stop at most its tile's end).
// NTL: tiles per block row (the N blocks of gm, or of the paired columns).
template <int BM, int NW, int SG, bool PAIR>
__device__ __forceinline__ void w4_sk_segment(char* lds, const uint16_t* xb, const GemmMats& gm, float* part,
                                              uint16_t* hout, unsigned* flags, unsigned* errors, unsigned epoch,
                                              int M, int K, int NTL, const SkGroup& gp, long it, long stop,
                                              const W4Src<BM, NW>& src, int tid, int wave, int lane) {
    typedef __attribute__((address_space(3))) void* lds_ptr;
    constexpr int TM = W4Layout<BM, NW>::TM, TN = W4Layout<BM, NW>::TN, NB = TM * TN;
    constexpr int NT = 64 * NW;
    constexpr int kDevice = 16;                                    // sc1: device-coherent
    constexpr uint32_t kSlotBytes = 256u * 256u * 4u;
    using u32x4 = unsigned int __attribute__((__vector_size__(16)));
    const int G = K >> 6;
    const long T = gp.T;
    const int P = gp.P, wg = gp.slot;
    W4Acc<BM, NW> acc;
    const int k0 = static_cast<int>(it % G);
    const int nk = static_cast<int>(stop - it);
    const long tile_start = it - k0;                               // in the group's iterations
    const int tile = gp.t0 + static_cast<int>(it / G);
    const int nt = tile % NTL, mk = PAIR ? 0 : gm_mat(gm, nt);
    const int N = gm.n_out[mk];
    float* const out = gm.out[mk];
    const W4Tile t = PAIR ? w4_tile_pair<BM>(xb, gm, M, N, K, tile / NTL, nt, wave)
                          : w4_tile<BM>(xb, gm.w[mk], gm.s[mk], gm.b[mk], M, N, K, tile / NTL, nt - gm.nb0[mk],
                                        wave);
    w4_zero<BM, NW>(acc);
    w4_segment<BM, NW, SG, PAIR>(acc, lds, t, src, k0, nk, wave, lane);
    if (stop < tile_start + G) {
        const __amdgpu_buffer_rsrc_t pr =
            buf_rsrc(part + static_cast<size_t>(gp.phys(wg)) * (kSlotBytes / 4), kSlotBytes);
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int v = 0; v < 16; v += 4) {
                    // by value: a bit cast of a vector element would read element 0
                    const u32x4 q = {__float_as_uint(acc[i][j][v]), __float_as_uint(acc[i][j][v + 1]),
                                     __float_as_uint(acc[i][j][v + 2]), __float_as_uint(acc[i][j][v + 3])};
                    const uint32_t o = static_cast<uint32_t>(((i * TN + j) * 4 + v / 4) * NT + tid) * 16u;
                    __builtin_amdgcn_raw_buffer_store_b128(q, pr, o, 0, kDevice);
                }
        __builtin_amdgcn_s_waitcnt(0x0F70);                    // this thread's stores have landed
        __syncthreads();
        if (tid == 0)
            __hip_atomic_store(flags + gp.phys(wg) * kSkFlagStride, epoch, __ATOMIC_RELEASE,
                               __HIP_MEMORY_SCOPE_AGENT);
    } else {
        // the partials of workgroups wg - 1, wg - 2, .. j1, whose ranges
        // end inside this tile
        int j1 = wg;
        while (j1 > 0 && T * j1 / P > tile_start) j1--;
        int missing = 0;
        if (tid == 0) {
            for (int j = wg - 1; j >= j1; j--) {
                if (T * (j + 1) / P == T * j / P) continue;        // an empty range
                const long long t0 = __builtin_amdgcn_s_memrealtime();
                while (__hip_atomic_load(flags + gp.phys(j) * kSkFlagStride, __ATOMIC_RELAXED,
                                         __HIP_MEMORY_SCOPE_AGENT) != epoch) {
                    if (__builtin_amdgcn_s_memrealtime() - t0 > kSkSpinTicks) {
                        __hip_atomic_fetch_add(errors, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        missing = 1;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(2);
                }
            }
        }
        // a tile whose partials did not all arrive is stored as NaN
        const bool poison = __syncthreads_or(missing) != 0;
        // the partials, not stale cache lines (only when there are any: the
        // invalidate also drops the operand lines the XCD's other
        // workgroups are streaming)
        if (j1 < wg) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        // part h of the tile (blocks h NB / kSkParts ..): each partial's part
        // in turn through LDS, then the part is stored, so only a quarter of
        // the accumulators is ever live in VGPRs
        constexpr int PB = NB / kSkParts;                          // blocks per part
        constexpr int PCH = PB * 4 * NW;                           // 1 KiB chunks per part
#pragma unroll
        for (int h = 0; h < kSkParts; h++) {
            for (int j = wg - 1; j >= j1; j--) {
                if (T * (j + 1) / P == T * j / P) continue;
                const __amdgpu_buffer_rsrc_t pr =
                    buf_rsrc(part + static_cast<size_t>(gp.phys(j)) * (kSlotBytes / 4), kSlotBytes);
#pragma unroll
                for (int c = 0; c < PCH / NW; c++) {
                    const int chunk = wave * (PCH / NW) + c;
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(
                        pr, (lds_ptr)(lds + chunk * 1024), 16, static_cast<uint32_t>(lane) * 16u,
                        static_cast<uint32_t>((h * PCH + chunk) * 1024), 0, kDevice);
                }
                __builtin_amdgcn_s_waitcnt(0x0F70);
                __syncthreads();
                const float4* hp = reinterpret_cast<const float4*>(lds);
#pragma unroll
                for (int b = 0; b < PB; b++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const int blk = h * PB + b, i = blk / TN, jj = blk % TN;
                        const float4 p4 = hp[(b * 4 + q) * NT + tid];
                        acc[i][jj][4 * q] = __fadd_rn(acc[i][jj][4 * q], p4.x);
                        acc[i][jj][4 * q + 1] = __fadd_rn(acc[i][jj][4 * q + 1], p4.y);
                        acc[i][jj][4 * q + 2] = __fadd_rn(acc[i][jj][4 * q + 2], p4.z);
                        acc[i][jj][4 * q + 3] = __fadd_rn(acc[i][jj][4 * q + 3], p4.w);
                    }
                __syncthreads();                               // before the next copies overwrite LDS
            }
            if constexpr (PAIR) {
#pragma unroll
                for (int b = 0; b < PB; b++) w4_store_pair(acc[h * PB + b][0], hout, t, M, N, h * PB + b, poison, wave, lane);
            }
            else w4_store_rows<BM, NW, kSkParts>(acc, out, t, M, N, h, poison, wave, lane);
        }
    }
}

template <int BM, int NW, int SG, bool PAIR>
__global__ __launch_bounds__(64 * NW) void gemm_w4_sk_kernel(const uint16_t* __restrict__ xb, GemmMats gm,
                                                             float* __restrict__ part, unsigned* __restrict__ flags,
                                                             unsigned* __restrict__ ctl, int M, int K, int nx,
                                                             uint16_t* __restrict__ hout) {
    static_assert(BM == 256 && (!PAIR || NW == 8), "stream-K slots hold 256 x 256 tiles");
    extern __shared__ uint4 w4_lds[];
    char* lds = reinterpret_cast<char*>(w4_lds);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = K >> 6;
    const int NTL = PAIR ? (gm.n_out[0] + 127) / 128 : gm.nb0[gm.count];
    const int tiles = ((M + BM - 1) / BM) * NTL;
    SkGroup gp;
    gp.xcd = blockIdx.x % nx;
    gp.nx = nx;
    gp.slot = blockIdx.x / nx;
    gp.P = gridDim.x / nx;
    gp.t0 = tiles * gp.xcd / nx;
    gp.T = static_cast<long>(tiles * (gp.xcd + 1) / nx - gp.t0) * G;
    const long begin = gp.T * gp.slot / gp.P, end = gp.T * (gp.slot + 1) / gp.P;
    // this launch's epoch (never 0: the flags start at 0)
    const unsigned epoch =
        __builtin_amdgcn_readfirstlane(__hip_atomic_load(ctl + kSkCtlGen, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) +
        1u;
    unsigned* errors = ctl + kSkCtlErrors;
    if (begin < end) {
        W4Src<BM, NW> src;
        w4_src<BM, NW, PAIR>(src, K, wave, lane);
        // the segments, last to first: [max(tile start, begin), seg_end)
        for (long seg_end = end; seg_end > begin;) {
            const long tile_start = (seg_end - 1) / G * G;
            const long seg_start = tile_start > begin ? tile_start : begin;
            w4_sk_segment<BM, NW, SG, PAIR>(lds, xb, gm, part, hout, flags, errors, epoch, M, K, NTL, gp, seg_start,
                                        seg_end, src, tid, wave, lane);
            seg_end = seg_start;
        }
    }
    // the last workgroup to leave advances the epoch (every workgroup has
    // read it by then: the release orders that read before the count)
    if (tid == 0) {
        const unsigned left =
            __hip_atomic_fetch_add(ctl + kSkCtlExited, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (left == gridDim.x - 1) {
            __hip_atomic_store(ctl + kSkCtlExited, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // epoch - 1 is the stored value; skip the one whose epoch would be 0
            const unsigned next = epoch == 0xFFFFFFFFu ? 0u : epoch;
            __hip_atomic_store(ctl + kSkCtlGen, next, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

// SG of a launch: the groups of scales and biases that one copy takes, by the
// group count and the alignment of every matrix's scales and biases.
int w4_groups(const GemmMats& gm, int K) {
    const int G = K >> 6;
    uintptr_t al = 0;
    for (int k = 0; k < gm.count; k++)
        al |= reinterpret_cast<uintptr_t>(gm.s[k]) | reinterpret_cast<uintptr_t>(gm.b[k]);
    return G % 8 == 0 && !(al & 15) ? 8 : G % 2 == 0 && !(al & 3) ? 2 : 1;
}

template <int BM, int NW, int SG>
int launch_w4(const uint16_t* xb, const GemmMats& gm, float* part, int M, int K, int S, int kt_split, int ldp,
              hipStream_t st) {
    auto kern = gemm_w4_kernel<BM, NW, SG>;
    constexpr size_t lds = w4_lds_bytes(BM, SG);
    static std::atomic<uint64_t> lds_raised{0};
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kern), lds, lds_raised)) return rc;
    hipLaunchKernelGGL(kern, dim3((M + BM - 1) / BM, gm.nb0[gm.count], S), dim3(64 * NW), lds, st, xb, gm, part, M, K,
                       kt_split, ldp);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(Q4_EHIP, "prefill gemm launch: %s", hipGetErrorString(e));
    return 0;
}

template <int BM, int NW, int SG, bool PAIR>
int launch_w4_sk(const uint16_t* xb, const GemmMats& gm, float* part, unsigned* flags, unsigned* ctl, int M, int K,
                 int P, int nx, uint16_t* hout, hipStream_t st) {
    auto kern = gemm_w4_sk_kernel<BM, NW, SG, PAIR>;
    constexpr size_t lds = w4_lds_bytes(BM, SG);
    static_assert(256 * 256 * 4 / kSkParts <= lds, "a part of a slot fits the LDS");
    static std::atomic<uint64_t> lds_raised{0};
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kern), lds, lds_raised)) return rc;
    hipLaunchKernelGGL(kern, dim3(P), dim3(64 * NW), lds, st, xb, gm, part, flags, ctl, M, K, nx, hout);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(Q4_EHIP, "prefill gemm (stream-K) launch: %s", hipGetErrorString(e));
    return 0;
}

template <int BM, int SG>
int launch_w4_pair(const uint16_t* xb, const GemmMats& gm, uint16_t* h, int M, int K, hipStream_t st) {
    auto kern = gemm_w4_pair_kernel<BM, 8, SG>;
    constexpr size_t lds = w4_lds_bytes(BM, SG);
    static std::atomic<uint64_t> lds_raised{0};
    if (int rc = raise_lds_limit(reinterpret_cast<const void*>(kern), lds, lds_raised)) return rc;
    hipLaunchKernelGGL(kern, dim3((M + BM - 1) / BM, (gm.n_out[0] + 127) / 128), dim3(64 * 8), lds, st, xb, gm, h, M, K);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(Q4_EHIP, "prefill gate/up gemm launch: %s", hipGetErrorString(e));
    return 0;
}

template <int BM>
int pair_by_groups(const uint16_t* xb, const GemmMats& gm, uint16_t* h, int M, int K, hipStream_t st) {
    const int sg = w4_groups(gm, K);
    return sg == 8 ? launch_w4_pair<BM, 8>(xb, gm, h, M, K, st)
                   : sg == 2 ? launch_w4_pair<BM, 2>(xb, gm, h, M, K, st) : launch_w4_pair<BM, 1>(xb, gm, h, M, K, st);
}

int gemm_w4_pair(const uint16_t* xb, const GemmMats& gm, uint16_t* h, int M, int K, int bm, hipStream_t st) {
    switch (bm) {
        case 64: return pair_by_groups<64>(xb, gm, h, M, K, st);
        case 128: return pair_by_groups<128>(xb, gm, h, M, K, st);
        case 192: return pair_by_groups<192>(xb, gm, h, M, K, st);
        default: return pair_by_groups<256>(xb, gm, h, M, K, st);
    }
}

template <int BM, int NW>
int w4_by_groups(const uint16_t* xb, const GemmMats& gm, float* part, int M, int K, int S, int kt_split, int ldp,
                 hipStream_t st) {
    const int sg = w4_groups(gm, K);
    return sg == 8 ? launch_w4<BM, NW, 8>(xb, gm, part, M, K, S, kt_split, ldp, st)
                   : sg == 2 ? launch_w4<BM, NW, 2>(xb, gm, part, M, K, S, kt_split, ldp, st)
                             : launch_w4<BM, NW, 1>(xb, gm, part, M, K, S, kt_split, ldp, st);
}

int gemm_w4(const uint16_t* xb, const GemmMats& gm, float* part, int M, int K, int bm, int S, int kt_split, int ldp,
            hipStream_t st) {
    switch (bm) {
        case 64: return w4_by_groups<64, 8>(xb, gm, part, M, K, S, kt_split, ldp, st);
        case 128: return w4_by_groups<128, 8>(xb, gm, part, M, K, S, kt_split, ldp, st);
        case 192: return w4_by_groups<192, 8>(xb, gm, part, M, K, S, kt_split, ldp, st);
        default: return w4_by_groups<256, 8>(xb, gm, part, M, K, S, kt_split, ldp, st);
    }
}

template <bool PAIR>
int sk_by_groups(const uint16_t* xb, const GemmMats& gm, float* part, unsigned* flags, unsigned* ctl, uint16_t* h, int M,
                 int K, int P, int nx, hipStream_t st) {
    const int sg = w4_groups(gm, K);
    return sg == 8 ? launch_w4_sk<256, 8, 8, PAIR>(xb, gm, part, flags, ctl, M, K, P, nx, h, st)
                   : sg == 2 ? launch_w4_sk<256, 8, 2, PAIR>(xb, gm, part, flags, ctl, M, K, P, nx, h, st)
                             : launch_w4_sk<256, 8, 1, PAIR>(xb, gm, part, flags, ctl, M, K, P, nx, h, st);
}

int gemm_w4_sk(const uint16_t* xb, const GemmMats& gm, float* part, unsigned* flags, unsigned* ctl, int M, int K,
               int P, int nx, hipStream_t st) {
    return sk_by_groups<false>(xb, gm, part, flags, ctl, nullptr, M, K, P, nx, st);
}

int gemm_w4_sk_pair(const uint16_t* xb, const GemmMats& gm, float* part, unsigned* flags, unsigned* ctl, uint16_t* h,
                    int M, int K, int P, int nx, hipStream_t st) {
    return sk_by_groups<true>(xb, gm, part, flags, ctl, h, M, K, P, nx, st);
}

}  // namespace q4k
