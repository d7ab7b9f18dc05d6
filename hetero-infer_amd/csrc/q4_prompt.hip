// Causal grouped-query attention of a prompt chunk over the fp16 KV cache
// (gfx950), the attention of the device-resident prompt forward.  Declared
// in q4decode.h (q4_prompt_attention_dev).
//
// hetero/cpu_model.py:233-252 (sdpa with causal=True, L > 1): query row r
// of a chunk that starts at position pos0 sits at position pos0 + r and
// sees the positions [0, pos0 + r] -- the reference's mask
// `arange(S) <= arange(L) + (S - L)` with S = pos0 + L; query head h reads
// kv head h / (nh / nkv); s = (q . k) * scale, softmax over the visible
// positions, o = sum p v.
//
#include <hip/hip_runtime.h>

#include <cstdint>

#include "q4_common.h"
#include "q4decode.h"

namespace q4k {
namespace {

constexpr int kPTile = 64;                  // positions per tile
constexpr int kPMaxG = 8;                   // query heads per kv head

struct PromptAttnArgs {
    const float* q;          // [rows][nh * d], rotated queries
    const uint16_t* kc;      // [nkv][cap][d] fp16
    const uint16_t* vc;
    void* out;               // [rows][nh * d], fp32 or (BF) bf16
    int rows;
    int64_t pos0;
    int nh, nkv, d, cap;
    float scale;
};

// ---------------------------------------------------------------------
// On the matrix cores (v_mfma_f32_16x16x32_f16).  A workgroup takes one kv
// head, 16 consecutive query rows and 2 or 4 of the kv head's query heads,
// in KS groups of one wave per head: group k walks the tiles k, k + KS, ...
// of 64 positions, its tile's K rows (k_s, row-major) and V rows (vt_s,
// transposed: [dim][pos]) staged in LDS once for its heads, the next tile's
// loads in flight while the current one is multiplied.  The groups' maxima,
// sums and outputs are merged in LDS at the end.
//
// Per tile and wave, with lane l: c = l % 16 (a query row of the block),
// qd = l / 16:
//   S^T = K Q^T: 4 x D / 32 MFMAs; lane l ends with query row c's scores at
//     positions 16 mt + 4 qd + v (mt, v = 0..3);
//   the running softmax of row c (its 64 scores sit in lanes c, c + 16,
//     c + 32, c + 48: a max and a sum over the lane's 16, then across the
//     four lanes), evaluated online: it agrees with one max and one sum over
//     the whole row to fp32 rounding, not bit for bit;
//   O^T += V^T P^T: D / 16 x 2 MFMAs; lane l holds query row c's outputs at
//     dims 16 dt + 4 qd + v, rescaled by the row's correction in place.
// The MFMA operands are fp16, the sums fp32.  Exact fp16 operands: the
// cache is fp16, and q and p enter as two fp16 terms each, two MFMAs per
// product, placed in fp16's range so that nothing that counts is rounded away:
//   q: a row is scaled by a power of two to a maximum in [2^14, 2^15)
//     (pa_split), each value to 2^-22 of itself or 2^-38 of the maximum;
//   p: relative to its tile's own maximum (the online softmax's running
//     maximum replaced by it), after the first tile to the power of two just
//     above, so that rescaling l and O^T is exact, and times 2^15, as hi + lo
//     (pa_split_p), to 2^-23 of itself or 2^-40 of the tile's largest.
// One dominant key (an attention sink, whose value is near zero) leaves
// thousands of small p to make the output: from p below the running maximum,
// unscaled and so to 2^-25, 6e-5 of them was lost 10 nats below that key and
// 0.19 at 18; now 2e-6, as with fp32 probabilities, in the same time (45 us
// against 46 for the case below; 1 to 2 % more at head_dim 64).
// q is multiplied by scale * log2(e) first and the softmax taken with exp2,
// which is exp of the scaled score.  Workgroups of the last rows, which see
// the most positions, are launched first, over all kv heads (block rows are the
// grid's slowest dimension): with heads the slowest, the last heads' longest rows
// made a second round as long as the first (700 rows, 28 heads 26 -> 20 us).
//
// Bound by the matrix and vector ALUs of the few waves there are: 16 rows of
// 28 heads are 28 waves, 512 rows 896, so the groups put two waves on every
// SIMD, and each wave hides its LDS reads itself (a wave's 32 reads of a tile
// one after the other, each waited for, were 4000 of its 7000 clocks).
// 512 rows after 1536 positions, 28 heads of 4 kv heads, head_dim 128: all
// heads of a kv head in one workgroup, one group 89 us; two groups of four
// heads 57; operands read a step ahead, unmasked tiles without the mask, sums
// across lanes once at the end 46-49; two tile buffers, one barrier a tile,
// 45 (590 TFLOP/s of MFMA).  512 rows from an empty cache 26 -> 16 us, 17 rows
// after 4000 positions 162 -> 57.  head_dim
// 64 (on the vector ALUs before) 300 -> 27, 17 rows after 4000 (32 heads)
// 497 -> 30; errors against float64 at these sizes are at most what they were.
constexpr int kMRows = 16;                         // query rows per workgroup
constexpr int kVRowH = kPTile + 8;                 // vt_s row: 64 fp16 + 8 pad (144 bytes: 16-byte reads spread)

typedef _Float16 pa_h8 __attribute__((ext_vector_type(8)));
typedef float pa_f4 __attribute__((ext_vector_type(4)));

template <int D, int NT>
struct PaShape {
    static constexpr int KROW = D + 8;             // k_s row in fp16: D + 8 pad (16-byte reads spread)
    static constexpr int KCH = kPTile * D / 8;     // 16-byte chunks of a K tile
    static constexpr int VIT = kPTile / 2 * D / 8; // (position pair, 8 dims) items of a V tile
    static constexpr int KI = (KCH + NT - 1) / NT, VI = (VIT + NT - 1) / NT;   // per thread
    static constexpr int TILE = kPTile * KROW + D * kVRowH;                    // fp16 of a group's tiles
};

template <int D, int NT>
struct PaStage {                                   // one thread's share of a tile's loads
    uint4 k[PaShape<D, NT>::KI];
    uint4 v0[PaShape<D, NT>::VI], v1[PaShape<D, NT>::VI];
};

// V item e: a wave's 64 items are 16 position pairs of 4 neighbouring 8-dim
// chunks (64-byte reads; stores of 32 banks, two lanes each).
__device__ __forceinline__ int pa_v_pair(int e) { return e >> 2 & 31; }
__device__ __forceinline__ int pa_v_dim(int e) { return ((e >> 7) * 4 + (e & 3)) * 8; }

// The tile at position c0 of the kv head's rows, `valid` positions of it
// (none: zeros).
template <int D, int NT>
__device__ __forceinline__ void pa_load(PaStage<D, NT>& st, const PromptAttnArgs& a, size_t head_row0, int64_t c0,
                                        int64_t valid, int tid) {
    using S = PaShape<D, NT>;
    valid = valid < 0 ? 0 : valid < kPTile ? valid : kPTile;
    const uint32_t bytes = static_cast<uint32_t>(valid) * D * 2u;
    const __amdgpu_buffer_rsrc_t kr = buf_rsrc(a.kc + (head_row0 + c0) * D, bytes);
    const __amdgpu_buffer_rsrc_t vr = buf_rsrc(a.vc + (head_row0 + c0) * D, bytes);
#pragma unroll
    for (int i = 0; i < S::KI; i++) {
        const int e = tid + i * NT;
        const uint32_t off = e < S::KCH ? static_cast<uint32_t>(e) * 16u : kOutOfRange;
        st.k[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(kr, off, 0, 0));
    }
#pragma unroll
    for (int i = 0; i < S::VI; i++) {
        const int e = tid + i * NT;
        const uint32_t off = e < S::VIT ? static_cast<uint32_t>(pa_v_pair(e) * 2 * D + pa_v_dim(e)) * 2u : kOutOfRange;
        st.v0[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(vr, off, 0, 0));
        st.v1[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(vr, off + D * 2, 0, 0));
    }
}

template <int D, int NT>
__device__ __forceinline__ void pa_store(const PaStage<D, NT>& st, _Float16* k_s, _Float16* vt_s, int tid) {
    using S = PaShape<D, NT>;
#pragma unroll
    for (int i = 0; i < S::KI; i++) {
        const int e = tid + i * NT;
        if (e < S::KCH) *reinterpret_cast<uint4*>(k_s + e / (D / 8) * S::KROW + e % (D / 8) * 8) = st.k[i];
    }
#pragma unroll
    for (int i = 0; i < S::VI; i++) {
        const int e = tid + i * NT;
        if (e < S::VIT) {
            // position 32 kk + 16 h + 4 qd + v sits at column 32 kk + 8 qd + 4 h + v:
            // the 8 positions of an MFMA operand's lane are one 16-byte read
            const int pp = pa_v_pair(e);
            const int col = (pp & 16) * 2 + (pp >> 1 & 3) * 8 + (pp >> 3 & 1) * 4 + (pp & 1) * 2;
            _Float16* dst = vt_s + pa_v_dim(e) * kVRowH + col;
            const uint32_t a[4] = {st.v0[i].x, st.v0[i].y, st.v0[i].z, st.v0[i].w};
            const uint32_t b[4] = {st.v1[i].x, st.v1[i].y, st.v1[i].z, st.v1[i].w};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                // dims 2j and 2j + 1: (pos 2pp, pos 2pp + 1) each
                *reinterpret_cast<uint32_t*>(dst + 2 * j * kVRowH) = __builtin_amdgcn_perm(b[j], a[j], 0x05040100u);
                *reinterpret_cast<uint32_t*>(dst + (2 * j + 1) * kVRowH) =
                    __builtin_amdgcn_perm(b[j], a[j], 0x07060302u);
            }
        }
    }
}

// x = hi + lo in fp16: hi is the next value below |x| with its low 13
// significand bits cleared, which fp16 holds exactly whenever it is at least
// 2^-14, so no conversion of it can round (the compiler may convert it again,
// packed, for the MFMA operand: any rounding mode gives the same value); lo =
// fp16(x - hi), x - hi exact in fp32.  Below 2^-14 the pair is within 2^-24 of
// x.  From 2^-2 on lo is never 0 and both have x's sign, so that an infinite
// key gives an infinite score and not a NaN.
__device__ __forceinline__ void pa_split(float x, _Float16& hi, _Float16& lo) {
    const float h = __uint_as_float(__float_as_uint(__fmul_rn(x, 0x1.fffffcp-1f)) & 0xFFFFE000u);
    hi = static_cast<_Float16>(h);
    lo = static_cast<_Float16>(__fsub_rn(x, h));
}

// Two values of p, times 2^15, as hi + lo: hi the nearest fp16 value, lo the
// rest.  (Vector conversions: the packed one, where a product converted alone
// becomes a half-register write of its own; opaque, so that lo is the rest of
// the very value that the MFMA takes and not of a second conversion.)
constexpr float kPScale = 32768.0f;
constexpr float kPDrop = 32.0f;                    // see the softmax of a tile
typedef float pa_f2 __attribute__((ext_vector_type(2)));
typedef _Float16 pa_h2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void pa_split_p(const float (&x)[2], pa_h2& hi, pa_h2& lo) {
    uint32_t h = __builtin_bit_cast(uint32_t, __builtin_convertvector((pa_f2{x[0], x[1]}), pa_h2));
    asm("" : "+v"(h));
    hi = __builtin_bit_cast(pa_h2, h);
    lo = __builtin_convertvector(
        (pa_f2{__fsub_rn(x[0], static_cast<float>(hi[0])), __fsub_rn(x[1], static_cast<float>(hi[1]))}), pa_h2);
}

// f over the four lanes of a query row (c, c + 16, c + 32, c + 48), in all of them.
template <class F>
__device__ __forceinline__ float pa_rows4(float x, F f) {
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = f(__uint_as_float(s[0]), __uint_as_float(s[1]));
    const auto t = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return f(__uint_as_float(t[0]), __uint_as_float(t[1]));
}

template <int HPW, int KS, int D, bool BF>
__global__ __launch_bounds__(64 * HPW * KS) __attribute__((amdgpu_waves_per_eu(2, 2))) void prompt_attn_kernel(PromptAttnArgs a) {
    constexpr int NT = 64 * HPW, KT = D / 32, DT = D / 16;
    using S = PaShape<D, NT>;
    // a wave's maximum, sum and outputs, when the groups are merged
    constexpr int PART = (2 + 4 * DT) * 64;
    static_assert((KS - 1) * HPW * PART * 4 <= KS * S::TILE * 2, "the parts reuse the tiles' LDS");
    constexpr int NB = 2 * KS * S::TILE * 2 <= 160 * 1024 ? 2 : 1;     // tile buffers
    __shared__ __attribute__((aligned(16))) _Float16 lds[NB * KS * S::TILE];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const int kg = wave / HPW;                                  // the wave's group
    const int tid = threadIdx.x - kg * NT;                      // thread of the group
    const int G = a.nh / a.nkv;
    // (7 heads are 4 and 3: an XCD, workgroups modulo 8, gets some of each)
    const int part = gridDim.y == 2 ? blockIdx.y ^ (blockIdx.z & 1) : blockIdx.y;
    const int h = part * HPW + wave % HPW;                // query head of the kv head
    const int c = lane & 15, qd = lane >> 4;
    const int kvh = blockIdx.x;
    const int r0 = (static_cast<int>(gridDim.z) - 1 - static_cast<int>(blockIdx.z)) * kMRows;
    const int last_row = (r0 + kMRows < a.rows ? r0 + kMRows : a.rows) - 1;
    const int64_t wg_last = a.pos0 + last_row;
    const int r = r0 + c;                                      // lane's query row
    const bool row_ok = h < G && r < a.rows;
    const int64_t my_last = a.pos0 + (r < last_row ? r : last_row);
    const int n_tiles = static_cast<int>(wg_last / kPTile) + 1;
    const int hd = a.nh * D;
    const size_t head_row0 = static_cast<size_t>(kvh) * a.cap;

    PaStage<D, NT> st;
    pa_load<D, NT>(st, a, head_row0, kg * kPTile, wg_last + 1 - kg * kPTile, tid);

    // q of row r, head kvh G + h, as the B operand of S^T: dims 32 ks + 8 qd ..
    const float qs = __fmul_rn(a.scale, 1.44269504088896341f);
    pa_h8 qh[KT], ql[KT];
    float up;                                                  // what the row's operands were scaled down by
    {
        const float* src = a.q + static_cast<size_t>(r) * hd + static_cast<size_t>(kvh * G + h) * D + 8 * qd;
        float xv[KT][8], am = 0.0f;
#pragma unroll
        for (int ks = 0; ks < KT; ks++) {
            float4 x0 = make_float4(0.f, 0.f, 0.f, 0.f), x1 = x0;
            if (row_ok) {
                x0 = reinterpret_cast<const float4*>(src + 32 * ks)[0];
                x1 = reinterpret_cast<const float4*>(src + 32 * ks)[1];
            }
            const float x[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
            for (int i = 0; i < 8; i++) {
                xv[ks][i] = __fmul_rn(x[i], qs);
                am = fmaxf(am, fabsf(xv[ks][i]));
            }
        }
        // the row's maximum to [2^14, 2^15) by a power of two, its scores back
        // by the inverse (exact; a maximum below 2^-86 is no matter to exp2)
        am = pa_rows4(am, [](float x, float y) { return fmaxf(x, y); });
        int e = static_cast<int>(__float_as_uint(am) >> 23) - 127 - 14;
        e = e < -100 ? -100 : e;
        const float down = __uint_as_float(static_cast<uint32_t>(127 - e) << 23);
        up = __uint_as_float(static_cast<uint32_t>(127 + e) << 23);
#pragma unroll
        for (int ks = 0; ks < KT; ks++)
#pragma unroll
            for (int i = 0; i < 8; i++) {
                _Float16 hi, lo;
                pa_split(__fmul_rn(xv[ks][i], down), hi, lo);
                qh[ks][i] = hi;
                ql[ks][i] = lo;
            }
    }
    pa_f4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o[dt] = pa_f4{0.f, 0.f, 0.f, 0.f};
    float m = -__builtin_inff(), l = 0.0f, top = m;             // top: the largest m

    for (int t0 = 0; t0 < n_tiles; t0 += KS) {
        const int64_t c0 = static_cast<int64_t>(t0 + kg) * kPTile;
        // with two buffers, the barrier below has every wave past the tiles
        // before the last, which this store replaces
        _Float16* k_s = lds + ((NB == 2 ? t0 / KS & 1 : 0) * KS + kg) * S::TILE;
        _Float16* vt_s = k_s + kPTile * S::KROW;
        if (NB == 1) __syncthreads();                          // every wave is done with the last tiles
        pa_store<D, NT>(st, k_s, vt_s, tid);
        __syncthreads();
        if (t0 + KS < n_tiles) pa_load<D, NT>(st, a, head_row0, c0 + KS * kPTile, wg_last + 1 - c0 - KS * kPTile, tid);
        if (t0 + kg >= n_tiles || h >= G) continue;            // uniform in the wave
        // S^T = K Q^T: s[mt][v] = score of row r at position c0 + 16 mt + 4 qd + v;
        // operands are read one step ahead of the MFMAs that take them
        pa_f4 s[4];
        pa_h8 kf[2][4], vf[2][4];
        const _Float16* krow = k_s + c * S::KROW + 8 * qd;
        const _Float16* vrow = vt_s + c * kVRowH + 8 * qd;
#pragma unroll
        for (int mt = 0; mt < 4; mt++) {
            s[mt] = pa_f4{0.f, 0.f, 0.f, 0.f};
            kf[0][mt] = *reinterpret_cast<const pa_h8*>(krow + 16 * mt * S::KROW);
        }
#pragma unroll
        for (int ks = 0; ks < KT; ks++) {
#pragma unroll
            for (int mt = 0; mt < 4; mt++) {
                if (ks + 1 < KT)
                    kf[(ks + 1) & 1][mt] = *reinterpret_cast<const pa_h8*>(krow + 16 * mt * S::KROW + 32 * (ks + 1));
                else   // the first operands of V^T P^T
                    vf[0][mt] = *reinterpret_cast<const pa_h8*>(vrow + 16 * (mt % DT) * kVRowH + 32 * (mt / DT));
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int mt = 0; mt < 4; mt++) s[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[ks & 1][mt], qh[ks], s[mt], 0, 0, 0);
#pragma unroll
            for (int mt = 0; mt < 4; mt++) s[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[ks & 1][mt], ql[ks], s[mt], 0, 0, 0);
        }
        // the softmax of row r (s times up are the scores), l and o relative to
        // 2^m: m the tile's maximum, rounded up after the group's first tile, but
        // at most kPDrop (64 where m's spacing is that wide) below the row's
        // largest so far, so that o stays below 2^(64 + 15 + 16 + 16).  In the
        // first tile the largest p is so exactly 1, and a row that sees one key
        // gives that key's value exactly (rounded up there too, one bf16 value in
        // sixteen of a prompt's first row was a unit off, as an eighth of the
        // fp16 values are ties of bf16; 1 % of the time at 512 rows after 1536).
        if (c0 + kPTile - 1 > a.pos0 + r0) {                   // uniform: some row does not see all of the tile
            const int vis = static_cast<int>(my_last - c0 < kPTile ? my_last - c0 : kPTile) - 4 * qd;
#pragma unroll
            for (int mt = 0; mt < 4; mt++)
#pragma unroll
                for (int v = 0; v < 4; v++) s[mt][v] = 16 * mt + v <= vis ? s[mt][v] : -__builtin_inff();
        }
        float mx = -__builtin_inff();
#pragma unroll
        for (int mt = 0; mt < 4; mt++)
#pragma unroll
            for (int v = 0; v < 4; v++) mx = fmaxf(mx, s[mt][v]);
        mx = pa_rows4(mx, [](float x, float y) { return fmaxf(x, y); });
        const float t = __fmul_rn(mx, up);
        float mc = t0 == 0 ? t : __builtin_ceilf(t);
        if constexpr (D == 128) asm("" : "+v"(mc));             // a schedule 1 % faster there
        top = fmaxf(top, mc);
        const float mn = fmaxf(mc, __fsub_rn(top, kPDrop));
        const float ms = mn == -__builtin_inff() ? 0.0f : mn;  // the row sees none of the group's positions so far
        const float corr = __builtin_amdgcn_exp2f(__fsub_rn(m, ms));
        m = mn;
        float ps = 0.0f;
        pa_h8 ph[2], pl[2];
#pragma unroll
        for (int mt = 0; mt < 4; mt++)
#pragma unroll
            for (int v = 0; v < 4; v += 2) {
                float p[2];
#pragma unroll
                for (int k = 0; k < 2; k++) {                  // 0 where masked
                    p[k] = __fmul_rn(kPScale, __builtin_amdgcn_exp2f(__fmaf_rn(s[mt][v + k], up, -ms)));
                    asm("" : "+v"(p[k]));                      // one product for l and hi
                    ps = __fadd_rn(ps, p[k]);
                }
                pa_h2 hi, lo;
                pa_split_p(p, hi, lo);
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    ph[mt >> 1][(mt & 1) * 4 + v + k] = hi[k];
                    pl[mt >> 1][(mt & 1) * 4 + v + k] = lo[k];
                }
            }
        l = __fadd_rn(__fmul_rn(l, corr), ps);
#pragma unroll
        for (int dt = 0; dt < DT; dt++) o[dt] *= corr;
        // O^T += V^T P^T in steps of four operands, (kk, dt) with dt innermost;
        // k index 8 qd + i of kk is position 32 kk + 4 qd + i (i < 4) or
        // 32 kk + 16 + 4 qd + i - 4
        constexpr int VG = 2 * DT / 4;
#pragma unroll
        for (int g = 0; g < VG; g++) {
            if (g + 1 < VG)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int f = 4 * (g + 1) + i;
                    vf[(g + 1) & 1][i] =
                        *reinterpret_cast<const pa_h8*>(vrow + 16 * (f % DT) * kVRowH + 32 * (f / DT));
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int f = 4 * g + i;
                o[f % DT] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[g & 1][i], ph[f / DT], o[f % DT], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int f = 4 * g + i;
                o[f % DT] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[g & 1][i], pl[f / DT], o[f % DT], 0, 0, 0);
            }
        }
    }
    l = pa_rows4(l, [](float x, float y) { return __fadd_rn(x, y); });

    // merge the groups: group 0 rescales every part to the common maximum
    if (KS > 1 && n_tiles > 1) {
        __syncthreads();                                           // the last tiles are read
        float* parts = reinterpret_cast<float*>(lds);
        if (kg > 0) {
            float* mine = parts + (wave - HPW) * PART + lane;
            mine[0] = m;
            mine[64] = l;
#pragma unroll
            for (int i = 0; i < 4 * DT; i++) mine[(2 + i) * 64] = o[i >> 2][i & 3];
        }
        __syncthreads();
        if (kg > 0) return;
        float mt = m;
#pragma unroll
        for (int k = 1; k < KS; k++) mt = fmaxf(mt, parts[((k - 1) * HPW + wave) * PART + lane]);
        const float ms = mt == -__builtin_inff() ? 0.0f : mt;
        {
            const float f = __builtin_amdgcn_exp2f(__fsub_rn(m, ms));
            l = __fmul_rn(l, f);
#pragma unroll
            for (int dt = 0; dt < DT; dt++) o[dt] *= f;
        }
#pragma unroll
        for (int k = 1; k < KS; k++) {
            const float* other = parts + ((k - 1) * HPW + wave) * PART + lane;
            const float f = __builtin_amdgcn_exp2f(__fsub_rn(other[0], ms));
            l = __fmaf_rn(other[64], f, l);
#pragma unroll
            for (int i = 0; i < 4 * DT; i++) o[i >> 2][i & 3] = __fmaf_rn(other[(2 + i) * 64], f, o[i >> 2][i & 3]);
        }
    } else if (kg > 0) {
        return;
    }
    if (row_ok) {
        const size_t at = static_cast<size_t>(r) * hd + static_cast<size_t>(kvh * G + h) * D + 4 * qd;
#pragma unroll
        for (int dt = 0; dt < DT; dt++) {
            const float v0 = __fdiv_rn(o[dt][0], l), v1 = __fdiv_rn(o[dt][1], l);
            const float v2 = __fdiv_rn(o[dt][2], l), v3 = __fdiv_rn(o[dt][3], l);
            if constexpr (BF) {
                *reinterpret_cast<uint2*>(static_cast<uint16_t*>(a.out) + at + 16 * dt) =
                    make_uint2(bf16x2_rne(v0, v1), bf16x2_rne(v2, v3));
            } else {
                *reinterpret_cast<float4*>(static_cast<float*>(a.out) + at + 16 * dt) = make_float4(v0, v1, v2, v3);
            }
        }
    }
}

template <int HPW, int KS, int D>
void launch_prompt(PromptAttnArgs a, bool bf, hipStream_t st) {
    constexpr int kMost = 65535 * kMRows;                      // the grid's z
    const int parts = (a.nh / a.nkv + HPW - 1) / HPW;
    for (int left = a.rows; left > 0; left -= a.rows) {
        a.rows = left < kMost ? left : kMost;
        const dim3 grid(a.nkv, parts, (a.rows + kMRows - 1) / kMRows);
        if (bf) hipLaunchKernelGGL((prompt_attn_kernel<HPW, KS, D, true>), grid, dim3(64 * HPW * KS), 0, st, a);
        else hipLaunchKernelGGL((prompt_attn_kernel<HPW, KS, D, false>), grid, dim3(64 * HPW * KS), 0, st, a);
        const size_t at = static_cast<size_t>(a.rows) * a.nh * D;
        a.q += at;
        a.out = static_cast<char*>(a.out) + at * (bf ? 2 : 4);
        a.pos0 += a.rows;
    }
}

// Query heads per workgroup and groups of waves, by the tiles of the last row
// and the workgroups per CU (us at head_dim 128; a wave without a head still
// stages its share of the tiles).
// Pairs of heads while those workgroups fit the chip at one per CU, and always
// for 1 or 2 heads per kv head: a group per tile up to two tiles, four groups
// from seven on (17 rows of 28 heads: 1 tile 6.9 / 7.4 / 8.6 us with 1 / 2 / 4
// groups, 2 tiles 8.8 / 8.0 / 9.9, 6 tiles 2 groups 12.1 and 4 12.9, 8 tiles 13.7
// and 13.2, 63 tiles 69 and 56).  1 or 2 heads and up to three tiles: fours, the
// extra waves staging (one head, 1 tile 5.7 against 6.2 us, 3 tiles 8.4 against
// 9.0).  1 or 2 heads past one pair per CU: what a CU holds two workgroups of,
// pairs in two groups (700 rows, 8 heads 17.1 us; one per CU in four groups
// 19.9) or, at head_dim 128 past 16 tiles or from two pairs per CU on, fours (700
// after 1000 positions 42.1 against 46.3; 1500 39.0 against 51.3).
// Else fours, which read each K and V operand for more heads (300 rows after
// 3000, 28 heads 94 -> 60 us, 512 after 1536 69 -> 43): two groups; one, two
// workgroups per CU, for up to three tiles, or past one workgroup per CU for up
// to eight tiles (300 rows, 64 heads of 8 kv heads 15.3 against 16.4 us) or from
// two per CU on (700 rows 30.4 against 38.6; with fewer and more tiles the other
// way, 700 rows of 32 heads 24.6 against 21.4).
template <int D>
void launch_prompt_heads(const PromptAttnArgs& a, bool bf, hipStream_t st) {
    const int G = a.nh / a.nkv, cus = num_cus();
    const int64_t tiles = (a.pos0 + a.rows - 1) / kPTile + 1;
    const int64_t blocks = static_cast<int64_t>((a.rows + kMRows - 1) / kMRows) * a.nkv;
    const bool fit = blocks * ((G + 1) / 2) <= cus;
    if (G <= 2 && tiles <= 3) return launch_prompt<4, 1, D>(a, bf, st);
    if (G <= 2 || fit) {
        if (!fit && D == 128 && (tiles > 16 || blocks >= 2 * cus)) return launch_prompt<4, 1, D>(a, bf, st);
        if (tiles == 1) return launch_prompt<2, 1, D>(a, bf, st);
        if (tiles <= 6 || !fit) return launch_prompt<2, 2, D>(a, bf, st);
        return launch_prompt<2, 4, D>(a, bf, st);
    }
    const int64_t wgs = blocks * ((G + 3) / 4);
    if (tiles <= 3 || (wgs > cus && tiles <= 8) || wgs >= 2 * cus) return launch_prompt<4, 1, D>(a, bf, st);
    return launch_prompt<4, 2, D>(a, bf, st);
}

int launch_failed(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(Q4_EHIP, "%s launch: %s", what, hipGetErrorString(e));
    return 0;
}

}  // namespace
}  // namespace q4k

using namespace q4k;

namespace {

int prompt_attention(const float* q, const uint16_t* k_cache, const uint16_t* v_cache, void* out, bool bf, int rows,
                     int64_t pos0, int n_heads, int n_kv, int head_dim, int cap, float scale, void* stream) {
    if (!q || !k_cache || !v_cache || !out) return fail(Q4_EARG, "q4_prompt_attention_dev: null pointer");
    if (n_heads <= 0 || n_kv <= 0 || n_heads % n_kv || n_heads / n_kv > kPMaxG ||
        (head_dim != 32 && head_dim != 64 && head_dim != 128) || cap <= 0)
        return fail(Q4_EARG, "q4_prompt_attention_dev: unsupported sizes (heads %d, kv heads %d, head_dim %d, cap %d)",
                    n_heads, n_kv, head_dim, cap);
    if (rows < 0 || pos0 < 0 || pos0 + rows > cap)
        return fail(Q4_EARG, "q4_prompt_attention_dev: rows at positions [%lld, %lld) outside the cache [0, %d)",
                    static_cast<long long>(pos0), static_cast<long long>(pos0 + rows), cap);
    if ((reinterpret_cast<uintptr_t>(q) & 15) || (reinterpret_cast<uintptr_t>(out) & 15) ||
        (reinterpret_cast<uintptr_t>(k_cache) & 15) || (reinterpret_cast<uintptr_t>(v_cache) & 15))
        return fail(Q4_EARG, "q4_prompt_attention_dev: q, out and the caches must be 16-byte aligned");
    if (rows == 0) return 0;
    const PromptAttnArgs a{q, k_cache, v_cache, out, rows, pos0, n_heads, n_kv, head_dim, cap, scale};
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (head_dim == 128) launch_prompt_heads<128>(a, bf, st);
    else if (head_dim == 64) launch_prompt_heads<64>(a, bf, st);
    else launch_prompt_heads<32>(a, bf, st);
    return launch_failed("q4_prompt_attention_dev");
}

}  // namespace

#pragma GCC visibility push(default)
extern "C" {

int q4_prompt_attention_dev(const float* q, const uint16_t* k_cache, const uint16_t* v_cache, float* out, int rows,
                            int64_t pos0, int n_heads, int n_kv, int head_dim, int cap, float scale, void* stream) {
    return prompt_attention(q, k_cache, v_cache, out, false, rows, pos0, n_heads, n_kv, head_dim, cap, scale, stream);
}

int q4_prompt_attention_bf16_dev(const float* q, const uint16_t* k_cache, const uint16_t* v_cache, uint16_t* out,
                                 int rows, int64_t pos0, int n_heads, int n_kv, int head_dim, int cap, float scale,
                                 void* stream) {
    return prompt_attention(q, k_cache, v_cache, out, true, rows, pos0, n_heads, n_kv, head_dim, cap, scale, stream);
}

}  // extern "C"
#pragma GCC visibility pop
