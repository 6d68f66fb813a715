// matmul_q8.hip -- W8A32 GEMM (prefill) for gfx950 on the matrix cores:
// out[n, m] = (sum_k a[n, k] * q[m, k]) * s[m], a f32 [N, K] (tokens),
// weight [M, ceil(K/4)] packed int8 (matvecQ8's wire format), out f32 [N, M].
//
// Reference: ops/matmul/reference.ts:124-137 (matmulQ8) -- the reference
// dequantizes each weight term to f32 (fround(q * s)) and runs the f64 triple
// loop of matmul (:37-49); its own doc defines the op as "N independent
// matvecQ8 calls against the same weight" (:76-77).  This kernel computes
// that matvecQ8 form: the exact dot product of codes and activations, then
// the row scale once.  Against the reference's per-term form the two differ
// by at most one f32 rounding of each term, 2^-24 of sum |a * q * s|, far
// inside the 1e-5 bar the tests hold.
//
// Numerics on the f16 matrix cores: a code q in [-128, 127] is exact in f16;
// an activation, scaled by its token's power of two, becomes a pair of f16 h +
// l / 2048, every product q * part is exact in f32, and
// v_mfma_f32_16x16x32_f16 sums the two planes in two f32 accumulators.  Each
// 1024-code slice of K is summed there (32 accumulations a plane) and then
// folded into an outer f32 sum, so no rounding chain exceeds 32 + K/1024 steps.
// Against 64 bits, 2-norm: 1.7e-7 at K = 2048 to 5632, where three bf16 parts
// in one accumulator (96 accumulations per fold) had 3.1e-7; and a third less
// matrix work, LDS traffic and splitting.
//
// What the pair holds of one activation: 2^-23 of it at worst (two 11-bit parts
// and the sign between them: a quarter of all f32 values lose their last bit)
// from 2^-22 of the token's largest value up, and 2^-45 of the largest one below
// (the parts turn subnormal).  A token's power of two starts from its first 64
// codes and falls when a larger value comes (rescale_split): the waves multiply
// their accumulators by the ratio, exactly, so the time hardly depends on the
// values and a token's sums depend on no other token.  The values below that
// window only matter to a weight row that has no code at the larger ones:
// small_sums takes sums that are small enough for it again, from an exact
// three-part bf16 split.
//
// Tiling (matmul_q8_kernel, short prompts): a workgroup of two K groups of 8
// waves (2 over the weight rows x 4 over the tokens) owns BM = 32 FB weight
// rows x BN = 64 tokens and walks K in steps of 64 codes.  Each step, the
// threads load the tile's packed codes (one dwordx4 of 16 codes per chunk) and
// activations (8 consecutive k of one token per thread), convert them once into
// LDS, and after one barrier every wave reads its operand fragments with
// ds_read_b128.  The LDS holds two stages: while a wave's matrix cores work on
// step i, its VALU converts step i + 1 into the other stage, and global loads
// run four steps ahead of their conversion.  Rows of 64 codes (128 bytes of
// f16) are stored with their 16-byte pieces swizzled by row (piece_offset).
//
// Operand layout of v_mfma_f32_16x16x32_{f16,bf16} (probed on gfx950): A lane l
// holds A[l % 16][8 (l / 16) + e], B lane l holds B[8 (l / 16) + e][l % 16],
// C lane l holds C[4 (l / 16) + v][l % 16].  A = weight rows (16 features),
// B = activations (16 tokens), so a lane's C values are 4 consecutive
// features of one token: one 16-byte store into out[token, :].
//
// Workgroups are numbered so that the 8 XCDs (which take workgroups
// round-robin) each hold a contiguous run of the tile sequence, and the
// sequence walks groups of 4 weight-row tiles, each group through all its
// token tiles (tile_coords).  So an XCD's L2 holds about an eighth of the
// weight, reused by every token tile, and its resident workgroups share 4
// weight tiles and a few activation tiles.  A token-major sequence (each XCD
// one token tile and every weight row) streamed the whole weight through
// every XCD's L2: 512-token layer 215 -> 182 us, 2048 tokens 629 -> 570.
//
// With a caller's workspace, a short prompt's launch, whose tiles would leave most
// CUs idle, may also split the tiles' K steps between 2, 4 or 8 workgroups: part 0
// stores its unscaled sums into the output, the other parts into tile-sized
// workspace blocks, and a second launch adds them in part order
// and scales them.  The stream order between the two launches is the only
// synchronisation, so every run gives the same bits.
//
// Launches with enough tiles for one workgroup per CU, and short prompts'
// 256-row tiles split 4 or 8 ways, run matmul_q8_direct_kernel instead: every
// wave owns 32 or 48 weight rows and all 64 tokens of the tile, and loads its
// rows' codes straight into VGPRs (one dwordx4 per 16-row block and step), so
// only the activation pairs pass through LDS.
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <type_traits>

#include "kernels.hpp"
#include "wave_ops.hpp"

namespace wxo {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2v __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));

constexpr uint32_t kBN = 64;            // tokens per workgroup
constexpr uint32_t kFoldCodes = 1024;   // fold the accumulator every 1024 codes
constexpr uint32_t kMaxMatmulProjections = 4;

// Up to four projections of the same activations in one launch: projection p
// owns weight-row tiles [mt0[p], mt0[p + 1]) of the launch's tile sequence
// (mt0[p] = 0xffffffff past the last one).  A split launch splits the K steps of
// its `tiles` tiles into `parts` runs, one workgroup each: part 0 stores its
// unscaled sums into the output, part j >= 1 into the workspace block (j - 1) *
// tiles + tile of BM x kBN floats ([token][row] within the tile), and
// split_sum_kernel adds the parts in part order and scales them.
struct MatmulProjections {
    const uint32_t* weight[kMaxMatmulProjections];
    const float* scale[kMaxMatmulProjections];
    float* out[kMaxMatmulProjections];
    uint32_t M[kMaxMatmulProjections];
    uint32_t mt0[kMaxMatmulProjections];
    float* part;
    uint32_t tiles, parts;
};

// Tile `tile` of the launch's sequence -> weight-row tile mt, token tile nt.
// The sequence takes kTileGroup row tiles at a time (fewer in the last
// group) and walks all token tiles of the group, its row tiles innermost:
// consecutive workgroups share activation tiles, and a group's weight tiles
// stay in one XCD's L2 while all token tiles use them.  Same-process sweep of
// the group size (1, 2, 4, 8, 16, all): 512-token layer 182 / 181 / 182 / 187
// / 199 / 215 us, 2048 tokens 574 / 573 / 570 / 572 / 581 / 629.
constexpr uint32_t kTileGroup = 4;
__device__ __forceinline__ void tile_coords(uint32_t tile, uint32_t mtiles, uint32_t ntiles, uint32_t& mt,
                                            uint32_t& nt) {
    const uint32_t gi = tile / (kTileGroup * ntiles), first = gi * kTileGroup;
    const uint32_t gs = min(kTileGroup, mtiles - first);
    const uint32_t r = tile - gi * (kTileGroup * ntiles);
    nt = r / gs;
    mt = first + (r - nt * gs);
}

__device__ __forceinline__ uint32_t hi_pair(uint32_t a, uint32_t b) {
    // upper halves of two f32 bit patterns, a in the low half
    return __builtin_amdgcn_perm(b, a, 0x07060302u);
}

// 4 codes (a packed word) -> 4 f16, exactly: code + 128 is the low byte of the
// f16 1024 + (code + 128), so a byte permute and one packed add convert two
// codes (2.5 VALU ops per two codes; through f32 and bf16 it was 3).
__device__ __forceinline__ void codes4_to_f16(uint32_t w, uint32_t& lo, uint32_t& hi) {
    const f16x2 bias = {(_Float16)-1152.0f, (_Float16)-1152.0f};
    const uint32_t u = w ^ 0x80808080u;
    lo = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + bias);
    hi = __builtin_bit_cast(uint32_t, __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + bias);
}

// 16 codes (4 packed words) -> 16 f16 in two 16-byte pieces.
__device__ __forceinline__ void codes16_to_f16(u32x4v w, u32x4v& lo, u32x4v& hi) {
    uint32_t r[8];
    codes4_to_f16(w.x, r[0], r[1]);
    codes4_to_f16(w.y, r[2], r[3]);
    codes4_to_f16(w.z, r[4], r[5]);
    codes4_to_f16(w.w, r[6], r[7]);
    lo = u32x4v{r[0], r[1], r[2], r[3]};
    hi = u32x4v{r[4], r[5], r[6], r[7]};
}

// 8 codes (2 packed words) -> 8 f16.
__device__ __forceinline__ f16x8 codes8_to_f16(uint32_t w0, uint32_t w1) {
    uint32_t r[4];
    codes4_to_f16(w0, r[0], r[1]);
    codes4_to_f16(w1, r[2], r[3]);
    return __builtin_bit_cast(f16x8, u32x4v{r[0], r[1], r[2], r[3]});
}

// 8 codes (2 packed words) -> 8 bf16 (the exact three-part step only).
__device__ __forceinline__ bf16x8 codes8_to_bf16(u32x2v w) {
    const uint32_t ws[2] = {w.x, w.y};
    uint32_t r[4];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const float c0 = (float)(int8_t)(ws[q]);
        const float c1 = (float)(int8_t)(ws[q] >> 8);
        const float c2 = (float)(int8_t)(ws[q] >> 16);
        const float c3 = (float)((int32_t)ws[q] >> 24);
        r[2 * q] = hi_pair(__float_as_uint(c0), __float_as_uint(c1));
        r[2 * q + 1] = hi_pair(__float_as_uint(c2), __float_as_uint(c3));
    }
    return __builtin_bit_cast(bf16x8, u32x4v{r[0], r[1], r[2], r[3]});
}

// Where 16-byte piece p (8 codes or activations) of a 128-byte LDS row sits:
// even pieces in the first half and odd ones in the second, so that the four
// lane groups of a fragment read (pieces 2 g + h, g = 0 .. 3) find theirs side
// by side, then XOR-swizzled by row.  Reads and writes are then free of bank
// conflicts (p ^ row alone cost a fifth of the 2048-token launch's cycles).
__device__ __forceinline__ uint32_t piece_offset(uint32_t p, uint32_t row) {
    return ((((p & 1u) << 2) | (p >> 1)) ^ (row & 7u)) * 16u;
}

// Two activations -> their f16 pairs.  t = x * up (up the token's power of two,
// exact), h = f16(t) and l = f16(2048 (t - h)), both rounded to nearest: t - h is
// exact, so h + l / 2048 is t to 2^-23 of it for 2^-13 <= |t| <= 65504, and to
// 2^-36 below.  hi collects the largest |t|.
constexpr float kPartScale = 2048.0f;
constexpr float kPartMax = 65504.0f;
__device__ __forceinline__ void split2(float x0, float x1, float up, uint32_t& h, uint32_t& l, float& hi) {
    const float t0 = x0 * up, t1 = x1 * up;
    const f16x2 hp = __builtin_convertvector((f32x2v){t0, t1}, f16x2);
    const float r0 = __builtin_fmaf(x0, up, -(float)hp.x), r1 = __builtin_fmaf(x1, up, -(float)hp.y);
    const f16x2 lp = __builtin_convertvector((f32x2v){r0 * kPartScale, r1 * kPartScale}, f16x2);
    h = __builtin_bit_cast(uint32_t, hp);
    l = __builtin_bit_cast(uint32_t, lp);
    hi = __builtin_fmaxf(__builtin_fmaxf(__builtin_fabsf(t0), __builtin_fabsf(t1)), hi);
}

// A token's power of two 2^(127 - c) stands as the byte c, the exponent field of
// its inverse.  c = kNoValue: nothing above 2^-113 seen yet.
constexpr uint32_t kNoValue = 1u;
constexpr int kTopExponent = 9;  // a new power takes the largest value to [2^9, 2^10): 64 to 128 times of room
__device__ __forceinline__ float up_of(uint32_t c) { return __uint_as_float((254u - c) << 23); }
__device__ __forceinline__ float down_of(uint32_t c) { return __uint_as_float(c << 23); }
__device__ __forceinline__ uint32_t code_of(float up) { return 254u - (__float_as_uint(up) >> 23); }

// The power of two for a token whose largest value is `most`.
__device__ __forceinline__ float up_for(float most) {
    const int c = (int)(__float_as_uint(most) >> 23) - kTopExponent;
    return up_of(c > (int)kNoValue ? (uint32_t)c : kNoValue);
}

// The largest of a token's values (not negative) over its 8 lanes.
__device__ __forceinline__ float token_max(float v) {
    uint32_t b = __float_as_uint(v);
    b = max(b, partner_u32<1>(b));
    b = max(b, partner_u32<2>(b));
    return __uint_as_float(max(b, partner_u32<4>(b)));
}

// A token's first power of two, from its first 64 activations (an infinity among
// them leaves it to rescale_split).
__device__ __forceinline__ float first_up(const uint32_t (&v)[8]) {
    float most = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) most = __builtin_fmaxf(most, __builtin_fabsf(__uint_as_float(v[e])));
    most = token_max(most);
    return most <= 3.402823466e38f ? up_for(most) : up_of(kNoValue);
}

// True (wave-uniform) if a value of the wave passes its token's window.
__device__ __forceinline__ bool past_window(float hi) {
    return __builtin_amdgcn_ballot_w64(!(hi <= kPartMax)) != 0;
}

// Then the pairs again, written over the first ones so that the conversion stays
// free of the branch (and under the matrix work): a token (8 lanes side by side)
// whose largest finite value passes 65504 gets its new power of two, and an
// infinity is h itself, beside l = 0.
__device__ __forceinline__ void rescale_split(const uint32_t (&v)[8], float& up, uint8_t* w, uint32_t plane) {
    uint32_t hp[4], lp[4];
    float most = 0.0f, hi = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const uint32_t b = v[e] & 0x7fffffffu;
        most = __builtin_fmaxf(most, b == 0x7f800000u ? 0.0f : __uint_as_float(b));
    }
    most = token_max(most);
    if (most * up > kPartMax) up = up_for(most);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const uint32_t a = v[2 * e], b = v[2 * e + 1];
        const bool ai = (a & 0x7fffffffu) == 0x7f800000u, bi = (b & 0x7fffffffu) == 0x7f800000u;
        split2(ai ? 0.0f : __uint_as_float(a), bi ? 0.0f : __uint_as_float(b), up, hp[e], lp[e], hi);
        if (ai) hp[e] |= 0x7c00u | ((a >> 16) & 0x8000u);
        if (bi) hp[e] |= 0x7c000000u | (b & 0x80000000u);
    }
    *reinterpret_cast<u32x4v*>(w) = u32x4v{hp[0], hp[1], hp[2], hp[3]};
    *reinterpret_cast<u32x4v*>(w + plane) = u32x4v{lp[0], lp[1], lp[2], lp[3]};
}

// What the converting waves tell the others of a K group, for the last four
// steps: [step][8 tokens] whether a power of two may have changed at the step,
// and then (at step 0 always) the tokens' codes.
struct TokenScales {
    uint8_t changed[4][8];
    uint8_t code[4][kBN];
};

// The pairs of a wave's 8 tokens, 8 activations v a lane, are in LDS at `w` and
// `w + plane`, the largest of them hi: makes them again if one passes its token's
// window, and notes that for step `step` (every lane the same byte: one lane's store
// alone is a branch, and with the read of it after the fragments' 2048 x 2048 x 5632
// takes 97.2 us for 99.4, 512 x 6144 x 2048 34.4 for 35.4).
__device__ __forceinline__ void settle(const uint32_t (&v)[8], float hi, float& up, uint8_t* w, uint32_t plane,
                                       TokenScales& sc, uint32_t step, uint32_t token) {
    const bool out = past_window(hi);
    if (__builtin_expect(out, 0)) {
        rescale_split(v, up, w, plane);
        sc.code[step % 4u][token] = (uint8_t)code_of(up);  // the token's 8 lanes alike
    }
    sc.changed[step % 4u][token >> 3] = out ? 1u : 0u;
}

// Eight consecutive activations of one token -> their pairs in LDS.
__device__ __forceinline__ void store_split(const uint32_t (&v)[8], float& up, uint8_t* w, uint32_t plane,
                                            TokenScales& sc, uint32_t step, uint32_t token) {
    uint32_t hp[4], lp[4];
    float hi = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) split2(__uint_as_float(v[2 * e]), __uint_as_float(v[2 * e + 1]), up, hp[e], lp[e], hi);
    *reinterpret_cast<u32x4v*>(w) = u32x4v{hp[0], hp[1], hp[2], hp[3]};
    *reinterpret_cast<u32x4v*>(w + plane) = u32x4v{lp[0], lp[1], lp[2], lp[3]};
    settle(v, hi, up, w, plane, sc, step, token);
}

// The first step's, with the tokens' first powers of two and their codes.
__device__ __forceinline__ void store_first(const uint32_t (&v)[8], float& up, uint8_t* w, uint32_t plane,
                                            TokenScales& sc, uint32_t token) {
    up = first_up(v);
    store_split(v, up, w, plane, sc, 0u, token);
    sc.code[0][token] = (uint8_t)code_of(up);
}

// The accumulators' factor when a token's code goes from `was` to `now` (>= was).
__device__ __forceinline__ float scale_ratio(uint32_t was, uint32_t now) {
    const int e = 127 + (int)was - (int)now;
    return __uint_as_float((uint32_t)(e > 1 ? e : 1) << 23);  // never 0: an infinite sum stays infinite
}

// Three bf16 parts of an activation, exactly, whatever its exponent: h keeps
// the top 8 significant bits by truncation, m the next 8, l the rest (r = a -
// h and r - m are exact).  A non-finite value keeps all of itself in h (a NaN
// canonicalised, so truncating its payload cannot make it Inf) and m = l = 0,
// so Inf reaches the products as IEEE arithmetic has it.
__device__ __forceinline__ void split3_any(uint32_t bits, uint32_t& h, uint32_t& m, uint32_t& l) {
    const bool finite = (bits & 0x7f800000u) != 0x7f800000u;
    const bool nan = (bits & 0x7fffffffu) > 0x7f800000u;
    const uint32_t hf = bits & 0xffff0000u;
    const float r = finite ? __uint_as_float(bits) - __uint_as_float(hf) : 0.0f;
    h = finite ? hf : (nan ? 0x7fc00000u : bits);
    m = __float_as_uint(r) & 0xffff0000u;
    l = __float_as_uint(r - __uint_as_float(m));
}

// 0 for a block's sums, and infinity for those of rows past the tile's, which
// small_sums then leaves alone (they are not stored).
__device__ __forceinline__ f32x4 no_sums(uint32_t row, uint32_t mrows) {
    f32x4 s;
#pragma unroll
    for (uint32_t v = 0; v < 4u; ++v) s[v] = row + v < mrows ? 0.0f : __builtin_inff();
    return s;
}

// Steps between folds of a run of `steps`: kFoldCodes' worth, and half of a run
// that is no longer than that (in whole multiples of U), for smallest_of.  Only
// where the sums are in registers: the second fold of sums in LDS costs what the
// sums taken again do (1098 x 7216 x 896 52.1 us with it, 51.8 without).
template <uint32_t U>
__device__ __forceinline__ uint32_t fold_steps(uint32_t steps) {
    constexpr uint32_t full = kFoldCodes / 64u;
    return steps > full ? full : ((steps + 1u) / 2u + U - 1u) / U * U;
}

// min(least, |now|) over a block's sums, or of the larger of |was| and |now|: for
// small_sums, a sum after the last fold and, where there are two, before it
// (either shows that its products are large enough, so that then next to none is
// small by cancellation).
__device__ __forceinline__ float smallest_of(f32x4 was, f32x4 now, bool two, float least) {
    float m[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) m[v] = two ? __builtin_fmaxf(__builtin_fabsf(was[v]), __builtin_fabsf(now[v])) : __builtin_fabsf(now[v]);
    return __builtin_fminf(__builtin_fminf(__builtin_fminf(m[0], m[1]), __builtin_fminf(m[2], m[3])), least);
}

// sum += (acc + accl / 2048) * down, and both accumulators start again.
__device__ __forceinline__ void fold(f32x4& sum, f32x4& acc, f32x4& accl, float down) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const float p = __builtin_fmaf(accl[v], 1.0f / kPartScale, acc[v]);
        sum[v] = __builtin_fmaf(p, down, sum[v]);
    }
    acc = f32x4{0.f, 0.f, 0.f, 0.f};
    accl = f32x4{0.f, 0.f, 0.f, 0.f};
}

// The sums of a wave's FW x TB blocks over its run of `gs` steps from step s0,
// where the pairs might not hold what they came from.  A pair is off by 2^-36 /
// up at most where it is off by more than 2^-23 of its value, so a sum of n
// products by 128 n 2^-36 / up: less than 2^-17 of the sum of the products'
// sizes unless that is below n 2^-12 / up.  A sum that is not that small itself
// passes; the others (about one in 10^7 of an ordinary prompt's, by
// cancellation) are taken again here, straight from memory with the activations
// in three exact parts, until the products' sizes add up to enough, which the
// first step shows, or to the end: rows whose only codes meet values far below
// the token's largest.  smallest[b]: the lane's smallest_of its token b;
// code(b): that token's code; get and put: a block's sums.
template <int FW, int TB, typename Code, typename Get, typename Put>
__device__ __forceinline__ void small_sums(const float (&smallest)[TB], __amdgpu_buffer_rsrc_t wrs,
                                           __amdgpu_buffer_rsrc_t ars, uint32_t wm, uint32_t wn, uint32_t rowbytes,
                                           uint32_t K, uint32_t s0, uint32_t gs, Code&& code, Get&& get, Put&& put) {
    const uint32_t lane = __lane_id(), j = lane & 15u, g = lane >> 4;
    // n 2^-12 / up, and 0 for a token without values (down_of(c - 1) is half of down_of(c) but for c = 1)
    const float per = (float)(gs * 64u) * 0.00048828125f;
    const auto least_of = [&](int b) { return per * down_of(code(b) - kNoValue); };
    bool any = false;
#pragma unroll
    for (int b = 0; b < TB; ++b) any |= smallest[b] < least_of(b);
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(any) == 0, 1)) return;
    uint32_t todo = 0u;  // bit f * TB + b: the block has such a sum
#pragma unroll
    for (int f = 0; f < FW; ++f)
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            const f32x4 y = get(f, b);
            const float least = least_of(b);
            bool small = false;
#pragma unroll
            for (int v = 0; v < 4; ++v)
                small |= __builtin_fabsf(y[v]) < least;
            todo |= __builtin_amdgcn_ballot_w64(small) != 0 ? 1u << (f * TB + b) : 0u;
        }
#pragma unroll 1
    while (todo != 0u) {  // wave-uniform
        const uint32_t at = (uint32_t)__builtin_ctz(todo);
        todo &= todo - 1u;
        f32x4 y = {0.f, 0.f, 0.f, 0.f};
        float least = 0.0f;
#pragma unroll
        for (int i = 0; i < FW * TB; ++i)
            if (at == (uint32_t)i) {
                y = get(i / TB, i % TB);
                least = least_of(i % TB);
            }
        const uint32_t row0 = wm + 16u * (at / (uint32_t)TB);
        const uint32_t tk = wn + 16u * (at % (uint32_t)TB) + j;
        uint32_t left = 0u;  // bit v: sum v of the lane is to be taken again
#pragma unroll
        for (uint32_t v = 0; v < 4u; ++v)
            left |= (__builtin_fabsf(y[v]) < least ? 1u : 0u) << v;
        f32x4 size = {0.f, 0.f, 0.f, 0.f}, part = size, total = size;
#pragma unroll 1
        for (uint32_t st = 0; st < gs; ++st) {
            const uint32_t k0 = (s0 + st) * 64u + 16u * g;
            uint32_t x[16];
            u32x2v w[2];
#pragma unroll
            for (uint32_t q = 0; q < 4u; ++q) {
                const u32x4v t = __builtin_amdgcn_raw_buffer_load_b128(ars, (int)((tk * K + k0 + 4u * q) * 4u), 0, 0);
                x[4u * q] = t.x; x[4u * q + 1u] = t.y; x[4u * q + 2u] = t.z; x[4u * q + 3u] = t.w;
            }
#pragma unroll
            for (uint32_t h = 0; h < 2u; ++h)
                w[h] = __builtin_bit_cast(u32x2v, __builtin_amdgcn_raw_buffer_load_b64(
                    wrs, (int)((row0 + j) * rowbytes + k0 + 8u * h), 0, 0));
#pragma unroll
            for (uint32_t e = 0; e < 16u; ++e)
                if (k0 + e >= K) x[e] = 0u;  // the next token's
#pragma unroll
            for (uint32_t h = 0; h < 2u; ++h) {
                uint32_t hp[4], mp[4], lp[4];
#pragma unroll
                for (uint32_t e = 0; e < 4u; ++e) {
                    uint32_t h0, m0, l0, h1, m1, l1;
                    split3_any(x[8u * h + 2u * e], h0, m0, l0);
                    split3_any(x[8u * h + 2u * e + 1u], h1, m1, l1);
                    hp[e] = hi_pair(h0, h1);
                    mp[e] = hi_pair(m0, m1);
                    lp[e] = hi_pair(l0, l1);
                }
                const bf16x8 q = codes8_to_bf16(w[h]);
                const u32x4v qa = __builtin_bit_cast(u32x4v, q) & 0x7fff7fffu, xa = u32x4v{hp[0], hp[1], hp[2], hp[3]} & 0x7fff7fffu;
                size = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, qa), __builtin_bit_cast(bf16x8, xa), size, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q, __builtin_bit_cast(bf16x8, u32x4v{hp[0], hp[1], hp[2], hp[3]}), part, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q, __builtin_bit_cast(bf16x8, u32x4v{mp[0], mp[1], mp[2], mp[3]}), part, 0, 0, 0);
                part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q, __builtin_bit_cast(bf16x8, u32x4v{lp[0], lp[1], lp[2], lp[3]}), part, 0, 0, 0);
            }
            if (st % (kFoldCodes / 64u) == kFoldCodes / 64u - 1u || st + 1u == gs) {
                total += part;
                part = f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (uint32_t v = 0; v < 4u; ++v)
                if (size[v] >= least) left &= ~(1u << v);
            if (st == 0u && __builtin_amdgcn_ballot_w64(left != 0u) != 0) {
                // rows without any code need not be walked to the end
                uint32_t any = 0u;
#pragma unroll 4
                for (uint32_t q = 0; q < gs; ++q) {
                    const uint32_t k = (s0 + q) * 64u + 16u * g;
                    const u32x4v c = __builtin_amdgcn_raw_buffer_load_b128(wrs, (int)((row0 + j) * rowbytes + k), 0, 0);
#pragma unroll
                    for (uint32_t e = 0; e < 4u; ++e) any |= k + 4u * e < rowbytes ? c[e] : 0u;
                }
                uint64_t rows = __builtin_amdgcn_ballot_w64(any != 0u);
                rows |= rows >> 32;
                rows |= rows >> 16;
                left &= (uint32_t)rows >> (4u * g);  // row 4 g + v of the block
            }
            if (__builtin_amdgcn_ballot_w64(left != 0u) == 0) break;
        }
#pragma unroll
        for (int i = 0; i < FW * TB; ++i)
            if (at == (uint32_t)i) {
                f32x4 z = y;
#pragma unroll
                for (uint32_t v = 0; v < 4u; ++v)
                    if ((left >> v) & 1u) z[v] = total[v];
                put(i / TB, i % TB, z);
            }
    }
}

// SPLIT instances take the split launch above.
template <int FB, int NW, int BK, int PD, int KS, bool SPLIT = false>
__global__ __launch_bounds__(64 * NW * KS, 4) void matmul_q8_kernel(const float* __restrict__ a, MatmulProjections P,
                                                        uint32_t N, uint32_t K, uint32_t W, uint32_t mtiles,
                                                        uint32_t ntiles) {
    constexpr uint32_t BM = 32u * FB;                 // weight rows per workgroup
    constexpr uint32_t kBK = (uint32_t)BK;            // codes per K step
    constexpr uint32_t kRowBytes = kBK * 2u;          // one LDS row: BK f16
    constexpr uint32_t CPR = kBK / 16u;               // 16-code chunks per row and step
    constexpr uint32_t AST = BM * kRowBytes;          // bytes of one A stage
    constexpr uint32_t BST = 2u * kBN * kRowBytes;    // bytes of one B stage (two planes)
    constexpr uint32_t NT = 64u * NW;                 // threads of one K group
    constexpr uint32_t ACH = BM * CPR;                // 16-code chunks of A per step
    constexpr int AL = (int)((ACH + NT - 1u) / NT);   // A loads per thread per step
    constexpr uint32_t FPT = kBK / NW;                // activations per thread per step
    constexpr int BL = (int)(FPT / 4u);               // B loads (dwordx4) per thread per step
    constexpr uint32_t WR = 2u;                        // waves over the rows
    constexpr int TB = (int)(4u * WR / NW);            // 16-token blocks per wave (2 or 1)
    constexpr int FW = (int)(BM / (16u * WR));         // 16-row blocks per wave
    static_assert(NW == 8 && BK == 64, "a wave converts 8 tokens of a 64-code step, 8 activations a thread");
    static_assert(PD == 2 || PD == 4, "2 or 4 register sets of loads in flight");
    static_assert(KS == 1 || KS == 2, "K split over 1 or 2 groups of NW waves");
    // Per K group: [A0 A1 B0 B1]
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ __attribute__((aligned(8))) TokenScales scales[KS];

    // XCD-aware tile order: workgroup i runs on XCD i % 8; give each XCD a
    // contiguous run of the tile sequence (tile_coords), of a split launch with a
    // tile's parts side by side.  Workgroups past the end return whole (no
    // barrier is skipped by part of one).
    const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3;
    uint32_t tile, xs = 0u, np = (uint32_t)KS;  // np: runs of this tile's K steps
    if constexpr (!SPLIT) {
        const uint32_t total = mtiles * ntiles;
        const uint32_t lin = xcd * ((total + 7u) / 8u) + slot;
        if (lin >= total) return;
        tile = lin;
    } else {
        const uint32_t all = P.tiles * P.parts, q = xcd * ((all + 7u) / 8u) + slot;
        if (q >= all) return;
        tile = q / P.parts;
        xs = q % P.parts;
        np = (uint32_t)KS * P.parts;
    }
    uint32_t mt, nt;
    tile_coords(tile, mtiles, ntiles, mt, nt);
    // the projection that owns weight-row tile mt (wave-uniform)
    const uint32_t pj = (mt >= P.mt0[1] ? 1u : 0u) + (mt >= P.mt0[2] ? 1u : 0u) + (mt >= P.mt0[3] ? 1u : 0u);
    const uint32_t* __restrict__ weight = P.weight[pj];
    const float* __restrict__ scale = P.scale[pj];
    float* __restrict__ out = P.out[pj];
    const uint32_t M = P.M[pj];
    const uint32_t m0 = (mt - P.mt0[pj]) * BM, n0 = nt * kBN;

    // KS groups of NW waves share the tile and split its K steps in halves;
    // their sums meet in LDS at the end.
    const uint32_t kg = KS == 1 ? 0u : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    const uint32_t gbase = kg * (2u * AST + 2u * BST);  // this group's stages (0 for KS = 1)
    const uint32_t t = KS == 1 ? threadIdx.x : threadIdx.x % NT;
    const uint32_t lane = t & 63u;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t wm = (wv % WR) * (BM / WR);                  // wave's first weight row in the tile
    const uint32_t wn = (wv / WR) * (16u * (uint32_t)TB);       // wave's first token in the tile
    const uint32_t j = lane & 15u, g = lane >> 4;

    const uint32_t mrows = min(BM, M - m0);
    const uint32_t ntok = min(kBN, N - n0);
    const uint32_t rowbytes = W * 4u;
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(weight + (size_t)m0 * W, mrows * rowbytes);
    const __amdgpu_buffer_rsrc_t ars = make_rsrc(a + (size_t)n0 * K, ntok * K * 4u);

    // Global load assignment.  A: thread t, load u -> chunk t + NT u: row
    // chunk / 4, codes 16 (chunk % 4) .. +15 of the step (threads past the
    // tile's chunks load nothing; with BM = 64 and 8 waves that is waves 4-7,
    // a wave-uniform split).  B: token t / NW, k FPT (t % NW) .. +FPT-1.
    const uint32_t ac = t % CPR;
    const uint32_t ar = t / CPR;
    const uint32_t btok = t / NW;
    const uint32_t bc = t % NW;
    const int boff = (int)((btok * K + bc * FPT) * 4u);

    // PD register sets of global loads: step i's data sits in set i % PD,
    // loaded PD steps ahead of its conversion.
    u32x4v ga[PD][AL], gb[PD][BL];
    auto issue = [&](int b, uint32_t k0) {
#pragma unroll
        for (int u = 0; u < AL; ++u)
            if (ACH % NT == 0u || t + NT * (uint32_t)u < ACH)  // wave-uniform
                ga[b][u] = load_nt_b128(wrs, (int)((ar + (NT / CPR) * (uint32_t)u) * rowbytes + ac * 16u), (int)k0);
#pragma unroll
        for (int q = 0; q < BL; ++q)
            gb[b][q] = __builtin_amdgcn_raw_buffer_load_b128(ars, boff + 16 * q, (int)(k0 * 4u), 0);
    };

    // Zeroes, in register set s, the activations at k >= K of step k0 (they
    // belong to the next token).  Only the last step of a ragged K needs it;
    // the caller branches before the matrix work, so the conversion that
    // follows stays in one block with it.
    auto mask_b = [&](int s, uint32_t k0) {
        const uint32_t kb = k0 + bc * FPT;
#pragma unroll
        for (int q = 0; q < BL; ++q) {
            if (kb + 4u * (uint32_t)q >= K) gb[s][q].x = 0u;
            if (kb + 4u * (uint32_t)q + 1u >= K) gb[s][q].y = 0u;
            if (kb + 4u * (uint32_t)q + 2u >= K) gb[s][q].z = 0u;
            if (kb + 4u * (uint32_t)q + 3u >= K) gb[s][q].w = 0u;
        }
    };
    auto load_b = [&](int s, uint32_t (&v)[FPT]) {
#pragma unroll
        for (int q = 0; q < BL; ++q) {
            v[4 * q] = gb[s][q].x;
            v[4 * q + 1] = gb[s][q].y;
            v[4 * q + 2] = gb[s][q].z;
            v[4 * q + 3] = gb[s][q].w;
        }
    };
    float up = up_of(kNoValue);  // the power of two of this thread's token
    // Writes the converted step into stage st.
    auto convert_store = [&](int s, int st, uint32_t step, auto first) {
        uint8_t* as = lds + gbase + (uint32_t)st * AST;
#pragma unroll
        for (int u = 0; u < AL; ++u) {
            if (!(ACH % NT == 0u || t + NT * (uint32_t)u < ACH)) continue;  // wave-uniform
            const uint32_t r = ar + (NT / CPR) * (uint32_t)u;
            u32x4v lo, hi;
            codes16_to_f16(ga[s][u], lo, hi);
            *reinterpret_cast<u32x4v*>(as + r * kRowBytes + piece_offset(2u * ac, r)) = lo;
            *reinterpret_cast<u32x4v*>(as + r * kRowBytes + piece_offset(2u * ac + 1u, r)) = hi;
        }
        uint32_t v[FPT];
        load_b(s, v);
        uint8_t* row = lds + gbase + 2u * AST + (uint32_t)st * BST + btok * kRowBytes + piece_offset(bc, btok);
        if constexpr (first) store_first(v, up, row, kBN * kRowBytes, scales[kg], btok);
        else store_split(v, up, row, kBN * kRowBytes, scales[kg], step, btok);
    };

    const uint32_t steps = (K + kBK - 1u) / kBK;
    const bool ragged = (K % kBK) != 0u;
    // This group's steps: [s0, s0 + gs), run xs * KS + kg of np; every group
    // runs `iters` iterations (the same barriers), skipping the matrix work
    // past its own steps.
    constexpr bool kOneRun = KS == 1 && !SPLIT;  // every group takes all the steps: no skip
    const uint32_t iters = kOneRun ? steps : (steps + np - 1u) / np;
    const uint32_t s0 = kOneRun ? 0u : (xs * (uint32_t)KS + kg) * iters;
    const uint32_t gs = kOneRun ? steps : (s0 < steps ? min(iters, steps - s0) : 0u);

    f32x4 acc[FW][TB], accl[FW][TB], sum[FW][TB];
#pragma unroll
    for (int f = 0; f < FW; ++f)
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            acc[f][b] = f32x4{0.f, 0.f, 0.f, 0.f};
            accl[f][b] = f32x4{0.f, 0.f, 0.f, 0.f};
            sum[f][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        }

    // Operands of half h (32 codes) of a stage: lane group g takes codes 16 g + 8 h
    // .. +7 of the step (the sum's k order is free; this one is the direct
    // kernel's, whose lanes load 16 consecutive codes).
    auto operands = [&](int s, int h, f16x8 (&af)[FW], f16x8 (&bf)[TB][2]) {
        const uint8_t* as = lds + gbase + (uint32_t)s * AST;
        const uint8_t* bs = lds + gbase + 2u * AST + (uint32_t)s * BST;
        const uint32_t piece = 2u * g + (uint32_t)h;
#pragma unroll
        for (int f = 0; f < FW; ++f) {
            const uint32_t r = wm + 16u * (uint32_t)f + j;
            af[f] = *reinterpret_cast<const f16x8*>(as + r * kRowBytes + piece_offset(piece, r));
        }
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            const uint32_t tk = wn + 16u * (uint32_t)b + j;
#pragma unroll
            for (int p = 0; p < 2; ++p)
                bf[b][p] = *reinterpret_cast<const f16x8*>(bs + ((uint32_t)p * kBN + tk) * kRowBytes +
                                                           piece_offset(piece, tk));
        }
    };
    auto matrix = [&](const f16x8 (&af)[FW], const f16x8 (&bf)[TB][2]) {
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int b = 0; b < TB; ++b)
                acc[f][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[f], bf[b][0], acc[f][b], 0, 0, 0);
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int b = 0; b < TB; ++b)
                accl[f][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[f], bf[b][1], accl[f][b], 0, 0, 0);
    };
    // Matrix work of one stage.  Where a token's power of two changed with this
    // step, the accumulators follow first.
    uint32_t code = kNoValue;  // of this lane's token
    static_assert(TB == 1, "one token per lane");
    auto compute = [&](int s, uint32_t step) {
        const u32x2v changed = *reinterpret_cast<const u32x2v*>(scales[kg].changed[step % 4u]);
        f16x8 af[FW], bf[TB][2];
        operands(s, 0, af, bf);
        const uint32_t c = __builtin_amdgcn_readfirstlane(wn < 32u ? changed.x : changed.y) >> (wn & 16u);
        if (__builtin_expect((c & 0xffffu) != 0u && step != 0u, 0)) {  // wave-uniform
            if ((c >> (j & 8u)) & 1u) {
                const uint32_t now = scales[kg].code[step % 4u][wn + j];
                const float r = scale_ratio(code, now);
                code = now;
#pragma unroll
                for (int f = 0; f < FW; ++f) {
                    acc[f][0] *= r;
                    accl[f][0] *= r;
                }
            }
        }
        matrix(af, bf);
        operands(s, 1, af, bf);
        matrix(af, bf);
    };

    // Software pipeline, one barrier per step: iteration i converts step
    // i + 1 (register set (i + 1) % PD, LDS stage (i + 1) & 1) and refills
    // that set with step i + 1 + PD, then runs step i's matrix work on stage
    // i & 1.  A step's loads thus have PD iterations to arrive.  The
    // conversion (VALU) and the matrix work are independent, so a wave
    // overlaps them.  Past the last step the conversion writes a stage nobody
    // reads and the loads fall outside the buffer resources (they return 0).
#pragma unroll
    for (int q = 0; q < PD; ++q) issue(q, (s0 + (uint32_t)q) * kBK);
    if (ragged && s0 + 1u == steps) mask_b(0, s0 * kBK);
    convert_store(0, 0, 0u, std::true_type{});
    issue(0, (s0 + (uint32_t)PD) * kBK);
    __syncthreads();
    code = scales[kg].code[0][wn + j];
    // The matrix work comes first in program order: its LDS reads then need
    // not wait behind the conversion's LDS writes, and the scheduler can fill
    // the matrix-core latency with the conversion's VALU work.  q = i % PD.
    auto iter = [&](int q, uint32_t i) {
        const int nx = (q + 1) % PD;
        if (ragged && s0 + i + 2u == steps) mask_b(nx, (s0 + i + 1u) * kBK);  // uniform
        if (kOneRun || i < gs) compute(q & 1, i);                              // uniform
        convert_store(nx, (q + 1) & 1, i + 1u, std::false_type{});
        issue(nx, (s0 + i + 1u + (uint32_t)PD) * kBK);
        __syncthreads();
    };
    // Steps run in groups of a multiple of PD, so a group starts on register
    // set 0 and stage 0; the accumulator is folded into the outer sum after
    // each group.
    const uint32_t group = fold_steps<(uint32_t)PD>(iters);
    float smallest[TB] = {__builtin_inff()};  // of this lane's sums, at the last fold
    for (uint32_t g0 = 0; g0 < iters; g0 += group) {
        const uint32_t gend = min(g0 + group, iters);
        uint32_t i = g0;
        for (; i + (uint32_t)PD <= gend; i += (uint32_t)PD) {
#pragma unroll
            for (int q = 0; q < PD; ++q) iter(q, i + (uint32_t)q);
        }
#pragma unroll
        for (int q = 0; q < PD - 1; ++q)
            if (i + (uint32_t)q < gend) iter(q, i + (uint32_t)q);
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                const f32x4 was = sum[f][b];
                fold(sum[f][b], acc[f][b], accl[f][b], down_of(code));
                smallest[b] = smallest_of(was, sum[f][b], true, f == 0 ? __builtin_inff() : smallest[b]);
            }
    }
    if (mrows < BM) {  // uniform
        smallest[0] = __builtin_inff();
#pragma unroll
        for (int f = 0; f < FW; ++f) {
            sum[f][0] += no_sums(wm + 16u * (uint32_t)f + 4u * g, mrows);
            smallest[0] = smallest_of(sum[f][0], sum[f][0], false, smallest[0]);
        }
    }
    small_sums<FW, TB>(smallest, wrs, ars, wm, wn, rowbytes, K, s0, gs, [&](int) { return code; },
                       [&](int f, int b) { return sum[f][b]; }, [&](int f, int b, f32x4 v) { sum[f][b] = v; });

    if constexpr (KS > 1) {
        // Group 1's sums through LDS (its stages are done) into group 0's.
        constexpr uint32_t E = (uint32_t)(FW * TB * 4);
        static_assert(E * NT * 4u <= 2u * AST + 2u * BST, "the reduction fits in group 0's stages");
        float* red = reinterpret_cast<float*>(lds);
        __syncthreads();
        if (kg == 1u) {
#pragma unroll
            for (int f = 0; f < FW; ++f)
#pragma unroll
                for (int b = 0; b < TB; ++b)
#pragma unroll
                    for (int v = 0; v < 4; ++v) red[((uint32_t)((f * TB + b) * 4 + v)) * NT + t] = sum[f][b][v];
        }
        __syncthreads();
        if (kg != 0u) return;  // after the last barrier
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int b = 0; b < TB; ++b)
#pragma unroll
                for (int v = 0; v < 4; ++v) sum[f][b][v] += red[((uint32_t)((f * TB + b) * 4 + v)) * NT + t];
    }

    // Epilogue: lane (j, g) of block (f, b) holds features m0 + wm + 16 f +
    // 4 g .. +3 of token n0 + wn + 16 b + j.  A split tile stores unscaled
    // sums: part 0 into the output, part xs into its workspace block.
    // The lane group is read again: kept from the start it costs the 64-row form on
    // two K groups (128 registers a lane) a spill.
    const uint32_t ge = __lane_id() >> 4;
    const __amdgpu_buffer_rsrc_t srs = make_rsrc(scale + m0, SPLIT ? 0u : mrows * 4u);
    float* const blk = SPLIT && xs > 0u
        ? P.part + ((size_t)(xs - 1u) * P.tiles + tile) * (size_t)(BM * kBN) : nullptr;
#pragma unroll
    for (int f = 0; f < FW; ++f) {
        const uint32_t fm = wm + 16u * (uint32_t)f + 4u * ge;  // within the tile
        const u32x4v sv = SPLIT ? u32x4v{0x3f800000u, 0x3f800000u, 0x3f800000u, 0x3f800000u}  // 1.0f
                                : __builtin_amdgcn_raw_buffer_load_b128(srs, (int)(fm * 4u), 0, 0);
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            const uint32_t tok = wn + 16u * (uint32_t)b + j;
            if (tok >= ntok) continue;
            f32x4 y;
            y[0] = sum[f][b][0] * __uint_as_float(sv.x);
            y[1] = sum[f][b][1] * __uint_as_float(sv.y);
            y[2] = sum[f][b][2] * __uint_as_float(sv.z);
            y[3] = sum[f][b][3] * __uint_as_float(sv.w);
            float* o = blk ? blk + tok * BM + fm : out + (size_t)(n0 + tok) * M + m0 + fm;
            if (fm + 3u < mrows) {
                *reinterpret_cast<f32x4_a4*>(o) = f32x4_a4{y[0], y[1], y[2], y[3]};
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (fm + (uint32_t)q < mrows) o[q] = y[q];
            }
        }
    }
}

// One-group workgroups of 8 waves keep the folded sums in LDS (touched once
// per 1024 codes): the 16 FW registers they would take hold the next step's
// operands instead.
constexpr bool direct_sums_in_lds(int NW, int KS) { return NW == 8 && KS == 1; }

// The GEMM with each wave's weight codes loaded straight into registers.  A
// group of NW waves owns BM = 16 FW NW weight rows x 64 tokens; wave w owns rows
// 16 FW w .. +16 FW - 1 and every token of the tile, so nothing it converts is
// shared and no code passes through LDS.  Per 64-code step, lane (j, g) of a
// 16-row block loads codes 16 g .. +15 of row j, one dwordx4, two steps ahead;
// the activations go through a ring of three LDS stages, split into their f16
// pairs once per group.  KS = 2: two groups share the tile and split its K steps
// in halves (their sums meet in LDS), or, as kTilePairs, each take a tile of
// their own.  kSplitTiles splits the P.tiles tiles' K steps into P.parts runs,
// one workgroup each.  Every form sums a run in the same order, so whole tiles
// have the same bits in all of them.
//
// What bounds it: at 2048 x 2048 x 5632 (256 tiles of 256 rows, one per CU) the
// step takes 1.1 us where its matrix ops alone, at the clock they leave (they
// sustain 1.5 PFLOP/s), take 0.69; loads, split, code conversion and LDS reads
// each add about 0.1 us to that (timing bounds with each taken out).  Two parts
// for three, the ring, and the order below took that shape from 122 to 98 us.
// One wave per SIMD (4 waves of 64 rows: 133), 32x32x16 matrix ops (109), waves
// over 4 x 2 row and token halves (113) and code conversion through masks in
// place of byte permutes (105) are all slower.
enum : int { kWholeTiles = 0, kSplitTiles = 1, kTilePairs = 2 };
template <int NW, int FW, int KS, int MODE>
__global__ __launch_bounds__(64 * NW * KS, 2) void matmul_q8_direct_kernel(const float* __restrict__ a,
                                                                           MatmulProjections P, uint32_t N, uint32_t K,
                                                                           uint32_t W, uint32_t mtiles,
                                                                           uint32_t ntiles) {
    constexpr int TB = 4, NS = 3, PD = 2;             // 16-token blocks per wave, LDS stages, code register sets
    constexpr int CH = 8 / NW;                        // 8-activation chunks a thread converts per step
    constexpr int GB = CH == 1 ? 2 : 1;               // activation register sets
    constexpr uint32_t NT = 64u * NW;                 // threads of one K group
    constexpr uint32_t BM = 16u * FW * NW;
    constexpr uint32_t kRowBytes = 128u;              // one LDS row: 64 codes of f16
    constexpr uint32_t BST = 2u * kBN * kRowBytes;    // one stage: two planes of 64 tokens
    constexpr bool kSumsInLds = direct_sums_in_lds(NW, KS);
    constexpr bool kOneRun = KS == 1 && MODE == kWholeTiles;  // every workgroup takes all the steps
    static_assert(NW == 4 || NW == 8, "whole chunks per thread");
    static_assert(KS == 1 || KS == 2, "one or two K groups");
    static_assert(MODE != kTilePairs || KS == 2, "pairs are the two groups of a workgroup");
    // [stages of group 0][stages of group 1][sums]
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    __shared__ __attribute__((aligned(8))) TokenScales scales[KS];

    // XCD-aware order: workgroup i runs on XCD i % 8; each XCD gets a
    // contiguous run of the tile sequence (tile_coords), of a split launch with a
    // tile's parts side by side.  Workgroups past the end return whole (no barrier
    // is skipped by part of one).
    const uint32_t kg = KS == 1 ? 0u : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    const uint32_t xcd = blockIdx.x & 7u, slot = blockIdx.x >> 3;
    uint32_t tile, xs = 0u, np = (uint32_t)KS;  // np: runs of this tile's K steps
    if constexpr (MODE == kTilePairs) {
        const uint32_t pairs = mtiles * ntiles / 2u;
        const uint32_t i = xcd * ((pairs + 7u) / 8u) + slot;
        if (i >= pairs) return;
        tile = 2u * i + kg;
        np = 1u;
    } else if constexpr (MODE == kWholeTiles) {
        const uint32_t total = mtiles * ntiles;
        tile = xcd * ((total + 7u) / 8u) + slot;
        if (tile >= total) return;
    } else {
        const uint32_t all = P.tiles * P.parts, q = xcd * ((all + 7u) / 8u) + slot;
        if (q >= all) return;
        tile = q / P.parts;
        xs = q % P.parts;
        np = (uint32_t)KS * P.parts;
    }
    uint32_t mt, nt;
    tile_coords(tile, mtiles, ntiles, mt, nt);
    // the projection that owns weight-row tile mt (wave-uniform)
    const uint32_t pj = (mt >= P.mt0[1] ? 1u : 0u) + (mt >= P.mt0[2] ? 1u : 0u) + (mt >= P.mt0[3] ? 1u : 0u);
    const uint32_t* __restrict__ weight = P.weight[pj];
    const float* __restrict__ scale = P.scale[pj];
    float* __restrict__ out = P.out[pj];
    const uint32_t M = P.M[pj];
    const uint32_t m0 = (mt - P.mt0[pj]) * BM, n0 = nt * kBN;

    const uint32_t t = KS == 1 ? threadIdx.x : threadIdx.x % NT, lane = t & 63u;
    const uint32_t wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t wm = wv * (16u * FW);
    const uint32_t j = lane & 15u, g = lane >> 4;
    const uint32_t mrows = min(BM, M - m0), ntok = min(kBN, N - n0);
    const uint32_t rowbytes = W * 4u;
    const __amdgpu_buffer_rsrc_t wrs = make_rsrc(weight + (size_t)m0 * W, mrows * rowbytes);
    const __amdgpu_buffer_rsrc_t ars = make_rsrc(a + (size_t)n0 * K, ntok * K * 4u);
    // this thread converts k 8 bc .. +7 of a step for tokens btok (and btok + 8 NW)
    const uint32_t btok = t >> 3, bc = t & 7u;
    const int boff = (int)((btok * K + bc * 8u) * 4u), bnext = (int)(8u * NW * K * 4u);
    uint8_t* const stages = lds + kg * (NS * BST);
    uint8_t* const brow = stages + btok * kRowBytes + piece_offset(bc, btok);
    f32x4* const lsum = reinterpret_cast<f32x4*>(lds + KS * NS * BST) + t;  // block i of the thread: lsum[i * NT]

    // PD register sets of codes (set i % PD: step i) and GB of activations
    // (step i, converted two steps before its matrix work).
    u32x4v ga[PD][FW];
    u32x4v gb[GB][CH][2];
    const int aoff = (int)((wm + j) * rowbytes + 16u * g);
    auto issue_a = [&](int b, uint32_t k0) {
#pragma unroll
        for (int f = 0; f < FW; ++f)
            ga[b][f] = __builtin_amdgcn_raw_buffer_load_b128(wrs, aoff + (int)(16u * (uint32_t)f * rowbytes), (int)k0, 0);
    };
    auto issue_b = [&](int b, uint32_t k0) {
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
            for (int q = 0; q < 2; ++q)
                gb[b][c][q] = __builtin_amdgcn_raw_buffer_load_b128(ars, boff + c * bnext + 16 * q, (int)(k0 * 4u), 0);
    };
    // activations at k >= K of step k0 belong to the next token: zero
    auto mask_b = [&](int s, uint32_t k0) {
        const uint32_t kb = k0 + bc * 8u;
#pragma unroll
        for (int c = 0; c < CH; ++c)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                if (kb + 4u * (uint32_t)q >= K) gb[s][c][q].x = 0u;
                if (kb + 4u * (uint32_t)q + 1u >= K) gb[s][c][q].y = 0u;
                if (kb + 4u * (uint32_t)q + 2u >= K) gb[s][c][q].z = 0u;
                if (kb + 4u * (uint32_t)q + 3u >= K) gb[s][c][q].w = 0u;
            }
    };
    float up[CH];  // the powers of two of this thread's tokens
    constexpr uint32_t kChunkBytes = 8u * NW * kRowBytes;  // from a thread's token to its next in a stage
    auto take = [&](int s, int c, uint32_t (&v)[8]) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            v[4 * q] = gb[s][c][q].x;
            v[4 * q + 1] = gb[s][c][q].y;
            v[4 * q + 2] = gb[s][c][q].z;
            v[4 * q + 3] = gb[s][c][q].w;
        }
    };
    // The two planes of register set s into the stage at `stage`.
    auto convert_b = [&](int s, uint32_t stage, uint32_t step, auto first) {
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            uint32_t v[8];
            take(s, c, v);
            uint8_t* const w = brow + stage + (uint32_t)c * kChunkBytes;
            const uint32_t token = btok + 8u * NW * (uint32_t)c;
            if constexpr (first) store_first(v, up[c], w, kBN * kRowBytes, scales[kg], token);
            else store_split(v, up[c], w, kBN * kRowBytes, scales[kg], step, token);
        }
    };

    f32x4 acc[FW][TB], accl[FW][TB], sum[kSumsInLds ? 1 : FW][kSumsInLds ? 1 : TB];
#pragma unroll
    for (int f = 0; f < FW; ++f)
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            acc[f][b] = f32x4{0.f, 0.f, 0.f, 0.f};
            accl[f][b] = f32x4{0.f, 0.f, 0.f, 0.f};
            const f32x4 none = no_sums(wm + 16u * (uint32_t)f + 4u * g, mrows);
            if constexpr (kSumsInLds) lsum[(uint32_t)(f * TB + b) * NT] = none;
            else sum[f][b] = none;
        }

    // Activation fragments of plane p of half h of a stage: lane group g takes
    // codes 16 g + 8 h .. +7 of the step, so a lane's 16 consecutive codes feed
    // both halves.
    const uint8_t* const brd0 = stages + j * kRowBytes + piece_offset(2u * g, j);
    const uint8_t* const brd1 = stages + j * kRowBytes + piece_offset(2u * g + 1u, j);
    auto read_b = [&](uint32_t stage, int h, int p, f16x8 (&bf)[TB]) {
#pragma unroll
        for (int b = 0; b < TB; ++b)
            bf[b] = *reinterpret_cast<const f16x8*>((h ? brd1 : brd0) + stage + (uint32_t)p * kBN * kRowBytes +
                                                    16u * (uint32_t)b * kRowBytes);
    };
    auto codes = [&](int q, int h, f16x8 (&af)[FW]) {
#pragma unroll
        for (int f = 0; f < FW; ++f)
            af[f] = h == 0 ? codes8_to_f16(ga[q][f].x, ga[q][f].y) : codes8_to_f16(ga[q][f].z, ga[q][f].w);
    };
    auto matrix = [&](const f16x8 (&af)[FW], const f16x8 (&bf)[TB], f32x4 (&c)[FW][TB]) {
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int b = 0; b < TB; ++b) c[f][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[f], bf[b], c[f][b], 0, 0, 0);
    };
    // One phase's instruction order: its LDS reads under its first matrix ops,
    // VALU work in the shadow of each.
    auto interleave = [&]() {
#pragma unroll
        for (int q = 0; q < FW * TB; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);               // a matrix op
            if (q < TB) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // an LDS read
            __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);               // VALU
        }
        __builtin_amdgcn_sched_barrier(0);
    };

    // This group's steps: [s0, s0 + gs), run xs * KS + kg of np; every group
    // runs `iters` iterations (the same barriers).  Loads past the run read
    // the next run's steps, the next token's or past the buffer (0), all
    // unused.
    const uint32_t steps = (K + 63u) / 64u;
    const bool ragged = (K % 64u) != 0u;
    const uint32_t iters = kOneRun ? steps : (steps + np - 1u) / np;
    const uint32_t s0 = kOneRun || MODE == kTilePairs ? 0u : (xs * (uint32_t)KS + kg) * iters;
    const uint32_t gs = kOneRun ? steps : (s0 < steps ? min(iters, steps - s0) : 0u);

    issue_b(0, 64u * s0);
    if constexpr (GB == 2) issue_b(1, 64u * (s0 + 1u));
#pragma unroll
    for (int q = 0; q < PD; ++q) issue_a(q, 64u * (s0 + (uint32_t)q));
    if (ragged && s0 + 1u == steps) mask_b(0, 64u * s0);
    convert_b(0, 0u, 0u, std::true_type{});
    if constexpr (GB == 2) issue_b(0, 64u * (s0 + 2u));
    else issue_b(0, 64u * (s0 + 1u));
    if (ragged && s0 + 2u == steps) mask_b(GB - 1, 64u * (s0 + 1u));
    convert_b(GB - 1, BST, 1u, std::false_type{});
    if constexpr (GB == 2) issue_b(1, 64u * (s0 + 3u));
    else issue_b(0, 64u * (s0 + 2u));
    __syncthreads();
    // The codes of this lane's tokens 16 b + j, a byte each, and what changes with
    // the next step (a byte per 8 tokens; wave-uniform).
    uint32_t code = 0u, changed0 = 0u, changed1 = 0u;  // (step 0 starts from its codes)
#pragma unroll
    for (int b = 0; b < TB; ++b) code |= (uint32_t)scales[kg].code[0][16u * (uint32_t)b + j] << (8 * b);
    auto code_at = [&](int b) { return (code >> (8 * b)) & 255u; };
    // A token's power of two changed with step `step`: its accumulators follow.
    auto rescale = [&](uint32_t step) {
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            const uint32_t c = ((b < 2 ? changed0 : changed1) >> (16 * (b & 1) + (j & 8u))) & 1u;
            const uint32_t now = c ? (uint32_t)scales[kg].code[step % 4u][16u * (uint32_t)b + j] : code_at(b);
            const float r = scale_ratio(code_at(b), now);
            code = (code & ~(255u << (8 * b))) | now << (8 * b);
#pragma unroll
            for (int f = 0; f < FW; ++f) {
                acc[f][b] *= r;
                accl[f][b] *= r;
            }
        }
    };

    // One barrier per step.  Iteration i works on stage i % NS, written two
    // iterations earlier, so the fragments of its first phase are read before
    // the barrier that starts it: matrix work runs across the barrier.  In
    // the shadow of the matrix ops it converts step i + 2's activations into
    // their stage and the codes of the next half, and refills the registers
    // those came from.  Four phases (half h, plane p), each reading the next
    // one's fragments.
    f16x8 bx[TB], by[TB], ax[FW], ay[FW];
    read_b(0u, 0, 0, bx);
    codes(0, 0, ax);
    uint32_t cur = 0u;  // the stage of step i
    auto iter = [&](int q, uint32_t i) {
        constexpr uint32_t kEnd = (uint32_t)NS * BST;
        const int s = q % GB;
        const uint32_t next = cur + BST == kEnd ? 0u : cur + BST, after = next + BST == kEnd ? 0u : next + BST;
        if (ragged && s0 + i + 3u == steps) mask_b(s, (s0 + i + 2u) * 64u);  // uniform
        if (__builtin_expect((changed0 | changed1) != 0u, 0)) rescale(i);    // uniform
        __builtin_amdgcn_sched_barrier(0);
        uint32_t v[CH][8], hp[CH][4], lp[CH][4];
        float hi[CH];
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            take(s, c, v[c]);
            hi[c] = 0.0f;
        }
        auto split = [&](int e) {  // pair e of the thread's 4 CH
            const int c = e >> 2, k = e & 3;
            split2(__uint_as_float(v[c][2 * k]), __uint_as_float(v[c][2 * k + 1]), up[c], hp[c][k], lp[c][k], hi[c]);
        };
        read_b(cur, 0, 1, by);
        matrix(ax, bx, acc);
        codes(q, 1, ay);
        interleave();
        issue_a(q, (s0 + i + (uint32_t)PD) * 64u);
        read_b(cur, 1, 0, bx);
        matrix(ax, by, accl);
#pragma unroll
        for (int e = 0; e < 2 * CH; ++e) split(e);
        interleave();
        read_b(cur, 1, 1, by);
        matrix(ay, bx, acc);
#pragma unroll
        for (int e = 2 * CH; e < 4 * CH; ++e) split(e);
        interleave();
        uint8_t* const w = brow + after;
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            *reinterpret_cast<u32x4v*>(w + (uint32_t)c * kChunkBytes) = u32x4v{hp[c][0], hp[c][1], hp[c][2], hp[c][3]};
            *reinterpret_cast<u32x4v*>(w + (uint32_t)c * kChunkBytes + kBN * kRowBytes) =
                u32x4v{lp[c][0], lp[c][1], lp[c][2], lp[c][3]};
        }
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            settle(v[c], hi[c], up[c], w + (uint32_t)c * kChunkBytes, kBN * kRowBytes, scales[kg], i + 2u,
                   btok + 8u * NW * (uint32_t)c);
        }
        issue_b(s, (s0 + i + 2u + (uint32_t)GB) * 64u);
        __builtin_amdgcn_sched_barrier(0);
        read_b(next, 0, 0, bx);
        const u32x2v changed = *reinterpret_cast<const u32x2v*>(scales[kg].changed[(i + 1u) % 4u]);
        matrix(ay, by, accl);
        codes(q ^ 1, 0, ax);
#pragma unroll
        for (int f = 0; f < FW; ++f) asm volatile("" : "+v"(ax[f]));  // converted here, not past the barrier
        interleave();
        changed0 = __builtin_amdgcn_readfirstlane(changed.x);
        changed1 = __builtin_amdgcn_readfirstlane(changed.y);
        cur = next;
    };
    float smallest[TB];  // of each of this lane's tokens' sums, at the last fold
#pragma unroll
    for (int b = 0; b < TB; ++b) smallest[b] = __builtin_inff();
    // (a group starts on register set 0; whole tiles fold alike in every form)
    const uint32_t group = KS == 2 && MODE != kTilePairs ? fold_steps<2>(iters) : kFoldCodes / 64u;
    for (uint32_t g0 = 0; g0 < iters; g0 += group) {
        const uint32_t gend = min(g0 + group, iters);
        for (uint32_t i = g0; i < gend; i += 2u) {
            if (kOneRun || i < gs) iter(0, i);  // uniform over the group
            __syncthreads();
            if (i + 1u < gend) {
                if (kOneRun || i + 1u < gs) iter(1, i + 1u);
                __syncthreads();
            }
        }
        if (!kOneRun && g0 >= gs) continue;  // nothing since the last fold
        auto fold_all = [&](auto look) {  // look: smallest_of too, of one fold (1) or two (2)
#pragma unroll
            for (int b = 0; b < TB; ++b) {
                if constexpr (look != 0) smallest[b] = __builtin_inff();
#pragma unroll
                for (int f = 0; f < FW; ++f) {
                    f32x4 v;
                    if constexpr (kSumsInLds) v = lsum[(uint32_t)(f * TB + b) * NT];
                    else v = sum[f][b];
                    const f32x4 was = v;
                    fold(v, acc[f][b], accl[f][b], down_of(code_at(b)));
                    if constexpr (kSumsInLds) lsum[(uint32_t)(f * TB + b) * NT] = v;
                    else sum[f][b] = v;
                    if constexpr (look != 0) smallest[b] = smallest_of(was, v, look == 2, smallest[b]);
                }
            }
        };
        if (g0 + group < gs) fold_all(std::integral_constant<int, 0>{});
        else if (g0 == 0u) fold_all(std::integral_constant<int, 1>{});
        else fold_all(std::integral_constant<int, 2>{});
    }
    auto get = [&](int f, int b) {
        if constexpr (kSumsInLds) return lsum[(uint32_t)(f * TB + b) * NT];
        else return sum[f][b];
    };
    small_sums<FW, TB>(smallest, wrs, ars, wm, 0u, rowbytes, K, s0, gs, code_at, get, [&](int f, int b, f32x4 v) {
        if constexpr (kSumsInLds) lsum[(uint32_t)(f * TB + b) * NT] = v;
        else sum[f][b] = v;
    });

    if constexpr (KS > 1 && MODE != kTilePairs) {
        // group 1's sums through LDS (every stage is done with) into group 0's
        static_assert(!kSumsInLds && (uint32_t)(FW * TB) * NT * 16u <= NS * BST, "the sums fit in group 0's stages");
        f32x4* const red = reinterpret_cast<f32x4*>(lds) + t;
        if (kg == 1u) {
#pragma unroll
            for (int f = 0; f < FW; ++f)
#pragma unroll
                for (int b = 0; b < TB; ++b) red[(uint32_t)(f * TB + b) * NT] = sum[f][b];
        }
        __syncthreads();
        if (kg != 0u) return;  // after the last barrier
#pragma unroll
        for (int f = 0; f < FW; ++f)
#pragma unroll
            for (int b = 0; b < TB; ++b) sum[f][b] += red[(uint32_t)(f * TB + b) * NT];
    }

    // lane (j, g) of block (f, b): rows m0 + wm + 16 f + 4 g .. +3 of token
    // n0 + 16 b + j.  A split tile's parts store unscaled sums: part 0 into
    // the output, part xs into its workspace block ([token][row] in the tile).
    constexpr bool split = MODE == kSplitTiles;
    const __amdgpu_buffer_rsrc_t srs = make_rsrc(scale + m0, split ? 0u : mrows * 4u);
    float* const blk = MODE == kSplitTiles && xs > 0u
        ? P.part + ((size_t)(xs - 1u) * P.tiles + tile) * (size_t)(BM * kBN) : nullptr;
#pragma unroll
    for (int f = 0; f < FW; ++f) {
        const uint32_t fm = wm + 16u * (uint32_t)f + 4u * g;
        const u32x4v sv = split ? u32x4v{0x3f800000u, 0x3f800000u, 0x3f800000u, 0x3f800000u}  // 1.0f
                                : __builtin_amdgcn_raw_buffer_load_b128(srs, (int)(fm * 4u), 0, 0);
#pragma unroll
        for (int b = 0; b < TB; ++b) {
            const uint32_t tok = 16u * (uint32_t)b + j;
            if (tok >= ntok) continue;
            f32x4 y = get(f, b);
            y[0] *= __uint_as_float(sv.x);
            y[1] *= __uint_as_float(sv.y);
            y[2] *= __uint_as_float(sv.z);
            y[3] *= __uint_as_float(sv.w);
            float* o = blk ? blk + tok * BM + fm : out + (size_t)(n0 + tok) * M + m0 + fm;
            if (fm + 3u < mrows) {
                *reinterpret_cast<f32x4_a4*>(o) = f32x4_a4{y[0], y[1], y[2], y[3]};
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (fm + (uint32_t)q < mrows) o[q] = y[q];
            }
        }
    }
}

// out = (part 0 + part 1 + ... + part parts-1) * scale, in part order (up to
// 8 parts), for every output of the split tiles of a split launch.  Grid x: split tile;
// grid y: BM / 16 slices of it; a thread takes 4 consecutive rows of one
// token (one 16-byte group of every part), all its loads in flight at once.
template <uint32_t BM>
__global__ __launch_bounds__(256) void split_sum_kernel(MatmulProjections P, uint32_t N, uint32_t mtiles) {
    constexpr uint32_t G = BM / 4u;  // 4-row groups per token
    static_assert(kBN * G == 256u * (BM / 16u), "one group per thread");
    const uint32_t tile = blockIdx.x;
    uint32_t mt, nt;
    tile_coords(tile, mtiles, (N + kBN - 1u) / kBN, mt, nt);
    const uint32_t pj = (mt >= P.mt0[1] ? 1u : 0u) + (mt >= P.mt0[2] ? 1u : 0u) + (mt >= P.mt0[3] ? 1u : 0u);
    const uint32_t M = P.M[pj];
    const uint32_t m0 = (mt - P.mt0[pj]) * BM, n0 = nt * kBN;
    const uint32_t mrows = min(BM, M - m0), ntok = min(kBN, N - n0);
    const uint32_t e = blockIdx.y * 256u + threadIdx.x;  // group index within the tile
    const uint32_t t = e / G, r = (e - t * G) * 4u;
    if (t >= ntok || r >= mrows) return;
    float* y = P.out[pj] + (size_t)(n0 + t) * M + m0 + r;
    const float* sc = P.scale[pj] + m0 + r;
    const uint32_t parts = P.parts;
    const size_t blk = (size_t)BM * kBN, off = (size_t)tile * blk + (size_t)t * BM + r;
    if (r + 3u < mrows) {
        f32x4 v = *reinterpret_cast<const f32x4_a4*>(y);
        const f32x4 s4 = *reinterpret_cast<const f32x4_a4*>(sc);
        f32x4 q[7];
#pragma unroll
        for (uint32_t j = 1; j < 8u; ++j)
            if (j < parts) q[j - 1u] = *reinterpret_cast<const f32x4*>(P.part + (size_t)(j - 1u) * P.tiles * blk + off);
#pragma unroll
        for (uint32_t j = 1; j < 8u; ++j)
            if (j < parts) v += q[j - 1u];
        *reinterpret_cast<f32x4_a4*>(y) = v * s4;
    } else {
        for (uint32_t k = 0; k < mrows - r; ++k) {
            float v = y[k];
            for (uint32_t j = 1; j < parts; ++j) v += P.part[(size_t)(j - 1u) * P.tiles * blk + off + k];
            y[k] = v * sc[k];
        }
    }
}

__global__ void fill_zero_kernel(float* __restrict__ y, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        y[i] = 0.0f;
}

// The launch's projection table for BM-row tiles; returns the row tiles of
// all projections together.
uint32_t fill_projections(const MatmulProjection* p, uint32_t count, uint32_t BM, MatmulProjections& P) {
    uint32_t mtiles = 0;
    for (uint32_t i = 0; i < kMaxMatmulProjections; ++i) {
        if (i < count) {
            P.weight[i] = p[i].weight;
            P.scale[i] = p[i].scale;
            P.out[i] = p[i].output;
            P.M[i] = p[i].M;
            P.mt0[i] = mtiles;
            mtiles += (p[i].M + BM - 1u) / BM;
        } else {
            P.mt0[i] = 0xffffffffu;
        }
    }
    return mtiles;
}

// One launch of matmul_q8_direct_kernel over `count` projections of the same
// activations.  kSplitTiles: the tiles' K steps split into `parts` runs, the
// workspace `part` holding (parts - 1) blocks of BM x kBN floats per tile, and
// split_sum_kernel sums them in a second launch.
template <int NW, int FW, int KS = 1, int MODE = kWholeTiles>
hipError_t launch_direct(const float* a, const MatmulProjection* p, uint32_t count, uint32_t N, uint32_t K,
                         hipStream_t stream, float* part = nullptr, uint32_t parts = 1) {
    constexpr uint32_t BM = 16u * FW * NW;
    const uint32_t W = (uint32_t)(((uint64_t)K + 3) / 4);
    MatmulProjections P = {};
    const uint32_t mtiles = fill_projections(p, count, BM, P);
    const uint32_t ntiles = (N + kBN - 1u) / kBN;
    const uint32_t tiles = mtiles * ntiles;
    P.part = part;
    P.tiles = tiles;
    P.parts = parts;
    uint32_t grid = ((tiles + 7u) / 8u) * 8u;
    if constexpr (MODE == kSplitTiles) grid = ((tiles * parts + 7u) / 8u) * 8u;
    if constexpr (MODE == kTilePairs) grid = 8u * ((tiles / 2u + 7u) / 8u);
    const size_t lds = KS * 3u * 2u * kBN * 128u + (direct_sums_in_lds(NW, KS) ? BM * kBN * 4u : 0u);
    hipLaunchKernelGGL((matmul_q8_direct_kernel<NW, FW, KS, MODE>), dim3(grid), dim3(64 * NW * KS), lds, stream, a, P, N,
                       K, W, mtiles, ntiles);
    if constexpr (MODE == kSplitTiles) {
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
        hipLaunchKernelGGL(split_sum_kernel<BM>, dim3(tiles, BM / 16u), dim3(256), 0, stream, P, N, mtiles);
    }
    return hipGetLastError();
}

// One launch of matmul_q8_kernel, alike.
template <int FB, int NW, int BK, int PD, int KS = 1, bool SPLIT = false>
hipError_t launch_fb(const float* a, const MatmulProjection* p, uint32_t count, uint32_t N, uint32_t K,
                     hipStream_t stream, float* part = nullptr, uint32_t parts = 1) {
    constexpr uint32_t kRowBytes = (uint32_t)BK * 2u;
    constexpr uint32_t BM = 32u * FB;
    const uint32_t W = (uint32_t)(((uint64_t)K + 3) / 4);
    MatmulProjections P = {};
    const uint32_t mtiles = fill_projections(p, count, BM, P);
    const uint32_t ntiles = (N + kBN - 1u) / kBN;
    const uint32_t tiles = mtiles * ntiles;
    P.part = part;
    P.tiles = tiles;
    P.parts = parts;
    uint32_t grid = ((tiles + 7u) / 8u) * 8u;
    if constexpr (SPLIT) grid = ((tiles * parts + 7u) / 8u) * 8u;
    const size_t lds = (size_t)KS * (2u * BM * kRowBytes + 2u * 2u * kBN * kRowBytes);
    hipLaunchKernelGGL((matmul_q8_kernel<FB, NW, BK, PD, KS, SPLIT>), dim3(grid), dim3(64 * NW * KS), lds, stream, a,
                       P, N, K, W, mtiles, ntiles);
    if constexpr (SPLIT) {
        const hipError_t err = hipGetLastError();
        if (err != hipSuccess) return err;
        hipLaunchKernelGGL(split_sum_kernel<BM>, dim3(tiles, BM / 16u), dim3(256), 0, stream, P, N, mtiles);
    }
    return hipGetLastError();
}

}  // namespace

hipError_t launch_matmul_q8_multi(const float* a, const MatmulProjection* projections, uint32_t count, uint32_t N,
                                  uint32_t K, const DeviceInfo& dev, hipStream_t stream, Variant* variant,
                                  float* workspace, size_t workspace_bytes) {
    static_assert(kMaxMatmulProjectionsPerLaunch == kMaxMatmulProjections, "one launch's projection table");
    MatmulProjection p[kMaxMatmulProjections];
    uint32_t n = 0;
    for (uint32_t i = 0; i < count; ++i) {
        if (projections[i].M == 0) continue;
        if (n == kMaxMatmulProjections) return hipErrorInvalidValue;
        p[n++] = projections[i];
    }
    if (N == 0 || n == 0) return hipSuccess;
    if (K == 0) {
        // matmul over an empty K: every sum is 0 (ops/matmul/reference.ts:17-18)
        for (uint32_t i = 0; i < n; ++i) {
            const size_t e = (size_t)N * p[i].M;
            const uint32_t grid = (uint32_t)((e + 255) / 256 < 65536 ? (e + 255) / 256 : 65536);
            hipLaunchKernelGGL(fill_zero_kernel, dim3(grid), dim3(256), 0, stream, p[i].output, e);
            set_variant(variant, "fill_zero", "matmul.k0", 4, 0, 0, 0, grid);
            const hipError_t err = hipGetLastError();
            if (err != hipSuccess) return err;
        }
        return hipSuccess;
    }
    // Up to 32 tokens: the batched single-vector path, one token per vector
    // (out[n, m] is y[vector n][row m], the same layout), one call per
    // projection.  The GEMM walks all of K in a serial chain of steps per
    // workgroup whatever the token count (20 us for 1 token at 2048 x 2048);
    // the batched path streams the weight once per 8 or 16 tokens (3.6 us
    // for 1 token, 7.0 us for 32).
    // Both compute the matvecQ8 form.
    Projection pv[kMaxMatmulProjections];
    for (uint32_t i = 0; i < n; ++i) pv[i] = Projection{p[i].weight, p[i].scale, p[i].output, p[i].M};
    if (N <= 32u) {
        // several projections in one launch where the k-split kernel pays for
        // their rows together (24 tokens, two of 5632 x 2048: 26.1 -> 12.8 us)
        if (n > 1u && matvec_q8_batched_multi_pays(pv, n, K, N, dev)) {
            const hipError_t e = launch_matvec_q8_batched_multi(pv, n, a, K, N, dev, stream, variant);
            if (variant && e == hipSuccess) variant->form = "matmul.tokens_as_vectors";
            return e;
        }
        for (uint32_t i = 0; i < n; ++i) {
            MatvecArgs mv{p[i].weight, p[i].scale, a, p[i].output, p[i].M, K, N, (uint32_t)(((uint64_t)K + 3) / 4)};
            const hipError_t e = launch_matvec_q8(mv, dev, stream, variant);
            if (e != hipSuccess) return e;
            if (variant) variant->form = "matmul.tokens_as_vectors";
        }
        return hipSuccess;
    }
    // The direct kernel where its tiles give (most of) the CUs one each, alone
    // or split through the workspace (D256, D128 and the FB4 forms below); short
    // prompts' smaller tiles, 64 or 32 rows, through LDS with two groups of 8
    // waves that split each tile's K steps.  Projections in one launch count
    // their tiles together.
    const uint32_t cus = (uint32_t)(dev.cu_count > 0 ? dev.cu_count : 256);
    const uint64_t ntiles = (N + kBN - 1u) / kBN;
    uint64_t t12 = 0, t8 = 0, t4 = 0, t2 = 0, t1 = 0;
    for (uint32_t i = 0; i < n; ++i) {
        t12 += (uint64_t)((p[i].M + 383u) / 384u) * ntiles;
        t8 += (uint64_t)((p[i].M + 255u) / 256u) * ntiles;
        t4 += (uint64_t)((p[i].M + 127u) / 128u) * ntiles;
        t2 += (uint64_t)((p[i].M + 63u) / 64u) * ntiles;
        t1 += (uint64_t)((p[i].M + 31u) / 32u) * ntiles;
    }
    const uint32_t steps = (uint32_t)(((uint64_t)K + 63u) / 64u);
    const char* kname = n > 1 ? "matmul_q8.multi" : "matmul_q8";
    // Short prompts on the batched k-split kernel, 16 tokens a pass, all passes in
    // one round of the CUs: it splits each activation once per 16-row tile range
    // instead of once per 32- or 64-row tile, and waits for no barrier per step.
    // A workgroup costs its start and its 16-row tiles, each as much as rows of whole
    // 1024s of codes; the tiles below cost their steps, more past one tile per CU.  So
    // the line is drawn by a workgroup's tiles times the codes they are priced at, per
    // code of a row.  From a sweep of 220 shapes of 33 to 4096 tokens, k-split / tiles,
    // us: at 8, 183 x 2595 x 4096 29.7 / 33.4, 3214 x 115 x 1024 12.1 / 13.4, 191 x 1894 x
    // 3073 26.3 / 30.3; past 9.5 against 32-row tiles 97 x 3881 x 2112 23.6 / 21.3, 282 x
    // 1327 x 1088 14.5 / 14.2; against 64-row ones up to 12.5, 43 x 10399 x 1300 17.3 /
    // 20.3, 2925 x 186 x 4038 38.4 / 47.4, past it 1377 x 400 x 2048 25.9 / 22.3, 2049 x
    // 272 x 2048 (17 tiles on each of 129 workgroups) 28.9 / 23.3.  Over nine tile
    // passes per CU in all the weight streams too often (33 x 15122 x 3996, 11: 49.6 /
    // 42.6).  Rows up to 768 codes have few steps to save: up to 4 tiles, or 7 at whole
    // rows' price (48 x 4096 x 512 8.0 / 8.4; 3469 x 68 x 640, 5 tiles: 10.5 / 9.4).
    // A workspace changes nothing here (64 x 2048 x 2048 8.2 us; its 32-row tiles split
    // in 4 parts 13.0, 425 x 128 x 1024 in 2 13.1 against 6.6).
    const uint64_t passes = (N + 15u) / 16u;
    uint64_t t16 = 0;
    for (uint32_t i = 0; i < n; ++i) t16 += (p[i].M + 15ull) / 16u;
    bool on_ksplit = false;
    if (K >= 512u && K <= 4096u && passes <= cus && t16 * passes <= 9ull * cus) {
        const uint64_t per_pass = cus / passes, load = (t16 + per_pass - 1u) / per_pass;
        const uint64_t priced = load * 1024u * ((K + 1023u) / 1024u);
        on_ksplit = K > 768u ? 2u * priced <= (t1 > cus ? 25u : 19u) * (uint64_t)K
                             : load <= 4u || priced <= 7u * (uint64_t)K;
    }
    if (on_ksplit) {
        const hipError_t e = launch_matvec_q8_batched_multi(pv, n, a, K, N, dev, stream, variant);
        if (variant && e == hipSuccess) variant->form = "matmul.tokens_as_vectors";
        return e;
    }
    // One workgroup of 8 waves per CU on the direct kernel, each wave 32 or 48
    // rows x 64 tokens.  The larger tile needs 1.26 times the smaller one's time
    // for 1.5 times its work (the activations' LDS reads, split and barriers per
    // step are the same), so the dispatch takes the one whose rounds of the CUs
    // cost less.  Same process, us, 256 / 384 rows: 512 x 11264 x 2048 (352 / 240
    // tiles) 65 / 50, 2048 x 11264 x 2048 (1408 / 960) 228 / 198, 512 x 6144 x
    // 2048 (192 / 128) 35.1 / 43.8, 2048 x 2048 x 5632 (256 / 192) 98.8 / 111.
    // 128-row tiles, two workgroups of 4 waves per CU, take 0.69 of a 256-row
    // round per tile and CU (704 tiles 67 us): they are left the launches whose
    // 256-row tiles would leave a round mostly empty.  The sums and their order
    // are the same in all three, so are the bits.
    const uint64_t r8 = (t8 + cus - 1u) / cus, r12 = (t12 + cus - 1u) / cus;
    const bool rows384 = t4 > 2ull * cus && 126u * r12 < 100u * r8;
    if (!rows384 && t8 >= cus && 100u * r8 * cus < 69u * t4) {
        set_variant(variant, kname, "D256", 8, 256, 0, (int)kBN, (uint32_t)((t8 + 7u) / 8u * 8u));
        return launch_direct<8, 2>(a, p, n, N, K, stream);
    }
    // Up to 6 steps (K <= 384) the two groups' own starts outweigh what they share in
    // one round of 128-row tiles: 64-row tiles, two workgroups per CU.  Same process,
    // us, 128 -> 64 rows: 210 x 5406 x 128 9.5 -> 7.5, 995 x 1068 x 256 10.3 -> 9.0,
    // 512 x 4096 x 256 11.0 -> 10.1, 75 x 11952 x 384 12.9 -> 12.4; past it 75 x 11952
    // x 448 12.9 -> 13.8.
    const bool halves = steps > 6u;
    if (t4 > cus || (t4 == cus && halves)) {
        if (t4 == cus) {
            set_variant(variant, kname, "FB4.ksplit2", 8, 128, 0, (int)kBN, (uint32_t)((t4 + 7u) / 8u * 8u));
            return launch_direct<4, 2, 2>(a, p, n, N, K, stream);
        }
        // One round of 256-row tiles beats an uneven round of 128-row ones, two
        // workgroups per CU: a 128-row workgroup beside another takes longer than a
        // 256-row one alone (us, 128 -> 256 rows: 700 x 3548 x 1030 28.0 -> 24.7, 640 x
        // 4200 x 2048 42.4 -> 36.7, 1280 x 2048 x 8192 142 -> 118, 320 x 7168 x 1024 24.5 ->
        // 20.6), and beats their last tiles' K steps split through a workspace as well
        // (33.2, 48.3, 127, 30.4).  More 256-row tiles than CUs (19000 x 128 x 2048, every
        // tile half empty) would take two rounds: 67.9 against 41.9.
        if (t4 < 2ull * cus && t8 <= cus) {
            set_variant(variant, kname, "D256", 8, 256, 0, (int)kBN, (uint32_t)((t8 + 7u) / 8u * 8u));
            return launch_direct<8, 2>(a, p, n, N, K, stream);
        }
        // Long rows whose 128-row tiles make two or more whole rounds of two per CU
        // where 256-row ones make neither whole rounds nor 2.75 of them: one
        // workgroup of 8 waves per two consecutive tiles of the sequence, 4 waves
        // each.  The same sums in the same order as the one-group form.
        // Past that line the larger tiles are faster (us, pairs -> 384-row): 4096 x 4096
        // x 4096 367 -> 281, 2048 x 8192 x 4096 356 -> 274, 1024 x 12288 x 4096 263 ->
        // 191; below it the two are even at K = 4096 (1024 x 8192: 174, 176).
        if (K >= 4096u && t4 >= 4ull * cus && t4 % (2ull * cus) == 0 && t8 % cus != 0 && 4u * t8 < 11ull * cus) {
            set_variant(variant, kname, "FB4.pairs", 8, 128, 0, (int)kBN, (uint32_t)((t4 / 2u + 7u) / 8u * 8u));
            return launch_direct<4, 2, 2, kTilePairs>(a, p, n, N, K, stream);
        }
        // Otherwise whole 128-row units: three per workgroup by the rule above,
        // or one per workgroup of 4 waves, two workgroups per CU.
        // Up to 6 steps (K <= 384) several rounds of 384-row tiles lose to the smaller
        // ones, whose two workgroups per CU cover each other's first loads and
        // stores: 1371 x 7327 x 64 25.2 -> 21.7 us, 519 x 16882 x 192 27.4 -> 24.8,
        // 928 x 8984 x 384 34.9 -> 34.1; past it 2412 x 3664 x 512 39.4 -> 40.9.
        if (rows384 && (r12 == 1u || steps > 6u)) {
            set_variant(variant, kname, "D384", 8, 384, 0, (int)kBN, (uint32_t)((t12 + 7u) / 8u * 8u));
            return launch_direct<8, 3>(a, p, n, N, K, stream);
        }
        set_variant(variant, kname, "D128", 4, 128, 0, (int)kBN, (uint32_t)((t4 + 7u) / 8u * 8u));
        return launch_direct<4, 2>(a, p, n, N, K, stream);
    }
    // With a workspace, 256-row tiles on the direct kernel with every tile's
    // K steps split into 4 or 8 parts, one workgroup each, when that fills
    // more than 7/8 of the CUs with at least 11 steps per part (the parts
    // meet in split_sum_kernel).  Same process, us, against the forms below: 512
    // tokens x 2048 x 5632 38.9 -> 36.3 (4 parts of 22 steps), 256 tokens 24.6 ->
    // 25.0 (8 parts of 11: even); with fewer steps per part the split's second
    // launch costs more than it saves.
    for (uint32_t xs : {4u, 8u}) {
        const size_t blk = (size_t)256u * kBN * 4u;
        if (workspace && t8 * xs <= cus && 8u * t8 * xs > 7u * cus && steps >= 11u * xs &&
            (xs - 1u) * t8 * blk <= workspace_bytes) {
            set_variant(variant, kname, xs == 4u ? "D256.split4" : "D256.split8", 8, 256, 0, (int)kBN,
                        (uint32_t)(t8 * xs));
            return launch_direct<8, 2, 1, kSplitTiles>(a, p, n, N, K, stream, workspace, xs);
        }
    }
    // 128-row tiles that fill most of the CUs, one per CU with two K groups of 4
    // waves on the direct kernel, beat smaller tiles that fill them all.  Same
    // process, us, against the 64-row form: 128 tokens gate and up (176 tiles) 32.5 ->
    // 24.8, 256 tokens q, k, v (192) 31.7 -> 24.8, 320 x 5120 x 2048 (200) 32.2 -> 24.9.
    if (halves && 5u * t4 >= 3u * cus) {
        set_variant(variant, kname, "FB4.ksplit2", 8, 128, 0, (int)kBN, (uint32_t)((t4 + 7u) / 8u * 8u));
        return launch_direct<4, 2, 2>(a, p, n, N, K, stream);
    }
    // With a workspace, 128-row tiles whose K steps split in 2 or 4 fill
    // (nearly) every CU, as long as each K group keeps at least 10 steps
    // (the split's second launch and every part's pipeline start cost a few
    // us): 512 tokens x 2048 x 2560 25.8 -> 24.7 us (2 parts, 10 steps per group)
    // against the 64-row form.
    for (uint32_t xs : {4u, 2u}) {
        const size_t blk = (size_t)128u * kBN * 4u;
        if (workspace && t4 * xs <= cus && 8u * t4 * xs > 7u * cus && steps >= 20u * xs &&
            (xs - 1u) * t4 * blk <= workspace_bytes) {
            set_variant(variant, kname, xs == 4u ? "FB4.ksplit2.wgsplit4" : "FB4.ksplit2.wgsplit2", 8, 128, 0, (int)kBN,
                        (uint32_t)(t4 * xs));
            return launch_direct<4, 2, 2, kSplitTiles>(a, p, n, N, K, stream, workspace, xs);
        }
    }
    if (t1 <= cus) {
        // With a workspace, 32-row tiles that fill at most a quarter (a half) of the
        // CUs also split their K steps between 4 (2) workgroups, each run at least 4
        // steps per K group; the parts' sums meet in a second launch.
        const size_t blk32 = (size_t)32u * kBN * 4u;
        if (workspace && 4u * t1 <= cus && steps >= 32u && 3u * t1 * blk32 <= workspace_bytes) {
            set_variant(variant, kname, "FB1.PD4.ksplit2.wgsplit4", 16, 32, 0, (int)kBN, (uint32_t)(4u * t1));
            return launch_fb<1, 8, 64, 4, 2, true>(a, p, n, N, K, stream, workspace, 4u);
        }
        if (workspace && 2u * t1 <= cus && steps >= 16u && t1 * blk32 <= workspace_bytes) {
            set_variant(variant, kname, "FB1.PD4.ksplit2.wgsplit2", 16, 32, 0, (int)kBN, (uint32_t)(2u * t1));
            return launch_fb<1, 8, 64, 4, 2, true>(a, p, n, N, K, stream, workspace, 2u);
        }
        set_variant(variant, kname, "FB1.PD4.ksplit2", 16, 32, 0, (int)kBN, (uint32_t)((t1 + 7u) / 8u * 8u));
        return launch_fb<1, 8, 64, 4, 2>(a, p, n, N, K, stream);
    }
    set_variant(variant, n > 1 ? "matmul_q8.multi" : "matmul_q8", t2 <= cus ? "FB2.PD4.ksplit2" : "FB2.PD4",
                t2 <= cus ? 16 : 8, 64, 0, (int)kBN, (uint32_t)((t2 + 7u) / 8u * 8u));
    return t2 <= cus ? launch_fb<2, 8, 64, 4, 2>(a, p, n, N, K, stream)
                     : launch_fb<2, 8, 64, 4, 1>(a, p, n, N, K, stream);
}

hipError_t launch_matmul_q8(const float* a, const uint32_t* weight, const float* scale, float* out, uint32_t N,
                            uint32_t M, uint32_t K, const DeviceInfo& dev, hipStream_t stream, Variant* variant) {
    const MatmulProjection p{weight, scale, out, M};
    return launch_matmul_q8_multi(a, &p, 1, N, K, dev, stream, variant, nullptr, 0);
}

}  // namespace wxo
