// GEMM for few tokens (2 to 48): out[t][r] = Σ_k x[t][k] · w[r][k] with n rows of FP16
// activations against Q4_K / Q6_K weights in the device layout (gh_kargs.h), each weight read and
// unpacked once for all tokens.
//
// Mapping: a 256-thread workgroup takes 128 weight rows and one K split of whole 256-weight blocks.
// The split's activations are staged once in LDS. Every wave streams two tiles of 16 rows straight
// into registers, two blocks in flight: lane l takes unit l / 16 of the block of row l % 16, so a
// load instruction reads 64 contiguous bytes of each of 16 rows (32 rows x 16 bytes, as a
// 32-row operand would need: gate 12288 x 4096 at 5 tokens 14.4 us with its reduce instead of 13.8,
// at 16 18.4 instead of 16.9). Products with v_mfma_f32_16x16x32_f16: A = 16 tokens,
// B = 16 weight rows, whose k-slots 8 (l / 16) .. + 8 are a lane's own 8 weights, so scales are applied
// per lane before the product and a lane's accumulators all belong to its weight row.
//
// Weights. From 8 tokens: the FP16-rounded weights of the tiled GEMMs (gh_w16_*), unpacked into
// B fragments in registers. Below 8 (EXACT), where a GEMV over exact weights ran before, nothing is
// rounded: the quants are multiplied by their sub-block's integer scale in FP16, which is exact, the
// matrix cores sum a whole block of x · (scale · quant), and the FP16 block scale enters once per
// block in FP32:
//   Q4_K: scale · quant <= 63 · 15 = 945; the minima as one more product over the block's eight
//     sub-blocks, min_j · Σx_j: Σx_j, an FP32 sum, goes in as the FP16 parts hi + 2^-11 mid + 2^-22 low
//     of the sub-block's mean, which hold all of it (33 bits; where a part is subnormal, down to 2^-46,
//     and a mean of 32 FP16 values is a multiple of 2^-29), so Σ = d · S - 32 dmin · M;
//   Q6_K: |scale · (quant - 32)| <= 4096, of which FP16 holds all up to 2048 and the even ones; the
//     +-1 that rounding leaves out goes in as a second product.
// There quants are used as FP16 subnormals (the integer q in the low bits is q · 2^-24), multiplied
// by 2^10 · scale (Q4_K, high nibbles in place: 2^6 · scale) or 2^8 · scale (Q6_K).
//
// What bounds it: the weight stream's 64-byte pieces. At 24576 x 4096 and 5 tokens (56.6 MB) a launch
// with its reduce takes 24.0 us, a copy that only loads 22.0 (19.5 with 128-byte pieces, which do not
// fit the operand layout) and one that only computes 12.7. Workgroups that kept the staged
// activations over several row tiles, the next tile's weights in flight, were slower (12288 x 4096
// 13.3 -> 15.6 us: half the waves), and so were nontemporal loads (22 -> 26.5) and four blocks in flight.
// With its split reduce, us before (the GEMV below 8 tokens, the 128-token tiles from 8) and now at
// 5 / 16 / 32 tokens: 12288 x 4096 Q4_K 32.7 / 28.0 / 29.4 -> 13.4 / 16.3 / 19.7; 4096 x 12288 Q6_K
// 47.2 / 32.1 / 33.5 -> 18.4 / 20.1 / 23.1; 5120 x 16384 Q6_K 73.0 / 51.7 / 53.2 -> 30.1 / 32.1 / 37.8.
//
// With a.part set: FP32 partials [split][n][row length] at the segment's part0, summed in split order
// by the tiled GEMMs' reduce and tail kernels; without it (one split) FP16 outputs. The split count
// depends on in_dim and n only, so a matrix gives the same bits alone and in a launch with others.
#include <type_traits>

#include "gh_common.h"

namespace {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));
constexpr uint32_t kQ4K = 12, kQ6K = 14;

__device__ __forceinline__ uint32_t pk_mul(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, gh_as_h2(a) * gh_as_h2(b));
}
__device__ __forceinline__ uint32_t pk_add(uint32_t a, uint32_t b) {
    return __builtin_bit_cast(uint32_t, gh_as_h2(a) + gh_as_h2(b));
}

// A lane's unit (64 weights) of one 256-weight block of its row, and the block's scales.
template <uint32_t FMT>
struct Unit;
template <>
struct Unit<kQ4K> {
    uint4 q[2];  // the two halves of the 32 qs bytes of group u
    uint4 hd;
};
template <>
struct Unit<kQ6K> {
    uint4 a, b, h;  // ql planes and qh of the unit (segment u / 2, half u % 2)
    uint4 sc;
    uint32_t d;
};

// unit u of block b of `row`
template <uint32_t FMT>
__device__ __forceinline__ void load_unit(uint64_t w, uint32_t rows, uint32_t nb, uint32_t row, uint32_t b, uint32_t u,
                                          Unit<FMT>& o) {
    const uint64_t blk = (uint64_t)row * nb + b;
    if constexpr (FMT == kQ4K) {
        const uint64_t q = w + (uint64_t)row * GH_Q4K_QS_BYTES * nb + b * 64 + u * 16;
        o.q[0] = *gh_gp<uint4>(q);
        o.q[1] = *gh_gp<uint4>(q + (uint64_t)nb * 64);
        o.hd = *gh_gp<uint4>(w + (uint64_t)rows * GH_Q4K_QS_BYTES * nb + blk * 16);
    } else {
        const uint64_t q = w + (uint64_t)row * GH_Q6K_QLH_BYTES * nb + b * 64 + u * 16;
        o.a = *gh_gp<uint4>(q);
        o.b = *gh_gp<uint4>(q + (uint64_t)nb * 64);
        o.h = *gh_gp<uint4>(q + 2ull * nb * 64);
        o.sc = *gh_gp<uint4>(w + (uint64_t)rows * GH_Q6K_QLH_BYTES * nb + blk * 16);
        o.d = *gh_gp<uint16_t>(w + (uint64_t)rows * 208 * nb + blk * 2);
    }
}

// The int8 scales of a Q6_K unit's quarters 0..3 in bytes 0, 2 of two words
__device__ __forceinline__ uint2 q6_scales(const uint4& sc, uint32_t u) {
    const bool s = u >= 2;
    return make_uint2((s ? sc.z : sc.x) >> (8 * (u & 1u)), (s ? sc.w : sc.y) >> (8 * (u & 1u)));
}

// The staged activations: row t (token) holds the split's k in 8-value chunks, for EXACT with the
// values in the order 0 2 1 3 4 6 5 7 that its quant dwords unpack to; `xp` halves a row. Sub-block
// means (EXACT Q4_K): for token t, block b and unit u the hi, mid and low parts (and a zero) of its two
// sub-blocks, 8 halves at sums + t · sp + 32 b + 8 u.
struct Staged {
    const _Float16* xs;
    const _Float16* sums;
    uint32_t xp, sp;
};

// halves from a block's first k to the lane's first: Q4_K units are 64 consecutive k, Q6_K units
// 16 of each of a segment's four 32-k quarters
template <uint32_t FMT>
__device__ __forceinline__ uint32_t lane_k(uint32_t u) {
    return FMT == kQ4K ? 64 * u : 128 * (u >> 1) + 16 * (u & 1u);
}

// 32 FP16-rounded weights of a unit: lo = the low nibbles of 16 quant bytes, hi = the high ones, as
// natural-order pairs. Q4_K: q = half of the group's qs bytes; Q6_K: q = 16 bytes of ql plane `part`.
__device__ __forceinline__ void w16_q4k(const uint4& q, const uint4& hd, uint32_t g, uint32_t (&lo)[8], uint32_t (&hi)[8]) {
    const GhW16Q4K c = gh_w16_q4k_scales(hd, g);
    const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint32_t lo4 = qw[j] & 0x0F0F0F0Fu, hi4 = (qw[j] >> 4) & 0x0F0F0F0Fu;
        asm volatile("" : "+v"(lo4), "+v"(hi4));  // bytes converted in place, as in the tiles' store_w
        lo[2 * j] = gh_w16_q4k_pair(lo4, 0, c.d1, c.m1);
        lo[2 * j + 1] = gh_w16_q4k_pair(lo4, 2, c.d1, c.m1);
        hi[2 * j] = gh_w16_q4k_pair(hi4, 0, c.d2, c.m2);
        hi[2 * j + 1] = gh_w16_q4k_pair(hi4, 2, c.d2, c.m2);
    }
}
__device__ __forceinline__ void w16_q6k(const uint4& q, const uint4& qhv, const uint2& sc, uint32_t dh, uint32_t part,
                                        uint32_t (&lo)[8], uint32_t (&hi)[8]) {
    const GhW16Q6K c = gh_w16_q6k_scales(make_uint4(sc.x, sc.y, 0u, 0u), dh, 0, 0, part);
    const uint32_t qw[4] = {q.x, q.y, q.z, q.w}, qh[4] = {qhv.x, qhv.y, qhv.z, qhv.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t qa4 = gh_w16_q6k_low(qw[j], qh[j], part), qb4 = gh_w16_q6k_high(qw[j], qh[j], part);
        lo[2 * j] = gh_w16_q6k_pair(qa4, 0, c.da, c.na);
        lo[2 * j + 1] = gh_w16_q6k_pair(qa4, 2, c.da, c.na);
        hi[2 * j] = gh_w16_q6k_pair(qb4, 0, c.db, c.nb);
        hi[2 * j + 1] = gh_w16_q6k_pair(qb4, 2, c.db, c.nb);
    }
}

// Two row tiles x NT token tiles of 16: acc += x · (B fragments of 16 weights, k offset `ko` halves
// from the lane's first), chunk by chunk.
template <int NT>
__device__ __forceinline__ void mma16(const _Float16* const (&xr)[NT], uint32_t ko, const uint32_t (&b0)[8],
                                      const uint32_t (&b1)[8], f4v (&acc)[2][NT]) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const h8 w0 = __builtin_bit_cast(h8, make_uint4(b0[4 * c], b0[4 * c + 1], b0[4 * c + 2], b0[4 * c + 3]));
        const h8 w1 = __builtin_bit_cast(h8, make_uint4(b1[4 * c], b1[4 * c + 1], b1[4 * c + 2], b1[4 * c + 3]));
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const h8 x = *(const h8*)(xr[t] + ko + 8 * c);
            acc[0][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, w0, acc[0][t], 0, 0, 0);
            acc[1][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, w1, acc[1][t], 0, 0, 0);
        }
    }
}

// acc += the contribution of the split's block `at` over FP16-rounded weights.
template <uint32_t FMT, int NT>
__device__ __forceinline__ void block_w16(const Unit<FMT> (&w)[2], const Staged& st, uint32_t at, uint32_t n,
                                          uint32_t fr, uint32_t u, f4v (&acc)[2][NT]) {
    const _Float16* xr[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
        xr[t] = st.xs + min(16u * t + fr, n - 1) * st.xp + at * 256 + lane_k<FMT>(u);
    uint32_t lo[2][8], hi[2][8];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if constexpr (FMT == kQ4K) {
#pragma unroll
            for (int r = 0; r < 2; ++r) w16_q4k(w[r].q[h], w[r].hd, u, lo[r], hi[r]);
            mma16<NT>(xr, 16 * h, lo[0], lo[1], acc);
            mma16<NT>(xr, 32 + 16 * h, hi[0], hi[1], acc);
            __builtin_amdgcn_sched_barrier(0);  // one half's fragments live at a time
        } else {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const uint2 sc = q6_scales(w[r].sc, u);
                w16_q6k(h ? w[r].b : w[r].a, w[r].h, sc, w[r].d, h, lo[r], hi[r]);
            }
            mma16<NT>(xr, 32 * h, lo[0], lo[1], acc);
            mma16<NT>(xr, 64 + 32 * h, hi[0], hi[1], acc);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
}

// The same over exact weights, for fewer than 8 tokens (one token tile).
template <uint32_t FMT>
__device__ __forceinline__ void block_exact(const Unit<FMT> (&w)[2], const Staged& st, uint32_t at, uint32_t n,
                                            uint32_t fr, uint32_t u, f4v (&acc)[2][1]) {
    const uint32_t row = min(fr, n - 1);
    const _Float16* xr[1] = {st.xs + row * st.xp + at * 256 + lane_k<FMT>(u)};
    f4v S[2][1] = {{f4v{}}, {f4v{}}};
    uint32_t p[2][8], q[2][8];
    if constexpr (FMT == kQ4K) {
        uint32_t s0[2], s1[2], mn[2];  // mn: the two minima
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            uint32_t sc0, mn0, sc1, mn1;
            gh_q4k_scale_min(w[r].hd, 2 * u, sc0, mn0);
            gh_q4k_scale_min(w[r].hd, 2 * u + 1, sc1, mn1);
            const _Float16 a = (_Float16)(float)(sc0 << 10), b = (_Float16)(float)(sc1 << 6);
            s0[r] = __builtin_bit_cast(uint32_t, gh_h2{a, a});
            s1[r] = __builtin_bit_cast(uint32_t, gh_h2{b, b});
            mn[r] = __builtin_bit_cast(uint32_t, gh_h2{(_Float16)(float)mn0, (_Float16)(float)mn1});
            asm volatile("" : "+v"(mn[r]));  // one register until the sums' product below
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const uint32_t v[4] = {w[r].q[h].x, w[r].q[h].y, w[r].q[h].z, w[r].q[h].w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t v8 = v[i] >> 8;
                    p[r][2 * i] = pk_mul(v[i] & 0x000F000Fu, s0[r]);
                    p[r][2 * i + 1] = pk_mul(v8 & 0x000F000Fu, s0[r]);
                    q[r][2 * i] = pk_mul(v[i] & 0x00F000F0u, s1[r]);
                    q[r][2 * i + 1] = pk_mul(v8 & 0x00F000F0u, s1[r]);
                }
            }
            mma16<1>(xr, 16 * h, p[0], p[1], S);
            mma16<1>(xr, 32 + 16 * h, q[0], q[1], S);
            __builtin_amdgcn_sched_barrier(0);  // one half's fragments live at a time
        }
        const h8 x = *(const h8*)(st.sums + row * st.sp + 32 * at + 8 * u);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            // min_j, 2^-11 min_j and 2^-22 min_j (an exact subnormal) against the parts
            const uint32_t e = 0x10001000u, m1 = pk_mul(mn[r], e), m2 = pk_mul(m1, e);
            const h8 mv = __builtin_bit_cast(h8, make_uint4(__builtin_amdgcn_perm(m1, mn[r], 0x05040100u), m2 & 0xFFFFu,
                                                            __builtin_amdgcn_perm(m1, mn[r], 0x07060302u), m2 >> 16));
            const f4v M = __builtin_amdgcn_mfma_f32_16x16x32_f16(x, mv, f4v{}, 0, 0, 0);
            const float d = gh_h2f(w[r].hd.x & 0xFFFFu) * 16384.0f, dm = gh_h2f(w[r].hd.x >> 16) * -32.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                acc[r][0][i] = __builtin_fmaf(dm, M[i], __builtin_fmaf(d, S[r][0][i], acc[r][0][i]));
        }
    } else {
        uint2 sc[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) sc[r] = q6_scales(w[r].sc, u);
#pragma unroll
        for (int k = 0; k < 4; ++k) {  // quarters
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                const uint32_t L[4] = {(k & 1) ? w[r].b.x : w[r].a.x, (k & 1) ? w[r].b.y : w[r].a.y,
                                       (k & 1) ? w[r].b.z : w[r].a.z, (k & 1) ? w[r].b.w : w[r].a.w};
                const uint32_t H[4] = {w[r].h.x, w[r].h.y, w[r].h.z, w[r].h.w};
                const _Float16 f = (_Float16)(float)((int32_t)(int8_t)((k >= 2 ? sc[r].y : sc[r].x) >> (16 * (k & 1))) * 256);
                const gh_h2 s = gh_h2{f, f};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t l4 = (k >= 2 ? L[i] >> 4 : L[i]) & 0x0F0F0F0Fu;
                    const uint32_t h2 = (k == 0 ? H[i] << 4 : k == 1 ? H[i] << 2 : k == 2 ? H[i] : H[i] >> 2) & 0x30303030u;
                    const uint32_t v = l4 | h2;
                    // (quant - 32) · 2^-24, exact subnormals; q: what rounding the product to FP16 left out
                    const gh_h2 x0 = gh_as_h2(pk_add(v & 0x003F003Fu, 0x80208020u));
                    const gh_h2 x1 = gh_as_h2(pk_add((v >> 8) & 0x003F003Fu, 0x80208020u));
                    const gh_h2 p0 = x0 * s, p1 = x1 * s;
                    p[r][2 * i] = __builtin_bit_cast(uint32_t, p0);
                    p[r][2 * i + 1] = __builtin_bit_cast(uint32_t, p1);
                    q[r][2 * i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(x0, s, -p0));
                    q[r][2 * i + 1] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(x1, s, -p1));
                }
            }
            mma16<1>(xr, 32 * k, p[0], p[1], S);
            mma16<1>(xr, 32 * k, q[0], q[1], S);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const float d = gh_h2f(w[r].d) * 65536.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[r][0][i] = __builtin_fmaf(d, S[r][0][i], acc[r][0][i]);
        }
    }
}

// 16 bytes of activations (8 values) reordered to 0 2 1 3 4 6 5 7
__device__ __forceinline__ uint4 reorder(const uint4& v) {
    return make_uint4(__builtin_amdgcn_perm(v.y, v.x, 0x05040100u), __builtin_amdgcn_perm(v.y, v.x, 0x07060302u),
                      __builtin_amdgcn_perm(v.w, v.z, 0x05040100u), __builtin_amdgcn_perm(v.w, v.z, 0x07060302u));
}

// Row tile blockIdx.y (128 rows) of the launch's matrices, in segment g of format FMT; K split
// blockIdx.x. NT: token tiles of 16; 0: EXACT, fewer than 8 tokens.
template <uint32_t FMT, int NT>
__device__ __forceinline__ void few_body(const GhGemmArgs& a, const GhGemmSeg& g) {
    constexpr bool EXACT = NT == 0;
    extern __shared__ __attribute__((aligned(16))) _Float16 lds[];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, fr = lane & 15u, u = lane >> 4;
    const uint32_t r = (blockIdx.y - g.tile0) * 128 + 32 * (tid >> 6) + fr;  // this lane's rows: r, r + 16
    const uint32_t z = blockIdx.x, nb = a.in_dim >> 8, per = gh_gemm_split_units(4 * nb, a.splits) / 4;
    const uint32_t b0 = z * per, cnt = min(per, nb - b0);  // the host leaves no split empty
    Staged st;
    st.xp = per * 256 + 8;
    st.sp = per * 32 + 8;
    st.xs = lds;
    st.sums = lds + a.n * st.xp;
    // activations: chunk i = 8 values c of token t; the first round is requested ahead of the weights
    // (loads complete in issue order)
    constexpr uint32_t kX = EXACT ? 2 : 8;              // chunks per thread and round
    const uint32_t cpt = cnt * 32, chunks = a.n * cpt;  // chunks per token, in all
    uint4 xv[kX];
    auto request = [&](uint32_t i0) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t k = 0; k < kX; ++k) {
            const uint32_t i = min(i0 + 256 * k + tid, chunks - 1), t = i / cpt, c = i % cpt;
            xv[k] = *gh_gp<uint4>(a.x + ((uint64_t)t * a.in_dim + b0 * 256 + 8 * c) * 2);
        }
    };
    auto stage = [&](uint32_t i0) __attribute__((always_inline)) {
#pragma unroll
        for (uint32_t k = 0; k < kX; ++k) {
            const uint32_t i = i0 + 256 * k + tid, t = i / cpt, c = i % cpt;
            const uint4 v = xv[k];
            if (i < chunks) *(uint4*)(lds + t * st.xp + 8 * c) = EXACT ? reorder(v) : v;
            if constexpr (EXACT && FMT != kQ6K) {
                // the sub-block's mean over the quad's four chunks (cpt is a multiple of 32)
                float s = gh_dot2(v.x, 0x3C003C00u, 0.0f);
                s = gh_dot2(v.y, 0x3C003C00u, s);
                s = gh_dot2(v.z, 0x3C003C00u, s);
                s = gh_dot2(v.w, 0x3C003C00u, s);
                s += GH_DPP(s, 0xB1, 0xF);
                s += GH_DPP(s, 0x4E, 0xF);
                s *= 0.03125f;
                const _Float16 hi = (_Float16)s;
                const float rest = (s - (float)hi) * 2048.0f;
                const _Float16 mid = (_Float16)rest, low = (_Float16)((rest - (float)mid) * 2048.0f);
                if (i < chunks && (tid & 3u) == 0) {
                    typedef _Float16 h4 __attribute__((ext_vector_type(4)));
                    *(h4*)(lds + a.n * st.xp + t * st.sp + (c >> 2) * 4) = h4{hi, mid, low, (_Float16)0.0f};
                }
            }
        }
    };
    request(0);
    __builtin_amdgcn_sched_barrier(0);
    Unit<FMT> wb[2][2];  // two blocks in flight: [block][row tile]
    auto load = [&](uint32_t i, Unit<FMT> (&o)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
            load_unit<FMT>(g.w, g.rows, nb, min(r + 16u * k, g.rows - 1), b0 + min(i, cnt - 1), u, o[k]);
    };
    load(0, wb[0]);
    load(1, wb[1]);
    __builtin_amdgcn_sched_barrier(0);
    stage(0);
    for (uint32_t i0 = 256 * kX; i0 < chunks; i0 += 256 * kX) {
        request(i0);
        stage(i0);
    }
    gh_lds_barrier();
    constexpr int kT = EXACT ? 1 : NT;
    f4v acc[2][kT];
#pragma unroll
    for (int t = 0; t < kT; ++t) acc[0][t] = acc[1][t] = f4v{};
    auto step = [&](const Unit<FMT> (&b)[2], uint32_t at) __attribute__((always_inline)) {
        if constexpr (EXACT) block_exact<FMT>(b, st, at, a.n, fr, u, acc);
        else block_w16<FMT, NT>(b, st, at, a.n, fr, u, acc);
    };
    for (uint32_t i = 0; i < cnt; i += 2) {
        step(wb[0], i);
        if (i + 2 < cnt) load(i + 2, wb[0]);
        if (i + 1 < cnt) {
            step(wb[1], i + 1);
            if (i + 3 < cnt) load(i + 3, wb[1]);
        }
    }
    // D: lane holds weight row r (+ 16 for its second tile), tokens 16 t + 4 u + i
#pragma unroll
    for (int k = 0; k < 2; ++k) {
        const uint32_t rk = r + 16 * k;
        if (rk >= g.rows) break;
#pragma unroll
        for (int t = 0; t < kT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t tok = 16 * t + 4 * u + i;
                if (tok >= a.n) continue;
                if (a.part) {
                    gh_gpw<float>(a.part)[g.part0 + ((uint64_t)z * a.n + tok) * a.rows + g.col0 + rk] = acc[k][t][i];
                } else {
                    const uint64_t o = (uint64_t)tok * g.rows + rk;
                    uint16_t h = gh_f2h(acc[k][t][i]);
                    if (a.epi == GH_GEMM_EPI_SILU) h = gh_silu_mul_h(gh_gp<uint16_t>(a.aux)[o], h);
                    gh_gpw<uint16_t>(g.out)[o] = h;
                }
            }
    }
}

// FMT 0: matrices of either format
template <uint32_t FMT, int NT>
__device__ __forceinline__ void few_tile(const GhGemmArgs& a) {
    uint32_t s = 0;
    for (uint32_t i = 1; i < a.nseg; ++i)
        if (blockIdx.y >= a.seg[i].tile0) s = i;
    const GhGemmSeg g = a.seg[s];
    if (FMT ? FMT == kQ4K : g.fmt == kQ4K) few_body<kQ4K, NT>(a, g);
    else few_body<kQ6K, NT>(a, g);
}

}  // namespace

// Grid (K splits, row tiles of 128 of all matrices): the splits of a row tile, neighbours in memory,
// start together (with the row tiles fastest: gate 13.8 us, down 21.4 at 5 tokens instead of 12.8,
// 17.8). Suffix _t8 / _t16 / _t32 / _t48: most tokens (_t8: fewer than 8). Up to three matrices of one
// format (q4k, q6k) or of both (mixed).
#define GH_GEMM_FEW(T, NT, W4, W6, WM)                                                                       \
    GH_KERNEL __launch_bounds__(256, W4) void gh_gemm_few_q4k_t##T(GhGemmArgs a) { few_tile<kQ4K, NT>(a); } \
    GH_KERNEL __launch_bounds__(256, W6) void gh_gemm_few_q6k_t##T(GhGemmArgs a) { few_tile<kQ6K, NT>(a); } \
    GH_KERNEL __launch_bounds__(256, WM) void gh_gemm_few_mixed_t##T(GhGemmArgs a) { few_tile<0, NT>(a); }
GH_GEMM_FEW(8, 0, 4, 3, 3)
GH_GEMM_FEW(16, 1, 4, 3, 2)
GH_GEMM_FEW(32, 2, 3, 3, 2)
GH_GEMM_FEW(48, 3, 3, 2, 2)
