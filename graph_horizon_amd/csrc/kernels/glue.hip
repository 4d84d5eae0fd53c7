// Decode/prefill glue: RMSNorm, YaRN RoPE, SiLU·up, residual add, KV append, argmax.
#include "gh_common.h"

// rmsnorm_x (backend/cpu/kernels/elementwise/normalization.rs:12-40): one 256-thread
// workgroup per row, Σx² in gh_rms_inverse_256's order (thread t: the 16-value items t, t + 256, ...),
// inverse = 1/sqrt(Σx²/dim + eps), out = f16((x*inverse)*w). dim % 4 == 0. Bound by memory (x in, out
// out): rows of up to 8192 values stay in registers between the sum and the scaling (2000 x 4096 read
// twice 15.2 us, now 12.6).
GH_KERNEL __launch_bounds__(256) void gh_rmsnorm_x(GhRmsnormArgs a) {
#pragma clang fp contract(off)
    const uint32_t row = blockIdx.x;
    if (row >= a.rows) return;
    const GH_GLOBAL float4* x = gh_gp<float4>(a.x + (uint64_t)row * a.dim * 4);
    const GH_GLOBAL uint2* w = gh_gp<uint2>(a.w);
    GH_GLOBAL uint2* out = gh_gpw<uint2>(a.out + (uint64_t)row * a.dim * 2);
    __shared__ float red[4];
    const uint32_t n4 = a.dim >> 2;
    auto scaled = [&](const float4& v, float inverse, uint32_t i) __attribute__((always_inline)) {
        const uint2 wv = w[i];
        const uint32_t o0 = gh_f2h(v.x * inverse * gh_h2f(wv.x & 0xFFFFu));
        const uint32_t o1 = gh_f2h(v.y * inverse * gh_h2f(wv.x >> 16));
        const uint32_t o2 = gh_f2h(v.z * inverse * gh_h2f(wv.y & 0xFFFFu));
        const uint32_t o3 = gh_f2h(v.w * inverse * gh_h2f(wv.y >> 16));
        out[i] = make_uint2(o0 | (o1 << 16), o2 | (o3 << 16));
    };
    if (a.dim > 8192) {
        const float inverse = gh_rms_inverse_256(x, a.dim, a.eps, red);
        for (uint32_t i = threadIdx.x; i < n4; i += 256) scaled(x[i], inverse, i);
        return;
    }
    float4 v[2][4];
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k)
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) v[k][q] = x[min(4 * (threadIdx.x + 256 * k) + q, n4 - 1)];
    float s = 0.0f;
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k)
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q)
            if (4 * (threadIdx.x + 256 * k) + q < n4) s = gh_rms_add(s, v[k][q]);
    const float inverse = gh_rms_finish_256(s, a.dim, a.eps, red);
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k)
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const uint32_t i = 4 * (threadIdx.x + 256 * k) + q;
            if (i < n4) scaled(v[k][q], inverse, i);
        }
}

// One pair of RoPE: (x0, x1) in v rotated by cs, times the post-scale
__device__ __forceinline__ uint32_t rope_pair(uint32_t v, float c, float s, float scale) {
#pragma clang fp contract(off)
    const float x0 = gh_h2f(v & 0xFFFFu), x1 = gh_h2f(v >> 16);
    const float y0 = (x0 * c - x1 * s) * scale;
    const float y1 = (x0 * s + x1 * c) * scale;
    return (uint32_t)gh_f2h(y0) | ((uint32_t)gh_f2h(y1) << 16);
}

// rope_yarn (cpu/kernels/elementwise/rope.rs:14-39): adjacent pairs rotated by the per
// (position, pair) YaRN (cos, sin) table, then the role's post-scale; FP16 in place. Query heads
// and, in the same launch, key heads (no post-scale). a.groups workgroups per row, a thread per a.per
// pairs: four (16 bytes) where the head and the addresses allow it, else one (a row of 32 + 8 heads
// in two launches of one pair per thread took 13.5 + 4.7 us at 2000 rows, now
// 9.9).
GH_KERNEL __launch_bounds__(256) void gh_rope(GhRopeArgs a) {
    const uint32_t row = blockIdx.x / a.groups;  // workgroup-uniform
    const uint32_t t = (blockIdx.x % a.groups) * 256 + threadIdx.x, quads = a.pairs / a.per;
    uint32_t head = t / quads;
    const uint32_t pair = (t % quads) * a.per;
    if (head >= a.heads + a.kheads) return;
    const uint32_t pos = (a.pos_ptr ? *gh_gp<uint32_t>(a.pos_ptr) : 0u) + a.base + row;
    const bool key = head >= a.heads;
    if (key) head -= a.heads;
    const float scale = !key && a.post ? gh_gp<float>(a.post)[pos] : 1.0f;
    const uint64_t p = (key ? a.k : a.x) + (((uint64_t)row * (key ? a.kheads : a.heads) + head) * a.head_dim + 2 * pair) * 2;
    const uint64_t cs = a.table + ((uint64_t)pos * a.pairs + pair) * 8;
    if (a.per == 4) {
        const uint4 v = *gh_gp<uint4>(p);
        const float4 c0 = *gh_gp<float4>(cs), c1 = *gh_gp<float4>(cs + 16);
        *gh_gpw<uint4>(p) = make_uint4(rope_pair(v.x, c0.x, c0.y, scale), rope_pair(v.y, c0.z, c0.w, scale),
                                       rope_pair(v.z, c1.x, c1.y, scale), rope_pair(v.w, c1.z, c1.w, scale));
    } else {
        const float2 c = *gh_gp<float2>(cs);
        *gh_gpw<uint32_t>(p) = rope_pair(*gh_gp<uint32_t>(p), c.x, c.y, scale);
    }
}

// The elementwise kernels below take 8 consecutive values per thread: 16-byte accesses where a.pad
// says that every address allows them (2-byte ones ran silu_mul of 24.6 M values at 3.0 TB/s, 50 us; now
// 26.2 us, 5.6 TB/s; kv_write of 2000 x 2 x 1024 values 7.0 -> 4.2), value by value otherwise and in the
// last, partial thread.
// silu_mul (cpu/kernels/elementwise/activation.rs:16-29): out = f16(f16(g/(1+exp(-g))) * u).
GH_KERNEL __launch_bounds__(256) void gh_silu_mul(GhEltArgs a) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (a.pad && i + 8 <= a.n) {
        const uint4 g = *gh_gp<uint4>(a.a + 2 * i), u = *gh_gp<uint4>(a.b + 2 * i);
        auto two = [](uint32_t g2, uint32_t u2) __attribute__((always_inline)) {
            return (uint32_t)gh_silu_mul_h(g2 & 0xFFFFu, u2 & 0xFFFFu) | ((uint32_t)gh_silu_mul_h(g2 >> 16, u2 >> 16) << 16);
        };
        *gh_gpw<uint4>(a.out + 2 * i) = make_uint4(two(g.x, u.x), two(g.y, u.y), two(g.z, u.z), two(g.w, u.w));
        return;
    }
    for (size_t k = i; k < a.n && k < i + 8; ++k)
        gh_gpw<uint16_t>(a.out)[k] = gh_silu_mul_h(gh_gp<uint16_t>(a.a)[k], gh_gp<uint16_t>(a.b)[k]);
}

// residual_add (cpu/kernels/elementwise/residual.rs:12-22): x(f32) += f16 y.
GH_KERNEL __launch_bounds__(256) void gh_residual_add(GhEltArgs a) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
    if (a.pad && i + 8 <= a.n) {
        GH_GLOBAL float4* x = gh_gpw<float4>(a.out + 4 * i);
        const uint4 y = *gh_gp<uint4>(a.b + 2 * i);
        float4 u = x[0], v = x[1];
        u.x += gh_h2f(y.x & 0xFFFFu);
        u.y += gh_h2f(y.x >> 16);
        u.z += gh_h2f(y.y & 0xFFFFu);
        u.w += gh_h2f(y.y >> 16);
        v.x += gh_h2f(y.z & 0xFFFFu);
        v.y += gh_h2f(y.z >> 16);
        v.z += gh_h2f(y.w & 0xFFFFu);
        v.w += gh_h2f(y.w >> 16);
        x[0] = u;
        x[1] = v;
        return;
    }
    for (size_t k = i; k < a.n && k < i + 8; ++k) gh_gpw<float>(a.out)[k] += gh_h2f(gh_gp<uint16_t>(a.b)[k]);
}

// Fill n u32 words at `out` with the value `pad`: a clear that a captured graph records as a
// kernel node, not a memset node.
GH_KERNEL __launch_bounds__(256) void gh_fill_u32(GhEltArgs a) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < a.n) gh_gpw<uint32_t>(a.out)[i] = a.pad;
}

// A plain streaming read, for measurement (no counterpart in the reference): the n 16-byte
// chunks at `a`, read with nontemporal loads (as the decode GEMVs read weights), four in
// flight per thread; thread i of the pad x 256 threads takes chunks i, i + 256 pad, ... . The
// chunks are XOR-folded and the fold is stored only if it equals 0xFFFFFFFF, so the loads stay
// live while the kernel writes (almost) nothing: its duration is what a pure weight stream of
// that size and launch shape takes on this chip.
GH_KERNEL __launch_bounds__(256) void gh_stream_probe(GhEltArgs a) {
    typedef uint32_t u4v __attribute__((ext_vector_type(4)));
    const GH_GLOBAL u4v* src = (const GH_GLOBAL u4v*)a.a;
    const uint32_t stride = a.pad * 256;
    uint32_t i = blockIdx.x * 256 + threadIdx.x, acc = 0;
    for (; i + 3 * stride < a.n; i += 4 * stride) {
        u4v v[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) v[k] = __builtin_nontemporal_load(src + i + k * stride);
#pragma unroll
        for (uint32_t k = 0; k < 4; ++k) acc ^= v[k].x ^ v[k].y ^ v[k].z ^ v[k].w;
    }
    for (; i < a.n; i += stride) {
        const u4v v = __builtin_nontemporal_load(src + i);
        acc ^= v.x ^ v.y ^ v.z ^ v.w;
    }
    if (acc == 0xFFFFFFFFu) gh_gpw<uint32_t>(a.out)[0] = blockIdx.x;
}

// kv_write f16 (cpu/kernels/attention/write.rs:50-63): raw FP16 copy of K and V into the
// caches at element offsets; with pos_ptr the offsets advance by stride * (*pos_ptr).
GH_KERNEL __launch_bounds__(256) void gh_kv_write(GhKvWriteArgs a) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 8;
    const size_t pos = a.pos_ptr ? *gh_gp<uint32_t>(a.pos_ptr) : 0u;
    auto copy = [&](uint64_t dst, uint64_t src, uint32_t count) __attribute__((always_inline)) {
        if (a.wide && i + 8 <= count) {
            *gh_gpw<uint4>(dst + 2 * i) = *gh_gp<uint4>(src + 2 * i);
            return;
        }
        for (size_t k = i; k < count && k < i + 8; ++k) gh_gpw<uint16_t>(dst)[k] = gh_gp<uint16_t>(src)[k];
    };
    copy(a.kc + 2 * (a.k_off + pos * a.k_stride), a.k, a.k_count);
    copy(a.vc + 2 * (a.v_off + pos * a.v_stride), a.v, a.v_count);
}

// argmax_f32 (backend/cpu/readback.rs:45-55): first index of the maximum, NaN never wins;
// if no logit exceeds -inf the answer is 0. Stage 1: one (value, index) per workgroup.
__device__ __forceinline__ void argmax_merge(float& v, uint32_t& i, float ov, uint32_t oi) {
    if (ov > v || (ov == v && oi < i)) {
        v = ov;
        i = oi;
    }
}

__device__ __forceinline__ void argmax_block(float& v, uint32_t& i) {
    __shared__ float sv[4];
    __shared__ uint32_t si[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float ov = __shfl_xor(v, off, 64);
        const uint32_t oi = __shfl_xor(i, off, 64);
        argmax_merge(v, i, ov, oi);
    }
    if ((threadIdx.x & 63) == 0) {
        sv[threadIdx.x >> 6] = v;
        si[threadIdx.x >> 6] = i;
    }
    __syncthreads();
    v = sv[0];
    i = si[0];
    for (int w = 1; w < 4; ++w) argmax_merge(v, i, sv[w], si[w]);
}

GH_KERNEL __launch_bounds__(256) void gh_argmax_partial(GhArgmaxArgs a) {
    const float* l = (const float*)a.logits;
    float v = -__builtin_inff();
    uint32_t idx = 0xFFFFFFFFu;
    const uint32_t stride = a.blocks * 256;
    for (uint32_t j = blockIdx.x * 256 + threadIdx.x; j < a.n; j += stride) {
        const float x = l[j];
        if (x > v) {  // strict: the first (lowest) index of this thread's subset wins
            v = x;
            idx = j;
        }
    }
    argmax_block(v, idx);
    if (threadIdx.x == 0) {
        ((float*)a.part_v)[blockIdx.x] = v;
        ((uint32_t*)a.part_i)[blockIdx.x] = idx;
    }
}

GH_KERNEL __launch_bounds__(256) void gh_argmax_final(GhArgmaxArgs a) {
    float v = -__builtin_inff();
    uint32_t idx = 0xFFFFFFFFu;
    for (uint32_t j = threadIdx.x; j < a.blocks; j += 256)
        argmax_merge(v, idx, ((const float*)a.part_v)[j], ((const uint32_t*)a.part_i)[j]);
    argmax_block(v, idx);
    if (threadIdx.x == 0) {
        const uint32_t r = (idx == 0xFFFFFFFFu) ? 0u : idx;
        *(uint32_t*)a.out = r;
        if (a.out2) *(uint32_t*)a.out2 = r;
        if (a.step_scalars) {  // end of a replayed greedy decode step
            uint32_t* s = (uint32_t*)a.step_scalars;
            const uint32_t pos = s[0];
            ((uint32_t*)a.step_history)[pos] = r;
            s[1] = r;
            s[0] = pos + 1;
        }
    }
}

// ---- top-k: read_topk (backend/contract.rs:303-318, cpu/readback.rs:59-69) on the device ----
// The min(k, n) largest logits under (logit descending by f32 total order, i.e.
// f32::total_cmp, then index ascending). Each logit becomes one 64-bit key that sorts
// ascending in exactly that order:
//   key = (~ord(bits) << 32) | index,   ord(b) = b ^ (b >> 31 ? 0xFFFFFFFF : 0x80000000),
// ord mapping the total order of f32 bit patterns (-NaN < -inf < ... < -0 < +0 < ... < +inf <
// +NaN) onto unsigned order. The all-ones key pads short stripes and lists and sorts after every
// real key.
// Everything is a sorted list of 64·V keys (V = 1 up to k = 64, else 2) in the registers of one
// wave, entry 64 v + lane in register v: bitonic networks over lane exchanges, no LDS and no barrier
// between their steps (sorted 2048 at a time in LDS by eight waves, 66 barriers, a stripe took 23 us
// and the merge of the 64 stripes 12.5; now 8.4 and 11.3 at 131072 logits and k = 40 with the result
// written to pinned host memory, one call in all 58.4 -> 31.5 us). Two lists of opposite directions merge by
// min(A[i], B[i]), which holds the smallest half as a bitonic list.
constexpr uint32_t kTopkChunk = 512;   // keys a wave sorts at a time (8 registers)

__device__ __forceinline__ uint64_t topk_key(uint32_t bits, uint32_t idx) {
    const uint32_t ord = bits ^ ((bits >> 31) ? 0xFFFFFFFFu : 0x80000000u);
    return ((uint64_t)~ord << 32) | idx;
}

// The smaller (keep_min) or larger of x and lane ^ stride's x: DPP moves within 16 lanes (xor 4 as
// xor 7 then xor 3), row swaps beyond, which leave the lane's own and its partner's value in the two
// registers (through ds_bpermute: partial 13.5 us, final 13.9 at k = 40).
template <int CTRL>
__device__ __forceinline__ uint64_t topk_dpp(uint64_t x) {
    const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)x, CTRL, 0xF, 0xF, false);
    const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(x >> 32), CTRL, 0xF, 0xF, false);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t topk_exchange(uint64_t x, uint32_t stride, bool keep_min) {
    uint64_t y;
    if (stride >= 16) {
        const uint32_t l = (uint32_t)x, h = (uint32_t)(x >> 32);
        const auto a = stride == 16 ? __builtin_amdgcn_permlane16_swap(l, l, false, false)
                                    : __builtin_amdgcn_permlane32_swap(l, l, false, false);
        const auto b = stride == 16 ? __builtin_amdgcn_permlane16_swap(h, h, false, false)
                                    : __builtin_amdgcn_permlane32_swap(h, h, false, false);
        x = ((uint64_t)b[0] << 32) | a[0];
        y = ((uint64_t)b[1] << 32) | a[1];
    } else if (stride == 8) {
        y = topk_dpp<0x128>(x);  // row_ror:8
    } else if (stride == 4) {
        y = topk_dpp<0x1B>(topk_dpp<0x141>(x));  // row_half_mirror, quad_perm [3,2,1,0]
    } else {
        y = stride == 2 ? topk_dpp<0x4E>(x) : topk_dpp<0xB1>(x);  // quad_perm [2,3,0,1], [1,0,3,2]
    }
    return ((x > y) == keep_min) ? y : x;
}

template <int V>
struct TopkList {
    uint64_t r[V];
};

// Sorts a bitonic list, ascending (up) or descending.
template <int V>
__device__ __forceinline__ void topk_merge(TopkList<V>& l, bool up) {
    const uint32_t lane = threadIdx.x & 63u;
    if constexpr (V == 2) {
        const uint64_t a = l.r[0], b = l.r[1];
        const bool swap = (a > b) == up;
        l.r[0] = swap ? b : a;
        l.r[1] = swap ? a : b;
    }
#pragma unroll
    for (uint32_t s = 32; s > 0; s >>= 1)
#pragma unroll
        for (int v = 0; v < V; ++v) l.r[v] = topk_exchange(l.r[v], s, ((lane & s) == 0) == up);
}

// The smallest 64 V of an ascending and a descending list, sorted.
template <int V>
__device__ __forceinline__ TopkList<V> topk_least(const TopkList<V>& a, const TopkList<V>& b, bool up) {
    TopkList<V> m;
#pragma unroll
    for (int v = 0; v < V; ++v) m.r[v] = min(a.r[v], b.r[v]);
    topk_merge<V>(m, up);
    return m;
}

// The smallest 64 V of eight vectors of 64 keys, descending.
template <int V>
__device__ __forceinline__ TopkList<V> topk_of_512(uint64_t (&x)[8]) {
    const uint32_t lane = threadIdx.x & 63u;
    // vectors 0, 2, .. ascending, 1, 3, .. descending
#pragma unroll
    for (uint32_t size = 2; size <= 64; size <<= 1)
#pragma unroll
        for (uint32_t s = size >> 1; s > 0; s >>= 1)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const bool up = ((lane & size) == 0) == ((i & 1) == 0);
                x[i] = topk_exchange(x[i], s, ((lane & s) == 0) == up);
            }
    TopkList<V> l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (V == 1) {
            l[i].r[0] = min(x[2 * i], x[2 * i + 1]);
        } else {  // all 128 of the pair: an ascending after a descending run is bitonic
            l[i].r[0] = x[2 * i + 1];
            l[i].r[1] = x[2 * i];
        }
        topk_merge<V>(l[i], (i & 1) == 0);
    }
    const TopkList<V> a = topk_least<V>(l[0], l[1], true), b = topk_least<V>(l[2], l[3], false);
    return topk_least<V>(a, b, false);
}

// One wave per stripe of a.per logits: its 64 V smallest keys, ascending, at part[stripe].
template <int V>
__device__ __forceinline__ void topk_partial(const GhTopkArgs& a) {
    const uint32_t lane = threadIdx.x;
    const uint64_t b0 = (uint64_t)blockIdx.x * a.per, e = min((uint64_t)a.n, b0 + a.per);
    const GH_GLOBAL uint32_t* bits = gh_gp<uint32_t>(a.logits);
    TopkList<V> acc;  // ascending
#pragma unroll
    for (int v = 0; v < V; ++v) acc.r[v] = ~0ull;
    for (uint64_t c = b0; c < e; c += kTopkChunk) {
        uint32_t raw[8];
        uint64_t x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) raw[i] = bits[min(c + 64 * i + lane, e - 1)];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint64_t at = c + 64 * i + lane;
            x[i] = at < e ? topk_key(raw[i], (uint32_t)at) : ~0ull;
        }
        acc = topk_least<V>(acc, topk_of_512<V>(x), true);
    }
#pragma unroll
    for (int v = 0; v < V; ++v) gh_gpw<uint64_t>(a.part)[((uint64_t)blockIdx.x * V + v) * 64 + lane] = acc.r[v];
}
GH_KERNEL __launch_bounds__(64) void gh_topk_partial(GhTopkArgs a) {
    if (a.width == 64) topk_partial<1>(a);
    else topk_partial<2>(a);
}

// The smallest 64 V of lists first, first + stride, ... < n at `src`, ascending: four lists at a time, the
// odd ones read backwards.
template <int V, class P>
__device__ __forceinline__ TopkList<V> topk_lists(const P src, uint32_t first, uint32_t stride, uint32_t n) {
    const uint32_t lane = threadIdx.x & 63u;
    TopkList<V> acc;  // ascending
#pragma unroll
    for (int v = 0; v < V; ++v) acc.r[v] = ~0ull;
    for (uint32_t l0 = first; l0 < n; l0 += 4 * stride) {
        TopkList<V> l[4];
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q)
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const uint32_t li = l0 + q * stride, i = 64 * v + lane;
                const uint64_t key = src[(uint64_t)min(li, n - 1) * 64 * V + ((q & 1) ? 64 * V - 1 - i : i)];
                l[q].r[v] = li < n ? key : ~0ull;
            }
        const TopkList<V> a = topk_least<V>(l[0], l[1], true), b = topk_least<V>(l[2], l[3], false);
        acc = topk_least<V>(acc, topk_least<V>(a, b, false), true);
    }
    return acc;
}

// One workgroup of 16 waves merges the stripes' lists, 16 apart per wave, then one wave the 16 lists
// left, and writes k u32 indices, then their f32 bits.
template <int V>
__device__ __forceinline__ void topk_final(const GhTopkArgs& a, uint64_t* s) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    TopkList<V> l = topk_lists<V>(gh_gp<uint64_t>(a.part), wave, 16, a.stripes);
#pragma unroll
    for (int v = 0; v < V; ++v) s[(wave * V + v) * 64 + lane] = l.r[v];
    __syncthreads();
    if (wave) return;
    l = topk_lists<V>((const uint64_t*)s, 0, 1, 16);
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const uint32_t t = 64 * v + lane, ord = ~(uint32_t)(l.r[v] >> 32);
        if (t >= a.k) continue;
        gh_gpw<uint32_t>(a.out)[t] = (uint32_t)l.r[v];
        gh_gpw<uint32_t>(a.out)[a.k + t] = ord ^ ((ord >> 31) ? 0x80000000u : 0xFFFFFFFFu);
    }
}
GH_KERNEL __launch_bounds__(1024) void gh_topk_final(GhTopkArgs a) {
    __shared__ uint64_t s[16 * 128];
    if (a.width == 64) topk_final<1>(a, s);
    else topk_final<2>(a, s);
}
